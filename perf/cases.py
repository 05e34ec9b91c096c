"""The work a user of this framework has it do, as cases that can be timed.

Each case is one pass through the public entry points (`plugins_amd.exl3`,
`plugins_amd.qwen3`): a quantized linear, linears that read the same rows, a
dense SwiGLU MLP, a grouped linear, a routed-expert layer, or a decoder's
decode step.  The shapes are those of the repository's own benchmark and tests
(Qwen3-8B-shaped linears, a DeepSeek-V3-shaped expert layer); `draw` takes
other sizes, rates, dtypes and options of the same ranges.  Weights are uniform
random trellis words (any bitstream decodes validly), suh +-1, svh f16(+-U[0.5,
1.5] * 0.02); activations N(0, 1).
"""
from __future__ import annotations

import math

import numpy as np
import torch

from plugins_amd import exl3 as X
from plugins_amd import qwen3 as Q

DEV = "cuda"
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
HEAD = 128


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # One projection (q or o) of a decode step at batch 1, called eagerly:
        # the smallest call, all latency.
        {"name": "linear_1", "kind": "linear", "rows": 1, "in": 4096, "out": 4096, "n": 64,
         "dtype": "f16", "codebook": "mul1"},
        # q, k and v of a speculative step of 3 tokens at a half-integer rate
        # (2.5 bits a weight), one call for the three linears.
        {"name": "qkv_half_3", "kind": "joint", "rows": 3, "in": 4096, "outs": "4096,1024,1024",
         "n": 40, "dtype": "bf16", "codebook": "mul1"},
        # A grouped output projection (8 linears side by side, each with its own
        # slice of the input) at 4 decode rows.
        {"name": "grouped_4", "kind": "grouped", "rows": 4, "groups": 8, "in": 4096, "out": 1024,
         "n": 48, "dtype": "bf16", "codebook": "mul1"},
        # A dense MLP at a small decode batch.
        {"name": "mlp_6", "kind": "mlp", "rows": 6, "hidden": 4096, "inter": 12288, "n": 64,
         "dtype": "bf16", "codebook": "mul1"},
        # One wide linear over the rows of a decode batch of 40 sequences.
        {"name": "linear_40", "kind": "linear", "rows": 40, "in": 4096, "out": 12288, "n": 64,
         "dtype": "f16", "codebook": "mul1"},
        # A dense MLP over a short, ragged prompt.
        {"name": "mlp_203", "kind": "mlp", "rows": 203, "hidden": 4096, "inter": 12288, "n": 64,
         "dtype": "bf16", "codebook": "mul1"},
        # Prefill of 2048 tokens through one wide linear.
        {"name": "linear_2048", "kind": "linear", "rows": 2048, "in": 4096, "out": 12288, "n": 64,
         "dtype": "f16", "codebook": "mul1"},
        # A routed-expert layer with its gated shared expert, one token.
        {"name": "moe_shared_1", "kind": "moe", "rows": 1, "hidden": 7168, "inter": 2048,
         "experts": 256, "topk": 8, "shared": True, "limit": 0, "n": 48, "dtype": "f16"},
        # The same routed experts at a decode batch of 16.
        {"name": "moe_16", "kind": "moe", "rows": 16, "hidden": 7168, "inter": 2048,
         "experts": 256, "topk": 8, "shared": False, "limit": 0, "n": 48, "dtype": "f16"},
        # ... and over a prompt of 1024 tokens, clamped, in bf16: the largest.
        {"name": "moe_1024", "kind": "moe", "rows": 1024, "hidden": 7168, "inter": 2048,
         "experts": 256, "topk": 8, "shared": False, "limit": 10, "n": 48, "dtype": "bf16"},
        # A whole decode step of a 36-layer decoder at context 2048, captured
        # in a HIP graph as a serving loop holds it: one sequence, ...
        {"name": "step_1", "kind": "step", "rows": 1, "ctx": 2048, "layers": 36, "hidden": 4096,
         "heads": 32, "kv_heads": 8, "inter": 12288, "vocab": 151936, "k_bits": 4},
        # ... and a batch of 16.
        {"name": "step_16", "kind": "step", "rows": 16, "ctx": 2048, "layers": 36, "hidden": 4096,
         "heads": 32, "kv_heads": 8, "inter": 12288, "vocab": 151936, "k_bits": 4},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A multiple of 128 between lo and hi, spread over its logarithm."""
    return 128 * max(1, min(hi // 128, _log_int(rng, lo, hi) // 128))


def _rate(rng):
    """Halfwords a tile: integer rates most often, half-integer rates, any even n."""
    return rng.choice([32, 48, 48, 64, 64, 64, 80, 96, 128, 24, 40, 2 * rng.randint(12, 50)])


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "joint", "grouped", "mlp", "mlp", "moe", "moe",
                       "step"])
    dtype = rng.choice(["f16", "f16", "bf16", "bf16", "f32"])
    codebook = rng.choice(["mul1", "mul1", "mul1", "mcg"])
    if kind == "linear":
        return {"kind": kind, "rows": _log_int(rng, 1, 2048), "in": _width(rng, 1024, 12288),
                "out": _width(rng, 512, 12288), "n": _rate(rng), "dtype": dtype,
                "codebook": codebook}
    if kind == "joint":
        outs = ",".join(str(_width(rng, 256, 12288)) for _ in range(rng.randint(2, 4)))
        return {"kind": kind, "rows": _log_int(rng, 1, 64), "in": _width(rng, 1024, 8192),
                "outs": outs, "n": _rate(rng), "dtype": dtype, "codebook": codebook}
    if kind == "grouped":
        return {"kind": kind, "rows": _log_int(rng, 1, 512), "groups": rng.choice([2, 4, 8, 16]),
                "in": _width(rng, 512, 4096), "out": _width(rng, 256, 2048),
                "n": rng.choice([32, 48, 64, 40]), "dtype": dtype, "codebook": codebook}
    if kind == "mlp":
        return {"kind": kind, "rows": _log_int(rng, 1, 1024), "hidden": _width(rng, 1024, 8192),
                "inter": _width(rng, 1024, 12288), "n": rng.choice([32, 48, 64, 80]),
                "dtype": dtype, "codebook": codebook}
    if kind == "moe":
        rows, experts = _log_int(rng, 1, 1024), rng.choice([16, 32, 64, 128])
        topk = rng.choice([2, 4, 6, 8])
        return {"kind": kind, "rows": rows, "hidden": _width(rng, 1024, 7168),
                "inter": _width(rng, 512, 2048), "experts": experts, "topk": topk,
                # the shared expert rides the routed launches at decode sizes only
                "shared": rows <= 16 and rng.random() < 0.5, "limit": rng.choice([0, 10]),
                "n": rng.choice([32, 48, 64]), "dtype": dtype}
    kv = rng.choice([2, 4, 8])
    return {"kind": "step", "rows": rng.randint(1, 16), "ctx": _log_int(rng, 16, 2048),
            "layers": rng.randint(1, 6), "hidden": _width(rng, 1024, 4096), "heads": 4 * kv,
            "kv_heads": kv, "inter": _width(rng, 2048, 12288), "vocab": _width(rng, 8192, 65536),
            "k_bits": rng.choice([2, 3, 4])}


# --------------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _tensors(g, i, o, n, lead=()):
    t = torch.randint(-32768, 32768, lead + (i // 16, o // 16, n), dtype=torch.int16, device=DEV,
                      generator=g)
    suh = (torch.randint(0, 2, lead + (i,), device=DEV, generator=g) * 2 - 1).to(torch.float16)
    sgn = torch.randint(0, 2, lead + (o,), device=DEV, generator=g) * 2 - 1
    svh = (sgn * (torch.rand(lead + (o,), device=DEV, generator=g) + 0.5) * 0.02).to(torch.float16)
    return t, suh, svh


def _acts(g, shape, dtype):
    return torch.randn(shape, device=DEV, generator=g).to(DTYPES[dtype])


def _outs(case):
    return [int(o) for o in case["outs"].split(",")]


def _inputs(case, seed):
    """The pass's tensors from the seed alone: weights (trellis, suh, svh) by
    name, activations, routes."""
    g = _gen(seed)
    k = case["kind"]
    if k in ("linear", "joint"):
        outs = [case["out"]] if k == "linear" else _outs(case)
        return {"w": [_tensors(g, case["in"], o, case["n"]) for o in outs],
                "x": _acts(g, (case["rows"], case["in"]), case["dtype"])}
    if k == "grouped":
        return {"w": [_tensors(g, case["in"], case["out"], case["n"])
                      for _ in range(case["groups"])],
                "x": _acts(g, (case["rows"], case["groups"], case["in"]), case["dtype"])}
    h, i, n = case["hidden"], case["inter"], case["n"]
    if k == "mlp":
        return {"w": [_tensors(g, h, i, n), _tensors(g, h, i, n), _tensors(g, i, h, n)],
                "x": _acts(g, (case["rows"], h), case["dtype"])}
    lead = (case["experts"],)
    d = {"w": [_tensors(g, h, i, n, lead), _tensors(g, h, i, n, lead), _tensors(g, i, h, n, lead)],
         "x": _acts(g, (case["rows"], h), case["dtype"])}
    probs = torch.softmax(torch.randn(case["rows"], case["experts"], device=DEV, generator=g), -1)
    top = probs.topk(case["topk"], -1)
    d["scores"] = (top.values / top.values.sum(-1, keepdim=True)).contiguous()
    d["inds"] = top.indices.to(torch.int32).contiguous()
    if case["shared"]:
        d["sw"] = [_tensors(g, h, i, n), _tensors(g, h, i, n), _tensors(g, i, h, n)]
        d["logit"] = _acts(g, (case["rows"],), case["dtype"])
    return d


class _Decoder:
    """A decoder with its key and value caches in two tensors [layers, batch,
    kv heads, positions, 128], and token ids from the seed."""

    def __init__(self, case, seed):
        cfg = Q.Qwen3Config(layers=case["layers"], hidden=case["hidden"], heads=case["heads"],
                            kv_heads=case["kv_heads"], inter=case["inter"], vocab=case["vocab"],
                            k_bits=case["k_bits"])
        self.ctx = case["ctx"]
        self.dec = Q.Qwen3Decoder(cfg, case["rows"], case["ctx"], seed=seed, max_new=16)
        g = _gen(seed + 1)
        self.dec.ids.copy_(torch.randint(0, case["vocab"], (case["rows"],), device=DEV,
                                         generator=g))
        shape = (case["layers"],) + tuple(self.dec.layers[0]["kc"].shape)
        self.kc, self.vc = (torch.empty(shape, dtype=torch.float16, device=DEV) for _ in range(2))
        for j, layer in enumerate(self.dec.layers):
            self.kc[j].copy_(layer["kc"])
            self.vc[j].copy_(layer["vc"])
            layer["kc"], layer["vc"] = self.kc[j], self.vc[j]


# ----------------------------------------------------------------- one pass

class _Owned:
    """A weight the library loaded, released with the state that holds it."""

    def __init__(self, loader, weight):
        self.loader, self.weight = loader, weight

    def __del__(self):
        try:
            X.release(self.weight)
            self.loader.close()
        except Exception:
            pass


def prepare(case, seed):
    k = case["kind"]
    if k == "step":
        d = _Decoder(case, seed)
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            d.dec.step()  # sizes the stream's scratch
        s.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            d.dec.step()
        torch.cuda.synchronize()
        return {"kind": k, "graph": graph, "d": d, "stream": s, "k": d.kc[:, :, :, d.ctx, :],
                "v": d.vc[:, :, :, d.ctx, :]}
    t = _inputs(case, seed)
    st = {"kind": k, "x": t["x"]}
    if k in ("linear", "joint", "mlp"):
        st["lin"] = [X.Linear(*w, codebook=case["codebook"]) for w in t["w"]]
        st["w"] = [lin.weight for lin in st["lin"]]
    elif k == "grouped":
        src = {}
        for j, (tr, suh, svh) in enumerate(t["w"]):
            src[f"m.slice.{j}.trellis"] = tr.cpu().numpy()
            src[f"m.slice.{j}.suh"] = suh.cpu().numpy()
            src[f"m.slice.{j}.svh"] = svh.cpu().numpy()
        loader = X.Loader('{"format":"exl3","codebook":"%s"}' % case["codebook"],
                          X.DictSource(src))
        X.check(loader.opened, "open")
        v, w = loader.load_tensor("m", case["in"])
        X.check(v, "load_tensor")
        st["owned"] = _Owned(loader, w)
        st["shape"] = (case["rows"], case["groups"], case["out"])
    else:
        st["t"] = t
        st["w"] = [X.wrap(*w) for w in t["w"]]
        st["limit"] = case["limit"]
        st["sw"] = [X.wrap(*w) for w in t["sw"]] if case["shared"] else None
    torch.cuda.synchronize()
    return st


def run(state):
    k = state["kind"]
    if k == "step":
        state["graph"].replay()
        return [state["d"].dec.logits, state["k"], state["v"]]
    x = state["x"]
    if k == "linear":
        return X.matmul(state["w"][0], x)
    if k == "joint":
        return X.matmul_shared(state["w"], x)
    if k == "grouped":
        return X.matmul(state["owned"].weight, x,
                        out=torch.empty(state["shape"], dtype=x.dtype, device=x.device))
    if k == "mlp":
        return X.swiglu(*state["w"], x)
    t = state["t"]
    if state["sw"]:
        return X.swiglu_shared(*state["w"], x, state["sw"], inds=t["inds"], scores=t["scores"],
                               logit=t["logit"])
    return X.swiglu(*state["w"], x, t["inds"], t["scores"], limit=state["limit"])


# --------------------------------------------------------------- what it needs

def _size(dtype):
    return 4 if dtype == "f32" else 2


def work(case):
    """Packed weights read once, activations in and out once; two operations
    per weight and row."""
    k, r = case["kind"], case["rows"]
    if k == "step":
        h, i, layers = case["hidden"], case["inter"], case["layers"]
        q, kv, bits = case["heads"] * HEAD, case["kv_heads"] * HEAD, case["k_bits"]
        weights = layers * (h * (2 * q + 2 * kv) + 3 * h * i) + h * case["vocab"]
        keys = case["ctx"] + 1
        return {"bytes": weights * bits // 8 + layers * 2 * kv * 2 * keys * r
                + r * 2 * (h + case["vocab"]),
                "flops": 2 * r * weights + 4 * layers * r * q * keys}
    b, n = _size(case["dtype"]), case["n"]
    if k in ("linear", "joint"):
        out = case["out"] if k == "linear" else sum(_outs(case))
        m = case["in"] * out
        return {"bytes": m * n // 128 + r * (case["in"] + out) * b, "flops": 2 * r * m}
    if k == "grouped":
        m = case["groups"] * case["in"] * case["out"]
        return {"bytes": m * n // 128 + r * case["groups"] * (case["in"] + case["out"]) * b,
                "flops": 2 * r * m}
    m = 3 * case["hidden"] * case["inter"]
    if k == "mlp":
        return {"bytes": m * n // 128 + 2 * r * case["hidden"] * b, "flops": 2 * r * m}
    e, top, sh = case["experts"], case["topk"], int(case["shared"])
    # distinct experts of the call's routes, as even routing gives them
    used = e * (1.0 - (1.0 - top / e) ** r) + sh
    return {"bytes": int(used * m * n / 128) + 2 * r * case["hidden"] * b,
            "flops": 2 * r * (top + sh) * m}


def tolerance(case):
    """About four times the distance to the 64-bit result that the rounding
    points of the format (f16 rotated rows, f16 inner products, the output's
    dtype) leave: 4e-4 a linear, more through an MLP's two and through the
    layers of a decoder."""
    if case["kind"] == "step":
        return {"rel": 8e-3 if case["layers"] <= 6 else 2e-2}
    base = 8e-3 if case["dtype"] == "bf16" else 2e-3
    if case["kind"] in ("mlp", "moe"):
        base = 8e-3 if case["dtype"] == "bf16" else 4e-3
    return {"rel": base}


# ------------------------------------------------------------ the 64-bit value

_TABLES = {}


def _table(codebook):
    """The 65536 codewords' weights (f16 values)."""
    if codebook not in _TABLES:
        c = torch.arange(65536, dtype=torch.int64, device=DEV)
        if codebook == "mul1":
            v = (c * 0x83DCD12D) & 0xFFFFFFFF
            s = sum(((v >> (8 * j)) & 255) for j in range(4)) + 1024
            a, b = (float(np.array([h], np.uint16).view(np.float16)[0]) for h in (0x1EEE, 0xC931))
            w = s.double() * a + b
        else:
            v = ((c * 0xCBAC1FED) & 0x8FFF8FFF) ^ 0x3B603B60
            halves = [h.to(torch.int32).to(torch.int16).view(torch.float16).double()
                      for h in (v & 0xFFFF, v >> 16)]
            w = halves[0] + halves[1]
        _TABLES[codebook] = w.float().to(torch.float16)  # exact in f32: one rounding
    return _TABLES[codebook]


def _weights(trellis, codebook):
    """Tiles [in/16, out/16, n] to W [in, out]: codeword t is the 16 stream
    bits ending at floor((t + 1) n / 16), circular; codeword 8 t + j sits at
    row (2q, 2q + 1, 2q + 8, 2q + 9)[j % 4], q = t % 4, column t / 4 + 8 (j / 4)."""
    it, ot, n = trellis.shape
    t = torch.arange(256, device=DEV)
    start = (((t + 1) * n) // 16 - 16) % (16 * n)
    s0, off = start // 16, (start % 16).to(torch.int32)
    # stream halfword s is stored at place s ^ 1
    place0, place1 = s0 ^ 1, ((s0 + 1) % n) ^ 1
    hw = trellis.view(it * ot, n)
    cw = (hw[:, place0].to(torch.int32) & 0xFFFF) << 16
    cw |= hw[:, place1].to(torch.int32) & 0xFFFF
    cw = (cw >> (16 - off)) & 0xFFFF
    q, j = (t // 8) % 4, t % 8
    row = 2 * q + (j % 2) + 8 * ((j % 4) // 2)
    col = t // 32 + 8 * (j // 4)
    dst = torch.empty(256, dtype=torch.int64, device=DEV)
    dst[row * 16 + col] = t
    w = _table(codebook)[cw[:, dst]]
    return w.view(it, ot, 16, 16).permute(0, 2, 1, 3).reshape(it * 16, ot * 16)


_H = {}


def _rotate(x):
    """The orthonormal 128-point Hadamard of every block of the last axis."""
    if not _H:
        h = torch.ones(1, 1, dtype=torch.float64, device=DEV)
        while h.shape[0] < 128:
            h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
        _H["h"] = h / math.sqrt(128.0)
    return (x.reshape(-1, 128) @ _H["h"]).reshape(x.shape)


def _linear64(x, w, codebook="mul1"):
    trellis, suh, svh = w
    z = []
    xp = _rotate(x * suh.double())
    for tr in trellis.split(4096, 1):  # by output columns: bounded memory
        z.append(xp @ _weights(tr.contiguous(), codebook).double())
    return _rotate(torch.cat(z, -1)) * svh.double()


def _mlp64(x, ws, limit=0, codebook="mul1"):
    g, u = _linear64(x, ws[0], codebook), _linear64(x, ws[1], codebook)
    if limit:
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    return _linear64(g * torch.sigmoid(g) * u, ws[2], codebook)


def _norm64(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _step64(case, seed):
    d = _Decoder(case, seed)
    c, dec, B, ctx = d.dec.cfg, d.dec, case["rows"], case["ctx"]
    inv = c.theta ** (-2.0 * torch.arange(64, dtype=torch.float64, device=DEV) / HEAD)
    cos, sin = torch.cos(ctx * inv), torch.sin(ctx * inv)

    def rope(v, w):
        v = _norm64(v.reshape(B, -1, HEAD), w, c.eps)
        a, b = v[..., :64], v[..., 64:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    h = dec.embed_table[dec.ids.long()].double()
    ks, vs = [], []
    for j, layer in enumerate(dec.layers):
        x = _norm64(h, layer["in_norm"], c.eps)
        q, k, v = (_linear64(x, layer[p].tensors) for p in ("q", "k", "v"))
        q, k = rope(q, layer["q_norm"]), rope(k, layer["k_norm"])
        v = v.reshape(B, -1, HEAD)
        ks.append(k)
        vs.append(v)
        att = []
        for b in range(B):
            kk = torch.cat([d.kc[j, b, :, :ctx].double(), k[b][:, None]], 1)
            vv = torch.cat([d.vc[j, b, :, :ctx].double(), v[b][:, None]], 1)
            qq = q[b].reshape(c.kv_heads, -1, HEAD)
            p = torch.softmax(qq @ kk.transpose(1, 2).contiguous() / math.sqrt(HEAD), -1)
            att.append((p @ vv).reshape(-1))
        h = h + _linear64(torch.stack(att), layer["o"].tensors)
        x = _norm64(h, layer["post_norm"], c.eps)
        h = h + _mlp64(x, [layer[p].tensors for p in ("gate", "up", "down")])
    logits = _linear64(_norm64(h, dec.final_norm, c.eps), dec.lm_head.tensors)
    return [logits, torch.stack(ks), torch.stack(vs)]


def exact(case, seed):
    """What `run` returns for these inputs, in 64 bits from the format's
    definition: W = diag(suh) H W_inner H diag(svh) with the decoded f16
    weights, no rounding between."""
    k = case["kind"]
    if k == "step":
        return _step64(case, seed)
    t = _inputs(case, seed)
    x = t["x"].double()
    cb = case.get("codebook", "mul1")
    if k == "linear":
        return _linear64(x, t["w"][0], cb)
    if k == "joint":
        return [_linear64(x, w, cb) for w in t["w"]]
    if k == "grouped":
        return torch.stack([_linear64(x[:, j], w, cb) for j, w in enumerate(t["w"])], 1)
    if k == "mlp":
        return _mlp64(x, t["w"], 0, cb)
    y = torch.zeros_like(x)
    for e in torch.unique(t["inds"]).tolist():
        row, slot = (t["inds"] == e).nonzero(as_tuple=True)
        ws = [tuple(a[e] for a in w) for w in t["w"]]
        y.index_add_(0, row, t["scores"][row, slot].double()[:, None]
                     * _mlp64(x[row], ws, case["limit"]))
    if case["shared"]:
        y = y + torch.sigmoid(t["logit"].double())[:, None] * _mlp64(x, t["sw"])
    return y
