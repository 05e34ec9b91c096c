"""The routed experts' grouped GEMM at the edges of its tiles: item sizes on
both sides of a row block (32), of the tile forms (64, 128) and of an item (64 or
128), a column tile that is half empty (widths of an odd number of 128-column
groups), rates on both sides of the word stages' limits, every codebook form at
the full and a narrowed window, arrays that are not 16-byte aligned, and the
rule that chooses it, against the oracle's composition."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402
from plugins_amd import exl3 as X  # noqa: E402
from tests import _synth as S  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _bank(rng, experts, in_f, out_f, n, codebook):
    t, u, v = S.linear(rng, in_f, out_f, n, experts=experts)
    d = [torch.from_numpy(t.view(np.int16)).to(DEV), torch.from_numpy(u.view(np.float16)).to(DEV),
         torch.from_numpy(v.view(np.float16)).to(DEV)]
    return (t, u, v), X.wrap(*d, codebook=codebook)


@pytest.mark.parametrize("counts", [(1, 31, 32, 33, 40), (63, 64, 65, 0, 20), (127, 128, 129, 1, 1),
                                    (260, 5, 96, 97, 17)])
@pytest.mark.parametrize("n,hidden,inter", [(48, 384, 640), (16, 128, 256), (112, 256, 384),
                                            (128, 512, 128)])
def test_grouped_gemm_item_edges(counts, n, hidden, inter):
    # to 64 workgroups and 32 slots an expert: this kernel, its items up to 64
    # slots; from 48 up to 128
    counts = counts + 27 * (34 if max(counts) <= 65 else 60,)
    rng = np.random.default_rng(sum(counts) + n)
    E = len(counts)
    inds = np.repeat(np.arange(E, dtype=np.int32), counts)
    rng.shuffle(inds)
    rows = inds.size
    inds = inds.reshape(rows, 1)
    scores = rng.uniform(0.2, 1.0, (rows, 1)).astype(np.float32)
    gn, g = _bank(rng, E, hidden, inter, n, "mul1")
    un, u = _bank(rng, E, hidden, inter, n, "mul1")
    dn, d = _bank(rng, E, inter, hidden, n, "mul1")
    x = S.activations(rng, rows, hidden)
    assert X.swiglu_path(g, u, d, rows, 1) == "routed-gemm"
    y = X.swiglu(g, u, d, torch.from_numpy(x).to(DEV), torch.from_numpy(inds).to(DEV),
                 torch.from_numpy(scores).to(DEV)).float().cpu().numpy()
    want = O.moe_swiglu(x.astype(np.float32), gn, un, dn, inds, scores, hidden, inter, n)
    # the repository's bar: three f16 rounding points a linear, 2^-11 each
    assert S.rel_fro(y, want) < 1e-3
    assert S.row_rel(y, want).max() < 3e-3


@pytest.mark.parametrize("E,topk,rows,hidden,inter,path", [
    (512, 4, 512, 256, 256, "routed-gemm"),   # 1024 workgroups, 4 slots an expert
    (512, 4, 511, 256, 256, "routed-gemv"),
    (256, 4, 320, 256, 256, "routed-gemm"),   # 512 workgroups, 5 slots
    (256, 4, 319, 256, 256, "routed-gemv"),
    (128, 4, 192, 256, 256, "routed-gemm"),   # 256 workgroups, 6 slots
    (128, 4, 191, 256, 256, "routed-gemv"),
    (64, 4, 192, 256, 256, "routed-gemm"),    # 128 workgroups, 12 slots: the work's bound
    (64, 4, 170, 256, 256, "routed-gemv"),
    (32, 4, 64, 512, 512, "routed-gemm"),     # 128 workgroups, 8 slots
    (32, 4, 63, 512, 512, "routed-gemv"),
    (8, 2, 68, 1024, 1024, "routed-gemm"),    # 64 workgroups, 17 slots
    (16, 2, 255, 128, 256, "routed-gemv"),    # 32 workgroups, no work: to 32 slots
    (16, 2, 256, 128, 256, "routed-gemm"),
    (16, 2, 512, 128, 256, "routed-gemm"),    # 64 slots: the 256-slot kernel
    (16, 2, 2048, 128, 256, "routed-gemm")])
def test_grouped_gemm_rule(E, topk, rows, hidden, inter, path):
    rng = np.random.default_rng(E + rows)
    n = 48
    gn, g = _bank(rng, E, hidden, inter, n, "mul1")
    un, u = _bank(rng, E, hidden, inter, n, "mul1")
    dn, d = _bank(rng, E, inter, hidden, n, "mul1")
    x = S.activations(rng, rows, hidden)
    inds, scores = O.route_topk(rng.standard_normal((rows, E)).astype(np.float32), topk)
    assert X.swiglu_path(g, u, d, rows, topk) == path
    y = X.swiglu(g, u, d, torch.from_numpy(x).to(DEV), torch.from_numpy(inds).to(DEV),
                 torch.from_numpy(scores).to(DEV)).float().cpu().numpy()
    want = O.moe_swiglu(x.astype(np.float32), gn, un, dn, inds, scores, hidden, inter, n)
    assert S.rel_fro(y, want) < 1e-3
    assert S.row_rel(y, want).max() < 3e-3


def test_last_window_of_few_rows_on_fresh_scratch():
    """8192 tokens x top-8 run as windows of 8191 rows (the grouped GEMM) and 1
    row (the GEMV items, which need split-K slots): as the first call on a
    stream whose scratch is empty."""
    rng = np.random.default_rng(8192)
    E, hidden, inter, n, topk, rows = 256, 128, 256, 48, 8, 8192
    gn, g = _bank(rng, E, hidden, inter, n, "mul1")
    un, u = _bank(rng, E, hidden, inter, n, "mul1")
    dn, d = _bank(rng, E, inter, hidden, n, "mul1")
    x = S.activations(rng, rows, hidden)
    inds, scores = O.route_topk(rng.standard_normal((rows, E)).astype(np.float32), topk)
    xd, ids, scs = (torch.from_numpy(a).to(DEV) for a in (x, inds, scores))
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    X.scratch_release(0, stream)
    y = X.swiglu(g, u, d, xd, ids, scs, stream=stream)
    stream.synchronize()
    assert X.stream_status(0, stream).is_ok()
    at = np.array([0, 4000, 8190, 8191])
    want = O.moe_swiglu(x[at].astype(np.float32), gn, un, dn, inds[at], scores[at], hidden, inter, n)
    assert S.rel_fro(y.float().cpu().numpy()[at], want) < 1e-3
    assert torch.equal(y[-1:], X.swiglu(g, u, d, xd[-1:], ids[-1:], scs[-1:]))


def _offset(a, halves):
    """The array's bits on the device, `halves` 2-byte places past a 16-byte
    boundary."""
    flat = torch.from_numpy(np.ascontiguousarray(a).view(np.int16).reshape(-1)).to(DEV)
    buf = torch.empty(flat.numel() + 8, dtype=torch.int16, device=DEV)
    view = buf[halves:halves + flat.numel()]
    view.copy_(flat)
    return view.view(a.shape)


@pytest.mark.parametrize("counts", [(63, 64, 1, 0), (260, 5, 96, 97)])
@pytest.mark.parametrize("n", [48, 128])
def test_unaligned_banks_keep_a_grouped_gemm(counts, n):
    """Trellises at a 4-byte boundary: from 32 slots an expert a grouped GEMM
    (256-slot items), as the aligned banks."""
    rng = np.random.default_rng(sum(counts) + n)
    E, hidden, inter = len(counts), 384, 256
    inds = np.repeat(np.arange(E, dtype=np.int32), counts)
    rng.shuffle(inds)
    rows = inds.size
    inds = inds.reshape(rows, 1)
    scores = rng.uniform(0.2, 1.0, (rows, 1)).astype(np.float32)
    nps, ws = [], []
    for i, o in ((hidden, inter), (hidden, inter), (inter, hidden)):
        t, u, v = S.linear(rng, i, o, n, experts=E)
        nps.append((t, u, v))
        ws.append(X.wrap(_offset(t, 2), torch.from_numpy(u.view(np.float16)).to(DEV),
                         torch.from_numpy(v.view(np.float16)).to(DEV)))
    assert X.swiglu_path(*ws, 32 * E, 1) == "routed-gemm"
    assert X.swiglu_path(*ws, 32 * E - 1, 1) == "routed-gemv"
    x = S.activations(rng, rows, hidden)
    y = X.swiglu(*ws, torch.from_numpy(x).to(DEV), torch.from_numpy(inds).to(DEV),
                 torch.from_numpy(scores).to(DEV)).float().cpu().numpy()
    want = O.moe_swiglu(x.astype(np.float32), *nps, inds, scores, hidden, inter, n)
    assert S.rel_fro(y, want) < 1e-3
    assert S.row_rel(y, want).max() < 3e-3


@pytest.mark.parametrize("topk", [1, 2, 3, 4, 5, 8, 9])
@pytest.mark.parametrize("rows", [1, 35])
def test_combine_at_every_width(topk, rows):
    """The weighted sum's passes of 2, 4 and 8 slots, full and not, a second
    pass, an out-of-range expert, and y at a 4-byte boundary; and the shared
    expert's sum beside them."""
    rng = np.random.default_rng(10 * topk + rows)
    E, hidden, inter, n = 12, 384, 128, 48
    gn, g = _bank(rng, E, hidden, inter, n, "mul1")
    un, u = _bank(rng, E, hidden, inter, n, "mul1")
    dn, d = _bank(rng, E, inter, hidden, n, "mul1")
    x = S.activations(rng, rows, hidden)
    inds, scores = O.route_topk(rng.standard_normal((rows, E)).astype(np.float32), topk)
    want = O.moe_swiglu(x.astype(np.float32), gn, un, dn, inds, scores, hidden, inter, n)
    xd, ids, scs = (torch.from_numpy(a).to(DEV) for a in (x, inds, scores))
    y = X.swiglu(g, u, d, xd, ids, scs)
    assert S.rel_fro(y.float().cpu().numpy(), want) < 1e-3
    odd = torch.empty(rows * hidden + 2, dtype=torch.float16, device=DEV)[2:].view(rows, hidden)
    assert torch.equal(X.swiglu(g, u, d, xd, ids, scs, out=odd), y)
    if topk > 1:  # the last route names no expert: as with a score of zero
        ids[:, -1] = E + 1
        zero = scores.copy()
        zero[:, -1] = 0.0
        got = X.swiglu(g, u, d, xd, ids, scs).float().cpu().numpy()
        want0 = O.moe_swiglu(x.astype(np.float32), gn, un, dn, inds, zero, hidden, inter, n)
        assert S.rel_fro(got, want0) < 1e-3
    sn, sw = zip(*(_bank(rng, 1, i, o, n, "mul1") for i, o in ((hidden, inter), (hidden, inter),
                                                               (inter, hidden))))
    sw = [X.wrap(*(torch.from_numpy(a[0].view(np.int16 if k == 0 else np.float16)).to(DEV)
                   for k, a in enumerate(s))) for s in sn]
    logit = torch.from_numpy(rng.standard_normal(rows).astype(np.float16)).to(DEV)
    ids = torch.from_numpy(inds).to(DEV)
    got = X.swiglu_shared(g, u, d, xd, sw, inds=ids, scores=scs, logit=logit).float().cpu().numpy()
    one = np.zeros((rows, 1), np.int32), np.ones((rows, 1), np.float32)
    sh = O.moe_swiglu(x.astype(np.float32), *sn, *one, hidden, inter, n)
    gate = torch.sigmoid(logit).float().cpu().numpy()
    assert S.rel_fro(got, want + gate[:, None] * sh) < 1e-3


# codebook, window, table, the oracle's
FORMS = {"mcg": ("mcg", 16, None, O.CB_MCG), "mcg-w10": ("mcg", 10, None, O.CB_MCG),
         "mul1-w12": ("mul1", 12, None, O.CB_MUL1),
         "spec1-w15": ("spec1", 16, "spec1-w15", O.spec1(O.TAB_SPEC1_W15)),
         "spec1-w9": ("spec1", 9, "spec1-w16", O.spec1(O.TAB_SPEC1_W16)),
         "pair1": ("pair1", 16, "pair1-w16-v1", O.CB_PAIR1)}


@pytest.mark.parametrize("fill", [34, 60])  # items of up to 64 and 128 slots
@pytest.mark.parametrize("form", FORMS)
def test_grouped_gemm_codebooks(form, fill):
    codebook, window, table, ocb = FORMS[form]
    counts = (33, 64, 5, 130) + 28 * (fill,)
    rng = np.random.default_rng(fill + len(form))
    E, hidden, inter, n = len(counts), 256, 384, 48
    inds = np.repeat(np.arange(E, dtype=np.int32), counts)
    rng.shuffle(inds)
    rows = inds.size
    inds = inds.reshape(rows, 1)
    scores = rng.uniform(0.2, 1.0, (rows, 1)).astype(np.float32)
    nps = [S.linear(rng, i, o, n, experts=E)
           for i, o in ((hidden, inter), (hidden, inter), (inter, hidden))]
    ws = [X.wrap(torch.from_numpy(t.view(np.int16)).to(DEV), torch.from_numpy(u.view(np.float16)).to(DEV),
                 torch.from_numpy(v.view(np.float16)).to(DEV), codebook, window, 0, table)
          for t, u, v in nps]
    x = S.activations(rng, rows, hidden)
    assert X.swiglu_path(*ws, rows, 1) == "routed-gemm"
    y = X.swiglu(*ws, torch.from_numpy(x).to(DEV), torch.from_numpy(inds).to(DEV),
                 torch.from_numpy(scores).to(DEV)).float().cpu().numpy()
    want = O.moe_swiglu(x.astype(np.float32), *nps, inds, scores, hidden, inter, n, codebook=ocb,
                        window=window)
    assert S.rel_fro(y, want) < 1e-3
    assert S.row_rel(y, want).max() < 3e-3


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_grouped_gemm_unaligned_arrays(dtype):
    """x, the scales and y off their 16-byte boundaries: narrower accesses, the
    same values."""
    rng = np.random.default_rng(44)
    E, hidden, inter, n, rows, topk = 32, 256, 384, 48, 300, 4
    nps = [S.linear(rng, i, o, n, experts=E)
           for i, o in ((hidden, inter), (hidden, inter), (inter, hidden))]

    def half(a):
        return torch.from_numpy(a.view(np.float16)).to(DEV)

    trs = [torch.from_numpy(t.view(np.int16)).to(DEV) for t, _, _ in nps]
    ws = [X.wrap(tr, half(u), half(v)) for tr, (_, u, v) in zip(trs, nps)]
    odd = [X.wrap(tr, _offset(u, 3).view(torch.float16), _offset(v, 1).view(torch.float16))
           for tr, (_, u, v) in zip(trs, nps)]
    x = torch.from_numpy(S.activations(rng, rows, hidden)).to(DEV).to(dtype)
    inds, scores = O.route_topk(rng.standard_normal((rows, E)).astype(np.float32), topk)
    ids, scs = torch.from_numpy(inds).to(DEV), torch.from_numpy(scores).to(DEV)
    assert X.swiglu_path(*ws, rows, topk) == "routed-gemm"
    y = X.swiglu(*ws, x, ids, scs)
    xo, yo = (torch.empty(x.numel() + 1, dtype=dtype, device=DEV)[1:].view(x.shape) for _ in range(2))
    xo.copy_(x)
    assert torch.equal(X.swiglu(*odd, xo, ids, scs, out=yo), y)
    want = O.moe_swiglu(x.float().cpu().numpy(), *nps, inds, scores, hidden, inter, n)
    # beside the bar a bf16 output's own rounding (2^-9)
    assert S.rel_fro(y.float().cpu().numpy(), want) < (3e-3 if dtype == torch.bfloat16 else 1e-3)
