"""The register-decode GEMM behind exl3_matmul_shared (several linears that
share their rows): rows on both sides of its row blocks and tiles (32, 64,
128), widths with a half-empty column tile, inputs of one block and of many
(split and unsplit k), rates on both sides of its word stages, the half-integer
rates, each codebook form, output type and a narrowed window, outputs that are
not 16-byte aligned, against x @ W_public in float64 from the oracle's decode; a
large linear alone; and the rules that choose the kernel."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402
from plugins_amd import exl3 as X  # noqa: E402
from tests import _synth as S  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda"
FORMS = {"mul1": ("mul1", None, O.CB_MUL1), "mcg": ("mcg", None, O.CB_MCG),
         "spec1-w15": ("spec1", "spec1-w15", O.spec1(O.TAB_SPEC1_W15)),
         "pair1": ("pair1", "pair1-w16-v1", O.CB_PAIR1)}


def _linear(rng, in_f, out_f, n, form):
    cb, table, _ = FORMS[form]
    t, u, v = S.linear(rng, in_f, out_f, n)
    lin = X.Linear(torch.from_numpy(t.view(np.int16)).to(DEV),
                   torch.from_numpy(u.view(np.float16)).to(DEV),
                   torch.from_numpy(v.view(np.float16)).to(DEV), cb, 16, table)
    return (t, u, v), lin


@pytest.mark.parametrize("rows", [17, 32, 33, 64, 65, 128, 129, 300])
@pytest.mark.parametrize("in_f,outs,n,form,dtype", [
    (128, (128, 384), 64, "mul1", torch.float16), (1024, (640, 128, 256), 48, "mcg", torch.float32),
    (2176, (256, 128), 128, "mul1", torch.float16), (512, (384, 128, 128, 256), 40, "mul1", torch.float16),
    (384, (256, 256), 24, "pair1", torch.float16), (640, (128, 256), 112, "spec1-w15", torch.float16)])
def test_shared_rows_every_linear(rows, in_f, outs, n, form, dtype):
    rng = np.random.default_rng(rows * 10 + in_f + n)
    lins = [_linear(rng, in_f, o, n, form) for o in outs]
    x = S.activations(rng, rows, in_f)
    ys = X.matmul_shared([lin.weight for _, lin in lins], torch.from_numpy(x).to(DEV).to(dtype))
    for ((t, u, v), _), o, y in zip(lins, outs, ys):
        w_inner = O.reconstruct_inner(t, in_f, o, n, FORMS[form][2])
        want = S.public_matmul(x.astype(np.float64), w_inner, u, v)
        got = y.float().cpu().numpy()
        # the repository's bar: three f16 rounding points, 2^-11 each
        assert S.rel_fro(got, want) < 1e-3
        assert S.row_rel(got, want).max() < 3e-3


@pytest.mark.parametrize("rows", [40, 4000])  # k split, and not
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_output_types_and_alignment(rows, dtype):
    rng = np.random.default_rng(rows)
    in_f, outs, n, window = 256, (640, 128, 256), 48, 12
    nps = [S.linear(rng, in_f, o, n) for o in outs]
    ws = [X.wrap(torch.from_numpy(t.view(np.int16)).to(DEV), torch.from_numpy(u.view(np.float16)).to(DEV),
                 torch.from_numpy(v.view(np.float16)).to(DEV), "mul1", window) for t, u, v in nps]
    x = torch.from_numpy(S.activations(rng, rows, in_f)).to(DEV).to(dtype)
    ys = X.matmul_shared(ws, x)
    odd = [torch.empty(rows * o + 1, dtype=dtype, device=DEV)[1:].view(rows, o) for o in outs]
    X.matmul_shared(ws, x, outs=odd)
    for (t, u, v), o, y, z in zip(nps, outs, ys, odd):
        assert torch.equal(y, z)
        w_inner = O.reconstruct_inner(t, in_f, o, n, O.CB_MUL1, window)
        want = S.public_matmul(x.double().cpu().numpy(), w_inner, u, v)
        got = y.float().cpu().numpy()
        # the repository's bar, and a bf16 output's own rounding (2^-9) beside it
        bar = 3e-3 if dtype == torch.bfloat16 else 1e-3
        assert S.rel_fro(got, want) < bar
        assert S.row_rel(got, want).max() < 3 * bar


def test_large_linear_alone():
    rng = np.random.default_rng(5)
    (t, u, v), lin = _linear(rng, 4096, 16384, 32, "mul1")
    x = S.activations(rng, 97, 4096)
    w_inner = O.reconstruct_inner(t, 4096, 16384, 32)
    for rows in (17, 50, 97):
        y = lin(torch.from_numpy(x[:rows]).to(DEV)).float().cpu().numpy()
        want = S.public_matmul(x[:rows].astype(np.float64), w_inner, u, v)
        assert S.rel_fro(y, want) < 1e-3
        assert S.row_rel(y, want).max() < 3e-3


def test_input_past_its_tile_count():
    """65536 k-tiles: beyond the register-decode kernel's range, the 256 x 128
    tiles take the call."""
    in_f, out_f = 16 * 65536, 128
    rng = np.random.default_rng(9)
    (t, u, v), lin = _linear(rng, in_f, out_f, 16, "mul1")
    x = S.activations(rng, 17, in_f)
    y = lin(torch.from_numpy(x).to(DEV)).float().cpu().numpy()
    want = S.public_matmul(x.astype(np.float64), O.reconstruct_inner(t, in_f, out_f, 16), u, v)
    assert S.rel_fro(y, want) < 1e-3
    assert S.row_rel(y, want).max() < 3e-3


@pytest.mark.parametrize("pieces", [(100, 100), (17, 183), (40, 40), (17, 64, 47), (96, 160)])
def test_pieces_sum_as_the_whole_call(pieces):
    """Row pieces on both sides of the register-decode kernel's row rule, and
    prepared rows that are not 16-byte aligned: the whole call's inner
    products, bit for bit."""
    rng = np.random.default_rng(sum(pieces))
    _, lin = _linear(rng, 4096, 12288, 64, "mul1")
    x = torch.from_numpy(S.activations(rng, sum(pieces), 4096)).to(DEV)
    whole = X.linear_split(lin.weight, x, inner=True)
    v, held = X.linear_pieces(lin.weight, pieces)
    assert v.is_ok() and held.data == lin.weight.w.data, v
    xp = X.prepare(lin.weight, x)
    at = 0
    for n in pieces:
        z = X.linear_piece(lin.weight, x[at:at + n], held)
        assert torch.equal(z, whole[at:at + n])
        odd = torch.empty(n * 4096 + 1, dtype=torch.float16, device=DEV)[1:].view(n, 4096)
        odd.copy_(xp[at:at + n])
        assert torch.equal(X.linear_piece(lin.weight, odd, held, prepared=True), z)
        at += n


def test_rule_of_one_linear():
    """4096 -> 8192 above 32 rows, where the 256 x 128 tiles are faster, takes
    them: a call's rows are then those of a 256-row call, bit for bit (the same
    tiles and k-splits)."""
    rng = np.random.default_rng(81)
    _, lin = _linear(rng, 4096, 8192, 48, "mul1")
    x = torch.from_numpy(S.activations(rng, 256, 4096)).to(DEV)
    whole = lin(x)
    for rows in (33, 64, 96, 128):
        assert torch.equal(lin(x[:rows]), whole[:rows])
    assert not torch.equal(lin(x[:32]), whole[:32])  # the register-decode kernel


@pytest.mark.parametrize("rows,apart", [(10880, False), (11008, True)])
def test_rule_of_linears_that_share_rows(rows, apart):
    """128 + 384 columns are 3 half-empty 256-column tiles: one launch up to 256
    workgroups (85 row tiles), beyond that each linear alone, bit for bit."""
    rng = np.random.default_rng(82)
    lins = [_linear(rng, 1024, o, 48, "mul1")[1] for o in (128, 384)]
    x = torch.from_numpy(S.activations(rng, rows, 1024)).to(DEV)
    ys = X.matmul_shared([lin.weight for lin in lins], x)
    assert all(torch.equal(y, lin(x)) for y, lin in zip(ys, lins)) == apart


def test_unaligned_inputs():
    """Rows and scales off their 16-byte boundaries: the prepare's narrower
    accesses, in a shared call and in an MLP (whose SwiGLU then runs apart from
    down's prepare), the same values."""
    rng = np.random.default_rng(85)

    def odd(a):
        buf = torch.empty(a.numel() + 1, dtype=a.dtype, device=DEV)[1:]
        buf.copy_(a.reshape(-1))
        return buf.view(a.shape)

    def pair(in_f, out_f):
        t, u, v = S.linear(rng, in_f, out_f, 64)
        t, u, v = (torch.from_numpy(a.view(k)).to(DEV)
                   for a, k in ((t, np.int16), (u, np.float16), (v, np.float16)))
        return X.wrap(t, u, v), X.wrap(t, odd(u), odd(v))

    (g, go), (u, uo), (d, do) = pair(512, 640), pair(512, 640), pair(640, 512)
    for dtype in (torch.float16, torch.bfloat16, torch.float32):
        x = torch.from_numpy(S.activations(rng, 70, 512)).to(DEV).to(dtype)
        xo = odd(x)
        for a, b in zip(X.matmul_shared([g, u], x), X.matmul_shared([go, uo], xo)):
            assert torch.equal(a, b)
        assert torch.equal(X.swiglu(g, u, d, x), X.swiglu(go, uo, do, xo))
