"""A dense SwiGLU MLP whose gate and up decode differently (codebook, window)
at one rate: each linear by its own rule at every row count, on both sides of
the GEMV's 16 rows and of the GEMM's row tiles, against the oracle's
projections."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402
from plugins_amd import exl3 as X  # noqa: E402
from tests import _synth as S  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda"
CODES = {"mul1": O.CB_MUL1, "mcg": O.CB_MCG}


def _linear(rng, in_f, out_f, n, codebook, window):
    t, u, v = S.linear(rng, in_f, out_f, n)
    lin = X.Linear(torch.from_numpy(t.view(np.int16)).to(DEV),
                   torch.from_numpy(u.view(np.float16)).to(DEV),
                   torch.from_numpy(v.view(np.float16)).to(DEV), codebook, window)
    return (t, u, v, in_f, out_f, n, CODES[codebook], window), lin


@pytest.mark.parametrize("rows", [1, 6, 16, 17, 40, 64, 203, 300])
@pytest.mark.parametrize("n,up", [(64, ("mcg", 16)), (48, ("mul1", 12)), (40, ("mcg", 16))])
def test_gate_and_up_decode_apart(rows, n, up):
    rng = np.random.default_rng(rows + n)
    hidden, inter = 512, 768
    gn, g = _linear(rng, hidden, inter, n, "mul1", 16)
    un, u = _linear(rng, hidden, inter, n, *up)
    dn, d = _linear(rng, inter, hidden, n, "mul1", 16)
    x = S.activations(rng, rows, hidden)
    y = X.swiglu(g.weight, u.weight, d.weight, torch.from_numpy(x).to(DEV)).float().cpu().numpy()
    gv, uv = (S.h2f(O.project(x.astype(np.float32), *w)) for w in (gn, un))
    h = (gv / (1.0 + np.exp(-gv)) * uv).astype(np.float16).astype(np.float32)
    want = S.h2f(O.project(h, *dn))
    # the bar of the repository's MLP tests: equal rounding points, sums in
    # another order
    assert S.rel_fro(y, want) < 1e-3
    assert S.row_rel(y, want).max() < 3e-3
