"""The dense GEMV's longer splits above 4 rows: 12288 -> 4096 runs 8 splits of
12 input blocks up to 10 rows (their prepare's last pass full), 12 of 8 beyond;
every row against the oracle's decode in float64."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402
from plugins_amd import exl3 as X  # noqa: E402
from tests import _synth as S  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def linear():
    rng = np.random.default_rng(12288)
    t, u, v = S.linear(rng, 12288, 4096, 32)
    lin = X.Linear(torch.from_numpy(t.view(np.int16)).to("cuda"),
                   torch.from_numpy(u.view(np.float16)).to("cuda"),
                   torch.from_numpy(v.view(np.float16)).to("cuda"))
    return rng, O.reconstruct_inner(t, 12288, 4096, 32), u, v, lin


@pytest.mark.parametrize("rows,dtype", [(5, torch.float16), (6, torch.float32), (10, torch.float16),
                                        (11, torch.float32), (16, torch.float16)])
def test_long_splits_every_row(linear, rows, dtype):
    rng, w_inner, u, v, lin = linear
    x = S.activations(rng, rows, 12288)
    y = lin(torch.from_numpy(x).to("cuda").to(dtype)).float().cpu().numpy()
    want = S.public_matmul(x.astype(np.float64), w_inner, u, v)
    # the repository's bar: three f16 rounding points, 2^-11 each
    assert S.rel_fro(y, want) < 1e-3
    assert S.row_rel(y, want).max() < 2e-3
    assert X.stream_status().is_ok()
