"""A grouped linear's decode rows in one GEMV launch: groups and rows on both
sides of the prepare forms (one batch, one pass, several), odd group counts,
an input long enough to split k, a rate without a GEMM over several windows of
16 rows, every activation type, against the oracle's projection group by
group."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402
from plugins_amd import exl3 as X  # noqa: E402
from tests import _synth as S  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G,in_f,out_f,n,rows,dtype", [
    (3, 256, 128, 48, 1, torch.float16), (3, 2048, 256, 64, 2, torch.bfloat16),
    (5, 1152, 384, 32, 5, torch.float32), (2, 4096, 128, 128, 16, torch.float16),
    (7, 384, 128, 40, 4, torch.bfloat16), (2, 512, 256, 50, 37, torch.float16)])
def test_grouped_gemv_every_group(G, in_f, out_f, n, rows, dtype):
    rng = np.random.default_rng(G * 1000 + in_f + rows)
    parts = [S.linear(rng, in_f, out_f, n) for _ in range(G)]
    src = {}
    for g, (t, u, v) in enumerate(parts):
        src[f"m.slice.{g}.trellis"] = t.view(np.int16)
        src[f"m.slice.{g}.suh"] = u.view(np.float16)
        src[f"m.slice.{g}.svh"] = v.view(np.float16)
    L = X.Loader('{"format":"exl3","codebook":"mul1"}', X.DictSource(src))
    v, w = L.load_tensor("m", in_f)
    assert v.is_ok(), v
    assert X.matmul_path(w, rows) == "gemv-groups"
    x = torch.from_numpy(S.activations(rng, rows * G, in_f).reshape(rows, G, in_f)).to("cuda").to(dtype)
    y = X.matmul(w, x, out=torch.empty(rows, G, out_f, dtype=dtype, device="cuda"))
    y = y.float().cpu().numpy()
    xs = x.float().cpu().numpy()
    # the repository's bar, and a bf16 output's own rounding (2^-9) beside it
    bar = 3e-3 if dtype == torch.bfloat16 else 1e-3
    for g, (t, u, vv) in enumerate(parts):
        want = S.h2f(O.project(np.ascontiguousarray(xs[:, g]), t, u, vv, in_f, out_f, n))
        assert S.rel_fro(y[:, g], want) < bar, g
        assert S.row_rel(y[:, g], want).max() < 2 * bar, g
    assert X.stream_status().is_ok()
    X.release(w)
    L.close()


def test_path_of_every_width():
    """One launch over the groups, or each group alone: prompts at a
    half-integer rate, whose GEMM takes one linear."""
    rng = np.random.default_rng(3)
    paths = {}
    for n in (48, 40, 50):
        src = {}
        for g in range(2):
            t, u, v = S.linear(rng, 256, 128, n)
            src[f"m.slice.{g}.trellis"] = t.view(np.int16)
            src[f"m.slice.{g}.suh"] = u.view(np.float16)
            src[f"m.slice.{g}.svh"] = v.view(np.float16)
        L = X.Loader('{"format":"exl3","codebook":"mul1"}', X.DictSource(src))
        v, w = L.load_tensor("m", 256)
        assert v.is_ok(), v
        paths[n] = [X.matmul_path(w, r) for r in (1, 16, 17, 300)]
        X.release(w)
        L.close()
    gv, gm = "gemv-groups", "gemm-groups"
    assert paths == {48: [gv, gv, gm, gm], 40: [gv, gv, "per-group", "per-group"], 50: [gv] * 4}
