"""Selection of small populations, whose stages between the sort and the
association run in one workgroup up to 2n = 4096 merged rows: both sides of that
line and of the 2048 in it, every objective count, rows left over in a wavefront, infeasible and NaN
rows; chosen rows, fronts, state, ideal point, extremes and intercepts (the
latter within the 1e-6 of the FP64 solve that the larger sizes are held to)
against the oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a ROCm GPU", allow_module_level=True)

import oracle as O  # noqa: E402
from cuda_moea import kernels as K  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _f(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


@pytest.mark.parametrize("n,m,kind", [(2, 2, "sphere"), (34, 7, "ties"), (66, 9, "rand"), (130, 6, "rand"),
                                      (512, 4, "infeasible"), (1022, 3, "nan"), (1024, 10, "sphere"),
                                      (1024, 2, "ties"), (1026, 3, "sphere"), (1026, 9, "ties"),
                                      (700, 7, "infeasible"), (2048, 5, "ties"), (2050, 4, "sphere")])
def test_small_selection(n, m, kind):
    rng = np.random.default_rng(n * 16 + m)
    if kind == "ties":
        fm = (rng.integers(0, 6, (m, 2 * n)) / 6).astype(np.float32)
    elif kind == "sphere":
        g = np.abs(rng.standard_normal((m, 2 * n)))
        fm = (rng.uniform(1.0, 1.2, 2 * n) * g / np.linalg.norm(g, axis=0)).astype(np.float32)
    else:
        fm = rng.random((m, 2 * n), dtype=np.float32)
    cvm = np.zeros(2 * n, np.float32)
    if kind == "infeasible":
        cvm = np.where(rng.random(2 * n) < 0.7, rng.random(2 * n), 0.0).astype(np.float32)
    w = O.das_dennis(n, m)
    ideal0 = fm[:, :n].min(axis=1).astype(np.float32)
    if kind == "nan":
        fm[:, rng.random(2 * n) < 0.05] = np.nan
    ua = rng.integers(0, 2**32, 2 * n, dtype=np.uint64).astype(np.uint32)
    ub = rng.integers(0, 2**32, 2 * n, dtype=np.uint64).astype(np.uint32)
    x = np.arange(2 * n, dtype=np.float32).reshape(-1, 1)
    print(f"small selection n={n} m={m} kind={kind}", flush=True)
    onorm, norm = {}, {}
    chosen, fr_o, st_o, ideal_o = O.nsga3_select(fm, cvm, w, ideal0, ua, ub, normalization=onorm)
    par = K.Population(_f(x[:n]), _f(fm[:, :n]), _f(cvm[:n]))
    ofs = K.Population(_f(x[n:]), _f(fm[:, n:]), _f(cvm[n:]))
    ideal_g = _f(ideal0)
    nxt, nfr, st = K.nsga3_select(par, ofs, _f(w), ideal_g, draws={"niche_a": ua, "niche_b": ub}, normalization=norm)
    st = st.cpu().numpy()
    np.testing.assert_array_equal(st[:3], st_o[:3])
    np.testing.assert_array_equal(nxt.x[:, 0].cpu().numpy().astype(np.int64), chosen)
    np.testing.assert_array_equal(nfr.cpu().numpy(), fr_o[chosen])
    np.testing.assert_array_equal(ideal_g.cpu().numpy(), ideal_o)
    if st[4] > 0:
        assert st[3] == st_o[3]
        np.testing.assert_array_equal(norm["extremes"].cpu().numpy(), onorm["extremes"])
        a64 = onorm["intercepts"]
        a = norm["intercepts"].cpu().numpy()
        assert np.all((np.abs(a - a64) <= 1e-6 * np.abs(a64)) | (np.isnan(a) & np.isnan(a64)) | (a == a64)), (a, a64)
