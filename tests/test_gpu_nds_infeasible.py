"""Fronts of infeasible rows (their order by cv, no dominance bitmask) against
the oracle's peeling: many distinct violations, ties, NaN violations, no
feasible row at all, and stop counts that fall inside the infeasible part."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a ROCm GPU", allow_module_level=True)

import oracle as O  # noqa: E402
from cuda_moea import kernels as K  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


# rows, objectives, feasible share, distinct violations (0: all distinct), NaN share
CASES = [(1, 2, 0.0, 0, 0.0), (1, 3, 0.0, 0, 1.0), (64, 3, 0.0, 0, 0.0), (65, 3, 0.0, 3, 0.2), (300, 2, 0.3, 0, 0.1),
         (700, 3, 0.0, 0, 1.0), (1000, 5, 0.5, 4, 0.0), (1500, 3, 0.7, 0, 0.3), (2049, 8, 0.02, 40, 0.02),
         (4100, 3, 0.9, 0, 0.0)]


@pytest.mark.parametrize("n,m,feasible,levels,nan", CASES)
def test_infeasible_fronts(n, m, feasible, levels, nan):
    rng = np.random.default_rng(n)
    f = rng.random((m, n), dtype=np.float32)
    v = rng.integers(1, levels + 1, n).astype(np.float32) if levels else rng.permutation(n).astype(np.float32) - n / 3
    v[v == 0] = 0.25
    cv = np.where(rng.random(n) < feasible, np.float32(0.0), v).astype(np.float32)
    cv[(cv != 0) & (rng.random(n) < nan)] = np.nan
    cv[(cv > 0) & (rng.random(n) < 0.05)] = np.inf
    n_feas = int((cv == 0).sum())
    n_nan = int(np.isnan(cv).sum())
    for stop in sorted({1, max(1, n_feas), n_feas + 1, n_feas + n_nan + 1, (n_feas + n) // 2 + 1, n - 1, n, n + 5} - {0}):
        print(f"infeasible case n={n} m={m} feasible={n_feas} nan={n_nan} stop={stop}", flush=True)
        fr_o, mf_o = O.nds(f, cv, stop)
        fr_g, mf_g = K.nds_rank(torch.from_numpy(f).to(DEV), torch.from_numpy(cv).to(DEV), stop)
        assert mf_g == mf_o
        np.testing.assert_array_equal(fr_g.cpu().numpy(), fr_o)
