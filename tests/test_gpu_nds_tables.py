"""Non-dominated ranks at the edges of the sort's pieces: rank-table chunks of
512 rows, word blocks of 64, the 32 row blocks (2048 rows) up to which one
workgroup peels, every objective count, exact ties, signed zeros and infinities;
fronts bit for bit against the oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a ROCm GPU", allow_module_level=True)

import oracle as O  # noqa: E402
from cuda_moea import kernels as K  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)

CASES = [(511, 2), (512, 3), (513, 9), (127, 10), (129, 9), (256, 10), (257, 8), (1023, 4), (1025, 7), (1025, 1),
         (2047, 3), (2048, 5), (2049, 3), (2048, 1), (2049, 10), (2112, 6)]


@pytest.mark.parametrize("n,m", CASES)
@pytest.mark.parametrize("kind", ["rand", "ties", "special", "chain"])
def test_ranks_at_edges(n, m, kind):
    rng = np.random.default_rng(n * 16 + m)
    if kind == "ties":
        f = (rng.integers(0, 4, (m, n)) / 4).astype(np.float32)
    elif kind == "chain":                # one row a front
        f = np.repeat(rng.permutation(n).astype(np.float32)[None], m, 0)
    else:
        f = rng.random((m, n), dtype=np.float32)
    if kind == "special":
        f[rng.random((m, n)) < 0.1] = np.float32(0.0)
        f[rng.random((m, n)) < 0.1] = np.float32(-0.0)
        f[rng.random((m, n)) < 0.03] = np.inf
        f[rng.random((m, n)) < 0.03] = -np.inf
    cv = np.zeros(n, np.float32)
    for stop in (n, (n + 1) // 2):
        print(f"nds edges n={n} m={m} kind={kind} stop={stop}", flush=True)
        fr_o, mf_o = O.nds(f, cv, stop)
        fr_g, mf_g = K.nds_rank(torch.from_numpy(f).to(DEV), torch.from_numpy(cv).to(DEV), stop)
        assert mf_g == mf_o
        np.testing.assert_array_equal(fr_g.cpu().numpy(), fr_o)


@pytest.mark.parametrize("n,m", [(2000, 1), (2500, 1), (2500, 2), (3001, 3), (2300, 5)])
@pytest.mark.parametrize("kind", ["band", "two chains"])
def test_many_fronts(n, m, kind):
    """Hundreds to thousands of fronts that the assigned set fills in sort order, and one where a second chain
    stays open below the first, with infeasible rows after both."""
    rng = np.random.default_rng(n + m)
    i = np.arange(n, dtype=np.float32)
    f = np.repeat(i[None], m, 0)
    if kind == "band":
        f += rng.uniform(0, 8, (m, n)).astype(np.float32)
    elif m > 1:                                      # the later half is not dominated by the earlier one
        f[1, n // 2:] -= n
    p = rng.permutation(n)
    f = np.ascontiguousarray(f[:, p])
    cv = np.where(rng.random(n) < 0.1, rng.integers(1, 9, n), 0).astype(np.float32)
    for stop in (n, n // 3):
        print(f"nds many fronts n={n} m={m} kind={kind} stop={stop}", flush=True)
        fr_o, mf_o = O.nds(f, cv, stop)
        fr_g, mf_g = K.nds_rank(torch.from_numpy(f).to(DEV), torch.from_numpy(cv).to(DEV), stop)
        assert mf_g == mf_o
        np.testing.assert_array_equal(fr_g.cpu().numpy(), fr_o)
