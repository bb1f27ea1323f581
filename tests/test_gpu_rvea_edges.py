"""RVEA's gamma at the edges of its tiles and the survivor list at the edge of
its LDS capacity, against the oracle."""
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


@pytest.mark.parametrize("k,m", [(1, 3), (2, 2), (31, 5), (33, 4), (69, 10), (70, 10), (150, 3), (151, 3), (225, 1), (226, 1), (256, 3), (511, 10), (512, 3), (513, 6), (1500, 2)])
def test_gamma_tile_edges(k, m):
    rng = np.random.default_rng(k)
    v = rng.standard_normal((m, k)).astype(np.float32)       # negative products too
    v /= np.linalg.norm(v, axis=0).astype(np.float32)
    if k > 40:
        v[:, 37] = v[:, 3]                                    # a duplicate: angle zero
    print(f"gamma k={k} m={m}", flush=True)
    np.testing.assert_array_equal(K.rvea_gamma(_f(v)).cpu().numpy(), O.rvea_gamma(v))


@pytest.mark.parametrize("n", [1, 33, 1001, 262144, 262145])   # 2n bits: 64 KiB of LDS at n = 262144
def test_survivor_list_sizes(n):
    m, k = 2, 24
    rng = np.random.default_rng(n)
    v = O.das_dennis(k, m, kind=2)
    gam = O.rvea_gamma(v)
    fm = (rng.random((m, 2 * n), dtype=np.float32) + 0.05).astype(np.float32)
    cvm = np.zeros(2 * n, np.float32)
    x = np.zeros((2 * n, 1), np.float32)
    x[:, 0] = np.arange(2 * n)
    pen = O.rvea_penalty(m, 3, 10, 2.0)
    print(f"rvea survivors n={n}", flush=True)
    sel, na, _, _, _ = O.rvea_select(fm, cvm, v, gam, n, pen)
    par = K.Population(_f(x[:n]), _f(fm[:, :n]), _f(cvm[:n]))
    ofs = K.Population(_f(x[n:]), _f(fm[:, n:]), _f(cvm[n:]))
    nxt, na_g = K.rvea_select(par, ofs, _f(v), _f(gam), n, pen)
    assert na_g == na
    np.testing.assert_array_equal(nxt.x[:na, 0].cpu().numpy().astype(np.int64), sel)
