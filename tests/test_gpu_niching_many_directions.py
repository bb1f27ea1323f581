"""Niching at and above 65535 directions, the most that a niche's 16-bit direction
word holds, with nearly every member of the last front in the directions of the
highest indices; survivors against the oracle in every niching mode."""
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


@pytest.mark.parametrize("m,k,spread", [(3, 65535, 40), (3, 65536, 40), (3, 65537, 40), (4, 66000, 464), (3, 73000, 7464)])
def test_survivors_equal_oracle(m, k, spread):
    rng = np.random.default_rng(k)
    n = 600
    fm = rng.random((m, 2 * n)) + 1e-3
    fm = (fm / fm.sum(axis=0)).astype(np.float32)
    cvm = np.zeros(2 * n, np.float32)
    xm = np.zeros((2 * n, 2), np.float32)
    xm[:, 0] = np.arange(2 * n, dtype=np.float32)
    w = rng.random((m, k)) + 1e-3                    # the last `spread` cover the plane
    w[0, : k - spread] += 500.0                      # the others lie around one axis
    w = (w / np.linalg.norm(w, axis=0)).astype(np.float32)
    ideal0 = fm[:, :n].min(axis=1).astype(np.float32)
    ua, ub = O.draw_niche(5, 3, 2 * n)
    chosen, fr_mix, st, _ = O.nsga3_select(fm, cvm, w, ideal0, ua, ub)
    assert st[2] > n                                 # the last front is cut
    for mode in (0, 2, 3):
        print(f"niching k={k} m={m} mode={mode}", flush=True)
        par = K.Population(_f(xm[:n]), _f(fm[:, :n]), _f(cvm[:n]))
        ofs = K.Population(_f(xm[n:]), _f(fm[:, n:]), _f(cvm[n:]))
        nxt, nfr, _ = K.nsga3_select(par, ofs, _f(w), _f(ideal0), seed=5, generation=3, niching=(mode, 0))
        np.testing.assert_array_equal(nxt.x[:, 0].cpu().numpy().astype(np.int64), chosen)
        np.testing.assert_array_equal(nfr.cpu().numpy(), fr_mix[chosen])
