"""Reproduction with its own draws, one and four variables a thread: rows of 1 to
9 variables and others that four does not divide, an odd last row, parents that
begin off a 16-byte line, equal parents, variables at their bounds, with and
without copying and with up to every variable mutated; offspring bit for bit
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


# the last two have the 2^24 pair-variables from which four go to a thread
SIZES = [(n, d, shift, copy_p, pm_p) for d in (1, 2, 3, 4, 5, 7, 8, 9, 63, 254, 1030)
         for n, shift, copy_p, pm_p in ((1, 0, 0.0, 1.0), (2, 1, 0.0, 1.0), (7, 1, 0.5, 40.0), (64, 2, 0.5, 1.0),
                                        (101, 3, 0.0, 4.0))] + [(8193, 4099, 1, 0.5, 4.0), (131074, 257, 0, 0.0, 1.0)]


@pytest.mark.parametrize("n,d,shift,copy_p,pm_p", SIZES)
def test_reproduce_rows(n, d, shift, copy_p, pm_p):
    rng = np.random.default_rng(n * 2048 + d)
    lo, hi = np.float32(-1.5), np.float32(2.25)
    x = (lo + (hi - lo) * rng.random((n, d), dtype=np.float32)).astype(np.float32)
    x[rng.random((n, d)) < 0.1] = lo
    x[rng.random((n, d)) < 0.1] = hi
    x[rng.random((n, d)) < 0.1] = np.float32(0.5)
    bounds = np.tile(np.array([lo, hi], np.float32), d)
    rank = rng.integers(0, 3, n).astype(np.int32)
    cv = np.zeros(n, np.float32)
    seed, gen = 1234 + d, 3
    buf = torch.zeros(n * d + 4, dtype=torch.float32, device=DEV)
    xg = buf[shift:shift + n * d].view(n, d)
    xg.copy_(_f(x))
    print(f"reproduce rows n={n} d={d} shift={shift} copy={copy_p} pm={pm_p}", flush=True)
    off_g, win_g = K.reproduce(xg, _f(bounds), rank=_f(rank), cv=_f(cv), sbx=(20.0, 0.9, copy_p), pm=(20.0, pm_p),
                               seed=seed, generation=gen)
    ca, cb = O.draw_mating(seed, gen, n, n)
    win = O.tournament(ca, cb, rank, cv)
    np.testing.assert_array_equal(win_g.cpu().numpy(), win)
    ub, up, sg, uc = O.draw_sbx(seed, gen, n // 2, d)
    off = O.sbx(x, win, bounds, ub, up, sg, uc, 20.0, 0.9, copy_p, n)
    ug, ud = O.draw_pm(seed, gen, n, d)
    off = O.pm(off, bounds, ug, ud, 20.0, pm_p)
    np.testing.assert_array_equal(off_g.cpu().numpy(), off)
