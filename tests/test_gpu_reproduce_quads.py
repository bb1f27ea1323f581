"""Reproduction with its own draws, one and four variables a thread, each with rows
of 1 to 9 variables and others that four does not divide, an odd last row, parents that
begin off a 16-byte line, equal parents, variables at their bounds, with and
without copying and with up to every variable mutated; offspring bit for bit
against the oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a ROCm GPU", allow_module_level=True)

import cuda_moea as cm  # noqa: E402
import oracle as O  # noqa: E402
from cuda_moea import kernels as K  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _f(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


# those with 2^24 pair-variables and at most a quarter of the used ones mutated take four a thread
SIZES = [(n, d, shift, copy_p, pm_p) for d in (1, 2, 3, 4, 5, 7, 8, 9, 63, 254, 1030)
         for n, shift, copy_p, pm_p in ((1, 0, 0.0, 1.0), (2, 1, 0.0, 1.0), (7, 1, 0.5, 40.0), (64, 2, 0.5, 1.0),
                                        (101, 3, 0.0, 4.0))] + [(8193, 4099, 1, 0.5, 4.0), (131074, 257, 0, 0.0, 1.0),
                                                  (33554433, 1, 3, 0.0, 0.05), (16777216, 2, 1, 0.5, 0.2),
                                                  (11184812, 3, 2, 0.0, 0.5), (8388609, 4, 1, 0.0, 1.0),
                                                  (5592406, 6, 3, 0.5, 1.1), (4793492, 7, 1, 0.0, 1.5),
                                                  (4194304, 8, 2, 0.5, 2.0), (3728273, 9, 3, 0.0, 1.6),
                                                  (33026, 1030, 0, 0.0, 1.0)]


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


def _philox(counter, stream, seed, gen):
    """The engine's counter draws (Philox4x32-10) of many elements."""
    c = [counter & 0xFFFFFFFF, counter >> 32, np.full_like(counter, gen), np.full_like(counter, stream)]
    k = [np.uint64(seed & 0xFFFFFFFF), np.uint64(seed >> 32)]
    mask = np.uint64(0xFFFFFFFF)
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ k[0], p1 & mask, (p0 >> np.uint64(32)) ^ c[3] ^ k[1], p0 & mask]
        k = [(k[0] + np.uint64(0x9E3779B9)) & mask, (k[1] + np.uint64(0xBB67AE85)) & mask]
    return c


def test_more_elements_than_31_bits():
    """Pairs on both sides of element 2^31, whose draw counter's 32-bit arithmetic and index division end there."""
    n, d, seed, gen = 16388, 262147, 77, 4
    assert (n // 2) * d > 1 << 31
    print(f"reproduce n={n} d={d}", flush=True)
    x = torch.rand(n, d, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1))
    bounds = np.tile(np.array([0.0, 1.0], np.float32), d)
    rank = torch.randint(0, 3, (n,), device=DEV, dtype=torch.int32)
    pm_p = 2000.0
    off, win = K.reproduce(x, _f(bounds), rank=rank, cv=torch.zeros(n, device=DEV), sbx=(20.0, 0.9, 0.5), pm=(20.0, pm_p),
                           seed=seed, generation=gen)
    for pair in (0, 5000, 8190, 8191, 8192, 8193):
        rs = _philox(np.uint64(pair) * np.uint64(d) + np.arange(d, dtype=np.uint64), 3, seed, gen)
        rp = _philox(np.uint64(pair) * np.uint64(d) + np.arange(d, dtype=np.uint64), 4, seed, gen)
        if pair == 0:
            np.testing.assert_array_equal([w[9] for w in rs], O.philox4x32_10([9, 0, gen, 3], [seed, 0]))
        u01 = lambda w: ((w >> np.uint64(8)).astype(np.float32) * np.float32(2.0 ** -24)).astype(np.float32)
        byte = np.uint64(0xFF)
        gate_b = ((rs[0] & byte) << np.uint64(16)) | ((rs[1] & byte) << np.uint64(8)) | (rs[2] & byte)
        ug = np.concatenate([u01(rs[3]), u01(gate_b << np.uint64(8))])
        ud = np.concatenate([u01(rp[0]), u01(rp[1])])
        sign = ((rs[3] >> np.uint64(7)) & np.uint64(1)).astype(np.int32)
        rows = win[2 * pair:2 * pair + 2].long()
        ref = O.sbx(x[rows].cpu().numpy(), np.array([0, 1], np.int32), bounds, u01(rs[0]), u01(rs[1]), sign, u01(rs[2]),
                    20.0, 0.9, 0.5, 2)
        ref = O.pm(ref, bounds, ug, ud, 20.0, pm_p)
        np.testing.assert_array_equal(off[2 * pair:2 * pair + 2].cpu().numpy(), ref)


class _Tournament(cm.PythonMating):
    """The built-in tournament's winners, handed in."""

    def select(self, parents, state, context):
        _, idx = K.reproduce(parents["variables"], parents["bounds"].reshape(-1).contiguous(), rank=state["rank"],
                             cv=parents["constraints"], seed=5, generation=context["generation"])
        return idx


class _Copy(cm.PythonCrossover):
    def apply(self, parents, parent_indices, context):
        return parents["variables"][parent_indices.long()]


def test_given_parents_and_mutation_alone():
    """Four variables a thread with parents from the caller, and for mutation alone: a run with either equals the
    run that draws its parents, or crosses with probability 0, by itself."""
    def run(**kw):
        alg = cm.NSGA3(population_size=8192, max_generations=2, problem=cm.QuadraticCenters(8203, 3, seed=1), seed=5,
                       reference_directions=cm.DasDennisDirections(partitions=12), print_progress=False, **kw)
        return alg.run().variables.cpu()

    print("reproduce through given parents", flush=True)
    assert torch.equal(run(), run(mating=_Tournament()))
    print("reproduce through mutation alone", flush=True)
    assert torch.equal(run(crossover=cm.SBX(probability=0.0)), run(crossover=_Copy()))
