"""Association with more directions than one kernel compares (8192): chunks of 1024
directions and their merge, at the edges of chunks and workgroups and for every
objective count, alone, in a selection and in a batch; bit for bit against the
oracle and the single run."""
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


def _directions(rng, m, k):
    w = rng.random((m, k)) + 1e-3
    w = (w / np.linalg.norm(w, axis=0)).astype(np.float32)
    w[:, k - 1] = w[:, 5]                            # equal directions in the first and the last chunk
    return w


@pytest.mark.parametrize("n,k,m", [(1, 8193, 1), (255, 8192, 2), (256, 8193, 3), (257, 9215, 4), (300, 9216, 5),
                                   (64, 9217, 6), (100, 12000, 7), (513, 8200, 8), (70, 66000, 9), (1000, 10240, 10),
                                   (90, 70000, 3)])
def test_chunks_equal_oracle(n, k, m):
    rng = np.random.default_rng(k + n)
    w = _directions(rng, m, k)
    fn = (rng.random((m, n)) * rng.uniform(0.1, 3.0, (1, n))).astype(np.float32)
    fn[:, : n // 3] = w[:, rng.integers(0, k, n // 3)]                     # on a direction
    fn[:, n // 2] = w[:, 5] * np.float32(1.5)
    if n > 60:
        fn[0, 40], fn[0, 41], fn[:, 42] = np.nan, np.inf, 0.0
    print(f"association chunks n={n} k={k} m={m}", flush=True)
    d, r = K.associate(_f(fn), torch.ones(m, device=DEV), _f(w), 1)
    do, ro = O.associate(fn, w)
    np.testing.assert_array_equal(r.cpu().numpy(), ro)
    np.testing.assert_array_equal(d.cpu().numpy().view(np.uint32), do.view(np.uint32))


@pytest.mark.parametrize("n,m,k", [(200, 5, 9000), (1024, 4, 12288), (300, 3, 66000)])
def test_selection_equals_oracle(n, m, k):
    rng = np.random.default_rng(n + k)
    u = np.abs(rng.standard_normal((m, 2 * n)))
    fm = (u / np.linalg.norm(u, axis=0) * rng.uniform(1.0, 1.1, 2 * n)).astype(np.float32)
    cvm = np.zeros(2 * n, np.float32)
    xm = np.zeros((2 * n, 2), np.float32)
    xm[:, 0] = np.arange(2 * n, dtype=np.float32)
    w = _directions(rng, m, k)
    ideal0 = fm[:, :n].min(axis=1).astype(np.float32)
    ua, ub = O.draw_niche(5, 3, 2 * n)
    chosen, fr_mix, st, _ = O.nsga3_select(fm, cvm, w, ideal0, ua, ub)
    print(f"selection n={n} m={m} k={k}: n_prior={st[1]} n_last={st[2]}", flush=True)
    par = K.Population(_f(xm[:n]), _f(fm[:, :n]), _f(cvm[:n]))
    ofs = K.Population(_f(xm[n:]), _f(fm[:, n:]), _f(cvm[n:]))
    nxt, nfr, _ = K.nsga3_select(par, ofs, _f(w), _f(ideal0), seed=5, generation=3)
    np.testing.assert_array_equal(nxt.x[:, 0].cpu().numpy().astype(np.int64), chosen)
    np.testing.assert_array_equal(nfr.cpu().numpy(), fr_mix[chosen])


@pytest.mark.parametrize("graph", [False, True])
def test_batch_equals_single_runs(graph):
    def runs():                                      # K = 91, 14950, 330 and 2600
        return [cm.NSGA3(population_size=n, max_generations=6, problem=cm.QuadraticCenters(d, m, seed=n), seed=n,
                         reference_directions=cm.DasDennisDirections(partitions=p), print_progress=False)
                for n, m, d, p in ((100, 3, 10, 12), (130, 5, 20, 22), (64, 8, 9, 4), (200, 4, 16, 23))]
    batch = cm.BatchNSGA3(runs(), graph=graph)
    batch.initialize()
    batch.step(6)
    for i, alone in enumerate(runs()):
        print(f"batch instance {i}", flush=True)
        r, s = batch.result(i), alone.run()
        for name in ("variables", "objectives", "constraints", "auxiliary_indices"):
            assert torch.equal(torch.as_tensor(getattr(r, name)).cpu(), torch.as_tensor(getattr(s, name)).cpu()), name
