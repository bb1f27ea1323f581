"""Niching with few directions (each niche holds hundreds to thousands of the
last front): the path that cuts niches into parts by value, its fallback for
values too uneven, and the counted selection of small fronts, against the
oracle."""
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


def _objectives(rng, kind, m, nm):
    g = rng.random((m, nm)) + 1e-3
    if kind == "narrow":                             # one niche takes nearly all, distances close together
        g = 1.0 + 0.01 * g
    if kind == "equal":                              # 60 % one point: equal distances, uneven parts
        g[:, : (3 * nm) // 5] = g[:, :1]
    return (g / g.sum(axis=0)).astype(np.float32)


# population, objectives, Das-Dennis partitions, kind
@pytest.mark.parametrize("n,m,parts,kind", [(192, 3, 1, "plane"), (194, 3, 2, "narrow"), (600, 3, 3, "plane"),
                                            (2048, 3, 12, "narrow"), (4096, 3, 12, "plane"), (4096, 8, 2, "plane"),
                                            (4096, 2, 5, "narrow"), (5120, 3, 4, "plane"), (5122, 3, 4, "plane"),
                                            (3000, 3, 4, "equal")])
def test_few_directions_equal_oracle(n, m, parts, kind):
    rng = np.random.default_rng(n + m)
    fm = _objectives(rng, kind, m, 2 * n)
    cvm = np.zeros(2 * n, np.float32)
    xm = np.zeros((2 * n, 2), np.float32)
    xm[:, 0] = np.arange(2 * n, dtype=np.float32)
    w = O.das_dennis(n, m, partitions=parts)
    ideal0 = fm[:, :n].min(axis=1).astype(np.float32)
    ua, ub = O.draw_niche(5, 3, 2 * n)
    chosen, fr_mix, st, _ = O.nsga3_select(fm, cvm, w, ideal0, ua, ub)
    print(f"niching n={n} m={m} k={w.shape[1]} kind={kind}: n_prior={st[1]} n_last={st[2]}", flush=True)
    for cap in (0, 1):
        par = K.Population(_f(xm[:n]), _f(fm[:, :n]), _f(cvm[:n]))
        ofs = K.Population(_f(xm[n:]), _f(fm[:, n:]), _f(cvm[n:]))
        nxt, nfr, _ = K.nsga3_select(par, ofs, _f(w), _f(ideal0), seed=5, generation=3, niching=(1, cap))
        np.testing.assert_array_equal(nxt.x[:, 0].cpu().numpy().astype(np.int64), chosen)
        np.testing.assert_array_equal(nfr.cpu().numpy(), fr_mix[chosen])


def test_one_direction_65532_members():
    """The largest niche whose members' positions fit 16 bits (its square needs 32)."""
    n, m = 32766, 3
    rng = np.random.default_rng(1)
    fm = _objectives(rng, "plane", m, 2 * n)
    cvm = np.zeros(2 * n, np.float32)
    xm = np.zeros((2 * n, 2), np.float32)
    xm[:, 0] = np.arange(2 * n, dtype=np.float32)
    w = np.full((m, 1), 1 / np.sqrt(3), np.float32)
    ideal0 = fm[:, :n].min(axis=1).astype(np.float32)
    ua, ub = O.draw_niche(5, 3, 2 * n)
    chosen, fr_mix, st, _ = O.nsga3_select(fm, cvm, w, ideal0, ua, ub)
    print(f"niching one direction: n_prior={st[1]} n_last={st[2]}", flush=True)
    assert st[2] > 46341
    par = K.Population(_f(xm[:n]), _f(fm[:, :n]), _f(cvm[:n]))
    ofs = K.Population(_f(xm[n:]), _f(fm[:, n:]), _f(cvm[n:]))
    nxt, nfr, _ = K.nsga3_select(par, ofs, _f(w), _f(ideal0), seed=5, generation=3)
    np.testing.assert_array_equal(nxt.x[:, 0].cpu().numpy().astype(np.int64), chosen)
    np.testing.assert_array_equal(nfr.cpu().numpy(), fr_mix[chosen])
