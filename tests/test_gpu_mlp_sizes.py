"""The MLP objective against FP64 at the edges of its tiles, slices and loads,
and its value for infinite and NaN variables."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a ROCm GPU", allow_module_level=True)

from cuda_moea import kernels as K  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _case(n, d, hidden, m):
    g = torch.Generator().manual_seed(n + d)
    x = torch.rand(n, d, generator=g)
    w1 = torch.randn(hidden, d, generator=g) / np.sqrt(d)
    w2 = torch.randn(m, hidden, generator=g) / np.sqrt(hidden)
    return x, w1, w2


def _fp64(x, w1, w2):
    xd = x.double()
    y = torch.tanh(xd @ w1.double().t()) @ w2.double().t()
    return (y.square() + 0.01 * (xd - 0.5).square().sum(1, keepdim=True)).t()


# tiles of 64 and 128 rows and columns, slices of 32, rows of every alignment,
# matrices of fewer than four numbers, rows of one to three numbers beside their
# matrix's end, folds at 4096, the large tile shape
@pytest.mark.parametrize("n,d,hidden,m", [(1, 1, 1, 1), (1, 3, 1, 2), (3, 1, 5, 3), (2, 2, 2, 1), (1, 5, 2, 1),
                                          (63, 31, 64, 3), (64, 32, 65, 5), (65, 33, 63, 2), (128, 35, 128, 10),
                                          (129, 64, 130, 4), (200, 4095, 100, 3), (130, 4097, 96, 3),
                                          (127, 8194, 40, 3), (12288, 37, 256, 5), (12289, 66, 255, 5),
                                          (4, 1, 4, 2), (5, 1, 3, 1), (9, 1, 64, 3), (70, 1, 65, 3), (300, 1, 256, 5),
                                          (24577, 1, 256, 3), (4, 2, 4, 1), (70, 2, 64, 3), (4, 3, 5, 2), (70, 3, 65, 3)])
def test_mlp_sizes_against_fp64(n, d, hidden, m):
    x, w1, w2 = _case(n, d, hidden, m)
    print(f"mlp n={n} d={d} hidden={hidden} m={m}", flush=True)
    f, cv = K.eval_mlp(x.to(DEV), w1.to(DEV), w2.to(DEV))
    ref = _fp64(x, w1, w2)
    # float sums of d terms: 64 sqrt(d) 2^-24 (1 + |f|), the objective tests' bound
    tol = 64 * np.sqrt(d) * 2.0 ** -24 * (1 + ref.abs())
    assert bool(((f.cpu().double() - ref).abs() <= tol).all())
    assert not cv.cpu().any()


# variables and weights far from one: parts that would fall under bf16's smallest
# exponents, subnormal variables, sums past the split's range
@pytest.mark.parametrize("n,d", [(70, 10), (200, 33), (24576, 64)])
@pytest.mark.parametrize("xe,we", [(-118, 118), (-126, 124), (-135, 125), (60, -60), (20, -110), (-3, 110)])
def test_mlp_far_magnitudes(n, d, xe, we):
    hidden = m = 10
    x, w1, _ = _case(n, d, hidden, m)
    x, w1 = torch.ldexp(x, torch.tensor(xe)), torch.ldexp(w1, torch.tensor(we))
    print(f"mlp far n={n} d={d} xe={xe} we={we}", flush=True)
    f, _ = K.eval_mlp(x.to(DEV), w1.to(DEV), torch.eye(hidden).to(DEV))
    xd, wd = x.double(), w1.double()
    ref = _fp64(x, w1, torch.eye(hidden))
    # d + 4 roundings of each hidden sum, d + 8 of the distance and the objective
    tol = 2.0 ** -24 * ((2 * (d + 4) * (xd.abs() @ wd.abs().t()).t()).clamp(max=2.0 ** 24) + (d + 8) * ref)
    if we == 110:                                    # saturated: the units' signs alone
        tol = 2.0 ** -24 * (d + 8) * ref
    assert bool(((f.cpu().double() - ref).abs() <= tol).all())


def test_mlp_infinite_and_nan_rows():
    n, d, hidden, m = 70, 45, 64, 3
    x, w1, w2 = _case(n, d, hidden, m)
    w1[3, 7] = 0.0
    x[5, 7], x[6, 9], x[7, 2], x[8, 4] = np.inf, -np.inf, np.nan, 3.4e38
    f, _ = K.eval_mlp(x.to(DEV), w1.to(DEV), w2.to(DEV))
    f = f.cpu()
    keep = [i for i in range(n) if i not in (5, 6, 7, 8)]
    ref = _fp64(x[keep], w1, w2)
    tol = 64 * np.sqrt(d) * 2.0 ** -24 * (1 + ref.abs())
    assert bool(((f[:, keep].double() - ref).abs() <= tol).all())
    assert bool(torch.isnan(f[:, 5]).all())               # 0 * inf in hidden unit 3, as in FP32
    assert bool(torch.isinf(f[:, 6]).all())               # every hidden unit saturates, the distance is infinite
    assert bool(torch.isnan(f[:, 7]).all())
    assert bool(torch.isinf(f[:, 8]).all())               # (3.4e38)^2 overflows in the distance only


# both tile shapes, each way of loading
@pytest.mark.parametrize("n,d,hidden,m", [(70, 45, 64, 3), (130, 64, 65, 2), (9, 1, 64, 3), (12289, 66, 255, 5), (12288, 4100, 256, 2)])
def test_mlp_nan_rows_leave_the_others_alone(n, d, hidden, m):
    x, w1, w2 = _case(n, d, hidden, m)
    print(f"mlp nan rows n={n} d={d} hidden={hidden} m={m}", flush=True)
    clean, _ = K.eval_mlp(x.to(DEV), w1.to(DEV), w2.to(DEV))
    x[1, d - 1], x[n - 1, 0], x[n // 2, d // 2] = np.nan, np.inf, -np.inf
    f, _ = K.eval_mlp(x.to(DEV), w1.to(DEV), w2.to(DEV))
    bad = [1, n // 2, n - 1]
    ref = _fp64(x[bad], w1, w2)
    f, clean = f.cpu(), clean.cpu()
    assert torch.equal(torch.isnan(f[:, bad]), torch.isnan(ref)) and torch.equal(torch.isinf(f[:, bad]), torch.isinf(ref))
    f[:, bad] = clean[:, bad]
    assert torch.equal(f, clean)


def test_mlp_time_with_nan_rows():
    """A NaN in every row costs about one more pass (2.6 times the time), not a loop per element (36 times)."""
    x, w1, w2 = (t.to(DEV) for t in _case(1024, 2048, 256, 3))
    bad = x.clone()
    bad[:, 1000] = np.nan

    def best(v):
        times = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(3):
                K.eval_mlp(v, w1, w2)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    clean, nan = best(x), best(bad)
    print(f"mlp 1024 x 2048 x 256: {clean / 3 * 1e3:.0f} us, with NaN rows {nan / 3 * 1e3:.0f} us", flush=True)
    assert nan < 8 * clean
