"""The FP32 solve's energy adds (MN/4) c K a^2 over the spectrum a in FP64, from
FP32 coefficients: it is that sum, formed here in FP64 from the same coefficients,
rounded once.  K comes to 2^-44, and the sum's order is another: a few thousand
FP64 additions of terms that are not negative; 2^-40 of it at most."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

ONE_ROUNDING = 2.0 ** -24 + 2.0 ** -40


def weight(M, N, u, v):
    """c_u c_v K (bins of equal sides)."""
    u, v = np.asarray(u), np.asarray(v)
    w2 = (2 * np.pi / M * u) ** 2 + (2 * np.pi / N * v) ** 2
    k = np.where(w2 > 0, 1 / np.where(w2 > 0, w2, 1), 0)
    return np.where(u > 0, 2, 1) * np.where(v > 0, 2, 1) * k


def check(plan, m, want):
    for phi in (True, False):
        e = float(plan.poisson(m, 1.0, 1.0, phi, True)[3])
        assert abs(e - want) <= ONE_ROUNDING * want, (e, want)


@pytest.mark.parametrize("shape", [(64, 64), (64, 1024), (2048, 32)], ids=str)
@pytest.mark.parametrize("precision", ["fp32", "bf16x3"])
def test_fast(gpu, precision, shape):
    """Rows of +A, -A, -A, +A ...: one coefficient, that of M/2 along the first
    side, whose sums are exact; it is 2 A M sqrt(1/2), rounded once, times 2/M."""
    from dreamplace_amd.spectral import get_plan
    print("case energy terms %s %s" % (precision, shape), flush=True)
    M, N = shape
    plan = get_plan(M, N, precision, gpu)
    sign = np.tile(np.array([1, -1, -1, 1], np.float32), M // 4)
    for A in np.random.default_rng(2).uniform(1, 2, 24).astype(np.float32):
        a = np.float32(2 * M) * A * np.float32(np.sqrt(0.5)) * np.float32(2.0 / M)
        m = torch.from_numpy(np.repeat((A * sign)[:, None], N, 1)).to(gpu)
        check(plan, m, M * N / 4.0 * float(weight(M, N, M // 2, 0)) * float(a) ** 2)


@pytest.mark.parametrize("shape", [(30, 44), (100, 84), (1000, 530)], ids=str)
def test_any_size(gpu, shape):
    """One odd mode along the first side, exactly antisymmetric (the map has no
    mean to take off): the solve's coefficients are the DCT2's, bit for bit."""
    from dreamplace_amd.spectral import get_plan
    print("case energy terms any %s" % (shape,), flush=True)
    M, N = shape
    plan = get_plan(M, N, "fp32", gpu)
    u, v = np.meshgrid(np.arange(M), np.arange(N), indexing="ij")
    c = weight(M, N, u, v)
    rng = np.random.default_rng(3)
    for _ in range(12):
        ku, kv = 2 * int(rng.integers(0, M // 2)) + 1, int(rng.integers(1, N))
        half = np.cos(np.pi * ku * (2 * np.arange(M // 2) + 1) / (2 * M))
        col = np.cos(np.pi * kv * (2 * np.arange(N) + 1) / (2 * N))
        m = (rng.uniform(1, 2) * np.outer(half, col)).astype(np.float32)
        m = torch.from_numpy(np.concatenate([m, -m[::-1]])).to(gpu)
        a = plan.dct2(m).double().cpu().numpy()
        check(plan, m, M * N / 4.0 * float((c * a * a).sum()))
