"""Every line length of the separable NUDFT (csrc/nufft.hip) in its four line
kernels, and more than one group of columns.  Tolerance as in
test_gpu_nufft.py."""
import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_nufft import TOL, _timer
from test_gpu_nufft_large import _grid

pytestmark = pytest.mark.gpu

LENGTHS = (96, 128, 144, 192, 256, 288, 384, 512, 576, 768, 1024, 1152, 1536, 2048, 2304, 3072,
           4096)


def _pick(want):
    return next(v for v in LENGTHS if v >= want)


def _axis(L, kind, r):
    """Coordinates and largest frequency of an axis whose lines have length L:
    the longest for integer points (read as bins; samples to 0.7 cycles per
    point: grids longer than the lines, folded), for points (i - n/2) / n rounded
    to FP32 (first-order step; frequencies that keep it within its bound), and
    for irregular ones (interpolated; as many points as the length admits)."""
    if kind == "free":
        kmax = L / 4.5 - 6
        n, x = L - 3, np.sort(r.uniform(-.5, .5, L - 3))
        x[0], x[-1] = -.5, .5
        nf = 2 * (np.ceil(1.5 * kmax + 5.5) + 1) + 1
        assert _pick(max(1.5 * nf, n)) == L
        return x, kmax
    n = 2 * (L // 3) + 1
    assert _pick(3 * (n // 2)) == L
    i = np.arange(n) - n // 2
    return (i, 0.7) if kind == "uniform" else (i / n, min(0.6 * n, 250.0))


@pytest.mark.parametrize("long_axis", ["A", "B"])
@pytest.mark.parametrize("kind", ["uniform", "near", "free"])
@pytest.mark.parametrize("L", LENGTHS)
def test_every_line_length(ctx, L, kind, long_axis):
    """A narrow image of one long axis, fastest in the voxel index (A: stored
    and spread from) or slowest (B: combined and formed), 3 coils."""
    from impatient import ops
    from oracle import oracle as orc
    r = np.random.default_rng(LENGTHS.index(L) + 40)
    # enough samples that the separable form is the faster one, also where F
    # lists the points of a long irregular axis
    nc, M = 3, 2500000 if kind == "free" and L >= 1024 else 500000
    a, ka = _axis(L, kind, r)
    n2 = max(4, 12000 // len(a))
    b = np.arange(n2) - n2 // 2
    f = lambda v: np.ascontiguousarray(v, np.float32)
    # x fastest; the long axis is x (A) or y (B)
    if long_axis == "A":
        x, y = _grid(len(a), n2, a, b)
        kx, ky = f(r.uniform(-ka, ka, M)), f(r.uniform(-.5, .5, M))
        kx[:2] = -ka, ka
    else:
        x, y = _grid(n2, len(a), b, a)
        kx, ky = f(r.uniform(-.5, .5, M)), f(r.uniform(-ka, ka, M))
        ky[:2] = -ka, ka
    N = len(x)
    t = f(r.uniform(1e-3, 6e-3, M))
    fm = f(2 * np.pi * r.uniform(-80, 80, N))
    c = lambda *s: r.standard_normal(s, np.float32) + np.complex64(1j) * r.standard_normal(
        s, np.float32)
    d, s, rho = c(nc, M), c(nc, N), c(N)
    got, (n,) = _timer(ctx, lambda: ops.nudft_adjoint(ctx, kx, ky, None, t, x, y, None, fm, d, s),
                       "nufft_adjoint")
    assert n == 1
    idx = np.unique(np.concatenate([[0, N - 1], r.integers(0, N, 24)]))
    ref = orc.nudft_adjoint(kx, ky, None, t, x[idx], y[idx], None, fm[idx], d, s[:, idx])
    ea = rel_l2(got[idx], ref)
    got, (n,) = _timer(ctx, lambda: ops.nudft_forward(ctx, kx, ky, None, t, x, y, None, fm, rho,
                                                      s), "nufft_forward")
    assert n == 1
    idx = np.unique(np.concatenate([[0, 1, M - 1], r.integers(0, M, 24)]))
    ref = orc.nudft_forward(kx[idx], ky[idx], None, t[idx], x, y, None, fm, rho, s)
    ef = rel_l2(np.asarray(got).reshape(nc, M)[:, idx], ref)
    print(f"{len(a)} x {n2}: adjoint {ea:.2e}, forward {ef:.2e}")
    assert ea < TOL and ef < TOL


@pytest.mark.parametrize("N,nc,M,hz,t_read,what", [
    (384, 32, 300000, 890.0, 10e-3, "more than 32 time terms"),
    (1024, 17, 100000, 100.0, 6e-3, "half-transformed grid"),
    (1000, 9, 100000, 400.0, 8e-3, "half-transformed grid, irregular")])
def test_several_column_groups(ctx, N, nc, M, hz, t_read, what):
    """Coils in more than one group: more time terms than the lanes beside 32
    coils hold, or a half-transformed grid beyond its limit."""
    from impatient import ops
    from oracle import oracle as orc
    r = np.random.default_rng(N)
    f = lambda v: np.ascontiguousarray(v, np.float32)
    i = (np.arange(N) - N // 2) / N
    x, y = _grid(N, N, i, i if "irregular" not in what else i + 2e-4 * np.sin(40 * i))
    kx, ky = f(r.uniform(-N / 2, N / 2, M)), f(r.uniform(-N / 2, N / 2, M))
    t = f(r.uniform(1e-3, 1e-3 + t_read, M))
    t[:2] = 1e-3, 1e-3 + t_read
    fm = f(2 * np.pi * hz * np.sin(5 * x) * np.cos(4 * y + 1))
    c = lambda *s: (r.standard_normal(s, np.float32) + 1j * r.standard_normal(s, np.float32))
    d, s = c(nc, M).astype(np.complex64), c(nc, N * N).astype(np.complex64)
    got, (n,) = _timer(ctx, lambda: ops.nudft_adjoint(ctx, kx, ky, None, t, x, y, None, fm, d, s),
                       "nufft_adjoint")
    assert n == 1
    idx = np.unique(np.concatenate([[0, N * N - 1], r.integers(0, N * N, 30)]))
    ref = orc.nudft_adjoint(kx, ky, None, t, x[idx], y[idx], None, fm[idx], d, s[:, idx])
    e = rel_l2(got[idx], ref)
    print(f"{what}: {e:.2e}")
    assert e < TOL
