"""The separable NUDFT (csrc/nufft.hip) at the ends of what its dispatch
admits: long and unequal axes, grids far beyond the image's band, many time
terms and samples.  Tolerance as in test_gpu_nufft.py."""
import ctypes as C

import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_nufft import TOL, _timer

pytestmark = pytest.mark.gpu


def _grid(Nx, Ny, x, y):
    """Voxel coordinates of the tensor grid, x fastest."""
    f = lambda a: np.ascontiguousarray(a, np.float32).reshape(-1)
    return f(np.broadcast_to(x, (Ny, Nx))), f(np.broadcast_to(np.asarray(y)[:, None], (Ny, Nx)))


def test_forward_half_transformed_grid_larger_than_32_bits(ctx):
    """2730 x 2730 voxels, 32 coils, samples in a strip: 75 x 4111 grid cells
    but 2730 x 4111 half-transformed ones, which for 13 time terms of 32 coils
    exceed 2^32 elements (the coils go in groups)."""
    from impatient import ops
    from oracle import oracle as orc
    N, nc, M = 2730, 32, 20000
    r = np.random.default_rng(31)
    i = np.arange(N) - N // 2
    x, y = _grid(N, N, i / N, i)            # y in voxels: ky in cycles per voxel
    kx, ky = r.uniform(-20, 20, M).astype(np.float32), r.uniform(-.5, .5, M).astype(np.float32)
    t = r.uniform(1e-3, 9e-3, M).astype(np.float32)
    fm = (2 * np.pi * 150 * np.cos(3 * x) * np.sin(2e-3 * y)).astype(np.float32)
    rho = (r.standard_normal(N * N) + 1j * r.standard_normal(N * N)).astype(np.complex64)
    got, (n,) = _timer(ctx, lambda: ops.nudft_forward(ctx, kx, ky, None, t, x, y, None, fm, rho,
                                                      None, nc), "nufft_forward")
    assert n == 1
    idx = np.array([0, 777, 12345, M - 1])
    ref = orc.nudft_forward(kx[idx], ky[idx], None, t[idx], x, y, None, fm, rho, None)
    got = np.asarray(got).reshape(nc, M)
    errs = [rel_l2(g[idx], ref) for g in got]
    print(f"worst coil {max(errs):.2e}")
    assert max(errs) < TOL


def test_q_of_more_weights_than_32_bits(ctx):
    """2^27 samples x 16 column slots: 2^31 weights.  The samples repeat 2^15
    of them, so the sums are the oracle's over those times the repetitions (at
    some points of each segment)."""
    from impatient import Context, ops
    from oracle import oracle as orc
    N, L, M, rep = 512, 16, 1 << 15, 1 << 12
    r = np.random.default_rng(32)
    kx, ky = r.uniform(-N / 2, N / 2, (2, M)).astype(np.float32)
    t = np.sort(r.uniform(1e-3, 9e-3, M)).astype(np.float32)
    big = Context(0)                        # its 90 GB go with it
    try:
        got, (n,) = _timer(big, lambda: ops.toeplitz_q(
            big, np.tile(kx, rep), np.tile(ky, rep), None, np.tile(t, rep), N, N, 1, L), "nufft_q")
    finally:
        big.close()
    assert n == 1
    pts = r.integers(0, 2 * N, (2, 100))
    ref = rep * orc.toeplitz_q(kx, ky, None, t, N, N, 1, L,
                               grid=((pts[0] - N) / N, (pts[1] - N) / N, None))
    errs = [rel_l2(a[pts[1] * 2 * N + pts[0]], b) for a, b in zip(got, ref)]
    print(f"worst segment {max(errs):.2e}")
    assert max(errs) < TOL


def test_q_of_more_than_2_24_cells(ctx):
    """Q of 1032 x 1032: 4101 x 4101 window starts, four digits in the sort."""
    from impatient import ops
    N, L, M = 1032, 2, 20001
    r = np.random.default_rng(33)
    kx, ky = r.uniform(-N / 2, N / 2, (2, M)).astype(np.float32)
    kx[:4], ky[:4] = N / 2 * np.array([-1, 1, -1, 1]), N / 2 * np.array([-1, -1, 1, 1])
    t = np.sort(r.uniform(1e-3, 9e-3, M)).astype(np.float32)
    got, (n,) = _timer(ctx, lambda: ops.toeplitz_q(ctx, kx, ky, None, t, N, N, 1, L), "nufft_q")
    assert n == 1
    from oracle import oracle as orc
    pts = r.integers(0, 2 * N, (2, 200))
    grid = ((pts[0] - N) / N, (pts[1] - N) / N, None)
    ref = orc.toeplitz_q(kx, ky, None, t, N, N, 1, L, grid=grid)
    errs = [rel_l2(a[pts[1] * 2 * N + pts[0]], b) for a, b in zip(got, ref)]
    print(f"worst segment {max(errs):.2e}")
    assert max(errs) < TOL


def _wide(N, nc, M, kmax, seed):
    """An N x N image and samples over +-kmax cycles (corners included)."""
    r = np.random.default_rng(seed)
    kx, ky = r.uniform(-kmax, kmax, (2, M)).astype(np.float32)
    kx[:4], ky[:4] = kmax * np.array([-1, 1, -1, 1]), kmax * np.array([-1, -1, 1, 1])
    t = r.uniform(1e-3, 6e-3, M).astype(np.float32)
    i = (np.arange(N) - N // 2) / N
    x, y = _grid(N, N, i, i)
    fm = (2 * np.pi * 60 * np.cos(4 * x + y)).astype(np.float32)
    c = lambda *s: (r.standard_normal(s) + 1j * r.standard_normal(s)).astype(np.complex64)
    return kx, ky, t, x, y, fm, c(nc, M), c(nc, N * N), c(N * N)


@pytest.mark.parametrize("kmax,M", [(1400.0, 300000), (2650.0, 2000000)])
def test_samples_far_beyond_the_band(ctx, kmax, M):
    """256 x 256 voxels with samples over 11 and 20 times the band: 4200^2 and
    7960^2 grid cells, folded up to 21 times onto the line transforms."""
    from impatient import ops
    from oracle import oracle as orc
    kx, ky, t, x, y, fm, d, s, rho = _wide(256, 2, M, kmax, 34)
    got, (n,) = _timer(ctx, lambda: ops.nudft_adjoint(ctx, kx, ky, None, t, x, y, None, fm, d, s),
                       "nufft_adjoint")
    assert n == 1
    r = np.random.default_rng(2)
    idx = np.unique(np.concatenate([[0, len(x) - 1], r.integers(0, len(x), 30)]))
    ref = orc.nudft_adjoint(kx, ky, None, t, x[idx], y[idx], None, fm[idx], d, s[:, idx])
    ea = rel_l2(got[idx], ref)
    got, (n,) = _timer(ctx, lambda: ops.nudft_forward(ctx, kx, ky, None, t, x, y, None, fm, rho,
                                                      s), "nufft_forward")
    assert n == 1
    idx = np.unique(np.concatenate([[0, 1, 2, 3, M - 1], r.integers(0, M, 30)]))
    ref = orc.nudft_forward(kx[idx], ky[idx], None, t[idx], x, y, None, fm, rho, s)
    ef = rel_l2(np.asarray(got).reshape(2, M)[:, idx], ref)
    print(f"adjoint {ea:.2e}, forward {ef:.2e}")
    assert ea < TOL and ef < TOL


@pytest.mark.parametrize("axes", ["x", "y", "xy"])
def test_volume_whose_first_voxel_is_not_a_number(ctx, axes):
    """The periods of a volume's axes are counted from voxel 0: where that is
    NaN there are none, and the sum stays direct (NaN at that voxel alone)."""
    from impatient import ops
    from oracle import oracle as orc
    from test_gpu_nufft import DIRECT_TOL, _stack
    q = _stack(48, 40, 8, 4, 30000, 16)
    for a in axes:
        q[a] = q[a].copy()
        q[a][0] = np.nan
    got, n = _timer(ctx, lambda: ops.nudft_adjoint(
        ctx, q["kx"], q["ky"], q["kz"], q["t"], q["x"], q["y"], q["z"], q["fm"], q["d"], q["s"]),
        "nufft_stack", "k_nudft_stack")
    assert n[0] == 0 and n[1] > 0
    assert np.isnan(got[0])
    idx = np.unique(np.concatenate([[1, len(q["x"]) - 1],
                                    np.random.default_rng(1).integers(1, len(q["x"]), 20)]))
    ref = orc.nudft_adjoint(q["kx"], q["ky"], q["kz"], q["t"], q["x"][idx], q["y"][idx],
                            q["z"][idx], q["fm"][idx], q["d"], q["s"][:, idx])
    assert rel_l2(got[idx], ref) < DIRECT_TOL


def test_large_workspaces_are_given_back(ctx):
    """F of 512 x 512 voxels with samples over ten times the band and 27 time
    terms needs 34 GB; the context keeps none of it (at most 16 GB stay)."""
    from impatient import Context, _lib, ops
    from oracle import oracle as orc
    lib = _lib.load()

    def free():
        a, b = C.c_size_t(), C.c_size_t()
        assert lib.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value
    N, M = 512, 2000000
    kx, ky, t, x, y, fm, _, _, rho = _wide(N, 1, M, 2650.0, 35)
    fm *= np.float32(1100 / 60)
    own = Context(0)
    try:
        ops.nudft_forward(own, kx[:64], ky[:64], None, t[:64], x, y, None, fm, rho)
        before = free()
        got, (n,) = _timer(own, lambda: ops.nudft_forward(own, kx, ky, None, t, x, y, None, fm,
                                                          rho), "nufft_forward")
        assert n == 1
        own.synchronize()
        kept = before - free()
    finally:
        own.close()
    idx = np.array([0, 1, 2, 3, 99999, M - 1])
    ref = orc.nudft_forward(kx[idx], ky[idx], None, t[idx], x, y, None, fm, rho, None)
    e = rel_l2(np.asarray(got).reshape(-1)[idx], ref)
    print(f"kept {kept / 1e9:.2f} GB, {e:.2e}")
    assert e < TOL
    assert kept < 17 << 30


def test_geometry_scans_behind_queued_work(ctx):
    """Calls queued without a wait between them, the scans of the later ones
    behind milliseconds of direct sums, each on other points and a grid of other
    structure (one not a grid): every result as of the call by itself."""
    from impatient._lib import call, ptr
    from test_gpu_nufft import _problem
    jobs = []
    for i, (Nx, Ny, move) in enumerate([(160, 160, True), (200, 120, False), (160, 160, True),
                                        (97, 251, False)]):
        p = _problem(Nx, Ny, 4, 60000, seed=50 + i)
        if move:
            p["x"][777] += np.float32(1e-4)
        up = lambda v: ctx.to_device(np.ascontiguousarray(v, np.float32).reshape(-1))
        g = [up(p[k]) for k in ("kx", "ky", "t", "x", "y", "fm")]
        v = [up(p["d"].real), up(p["d"].imag), up(p["s"].real), up(p["s"].imag)]
        out = [ctx.alloc((Nx * Ny,)) for _ in range(2)]
        jobs.append((g, v, out, Nx * Ny))

    def run(j):
        g, v, out, n = j
        call("imp_nudft_adjoint", ctx.h, C.c_int(60000), C.c_int(n), C.c_int(4), ptr(g[0]),
             ptr(g[1]), None, ptr(g[2]), ptr(g[3]), ptr(g[4]), None, ptr(g[5]), None, None,
             *(ptr(q) for q in (*v, *out)))

    def results():
        ctx.synchronize()
        return [np.stack([o.get() for o in j[2]]) for j in jobs]
    alone = []
    for j in jobs:
        run(j)
        alone.append(results()[len(alone)])
    for j in jobs:
        for o in j[2]:
            o.zero()
    for j in jobs:
        run(j)
    for a, b in zip(alone, results()):
        assert np.array_equal(a, b)
