"""The separable F^H d and F of large 2D problems and the 2D Q_l
(csrc/nufft.hip) against the FP64 oracle and against the direct kernels.

Tolerance: 2e-7 relative L2.  The separable form sums in FP64 and rounds once
to FP32 (at most 6e-8 per value); its time expansion and its two kernel
separations are each good to 1e-8 of the largest term.
"""
import ctypes as C

import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

TOL = 2e-7
DIRECT_TOL = 2e-6   # the direct kernels' own tolerance (test_gpu_nudft.py)


def _timer(ctx, fn, *names):
    from impatient._lib import call
    call("imp_profile_enable", ctx.h, C.c_int(1))
    call("imp_profile_reset", ctx.h)
    r = fn()
    counts = []
    for name in names:
        tot, n = C.c_double(), C.c_int()
        call("imp_profile_read", ctx.h, name.encode(), C.byref(tot), C.byref(n))
        counts.append(n.value)
    call("imp_profile_enable", ctx.h, C.c_int(0))
    return r, counts


def _problem(Nx, Ny, nc, M, seed=3, kscale=1.0, max_hz=120.0, t_read=8e-3, clump=False):
    rng = np.random.default_rng(seed)
    f = lambda a: np.ascontiguousarray(a, np.float32)
    if clump:   # every sample within half a cycle: a handful of grid cells
        kx, ky = rng.uniform(-0.4, 0.4, (2, M))
    else:       # dense centre, ragged edge
        r = 0.5 * rng.uniform(0, 1, M) ** 1.3 * kscale
        th = rng.uniform(0, 2 * np.pi, M)
        kx, ky = Nx * r * np.cos(th) + 0.3, Ny * r * np.sin(th) - 0.2
    t = rng.uniform(0, t_read, M) + 1e-3
    Y, X = np.meshgrid((np.arange(Ny) - Ny // 2) / Ny, (np.arange(Nx) - Nx // 2) / Nx,
                       indexing="ij")
    fm = 2 * np.pi * max_hz * (np.exp(-((X - .1) ** 2 + Y ** 2) / .05) - 0.3 * X)
    d = rng.standard_normal((nc, M)) + 1j * rng.standard_normal((nc, M))
    s = rng.standard_normal((nc, Nx * Ny)) + 1j * rng.standard_normal((nc, Nx * Ny))
    return dict(kx=f(kx), ky=f(ky), t=f(t), x=f(X).reshape(-1), y=f(Y).reshape(-1),
                fm=f(fm).reshape(-1), d=d.astype(np.complex64), s=s.astype(np.complex64))


def _check(ctx, p, separable=True, sens=True, phi=None, tol=TOL):
    from impatient import ops
    from oracle import oracle as orc
    s = p["s"] if sens else None
    got, (n,) = _timer(ctx, lambda: ops.nudft_adjoint(
        ctx, p["kx"], p["ky"], None, p["t"], p["x"], p["y"], None, p["fm"], p["d"], s, phi),
        "nufft_adjoint")
    assert (n > 0) == separable
    idx = np.unique(np.concatenate([[0, len(p["x"]) - 1],
                                    np.random.default_rng(1).integers(0, len(p["x"]), 60)]))
    ref = orc.nudft_adjoint(p["kx"], p["ky"], None, p["t"], p["x"][idx], p["y"][idx], None,
                            None if p["fm"] is None else p["fm"][idx], p["d"],
                            None if s is None else s[:, idx], phi)
    err = rel_l2(got[idx], ref)
    print(f"rel_l2 {err:.2e}")
    assert err < tol
    return got


# sizes: uniform axes at exact and rounded line lengths, rounded coordinates,
# odd and unequal axes; coil counts on both sides of every wave layout
@pytest.mark.parametrize("Nx,Ny,nc,M", [
    (128, 128, 1, 60001), (160, 128, 2, 50000), (150, 131, 3, 70001), (192, 97, 5, 80000),
    (129, 256, 8, 65537), (144, 144, 9, 90000), (128, 256, 16, 70000), (200, 187, 17, 60013),
    (160, 160, 31, 80000), (128, 200, 32, 70001)])
def test_adjoint_separable(ctx, Nx, Ny, nc, M):
    _check(ctx, _problem(Nx, Ny, nc, M))


@pytest.mark.parametrize("what", ["x_outer", "x_falling", "y_falling", "no_field_map",
                                  "no_sens", "phi", "beyond_nyquist", "wide_time", "clump",
                                  "axis_shuffled"])
def test_adjoint_separable_forms(ctx, what):
    """Voxel orders, axis directions and spacings, optional operands, samples
    beyond the band, many time terms, all samples in a few cells."""
    N, nc, M = 160, 4, 60000
    kw = dict(beyond_nyquist=dict(kscale=1.7), wide_time=dict(max_hz=900.0, t_read=10e-3),
              clump=dict(clump=True)).get(what, {})
    p = _problem(N, N, nc, M, **kw)
    grid = lambda a: a.reshape(N, N)
    if what == "x_outer":
        for k in ("x", "y", "fm"):
            p[k] = np.ascontiguousarray(grid(p[k]).T).reshape(-1)
    if what in ("x_falling", "y_falling"):
        p[what[0]] = -p[what[0]]
    if what == "axis_shuffled":
        o = np.random.default_rng(9).permutation(N)
        p["x"] = np.ascontiguousarray(grid(p["x"])[:, o]).reshape(-1)
    if what == "no_field_map":
        p["fm"] = None
    phi = None
    if what == "phi":
        r = np.random.default_rng(5)
        phi = (1 + 0.3 * r.standard_normal((nc, M)) + 0.2j * r.standard_normal((nc, M))).astype(
            np.complex64)
    if what == "no_sens":
        p["d"] = p["d"][:1]
    _check(ctx, p, sens=what != "no_sens", phi=phi)


@pytest.mark.parametrize("what", ["points", "nan_point", "inf_time", "one_row_moved"])
def test_adjoint_other_points_stay_direct(ctx, what):
    """Points that form no tensor grid, and operands that are not finite, take
    the direct kernels as before."""
    p = _problem(160, 160, 4, 40000)
    if what == "points":
        r = np.random.default_rng(2)
        p["x"] = (p["x"] + r.uniform(-1e-3, 1e-3, len(p["x"]))).astype(np.float32)
    if what == "one_row_moved":
        p["x"] = p["x"].copy()
        p["x"][160 * 71 + 5] += np.float32(1e-4)
    if what in ("points", "one_row_moved"):
        _check(ctx, p, separable=False, tol=DIRECT_TOL)
        return
    from impatient import ops
    if what == "nan_point":
        p["x"] = p["x"].copy()
        p["x"][77] = np.nan
    else:
        p["t"] = p["t"].copy()
        p["t"][77] = np.inf
    got, n = _timer(ctx, lambda: ops.nudft_adjoint(
        ctx, p["kx"], p["ky"], None, p["t"], p["x"], p["y"], None, p["fm"], p["d"], p["s"]),
        "nufft_adjoint", "k_nudft_mfma")
    assert n == [0, 1]
    assert np.isnan(got[77])


def test_adjoint_separable_repeats_bits_and_matches_direct(ctx):
    """Repeated calls give the same bits (no atomics on the grid), and the
    allocation-free entry point (always direct) the same image."""
    from impatient import ops
    from impatient._lib import call, ptr
    p = _problem(128, 128, 8, 40000)
    run = lambda: ops.nudft_adjoint(ctx, p["kx"], p["ky"], None, p["t"], p["x"], p["y"], None,
                                    p["fm"], p["d"], p["s"])
    (a, (n,)) = _timer(ctx, run, "nufft_adjoint")
    assert n > 0
    assert np.array_equal(a, run())
    up = lambda v: ctx.to_device(np.ascontiguousarray(v, np.float32).reshape(-1))
    dev = [up(p[k]) for k in ("kx", "ky", "t", "x", "y", "fm")]
    dr, di, sr, si = (up(v) for v in (p["d"].real, p["d"].imag, p["s"].real, p["s"].imag))
    o = [ctx.alloc((len(p["x"]),)) for _ in range(2)]
    call("imp_nudft_adjoint_noalloc", ctx.h, C.c_int(40000), C.c_int(128 * 128), C.c_int(8),
         ptr(dev[0]), ptr(dev[1]), None, ptr(dev[2]), ptr(dev[3]), ptr(dev[4]), None, ptr(dev[5]),
         None, None, ptr(dr), ptr(di), ptr(sr), ptr(si), ptr(o[0]), ptr(o[1]))
    ctx.synchronize()
    assert rel_l2(a, o[0].get() + 1j * o[1].get()) < DIRECT_TOL


@pytest.mark.parametrize("Nx,Ny,L,M,phi,flags", [
    (8, 8, 0, 40, False, 0), (16, 12, 1, 300, True, 0), (21, 17, 4, 501, False, 1),
    (32, 33, 7, 2000, True, 1), (64, 48, 12, 3001, False, 0), (24, 32, 31, 1000, False, 0)])
def test_q_separable(ctx, Nx, Ny, L, M, phi, flags):
    """Q_l on the 2D standard grid: even and odd segment counts, cumulative
    sums, odd sizes; exactly conjugate-symmetric."""
    from impatient import ops
    from oracle import oracle as orc
    p = _problem(Nx, Ny, 1, M, seed=7)
    r = np.random.default_rng(8)
    ph = (1 + 0.2 * r.standard_normal(M) + 0.2j * r.standard_normal(M)).astype(np.complex64)
    ph = ph if phi else None
    t = np.sort(p["t"])
    got, (n,) = _timer(ctx, lambda: ops.toeplitz_q(ctx, p["kx"], p["ky"], None, t, Nx, Ny, 1, L, ph,
                                                   flags), "nufft_q")
    assert n == 1
    ref = orc.toeplitz_q(p["kx"], p["ky"], None, t, Nx, Ny, 1, L, ph, cumulative=bool(flags & 1))
    errs = [rel_l2(a, b) for a, b in zip(got, ref)]
    print(f"worst segment {max(errs):.2e}")
    assert max(errs) < TOL
    q = got.reshape(L + 1, 2 * Ny, 2 * Nx)[:, 1:, 1:]
    assert np.array_equal(q, np.conj(q[:, ::-1, ::-1]))


def test_q_beyond_transforms_stays_gemm(ctx):
    """Samples far beyond the grid's band and non-finite ones keep the table
    GEMM."""
    from impatient import ops
    p = _problem(16, 16, 1, 200)
    for v in (3e5, np.nan):
        kx = p["kx"].copy()
        kx[5] = v
        _, n = _timer(ctx, lambda: ops.toeplitz_q(ctx, kx, p["ky"], None, np.sort(p["t"]), 16, 16,
                                                  1, 2), "nufft_q", "k_q_sep")
        assert n == [0, 1]


def test_batch_mixes_separable_and_direct_jobs(ctx):
    """Large jobs of a batch take the separable form and equal the single call
    bit for bit; small ones share the direct launch."""
    from impatient import ops
    ps = [_problem(48, 48, 5, 3000, seed=1), _problem(200, 187, 6, 60013, seed=2),
          _problem(64, 40, 3, 2000, seed=3), _problem(192, 192, 8, 70000, seed=4)]
    jobs = [dict(kx=p["kx"], ky=p["ky"], t=p["t"], x=p["x"], y=p["y"], fm=p["fm"], d=p["d"],
                 sens=p["s"]) for p in ps]
    got, n = _timer(ctx, lambda: ops.nudft_adjoint_batch(ctx, jobs), "nufft_adjoint",
                    "k_nudft_mfma_batch")
    assert n == [2, 1]
    for p, g, big in zip(ps, got, (False, True, False, True)):
        one = ops.nudft_adjoint(ctx, p["kx"], p["ky"], None, p["t"], p["x"], p["y"], None, p["fm"],
                                p["d"], p["s"])
        assert np.array_equal(g, one) if big else rel_l2(g, one) < DIRECT_TOL


def _check_forward(ctx, p, nc, sens=True, separable=True, tol=TOL):
    from impatient import ops
    from oracle import oracle as orc
    r = np.random.default_rng(12)
    n = len(p["x"])
    rho = (r.standard_normal(n) + 1j * r.standard_normal(n)).astype(np.complex64)
    s = p["s"] if sens else None
    got, (k,) = _timer(ctx, lambda: ops.nudft_forward(
        ctx, p["kx"], p["ky"], None, p["t"], p["x"], p["y"], None, p["fm"], rho, s, nc),
        "nufft_forward")
    assert (k > 0) == separable
    M = len(p["kx"])
    idx = np.unique(np.concatenate([[0, M - 1], r.integers(0, M, 60)]))
    ref = orc.nudft_forward(p["kx"][idx], p["ky"][idx], None, p["t"][idx], p["x"], p["y"], None,
                            p["fm"], rho, s)
    err = rel_l2(got[:, idx], ref)
    print(f"rel_l2 {err:.2e}")
    assert err < tol
    return got, rho


@pytest.mark.parametrize("Nx,Ny,nc,M", [
    (128, 192, 1, 60001), (160, 128, 2, 70000), (150, 151, 3, 90001), (192, 197, 8, 80000),
    (256, 257, 9, 65537), (256, 256, 16, 70000), (300, 287, 17, 60013), (320, 320, 32, 80000)])
def test_forward_separable(ctx, Nx, Ny, nc, M):
    _check_forward(ctx, _problem(Nx, Ny, nc, M), nc)


@pytest.mark.parametrize("what", ["x_outer", "y_falling", "no_field_map", "no_sens",
                                  "beyond_nyquist", "wide_time", "clump", "axis_shuffled",
                                  "points"])
def test_forward_separable_forms(ctx, what):
    N, nc, M = 200, 4, 60000
    kw = dict(beyond_nyquist=dict(kscale=1.7), wide_time=dict(max_hz=600.0),
              clump=dict(clump=True)).get(what, {})
    p = _problem(N, N, nc, M, **kw)
    if what == "x_outer":
        for k in ("x", "y", "fm"):
            p[k] = np.ascontiguousarray(p[k].reshape(N, N).T).reshape(-1)
    if what == "y_falling":
        p["y"] = -p["y"]
    if what == "axis_shuffled":
        o = np.random.default_rng(9).permutation(N)
        p["x"] = np.ascontiguousarray(p["x"].reshape(N, N)[:, o]).reshape(-1)
    if what == "no_field_map":
        p["fm"] = None
    if what == "points":
        p["x"] = (p["x"] + np.random.default_rng(2).uniform(-1e-3, 1e-3, N * N)).astype(np.float32)
    direct = what == "points"
    _check_forward(ctx, p, 1 if what == "no_sens" else nc, sens=what != "no_sens",
                   separable=not direct, tol=DIRECT_TOL if direct else TOL)


def test_forward_separable_repeats_and_is_the_adjoint(ctx):
    """Same bits on repeat, and <F x, y> = <x, F^H y> with both separable."""
    from impatient import ops
    p = _problem(256, 200, 4, 60000)
    got, rho = _check_forward(ctx, p, 4)
    again = ops.nudft_forward(ctx, p["kx"], p["ky"], None, p["t"], p["x"], p["y"], None, p["fm"],
                              rho, p["s"], 4)
    assert np.array_equal(got, again)
    back = ops.nudft_adjoint(ctx, p["kx"], p["ky"], None, p["t"], p["x"], p["y"], None, p["fm"],
                             p["d"], p["s"])
    a = np.vdot(p["d"].astype(np.complex128), got.astype(np.complex128))
    b = np.vdot(back.astype(np.complex128), rho.astype(np.complex128))
    scale = np.linalg.norm(p["d"]) * np.linalg.norm(got)
    assert abs(a - b) < TOL * scale


def _stack(Nx, Ny, Nz, nc, K, P, seed=4):
    p = _problem(Nx, Ny, nc, K, seed=seed)
    r = np.random.default_rng(seed + 1)
    kz = r.uniform(-Nz / 2, Nz / 2, P).astype(np.float32)
    vox = lambda a: np.repeat(a, Nz)
    z = np.tile(((np.arange(Nz) - Nz // 2) / Nz).astype(np.float32), Nx * Ny)
    q = dict(kx=np.tile(p["kx"], P), ky=np.tile(p["ky"], P), kz=np.repeat(kz, K),
             t=np.tile(p["t"], P), x=vox(p["x"]), y=vox(p["y"]), z=z)
    q["fm"] = (vox(p["fm"]) + 200 * z).astype(np.float32)
    c = lambda *s: (r.standard_normal(s) + 1j * r.standard_normal(s)).astype(np.complex64)
    q["d"], q["s"], q["phi"] = c(nc, P * K), c(nc, len(z)), c(nc, P * K)
    return q


@pytest.mark.parametrize("Nx,Ny,Nz,nc,K,P,what", [
    (64, 48, 8, 4, 30000, 16, "plain"), (33, 41, 12, 3, 40001, 33, "phi"),
    (64, 64, 4, 2, 40000, 34, "no_field_map"), (40, 56, 10, 9, 30000, 20, "y_fast"),
    (48, 48, 16, 1, 30000, 70, "no_sens"), (48, 48, 12, 4, 30000, 16, "z_slow")])
def test_adjoint_stack_separable(ctx, Nx, Ny, Nz, nc, K, P, what):
    """A stack of large partitions: the separable 2D sums of the coil-partition
    columns, combined over z.  Volumes whose z does not run fastest keep the
    z-separable direct sum."""
    from impatient import ops
    from oracle import oracle as orc
    q = _stack(Nx, Ny, Nz, nc, K, P)
    if what in ("y_fast", "z_slow"):   # other voxel orders of [Ny][Nx][Nz]
        o = (1, 0, 2) if what == "y_fast" else (2, 0, 1)
        perm = np.transpose(np.arange(Nx * Ny * Nz).reshape(Ny, Nx, Nz), o).reshape(-1)
        for k in ("x", "y", "z", "fm"):
            q[k] = np.ascontiguousarray(q[k][perm])
    if what == "no_field_map":
        q["fm"] = None
    phi = q["phi"] if what == "phi" else None
    s = None if what == "no_sens" else q["s"]
    got, n = _timer(ctx, lambda: ops.nudft_adjoint(
        ctx, q["kx"], q["ky"], q["kz"], q["t"], q["x"], q["y"], q["z"], q["fm"], q["d"], s, phi),
        "nufft_stack", "k_nudft_stack")
    assert (n[0] > 0, n[1] > 0) == ((False, True) if what == "z_slow" else (True, False))
    idx = np.unique(np.concatenate([[0, len(q["x"]) - 1],
                                    np.random.default_rng(1).integers(0, len(q["x"]), 60)]))
    ref = orc.nudft_adjoint(q["kx"], q["ky"], q["kz"], q["t"], q["x"][idx], q["y"][idx],
                            q["z"][idx], None if q["fm"] is None else q["fm"][idx], q["d"],
                            None if s is None else s[:, idx], phi)
    err = rel_l2(got[idx], ref)
    print(f"rel_l2 {err:.2e}")
    assert err < (DIRECT_TOL if what == "z_slow" else TOL)
