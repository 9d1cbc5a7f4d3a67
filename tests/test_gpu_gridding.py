"""The gridding path (-toeplitzGridding): Q_l and F^H d by Kaiser-Bessel
gridding on the GPU against the FP64 restatement of the reference's
gridding (oracle.gridding_q / gridding_fhd), and against the direct
operators (the method's own approximation error, "around 1%",
README:151-154)."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

GRID_TOL = 5e-6   # FP32 gridding + FFT against the FP64 restatement


@pytest.mark.parametrize("N,Nz,os_", [(32, 1, 1.375), (32, 1, 1.25), (24, 1, 2.0), (16, 8, 1.5)])
def test_q_gridding_matches_oracle(ctx, N, Nz, os_):
    """Grids of odd factor 11 (88 = 11 x 8), 5 (80 = 5 x 16), a power of
    two (96) and 3D (48 x 48 x 24)."""
    from impatient import ops, synth
    from oracle import oracle as orc
    p = synth.tiny(N=N, Nz=Nz, ncoils=1, J=8, S=256, ntime_segs=3)
    q = ops.toeplitz_q_gridding(ctx, p.kx, p.ky, p.kz, p.t, N, N, Nz, 3, os_)
    ref = orc.gridding_q(p.kx, p.ky, p.kz, p.t, N, N, Nz, 3, os_)
    img = (2 * N, 2 * N, 2 * Nz if Nz > 1 else 1)
    e = rel_l2(q, ref)
    print(f"Q gridding {N}x{N}x{Nz} os {os_} grid {orc.gridding_params(img, os_)[2]}: "
          f"vs FP64 {e:.2e}")
    assert e < GRID_TOL


@pytest.mark.parametrize("N,Nz,ncoils,os_", [(32, 1, 4, 1.375), (16, 8, 2, 1.5), (16, 1, 34, 1.25)])
def test_fhd_gridding_matches_oracle(ctx, N, Nz, ncoils, os_):
    """Time-segmented F^H d with field map and coils (34 coils: two coil
    groups of the gather), 2D and 3D."""
    from impatient import ops, synth
    from oracle import oracle as orc
    p = synth.tiny(N=N, Nz=Nz, ncoils=ncoils, J=8, S=256, ntime_segs=3)
    rng = np.random.default_rng(61)
    d = (rng.standard_normal((ncoils, p.nk)) + 1j * rng.standard_normal((ncoils, p.nk)))
    got = ops.fhd_gridding(ctx, p.kx, p.ky, p.kz, p.t, N, N, Nz, p.fm, d.astype(np.complex64),
                           p.sens, 3, os_)
    ref = orc.gridding_fhd(p.kx, p.ky, p.kz, p.t, p.fm, d, p.sens, N, N, Nz, 3, os_)
    e = rel_l2(got, ref)
    print(f"F^H d gridding {N}x{N}x{Nz}, {ncoils} coils, os {os_}: vs FP64 {e:.2e}")
    assert e < GRID_TOL


def test_gridding_is_deterministic(ctx):
    """Samples are gathered in a fixed order (no atomics on the grid): two
    calls give identical bits."""
    from impatient import ops, synth
    p = synth.tiny(N=32, ncoils=4, J=8, S=256, ntime_segs=3)
    rng = np.random.default_rng(62)
    d = (rng.standard_normal((4, p.nk)) + 1j * rng.standard_normal((4, p.nk))).astype(np.complex64)
    a = ops.fhd_gridding(ctx, p.kx, p.ky, None, p.t, 32, 32, 1, p.fm, d, p.sens, 3, 1.375)
    b = ops.fhd_gridding(ctx, p.kx, p.ky, None, p.t, 32, 32, 1, p.fm, d, p.sens, 3, 1.375)
    assert np.array_equal(a, b)


def test_gridding_against_direct_at_config3_size(ctx):
    """512^2, 48 x 8192 spiral, L = 10 (the 32-coil workload's trajectory) at
    the reference's demo oversampling (gridOS_Q 1.25, gridOS_FHD 1.375;
    run_all_demos.sh:4), against the direct operators: the method's own
    approximation error, "around 1%" (README:151-154).

    Q_l on the 2N grid is checked over its central half: at gridOS 1.25 the
    Kaiser-Bessel aliasing concentrates in the outer half (3.5% there on a
    64^2 oracle run, 0.3% in the centre), where Q_l only pairs voxels more
    than N/2 apart.  What the solve sees is the Toeplitz apply, checked on
    the phantom with 4 of the coils, and F^H d with the same time
    segmentation."""
    from impatient import ops, synth
    from oracle import oracle as orc
    p = synth.config(3)
    L, N = p.ntime_segs, p.Nx
    qg = np.asarray(ops.toeplitz_q_gridding(ctx, p.kx, p.ky, None, p.t, p.Nx, p.Ny, 1, L, 1.25))
    qd = np.asarray(ops.toeplitz_q(ctx, p.kx, p.ky, None, p.t, p.Nx, p.Ny, 1, L))
    c = (slice(None), slice(N // 2, 3 * N // 2), slice(N // 2, 3 * N // 2))
    eq_all = rel_l2(qg, qd)
    eq_mid = rel_l2(qg.reshape(L + 1, 2 * N, 2 * N)[c], qd.reshape(L + 1, 2 * N, 2 * N)[c])
    tau, t0 = orc.segment_timing(p.t, L)
    sens = p.sens[::8]
    opg = ops.Toeplitz(ctx, p.shape, qg, tau, t0, p.fm, sens, 0.0)
    opd = ops.Toeplitz(ctx, p.shape, qd, tau, t0, p.fm, sens, 0.0)
    rho = p.rho.astype(np.complex64)
    ea = rel_l2(opg.apply(rho), opd.apply(rho))
    opg.close()
    opd.close()
    rng = np.random.default_rng(63)
    d = (rng.standard_normal((4, p.nk)) + 1j * rng.standard_normal((4, p.nk))).astype(np.complex64)
    bg = ops.fhd_gridding(ctx, p.kx, p.ky, None, p.t, p.Nx, p.Ny, 1, p.fm, d, sens, L, 1.375)
    # the direct F^H d with the same time segmentation
    bd = np.zeros(p.nvox, np.complex128)
    for l in range(L + 1):
        a = orc.hanning(p.t, tau, l, t0).astype(np.float32)
        part = ops.nudft_adjoint(ctx, p.kx, p.ky, None, p.t, p.x, p.y, None, None,
                                 d * a[None, :], sens)
        bd += np.exp(1j * p.fm.astype(np.float64) * (tau * l + t0)) * part
    ef = rel_l2(bg, bd)
    print(f"config-3 size: gridded Q (os 1.25) vs direct {eq_all:.2e} (central half "
          f"{eq_mid:.2e}); Toeplitz apply on the phantom {ea:.2e}; gridded F^H d (os 1.375) vs "
          f"direct time-segmented {ef:.2e}")
    assert eq_mid < 0.01 and ea < 0.01 and ef < 0.03


# Both forms sum the same FP32 kernel weights and transform in FP32, in another
# order: sums of up to about 10^3 terms (a few 1e-7) and some ten rounded
# stages (1e-7).
TILES_TOL = 1e-6


@pytest.mark.parametrize("N,Nx,ncoils,os_,S", [
    (32, 32, 8, 1.5, 256), (32, 32, 32, 1.5, 1024), (48, 48, 9, 2.0, 300), (16, 24, 17, 1.0, 128),
    (64, 64, 33, 1.5, 200), (20, 32, 32, 1.5, 256), (128, 128, 16, 1.5, 700),
    (64, 64, 32, 1.375, 400), (128, 64, 20, 1.25, 300), (32, 32, 8, 1.75, 256),
    (64, 64, 12, 1.125, 256), (64, 40, 4, 1.375, 300)])
def test_fhd_gridding_coil_tiles(ctx, N, Nx, ncoils, os_, S):
    """Several coils in 2D (tiles of grid points with coil lanes: 4 to 32 of
    them, full and padded; tiles summed by one wave and by many; grid edges
    inside a tile; every odd factor of the line transforms) against the sum
    over groups of 2 coils, which keep one thread per grid point."""
    from impatient import ops, synth
    p = synth.make_problem("tiles", N, 1, ncoils, 8, S, 4e-3, 60.0, 2, 3, 11, Nx=Nx)
    rng = np.random.default_rng(62)
    d = (rng.standard_normal((ncoils, p.nk)) + 1j * rng.standard_normal((ncoils, p.nk)))
    d = d.astype(np.complex64)

    def fhd(c0, c1):
        return ops.fhd_gridding(ctx, p.kx, p.ky, p.kz, p.t, p.Nx, p.Ny, 1, p.fm, d[c0:c1],
                                p.sens[c0:c1], 3, os_)
    got = fhd(0, ncoils)
    ref = sum(fhd(c, min(c + 2, ncoils)).astype(np.complex128) for c in range(0, ncoils, 2))
    e = rel_l2(got, ref)
    print(f"F^H d gridding tiles {Nx}x{N}, {ncoils} coils, os {os_}: {e:.2e}")
    assert e < TILES_TOL
    assert np.array_equal(got, fhd(0, ncoils))
