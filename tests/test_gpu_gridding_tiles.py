"""The tiled gridded F^H d (csrc/grid.hip) at both listing thresholds and on
long lines, against the sum over groups of 2 coils (one thread per grid point,
tolerance as in test_gpu_gridding.py)."""
import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_gridding import TILES_TOL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Ny,Nx,ncoils,os_,S", [
    # up to 40000 samples tiles are listed from 65 on, beyond from 257 on
    (64, 64, 3, 1.5, 2000), (96, 96, 4, 1.5, 5000), (96, 96, 4, 1.5, 5001), (48, 48, 9, 2.0, 6000),
    (64, 64, 32, 1.25, 8000),
    # lines of 768, 1024, 1280, 1792, 2304 and 2816 points
    (512, 32, 4, 1.5, 600), (512, 64, 5, 2.0, 600), (1024, 64, 4, 1.25, 600),
    (1024, 64, 8, 1.75, 600), (2048, 64, 4, 1.125, 600), (2048, 64, 17, 1.375, 600)])
def test_fhd_gridding_tiles_against_points(ctx, Ny, Nx, ncoils, os_, S):
    from impatient import ops, synth
    p = synth.make_problem("tiles", Ny, 1, ncoils, 8, S, 4e-3, 60.0, 2, 3, 12, Nx=Nx)
    # the spiral covers Ny cycles: scaled to the image's shorter axis
    kx = (p.kx * (Nx / Ny)).astype(np.float32)
    rng = np.random.default_rng(63)
    d = (rng.standard_normal((ncoils, p.nk)) + 1j * rng.standard_normal((ncoils, p.nk)))
    d = d.astype(np.complex64)

    def fhd(c0, c1):
        return ops.fhd_gridding(ctx, kx, p.ky, p.kz, p.t, p.Nx, p.Ny, 1, p.fm, d[c0:c1],
                                p.sens[c0:c1], 3, os_)
    got = fhd(0, ncoils)
    ref = sum(fhd(c, min(c + 2, ncoils)).astype(np.complex128) for c in range(0, ncoils, 2))
    e = rel_l2(got, ref)
    print(f"{Nx}x{Ny}, {ncoils} coils, {p.nk} samples, os {os_}: {e:.2e}")
    assert e < TILES_TOL
    assert np.array_equal(got, fhd(0, ncoils))
