"""Segments of the Toeplitz apply that go through the passes together: all of
them on small grids, uneven parts on larger ones, one at a time on the largest
(tests of the operator), against the FP64 operator."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

# FP32: four transforms of some 20 rounded stages in all and two map products
# per segment, a few 1e-7; random over the segments and coils summed.
TOL = 2e-6


@pytest.mark.parametrize("N,Nz,ncoils,L", [
    (16, 1, 1, 0), (24, 1, 3, 4), (64, 1, 8, 10), (256, 1, 32, 10), (256, 1, 20, 12),
    (16, 8, 2, 5), (64, 16, 16, 6)])
def test_apply_segments_together(ctx, N, Nz, ncoils, L):
    """256^2 x 32 coils, 11 segments: parts of 4, 4 and 3; x 20, 13: 5, 5 and 3;
    64^2 x 16 x 16 coils, 7: 4 and 3."""
    import fp64_torch as ft
    from impatient import ops, synth
    p = synth.tiny(N=N, Nz=Nz, ncoils=ncoils, J=8, S=128, ntime_segs=max(L, 1))
    r = np.random.default_rng(5)
    M = (2 * N) ** 2 * (2 * Nz if Nz > 1 else 1)
    q = (r.standard_normal((L + 1, M)) + 1j * r.standard_normal((L + 1, M))).astype(np.complex64)
    x = (r.standard_normal(N * N * Nz) + 1j * r.standard_normal(N * N * Nz)).astype(np.complex64)
    tau, t0 = float(np.float32(p.t.max() / max(L, 1))), float(p.t[0])
    op = ops.Toeplitz(ctx, p.shape, q, tau, t0, p.fm, p.sens, 0.0)
    got = op.apply(x)
    again = op.apply(x)
    op.close()
    ref = ft.ToeplitzOperator(q, tau, t0, p.shape, p.fm, p.sens, 0.0)(x.astype(np.complex128))
    e = rel_l2(got, ref.cpu().numpy().reshape(-1))
    print(f"apply {N}x{N}x{Nz}, {ncoils} coils, {L + 1} segments: {e:.2e}")
    assert e < TOL
    assert np.array_equal(got, again)
