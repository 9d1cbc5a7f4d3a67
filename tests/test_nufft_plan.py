"""Host-side planning of the separable NUDFT (csrc/nufft.hip), called in the
built library without a GPU."""
import ctypes as C

from impatient import _lib


def _fn(name, res, *args):
    f = _lib.load()[name]
    f.restype, f.argtypes = res, args
    return f


def test_forward_groups_bound_both_grids():
    """Both grids of a group of coils of F stay within 2 and 3 GB unless one
    coil alone is larger, and a group's elements within k_fline's 32-bit
    offsets: 2730 x 2730 voxels with 75 x 4111 grid cells, 13 time terms and 32
    coils would need 4.7e9 elements side by side."""
    group = _fn("_ZN3imp19nufft_forward_groupEmmi", C.c_int, C.c_size_t, C.c_size_t, C.c_int)
    for nA, nfA, nfB, nt in ((2730, 75, 4111, 13), (4096, 31, 4111, 48), (512, 783, 783, 13),
                             (256, 399, 399, 11), (64, 8205, 8205, 48), (4096, 8205, 8205, 48),
                             (2, 15, 15, 1)):
        for ncoils in (1, 3, 8, 17, 32, 40):
            grid, mid = 16 * nfA * nfB * nt, 16 * nA * nfB * nt
            cg = group(grid, mid, ncoils)
            assert 1 <= cg <= min(32, ncoils)
            if cg > 1:
                assert cg * grid <= 2 << 30 and cg * mid <= 3 << 30
            assert nA * nfB * nt * cg < 2 ** 32 and nfA * nt * cg < 2 ** 32
    assert group(16 * 783 * 783 * 13, 16 * 512 * 783 * 13, 32) == 16
    assert group(16 * 75 * 4111 * 13, 16 * 2730 * 4111 * 13, 32) == 1


def test_sort_passes_cover_every_cell_and_end():
    """8-bit radix passes: enough digits for the last cell's number, no more,
    and at most the four of a 32-bit key (plan_axis admits 8195^2 cells)."""
    passes = _fn("_ZN3imp17nufft_sort_passesEi", C.c_int, C.c_int)
    for n in (1, 2, 255, 256, 257, 65535, 65536, 65537, 2 ** 24 - 1, 2 ** 24, 2 ** 24 + 1,
              4101 ** 2, 8195 ** 2, 2 ** 31 - 1):
        assert passes(n) == max(1, ((n - 1).bit_length() + 7) // 8)
