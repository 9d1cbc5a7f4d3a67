"""Host-side planning of the separable NUDFT (csrc/nufft.hip), called in the
built library without a GPU."""
import ctypes as C

import numpy as np
import pytest

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


class _Axis(C.Structure):   # NuAxis
    _fields_ = ([(f, C.c_int) for f in ("n", "L", "nf", "kind", "flip", "shift")] +
                [(f, C.c_double) for f in ("kc", "xc", "inv_d", "j0")])


class _Geometry(C.Structure):   # NuGeometry
    _fields_ = ([("ok", C.c_bool), ("a_is_y", C.c_bool), ("A", _Axis), ("B", _Axis),
                 ("nz", C.c_int)] + [(f, C.c_double) for f in ("tc", "th", "wc", "wh")])


# Single calls timed on an MI355X in both forms (microseconds).  Axes: points,
# line length, grid cells, kind (0 uniform, 1 rounded, 2 free); half widths of t
# and w multiplied; coils; samples; direct sum, separable form.
TIMED = [
    # sparse samples on large grids, free axes, few coils on long lines
    ("forward", (527, 4096, 2261, 2), (381, 576, 1653, 0), 9.512, 17, 130640, 18654, 110898),
    ("forward", (428, 2048, 1289, 2), (568, 3072, 1705, 2), 2.182, 32, 94369, 18815, 48118),
    ("forward", (514, 2048, 1097, 2), (492, 2048, 1045, 2), 7.223, 12, 40831, 5843, 14033),
    ("adjoint", (559, 1536, 857, 2), (499, 1152, 767, 2), 7.576, 32, 28657, 6693, 14991),
    ("forward", (423, 512, 319, 2), (338, 512, 257, 2), 17.866, 9, 13962, 1375, 3061),
    ("forward", (829, 2048, 1059, 2), (100, 256, 139, 2), 1.572, 4, 11675, 705, 1514),
    ("forward", (468, 768, 1531, 0), (401, 768, 1529, 0), 19.14, 3, 32385, 3467, 7300),
    ("adjoint", (91, 144, 53, 1), (17, 96, 39, 1), 0.0, 2, 580170, 1052, 2153),
    ("adjoint", (542, 1024, 939, 1), (542, 1152, 749, 2), 10.939, 16, 23677, 4057, 8274),
    ("forward", (191, 192, 125, 2), (235, 256, 151, 2), 18.277, 8, 13799, 494, 1245),
    # and calls that the separable form does faster
    ("forward", (60, 96, 107, 0), (204, 384, 379, 0), 0.42, 9, 165741, 1347, 731),
    ("adjoint", (273, 512, 1083, 1), (336, 2048, 1065, 2), 15.642, 1, 42984, 3142, 899),
    ("adjoint", (106, 192, 221, 1), (125, 192, 221, 1), 1.283, 4, 183972, 1639, 718),
    ("adjoint", (441, 768, 745, 0), (549, 1024, 989, 0), 8.643, 3, 68252, 8759, 1421),
    ("forward", (299, 512, 1327, 0), (773, 1536, 3953, 0), 0.0, 12, 19815, 2971, 914),
    ("adjoint", (359, 576, 507, 0), (346, 576, 507, 0), 1.957, 16, 50683, 3858, 1007),
    ("adjoint", (187, 288, 413, 1), (263, 512, 723, 1), 0.901, 12, 133601, 4174, 1207),
    ("forward", (324, 512, 311, 2), (644, 1024, 605, 2), 0.393, 2, 11166, 2001, 879),
    ("adjoint", (646, 1536, 1001, 2), (16, 96, 33, 2), 0.616, 8, 722497, 4901, 2493),
]


def test_the_faster_form_is_chosen():
    """Predicted times against timed calls, of those the ones that prices
    without axis kinds, padding and empty tiles got wrong by the most: the form
    timed as the slower is not taken, and each price is within a factor of two."""
    g = C.POINTER(_Geometry)
    adj = _fn("_ZN3imp16nufft_adjoint_usERKNS_10NuGeometryEii", C.c_double, g, C.c_int, C.c_int)
    fwd = _fn("_ZN3imp16nufft_forward_usERKNS_10NuGeometryEii", C.c_double, g, C.c_int, C.c_int)
    direct = _fn("_ZN3imp9direct_usEiiibi", C.c_double, C.c_int, C.c_int, C.c_int, C.c_bool,
                 C.c_int)
    pays = _fn("_ZN3imp14separable_paysEdd", C.c_bool, C.c_double, C.c_double)
    for op, a, b, theta, nc, m, t_direct, t_sep in TIMED:
        G = _Geometry(ok=True, nz=1, th=theta, wh=1.0)
        for X, v in ((G.A, a), (G.B, b)):
            X.n, X.L, X.nf, X.kind = v
        n = a[0] * b[0]
        if op == "adjoint":
            us, d = adj(C.byref(G), m, nc), direct(m, n, nc, False, 256)
        else:
            us, d = fwd(C.byref(G), m, nc), direct(n, m, nc, True, 256)
        assert 0.5 < us / t_sep < 2 and 0.5 < d / t_direct < 2, (op, a, b, us, d)
        assert pays(us, d) == (t_sep < t_direct), (op, a, b, us, d)


class _Vector(C.Structure):   # std::vector<double>
    _fields_ = [("begin", C.c_void_p), ("end", C.c_void_p), ("cap", C.c_void_p)]

    def array(self):
        n = (self.end - self.begin) // 8
        return np.ctypeslib.as_array((C.c_double * n).from_address(self.begin)).copy()


@pytest.mark.parametrize("theta", [1e-6, 1e-3, 0.1, 1.0, 3.77, 8.0, 12.5, 20.0, 31.0, 40.0])
def test_time_expansion(theta):
    """e^{i theta s u} from the expansion's terms over [-1, 1]^2 to the tolerance
    it is cut at (5e-8 at the corners), its functions orthonormal, and no more
    of them than that tolerance asks for."""
    f = _fn("_ZN3imp14prolate_expandEdRSt6vectorIdSaIdEES3_PiS4_", C.c_bool, C.c_double,
            C.POINTER(_Vector), C.POINTER(_Vector), C.POINTER(C.c_int), C.POINTER(C.c_int))
    a, b, nt, nleg = _Vector(), _Vector(), C.c_int(), C.c_int()
    assert f(theta, C.byref(a), C.byref(b), C.byref(nt), C.byref(nleg))
    nt, nleg = nt.value, nleg.value
    coef, mul = a.array()[:nt * nleg].reshape(nt, nleg), b.array()
    assert len(mul) == nt

    def psi(u):
        out = []
        for l in range(nt):
            k = np.zeros(2 * nleg + 1)
            k[l % 2:l % 2 + 2 * nleg:2] = coef[l]
            out.append(np.polynomial.legendre.legval(u, k))
        return np.array(out)
    s = np.linspace(-1, 1, 101)
    w = mul * 1j ** (np.arange(nt) % 2)
    p = psi(s)
    exact = np.exp(1j * theta * np.outer(s, s))
    assert np.abs((p.T * w) @ p - exact).max() < 5e-8 + 1e-12
    if nt > 1:   # one term less would not do
        assert np.abs((p[:-1].T * w[:-1]) @ p[:-1] - exact).max() > 2e-8
    x, g = np.polynomial.legendre.leggauss(120)
    q = psi(x)
    assert np.abs((q * g) @ q.T - np.eye(nt)).max() < 1e-12


def test_q_takes_the_faster_form():
    """Q_l on the standard grid, calls timed in both forms (N, L, samples;
    microseconds of the GEMM over tables and of the separable sums): few samples
    on a large grid are the GEMM's."""
    us = _fn("_ZN3imp10nufft_q_usERKNS_10NuGeometryEii", C.c_double, C.POINTER(_Geometry), C.c_int,
             C.c_int)
    gemm = _fn("_ZN3imp9q_gemm_usEiiii", C.c_double, C.c_int, C.c_int, C.c_int, C.c_int)
    pays = _fn("_ZN3imp14separable_paysEdd", C.c_bool, C.c_double, C.c_double)
    lengths = {16: 96, 64: 192, 512: 1536, 700: 2304, 1024: 3072, 1300: 4096}
    for N, L, m, t_gemm, t_sep in ((1300, 31, 500, 1663, 12058), (1024, 31, 500, 1213, 7111),
                                   (700, 31, 500, 754, 3885), (1024, 10, 500, 624, 2377),
                                   (700, 31, 10000, 1759, 3980), (512, 31, 10000, 1067, 1683),
                                   (512, 10, 393216, 16300, 1070), (64, 3, 10000, 374, 229),
                                   (16, 10, 500, 270, 158)):
        G = _Geometry(ok=True, nz=1)
        for X in (G.A, G.B):
            X.n, X.L = 2 * N + 1, lengths[N]
            X.nf = 2 * int(np.ceil(0.49 * X.L + 5.5) + 1) + 1
        a, b = us(C.byref(G), m, L + 1), gemm(m, N, N, L + 1)
        assert 0.5 < a / t_sep < 2 and 0.5 < b / t_gemm < 2, (N, L, m, a, b)
        assert pays(a, b) == (t_sep < t_gemm), (N, L, m, a, b)
