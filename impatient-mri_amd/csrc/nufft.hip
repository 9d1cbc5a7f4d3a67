// F^H d on image grids by wide-kernel spreading and FP64 line transforms.
//
//     out(r) = sum_c conj(S_c(r)) sum_k conj(phi_c(k)) d_c(k) e^{i(2pi k.r + w(r) t_k)}
//
// evaluated to rounding level without visiting every (sample, voxel) pair.
// Three separations, each exact to about 1e-8 of the largest term (the
// hardware sine of the direct kernel is good to 1.2e-7):
//   time    e^{i w t} = sum_l mu_l psi_l(w) psi_l(t), psi_l the prolate
//           spheroidal wave functions of the (w, t) rectangle the operands
//           span (Slepian and Pollak 1961; computed in a Legendre basis as in
//           Xiao, Rokhlin and Yarvin, Inverse Problems 17, 2001): the shortest
//           such sum, nt terms, real factors;
//   space   each sample is spread over NW x NW cells of a regular k grid with
//           the Kaiser-Bessel kernel at 1.5x oversampling, the grid is summed
//           onto the image axes one axis at a time and the kernel's transform
//           divided out (nonuniform FFT of types 1 and 3: Dutt and Rokhlin
//           1993, Greengard and Lee 2004, Lee and Greengard 2005);
//   axes    the image points must form a tensor grid (checked on the device,
//           bit for bit).  Uniform axes read the FFT's bins, nearly uniform
//           ones ((i - N/2)/N rounded to float with N no power of two) take
//           a first-order step from them, others interpolate in the
//           transformed line with the same kernel.
// All sums, grids and transforms are FP64 (half the FP32 rate here), so the
// result carries the rounding of its final FP32 store only.
//
// Layout.  Columns q = (l, c), l time term and c coil, are innermost in every
// grid: grid[gB][gA][q] -> mid[ia][gB][q] -> image.  A is the image axis that
// varies fastest in the voxel index.  Rows gB go through the spread and the
// A transform in blocks, so the spread grid stays small.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <numeric>
#include <utility>
#include <vector>

#include "common.h"
#include "fftcore.h"
#include "nufft.h"

namespace imp {

namespace {

using fftc::cmul;

// Kernel width in cells.  One axis at 1.5x is off by 7e-10 (rms over the band;
// worst 5e-9) at 12 cells, 4e-9 (2.5e-8) at 11, 2.4e-8 (1.4e-7) at 10; the
// results are stored in FP32, 2.5e-8 rms.  11 costs 1/6 less work than 12.
constexpr int NW = 11;
constexpr double NU_SIGMA = 1.5; // oversampling of both grids
// KB shape pi NW (1 - 1/(2 sigma)), 1% lower: the smallest error over the band
// by a scan of the factor
constexpr double NU_BETA = 0.99 * M_PI * NW * (1.0 - 1.0 / (2.0 * NU_SIGMA));
// Largest error of the time expansion, at the corner |t|, |w| = their largest:
// about 27 times the error's rms (the first functions left out reach sqrt(l +
// 1/2) at the ends), so 5e-8 is 2e-9 rms, a twelfth of the FP32 store's
// rounding.  1e-8 took one term more of about 12.
constexpr double NU_TIME_TOL = 5e-8;
constexpr int NU_MAX_TERMS = 48;       // time terms above which the direct kernel runs
                                       // (16 per lane, 3 groups of a 4-group wave)
constexpr double NU_MAX_THETA = 40.0;  // half widths of t and w multiplied: 43 terms
constexpr int NU_MAX_LEG = 160;        // Legendre coefficients per prolate function

// ------------------------------------------------------------------ geometry
// Words of the scan result (device and host).
enum {
    G_MIN = 0,        // kx, ky, t, x, y, w: smallest, as ordered integers
    G_MAX = 6,        // largest
    G_FCX = 12,       // first index where x / y differs from index 0
    G_FCY,
    G_FLAGS,          // 1: a voxel value is not finite, 2: not a tensor grid
    G_DEVA,           // largest distance of an axis from uniform spacing (float bits)
    G_DEVB,
    G_A0, G_A1, G_B0, G_B1,   // first and last coordinate of each axis (float bits)
    G_KFLAG,          // a sample value is not finite
    G_WORDS = 32
};

__host__ __device__ inline unsigned enc_f(unsigned u) {
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
static_assert(G_WORDS < GEO_HOST_WORDS, "the call's number follows the words");
inline float dec_f(unsigned e) {
    const unsigned u = (e & 0x80000000u) ? (e & 0x7fffffffu) : ~e;
    float f;
    std::memcpy(&f, &u, 4);
    return f;
}
inline float bits_f(unsigned u) {
    float f;
    std::memcpy(&f, &u, 4);
    return f;
}

// One block range scans the samples, the other the voxels; block results
// [block][GB_WORDS] are reduced by k_geo_final (atomics on the few shared
// words cost 0.2 ms at 512^2 x 393216).
constexpr int GB_WORDS = 9;   // 3 min, 3 max, first change of a and b, flags

__global__ __launch_bounds__(256) void k_geo_scan(int m, const float *kx, const float *ky,
                                                  const float *t, int n, const float *x,
                                                  const float *y, const float *fm, int kblocks,
                                                  unsigned *part) {
    const bool ks = (int)blockIdx.x < kblocks;
    const float *a = ks ? kx : x, *b = ks ? ky : y, *c = ks ? t : fm;
    const int cnt = ks ? m : n;
    const int nb = ks ? kblocks : (int)gridDim.x - kblocks;
    const int bi = ks ? blockIdx.x : blockIdx.x - kblocks;
    unsigned w[GB_WORDS] = {~0u, ~0u, ~0u, 0u, 0u, 0u, (unsigned)cnt, (unsigned)cnt, 0u};
    const float a0 = cnt ? a[0] : 0.f, b0 = cnt ? b[0] : 0.f;
    for (int i = bi * 256 + threadIdx.x; i < cnt; i += nb * 256) {
        const float v[3] = {a[i], b[i], c ? c[i] : 0.f};
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            if (!isfinite(v[q])) w[8] = 1u;
            const unsigned e = enc_f(__float_as_uint(v[q]));
            w[q] = min(w[q], e);
            w[3 + q] = max(w[3 + q], e);
        }
        if (v[0] != a0) w[6] = min(w[6], (unsigned)i);
        if (v[1] != b0) w[7] = min(w[7], (unsigned)i);
    }
    __shared__ unsigned sm[4][GB_WORDS];
#pragma unroll
    for (int q = 0; q < GB_WORDS; ++q) {
        const bool mx = (q >= 3 && q < 6) || q == 8;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const unsigned o = (unsigned)__shfl_xor((int)w[q], off, 64);
            w[q] = mx ? max(w[q], o) : min(w[q], o);
        }
        if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6][q] = w[q];
    }
    __syncthreads();
    if (threadIdx.x < GB_WORDS) {
        const int q = threadIdx.x;
        const bool mx = (q >= 3 && q < 6) || q == 8;
        unsigned v = sm[0][q];
        for (int u = 1; u < 4; ++u) v = mx ? max(v, sm[u][q]) : min(v, sm[u][q]);
        part[blockIdx.x * GB_WORDS + q] = v;
    }
}

// The result words straight into pinned host memory, then the call's number (one
// block).  A copy and a wait for the stream instead take some 10 us more.
__device__ __forceinline__ void geo_export(const unsigned *geo, unsigned *host, unsigned seq) {
    if (threadIdx.x < G_WORDS)
        __hip_atomic_store(&host[threadIdx.x], geo[threadIdx.x], __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0)
        __hip_atomic_store(&host[G_WORDS], seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
// After k_geo_check, in a launch of its own: counting ended blocks there takes
// a device-wide fence from each of them, which made its 6 us 24.
__global__ void k_geo_export(const unsigned *geo, unsigned *host, unsigned seq) {
    geo_export(geo, host, seq);
}

__global__ __launch_bounds__(256) void k_geo_final(int kblocks, int xblocks, const unsigned *part,
                                                   unsigned *geo, unsigned *host, unsigned seq) {
    // one wave per result word and block range
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int r = wave; r < 2 * GB_WORDS; r += 4) {
        const int q = r % GB_WORDS;
        const bool ks = r < GB_WORDS, mx = (q >= 3 && q < 6) || q == 8;
        unsigned v = mx ? 0u : ~0u;
        const int b0 = ks ? 0 : kblocks, nb = ks ? kblocks : xblocks;
        for (int b = lane; b < nb; b += 64) {
            const unsigned o = part[(b0 + b) * GB_WORDS + q];
            v = mx ? max(v, o) : min(v, o);
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const unsigned o = (unsigned)__shfl_xor((int)v, off, 64);
            v = mx ? max(v, o) : min(v, o);
        }
        if (lane == 0) {
            if (q < 3) geo[G_MIN + (ks ? 0 : 3) + q] = v;
            else if (q < 6) geo[G_MAX + (ks ? 0 : 3) + q - 3] = v;
            else if (q == 8) geo[ks ? G_KFLAG : G_FLAGS] = v;
            else if (!ks) geo[q == 6 ? G_FCX : G_FCY] = v;
        }
    }
    if (threadIdx.x == 0) geo[G_DEVA] = geo[G_DEVB] = 0u;
    if (!host) return;   // the voxels are checked first
    __syncthreads();
    geo_export(geo, host, seq);
}

// Axis structure implied by the first changes.  In 3D (nz_known = 0) z runs
// fastest and its period is where x or y first changes; then the coordinate
// that changes first is axis A, of nA points.  false: none.  (Index 0 differs
// from itself where it is NaN: no periods to divide by.)
__host__ __device__ inline bool geo_axes(unsigned fcx, unsigned fcy, int n, bool d3, bool *a_is_y,
                                         int *nA, int *nz) {
    const unsigned f = fcx < fcy ? fcx : fcy;
    if (f == 0) return false;
    *a_is_y = fcy < fcx;
    *nz = d3 ? (int)f : 1;
    const unsigned slow = *a_is_y ? fcx : fcy;
    *nA = (int)(slow / (unsigned)*nz);
    return (d3 || f == 1) && fcx != fcy && slow % (unsigned)*nz == 0 &&
           (unsigned)n % slow == 0;
}

// Whether the voxels form the grid that their first changes imply, bit for bit,
// and how far its axes are from uniform.
__global__ __launch_bounds__(256) void k_geo_check(int n, const float *x, const float *y,
                                                   const float *z, unsigned *geo) {
    bool a_is_y, bad = false;
    int nA, nz;
    float devA = 0.f, devB = 0.f;
    if (!geo_axes(geo[G_FCX], geo[G_FCY], n, z != nullptr, &a_is_y, &nA, &nz)) {
        bad = true;
    } else {
        const float *a = a_is_y ? y : x, *b = a_is_y ? x : y;
        const unsigned sa = nz, sb = sa * nA, nB = n / sb;
        const float a1 = a[(size_t)(nA - 1) * sa], b1 = b[(size_t)(nB - 1) * sb];
        const double a0 = a[0], da = nA > 1 ? ((double)a1 - a0) / (nA - 1) : 0.0;
        const double b0 = b[0], db = nB > 1 ? ((double)b1 - b0) / (nB - 1) : 0.0;
        for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < (unsigned)n; i += gridDim.x * 256) {
            const unsigned ia = i / sa % nA, ib = i / sb;
            bad = bad || a[i] != a[(size_t)ia * sa] || b[i] != b[(size_t)ib * sb];
            if (z) bad = bad || z[i] != z[i % sa] || !isfinite(z[i]);
            if (i % sa) continue;
            if (i < sb)
                devA = fmaxf(devA, (float)(fabs((double)a[i] - (a0 + ia * da)) * 1.000001));
            if (i % sb == 0)
                devB = fmaxf(devB, (float)(fabs((double)b[i] - (b0 + ib * db)) * 1.000001));
        }
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            geo[G_A0] = __float_as_uint(a[0]);
            geo[G_A1] = __float_as_uint(a1);
            geo[G_B0] = __float_as_uint(b[0]);
            geo[G_B1] = __float_as_uint(b1);
        }
    }
    // one atomic per wave at most
    const bool any = __ballot(bad) != 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        devA = fmaxf(devA, __shfl_xor(devA, off, 64));
        devB = fmaxf(devB, __shfl_xor(devB, off, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        if (any) atomicOr(&geo[G_FLAGS], 2u);
        if (devA > 0.f) atomicMax(&geo[G_DEVA], __float_as_uint(devA));
        if (devB > 0.f) atomicMax(&geo[G_DEVB], __float_as_uint(devB));
    }
}

// ------------------------------------------------------- prolate expansion
// Unit eigenvectors of a symmetric tridiagonal matrix, one at a time from the
// lowest eigenvalue up.  The pivots of T - s from the top, p_i, and from the
// bottom, q_i, hold everything wanted at a shift s: as many p_i are negative as
// eigenvalues lie below s (Sylvester's law of inertia), and where the two
// eliminations are joined at row k the vector x with x_k = 1 that solves all
// rows but k misses that one by g = p_k + q_k - (d_k - s) (Parlett and Dhillon,
// Linear Algebra Appl. 267, 1997).  So the counts bracket one eigenvalue, and x
// at the k of the smallest |g| gives the next shift, its Rayleigh quotient s +
// g / x.x.  Six to nine shifts per vector; the expansions below need about four
// vectors more than they keep (on the host, 36 us for 11 terms, 130 for 28).
class LowestEigenvectors {
  public:
    // off[i] couples rows i and i + 1
    LowestEigenvectors(std::vector<double> diag, std::vector<double> off)
        : d_(std::move(diag)), e_(std::move(off)), n_((int)d_.size()), p_(n_), q_(n_) {
        double lo = d_[0], hi = d_[0];
        for (int i = 0; i < n_; ++i) {
            const double r = (i ? std::fabs(e_[i - 1]) : 0.0) + (i + 1 < n_ ? std::fabs(e_[i]) : 0.0);
            lo = std::min(lo, d_[i] - r);
            hi = std::max(hi, d_[i] + r);
        }
        norm_ = std::max(std::fabs(lo), std::fabs(hi));
        below_ = lo - 1e-12 * norm_;
        step_ = (hi - lo) / (n_ * n_);   // eigenvalues grow like squares
    }
    // x: the next eigenvector.  false: none left, or no convergence.
    bool next(std::vector<double> &x) {
        if (found_ >= n_) return false;
        double lo = below_, hi = lo + step_;
        int count = pivots_down(hi);
        for (int i = 0; count <= found_; ++i, count = pivots_down(hi)) {
            if (i > 200) return false;
            lo = hi;
            step_ *= 2.0;
            hi = lo + step_;
        }
        for (int i = 0; count > found_ + 1; ++i) {
            if (i > 200) return false;
            const double mid = 0.5 * (lo + hi);
            const int c = pivots_down(mid);
            if (c <= found_) lo = mid;
            else { hi = mid; count = c; }
        }
        double s = 0.5 * (lo + hi), last = norm_;
        for (int i = 0; i < 100; ++i) {
            (pivots_down(s) <= found_ ? lo : hi) = s;
            pivots_up(s);
            const double g = joined(s, x), len = std::sqrt(std::inner_product(
                x.begin(), x.end(), x.begin(), 0.0));
            const double miss = std::fabs(g) / len;
            if (miss <= 1e-16 * norm_ || (miss < 1e-10 * norm_ && miss > 0.25 * last)) {
                for (double &v : x) v /= len;
                step_ = std::max(hi - below_, 1e-6 * norm_);
                below_ = hi;
                ++found_;
                return true;
            }
            last = miss;
            s += g / (len * len);
            if (!(s > lo && s < hi)) s = 0.5 * (lo + hi);
        }
        return false;
    }

  private:
    double pivot(double v) const {
        const double tiny = 1e-30 * norm_;
        return std::fabs(v) < tiny ? -tiny : v;
    }
    int pivots_down(double s) {
        int negative = 0;
        for (int i = 0; i < n_; ++i) {
            p_[i] = pivot(d_[i] - s - (i ? e_[i - 1] * e_[i - 1] / p_[i - 1] : 0.0));
            negative += p_[i] < 0.0;
        }
        return negative;
    }
    void pivots_up(double s) {
        for (int i = n_ - 1; i >= 0; --i)
            q_[i] = pivot(d_[i] - s - (i + 1 < n_ ? e_[i] * e_[i] / q_[i + 1] : 0.0));
    }
    // the joined solution and what it misses its row by
    double joined(double s, std::vector<double> &x) const {
        int k = 0;
        auto miss = [&](int i) { return p_[i] + q_[i] - (d_[i] - s); };
        for (int i = 1; i < n_; ++i)
            if (std::fabs(miss(i)) < std::fabs(miss(k))) k = i;
        x.assign(n_, 1.0);
        for (int i = k - 1; i >= 0; --i) x[i] = -e_[i] * x[i + 1] / p_[i];
        for (int i = k + 1; i < n_; ++i) x[i] = -e_[i - 1] * x[i - 1] / q_[i];
        return miss(k);
    }

    std::vector<double> d_, e_;
    int n_, found_ = 0;
    std::vector<double> p_, q_;
    double norm_, below_, step_;   // below_: found_ eigenvalues lie under it
};

}  // namespace

// e^{i theta s u} = sum_l i^(l mod 2) m_l psi_l(s) psi_l(u) on [-1, 1]^2 (m_l
// real, sign included; i for odd l), psi_l = sum_k coef[l][k] P_(2k + l%2);
// the recurrence constants of prolate() follow the coefficients.
// False when more than NU_MAX_TERMS terms are needed.
bool prolate_expand(double theta, std::vector<double> &coef, std::vector<double> &mul, int *nt,
                    int *nleg) {
    if (!(theta >= 0.0) || theta > NU_MAX_THETA) return false;
    if (theta == 0.0) {   // one constant term
        coef.assign({1.0, 0.0, 0.0, 0.0, 0.0});
        mul.assign(1, 1.0);
        *nt = *nleg = 1;
        return true;
    }
    const int K = 2 * (((int)(0.75 * theta) + 36) / 2);   // Legendre degrees, both parities
    const int H = K / 2;
    if (K > NU_MAX_LEG) return false;
    auto matrix = [&](int par) {   // of the Legendre coefficients of one parity
        const double c2 = theta * theta;
        std::vector<double> d(H), e(H - 1);
        for (int i = 0; i < H; ++i) {
            const double k = 2 * i + par;
            d[i] = k * (k + 1) + (2 * k * (k + 1) - 1) / ((2 * k + 3) * (2 * k - 1)) * c2;
            if (i + 1 < H)
                e[i] = (k + 2) * (k + 1) / ((2 * k + 3) * std::sqrt((2 * k + 1) * (2 * k + 5))) * c2;
        }
        return LowestEigenvectors(std::move(d), std::move(e));
    };
    LowestEigenvectors vectors[2] = {matrix(0), matrix(1)};
    const int most = std::min(NU_MAX_TERMS + 1, K - 8);
    std::vector<double> m, at1, c, z;
    for (int l = 0; l < most; ++l) {
        const int par = l & 1;
        if (!vectors[par].next(z)) return false;
        double s1 = 0.0, v0 = 0.0, p = 1.0;
        // P_k(0) for even k and P_k'(0) for odd k, by their recurrences:
        // P_(k+2)(0) = -(k+1)/(k+2) P_k(0); P_(k+2)'(0) = -(k+2)/(k+1) P_k'(0)
        for (int i = 0; i < H; ++i) {
            const double k = 2 * i + par;
            const double a = z[i] * std::sqrt(k + 0.5);
            c.push_back(a);
            s1 += a;
            v0 += a * p;
            p *= par ? -(k + 2) / (k + 1) : -(k + 1) / (k + 2);
        }
        at1.push_back(s1);
        // int e^{i theta s u} psi(s) ds = mu psi(u), at u = 0 (its derivative
        // for odd l); only the Legendre degree 0 (1) of psi integrates
        const double a0 = c[(size_t)l * H];
        m.push_back((par ? theta * (2.0 / 3.0) : 2.0) * a0 / v0);
        // past their largest the terms fall faster than any power: those after
        // one of a thousandth of the tolerance do not matter to the tail
        if (l > theta && std::fabs(m[l]) * s1 * s1 < 1e-3 * NU_TIME_TOL) break;
    }
    const int nmax = (int)m.size();
    // tail beyond the kept terms, at the corner where it is largest
    int keep = nmax;
    double tail = 0.0;
    while (keep > 1) {
        const double next = tail + std::fabs(m[keep - 1]) * at1[keep - 1] * at1[keep - 1];
        if (!(next < NU_TIME_TOL)) break;
        tail = next;
        --keep;
    }
    if (keep >= nmax) return false;
    *nt = keep;
    *nleg = H;
    coef.assign(c.begin(), c.begin() + (size_t)keep * H);
    // (k+1) P_(k+1) = (2k+1) u P_k - k P_(k-1) for the degrees 2i + 2, 2i + 3
    for (int i = 0; i < H; ++i) {
        const double k = 2 * i;
        coef.push_back((2 * k + 3) / (k + 2));
        coef.push_back((k + 1) / (k + 2));
        coef.push_back((2 * k + 5) / (k + 3));
        coef.push_back((k + 2) / (k + 3));
    }
    mul.assign(m.begin(), m.begin() + keep);
    return true;
}

namespace {

// -------------------------------------------------------------- device maths
__device__ __forceinline__ double kb(double z) {
    const double a = 1.0 - z * z * (4.0 / (NW * NW));
    return a >= 0.0 ? cyl_bessel_i0(NU_BETA * sqrt(a)) : 0.0;
}
// kb on one cell of a window as a polynomial: a point NW/2 - 1 + g behind the
// window's last whole cell, g in [0, 1], is NW/2 - 1 + g - c from cell c, and
// kb there is a polynomial in x = 2 g - 1 (degree KB_DEG, fitted on the host
// at Chebyshev nodes).  A tenth of the work of I0.
constexpr int KB_DEG = 9;   // off by 7e-11 of the peak (10: 2e-12, 8: 8e-10)
constexpr int KB_WORDS = NW * (KB_DEG + 1);
__device__ __forceinline__ double kb_cell(const double *poly, int cell, double x) {
    const double *c = poly + cell * (KB_DEG + 1);
    double v = c[KB_DEG];
#pragma unroll
    for (int d = KB_DEG - 1; d >= 0; --d) v = fma(v, x, c[d]);
    return v;
}

const double *kb_poly_table() {
    static const std::vector<double> table = [] {
        std::vector<double> t(KB_WORDS);
        constexpr int n = KB_DEG + 1;
        for (int cell = 0; cell < NW; ++cell) {
            double f[n], cheb[n], mono[n] = {}, tp[n] = {}, tc[n] = {};
            for (int i = 0; i < n; ++i) {
                const double z = 0.5 * NW - 1 + 0.5 * (std::cos(M_PI * (i + 0.5) / n) + 1) - cell;
                f[i] = std::cyl_bessel_i(0.0, NU_BETA * std::sqrt(std::max(0.0, 1 - z * z * 4.0 / (NW * NW))));
            }
            for (int k = 0; k < n; ++k) {
                double v = 0.0;
                for (int i = 0; i < n; ++i) v += f[i] * std::cos(M_PI * k * (i + 0.5) / n);
                cheb[k] = v * (k ? 2.0 : 1.0) / n;
            }
            // sum cheb[k] T_k in powers of x, T_(k+1) = 2 x T_k - T_(k-1)
            tp[0] = 1.0;
            tc[1] = 1.0;
            for (int d = 0; d < n; ++d) mono[d] = cheb[0] * tp[d] + cheb[1] * tc[d];
            for (int k = 2; k < n; ++k) {
                double tn[n] = {};
                for (int d = 0; d < n; ++d) tn[d] = (d ? 2.0 * tc[d - 1] : 0.0) - tp[d];
                for (int d = 0; d < n; ++d) {
                    mono[d] += cheb[k] * tn[d];
                    tp[d] = tc[d];
                    tc[d] = tn[d];
                }
            }
            for (int d = 0; d < n; ++d) t[cell * n + d] = mono[d];
        }
        return t;
    }();
    return table.data();
}

// Fourier transform of kb at u cycles per cell; pi NW |u| < NU_BETA for
// |u| <= 1/(2 sigma)
__device__ __forceinline__ double kb_hat(double u) {
    const double s = sqrt(NU_BETA * NU_BETA - (M_PI * NW * u) * (M_PI * NW * u));
    return NW * sinh(s) / s;
}

// psi_l(u): Legendre sum over one parity.  rec holds, per pair of degrees,
// the constants of P_(k+1) = a u P_k - b P_(k-1) (two steps).
__device__ __forceinline__ double prolate(const double *coef, const double *rec, int nleg, int par,
                                          double u) {
    double p0 = 1.0, p1 = u, s = 0.0;   // P_k, P_(k+1), k = 2 i
    for (int i = 0; i < nleg; ++i) {
        s = fma(coef[i], par ? p1 : p0, s);
        const double p2 = rec[4 * i] * (u * p1) - rec[4 * i + 1] * p0;
        p1 = rec[4 * i + 2] * (u * p2) - rec[4 * i + 3] * p1;
        p0 = p2;
    }
    return s;
}

__device__ __forceinline__ double clamp1(double u) { return fmin(1.0, fmax(-1.0, u)); }

// first cell of a sample's window on one axis, and its position in cells
__device__ __forceinline__ int window(const NuAxis &X, float k, double *s) {
    *s = ((double)k - X.kc) * X.inv_d + X.j0;
    const int b = (int)ceil(*s - 0.5 * NW);
    return min(max(b, 0), X.nf - NW);
}

// ------------------------------------------------------------ sort by cell
__global__ void k_nu_keys(int m, const float *kA, const float *kB, NuAxis A, NuAxis B, int *key,
                          int *val) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= m) return;
    double s;
    const int a = window(A, kA[j], &s), b = window(B, kB[j], &s);
    key[j] = b * (A.nf - NW + 1) + a;
    val[j] = j;
}

// Stable LSD radix sort of (cell, sample), 8-bit digits: each wave owns
// RX_WAVE consecutive elements, so ranks need no order between waves beyond
// their histograms, and equal cells keep the sample order (every run sums in
// the same order).
constexpr int RX_BINS = 256, RX_WAVES = 4, RX_ROUNDS = 8;
constexpr int RX_WAVE = 64 * RX_ROUNDS, RX_BLOCK = RX_WAVES * RX_WAVE;

__global__ __launch_bounds__(256) void k_rx_count(const int *__restrict__ key, int m, int shift,
                                                  int *__restrict__ hist) {
    __shared__ int cnt[RX_BINS];
    cnt[threadIdx.x] = 0;
    __syncthreads();
    for (int r = 0; r < RX_BLOCK / 256; ++r) {
        const int i = blockIdx.x * RX_BLOCK + r * 256 + threadIdx.x;
        if (i < m) atomicAdd(&cnt[(key[i] >> shift) & (RX_BINS - 1)], 1);
    }
    __syncthreads();
    hist[blockIdx.x * RX_BINS + threadIdx.x] = cnt[threadIdx.x];
}

__global__ __launch_bounds__(256) void k_rx_scatter(const int *__restrict__ key,
                                                    const int *__restrict__ val, int m, int shift,
                                                    int nblk, const int *__restrict__ hist,
                                                    int *__restrict__ key_out,
                                                    int *__restrict__ val_out) {
    __shared__ int cnt[RX_WAVES][RX_BINS];
    __shared__ int wsum[RX_WAVES];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // first output position of this block's elements with digit threadIdx.x:
    // all smaller digits, then the same digit in earlier blocks
    int first = 0;
    {
        int total = 0, before = 0;
#pragma unroll 16
        for (int b = 0; b < nblk; ++b) {
            const int c = hist[b * RX_BINS + threadIdx.x];
            total += c;
            before += b < (int)blockIdx.x ? c : 0;
        }
        int inc = total;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int o = __shfl_up(inc, off, 64);
            if (lane >= off) inc += o;
        }
        if (lane == 63) wsum[wave] = inc;
        __syncthreads();
        for (int w = 0; w < wave; ++w) first += wsum[w];
        first += inc - total + before;
    }
    for (int i = threadIdx.x; i < RX_WAVES * RX_BINS; i += 256) cnt[i / RX_BINS][i % RX_BINS] = 0;
    __syncthreads();
    const int base = blockIdx.x * RX_BLOCK + wave * RX_WAVE;
    int k[RX_ROUNDS];
#pragma unroll
    for (int r = 0; r < RX_ROUNDS; ++r) {
        const int i = base + r * 64 + lane;
        k[r] = i < m ? key[i] : 0;
        if (i < m) atomicAdd(&cnt[wave][(k[r] >> shift) & (RX_BINS - 1)], 1);
    }
    __syncthreads();
    {   // per wave and bin: first output position
        int run = first;
#pragma unroll
        for (int w = 0; w < RX_WAVES; ++w) {
            const int c = cnt[w][threadIdx.x];
            cnt[w][threadIdx.x] = run;
            run += c;
        }
    }
    __syncthreads();
    const unsigned long long lt = (1ull << lane) - 1ull;
#pragma unroll
    for (int r = 0; r < RX_ROUNDS; ++r) {
        const int i = base + r * 64 + lane;
        const bool ok = i < m;
        const int d = (k[r] >> shift) & (RX_BINS - 1);
        unsigned long long same = __ballot(ok);   // lanes with this lane's digit
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const unsigned long long set = __ballot((d >> b) & 1);
            same &= ((d >> b) & 1) ? set : ~set;
        }
        int pos = 0;
        if (ok) pos = cnt[wave][d] + __popcll(same & lt);
        __builtin_amdgcn_wave_barrier();
        if (ok) {
            key_out[pos] = k[r];
            val_out[pos] = val[i];
            if ((same >> lane) == 1ull) cnt[wave][d] = pos + 1;   // the last lane of the digit
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// start[c] = first sorted sample whose cell is >= c, c = 0..ncells
// (clears the work-list counters on the way)
__global__ void k_nu_starts(int m, const int *key, int ncells, int *start, int *zero, int nzero) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c < nzero) zero[c] = 0;
    if (c > ncells) return;
    int lo = 0, hi = m;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (key[mid] < c) lo = mid + 1;
        else hi = mid;
    }
    start[c] = lo;
}

// Per sorted sample: window start on A, kernel weights on both axes (zeros on
// either side so a tile may read past the window), time factors.  A workgroup
// fills PREP_S samples, one thread per table entry (coalesced stores).
constexpr int PREP_S = 32;
__global__ __launch_bounds__(256) void k_nu_prep(int m, const int *perm, const float *kA,
                                                 const float *kB, const float *t, NuAxis A,
                                                 NuAxis B, double tc, double tinv,
                                                 const double *coef, const double *poly, int nt,
                                                 int ntp, int nleg, int padA, int padB, int *bx,
                                                 double *wx, double *wy, double *u) {
    __shared__ double px[PREP_S], py[PREP_S], pt[PREP_S], pl[KB_WORDS];
    const int s0 = blockIdx.x * PREP_S, ns = min(PREP_S, m - s0);
    for (int i = threadIdx.x; i < KB_WORDS; i += 256) pl[i] = poly[i];
    if ((int)threadIdx.x < ns) {
        const int i = threadIdx.x, j = perm[s0 + i];
        double p;
        const int a = window(A, kA[j], &p);
        px[i] = 2.0 * (p - a - (0.5 * NW - 1)) - 1.0;
        bx[s0 + i] = a;
        const int b = window(B, kB[j], &p);
        py[i] = 2.0 * (p - b - (0.5 * NW - 1)) - 1.0;
        pt[i] = clamp1(((double)t[j] - tc) * tinv);
    }
    __syncthreads();
    const int nx = NW + 2 * padA, ny = NW + 2 * padB;
    for (int e = threadIdx.x; e < ns * nx; e += 256) {
        const int s = e / nx, g = e - s * nx - padA;
        wx[(size_t)s0 * nx + e] = g >= 0 && g < NW ? kb_cell(pl, g, px[s]) : 0.0;
    }
    for (int e = threadIdx.x; e < ns * ny; e += 256) {
        const int s = e / ny, g = e - s * ny - padB;
        wy[(size_t)s0 * ny + e] = g >= 0 && g < NW ? kb_cell(pl, g, py[s]) : 0.0;
    }
    for (int e = threadIdx.x; e < ns * ntp; e += 256) {
        const int s = e / ntp, l = e - s * ntp;
        u[(size_t)s0 * ntp + e] =
            l < nt ? prolate(coef + (size_t)l * nleg, coef + (size_t)nt * nleg, nleg, l & 1, pt[s])
                   : 0.0;
    }
}

// Sample weights conj(phi) d e^{i(2pi (kA - kcA) xcA + ... + wc (t - tc))},
// [sample][coil slot] FP64 pairs, zero in the slots beyond the group.
constexpr int WD_S = 64;
__global__ __launch_bounds__(256) void k_nu_data(int m, int c0, int nc, int slots,
                                                 const float *kA, const float *kB,
                                                 const float *t, NuAxis A, NuAxis B, double tc,
                                                 double wc_cyc, const float *phi_r,
                                                 const float *phi_i, const float *d_r,
                                                 const float *d_i, double2 *wd) {
    __shared__ double2 rot[WD_S];
    __shared__ double2 tile[8][WD_S + 1];
    const int j0 = blockIdx.x * WD_S, tj = threadIdx.x & (WD_S - 1), tc4 = threadIdx.x / WD_S;
    if (threadIdx.x < WD_S) {
        const int j = min(j0 + (int)threadIdx.x, m - 1);
        const double rev = ((double)kA[j] - A.kc) * A.xc + ((double)kB[j] - B.kc) * B.xc +
                           ((double)t[j] - tc) * wc_cyc;
        double s, c;
        sincospi(2.0 * (rev - rint(rev)), &s, &c);
        rot[threadIdx.x] = make_double2(c, s);
    }
    __syncthreads();
    for (int cb = 0; cb < slots; cb += 8) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int c = cb + tc4 + 4 * h, j = j0 + tj;
            double2 v = make_double2(0.0, 0.0);
            if (c < nc && j < m) {
                const size_t o = (size_t)(c0 + c) * m + j;
                double re = d_r[o], im = d_i[o];
                if (phi_r) {
                    const double pr = phi_r[o], pi = phi_i[o], x = pr * re + pi * im;
                    im = pr * im - pi * re;
                    re = x;
                }
                v = cmul(make_double2(re, im), rot[tj]);
            }
            tile[tc4 + 4 * h][tj] = v;
        }
        __syncthreads();
        const int nw = min(8, slots - cb);
        for (int e = threadIdx.x; e < WD_S * nw; e += 256) {
            const int j = e / nw, c = e % nw;
            if (j0 + j < m) wd[(size_t)(j0 + j) * slots + cb + c] = tile[c][j];
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------- spread
// Tile: `T` cells along A on `yg` rows of one row block.  Work entries split
// a tile's visits (sample, row) into runs of the chunk length the count pass
// settled on; a tile with several runs sums them from slots.  Tiles are split
// above twice the chunk length, since a slot costs its store and a second read.
constexpr int SP_CH0 = 64;         // shortest chunk, visits
constexpr int SP_WAVES = 3072;     // waves in flight: 256 CUs, 4 SIMDs, 3 each
// Chunks per wave in flight.  2, 4, 8: 539, 507, 514 us for the spread and its
// second pass on 250 x 234 x 8 coils, 483, 442, 495 on the Q of 512^2.
constexpr int SP_SHARE = 4;
constexpr int SP_RUN = 64;         // tiles of a super-block
constexpr int SP_LEVELS = 12;      // chunk lengths SP_CH0 << level
constexpr int SP_SLOTS = 8192;     // partial tiles a row block may use

struct SpEntry {
    int tile, v0, v1, slot;
};
struct SpMulti {
    int tile, slot, n, pad;
};
// Per row block counters: runs of split tiles (each with a slot), whole tiles
// of more than half a chunk and shorter ones, split tiles; slot demand per level
struct SpCount {
    int heavy, medium, light, multis;
    int visits, pad[3];     // of the block, in units of SP_CH0
    int need[SP_LEVELS];
};

struct SpGeom {
    int T, yg, rb;          // tile cells, rows, rows per block (multiple of yg)
    int ntx, nty;           // tiles along A, tile rows per block
    int bw;                 // tiles along A of a super-block (SP_RUN tiles in all)
    int ntile;              // tiles per block, whole super-blocks
    int ncA, ncB;           // cells (window starts) per axis
    int nfA, nfB;
    int entry_cap;          // per row block: SP_SLOTS runs, then whole tiles
};

// first grid row of local tile row ty of a block
__device__ __forceinline__ int tile_row(const SpGeom &G, int block, int ty) {
    return block * G.rb + ty * G.yg;
}

__device__ __forceinline__ int row_range(const SpGeom &G, const int *start, int gy0, int gx0,
                                         int row, int *s0) {
    const int by = gy0 - (NW - 1) + row;
    *s0 = 0;
    if (by < 0 || by >= G.ncB || gy0 >= G.nfB) return 0;
    const int lo = max(0, gx0 - (NW - 1)), hi = min(G.ncA - 1, gx0 + G.T - 1);
    if (lo > hi) return 0;
    *s0 = start[by * G.ncA + lo];
    return start[by * G.ncA + hi + 1] - *s0;
}

// Tiles are numbered by super-blocks of SP_RUN (about 16 rows x 64 cells): a
// sample is visited by tiles of neighbouring rows and columns, so tiles with
// near numbers read the same samples.  Raster index of tile t of a block, or
// -1 for the padding of the last super-blocks.
__device__ __forceinline__ int tile_raster(const SpGeom &G, int t) {
    const int nbx = (G.ntx + G.bw - 1) / G.bw, sb = t / SP_RUN, in = t % SP_RUN;
    const int ty = (sb / nbx) * (SP_RUN / G.bw) + in / G.bw, tx = (sb % nbx) * G.bw + in % G.bw;
    return ty < G.nty && tx < G.ntx ? ty * G.ntx + tx : -1;
}

__global__ __launch_bounds__(256) void k_sp_count(SpGeom G, const int *start, int *visits,
                                                  SpCount *cnt) {
    __shared__ int need[SP_LEVELS], sum;
    if (threadIdx.x < SP_LEVELS) need[threadIdx.x] = 0;
    if (threadIdx.x == 0) sum = 0;
    __syncthreads();
    const int t = blockIdx.x * 256 + threadIdx.x, block = blockIdx.y;
    if (t < G.ntile) {
        const int tile = tile_raster(G, t);
        int n = -1;
        if (tile >= 0) {
            const int gy0 = tile_row(G, block, tile / G.ntx), gx0 = (tile % G.ntx) * G.T;
            int s0;
            n = 0;
            for (int r = 0; r < NW + G.yg - 1; ++r) n += row_range(G, start, gy0, gx0, r, &s0);
        }
        visits[(size_t)block * G.ntile + t] = n;
        atomicAdd(&sum, (max(n, 0) + SP_CH0 - 1) / SP_CH0);
        if (n > 2 * SP_CH0) {
#pragma unroll
            for (int k = 0; k < SP_LEVELS; ++k) {
                const int ch = SP_CH0 << k;
                if (n > 2 * ch) atomicAdd(&need[k], (n + ch - 1) / ch);
            }
        }
    }
    __syncthreads();
    if (threadIdx.x < SP_LEVELS && need[threadIdx.x])
        atomicAdd(&cnt[block].need[threadIdx.x], need[threadIdx.x]);
    if (threadIdx.x == 0 && sum) atomicAdd(&cnt[block].visits, sum);
}

// The chunk length is the shortest whose slot demand fits and that leaves at
// most SP_SHARE chunks per wave in flight, so it depends on the operands only; which slot a run gets does not change what is summed.
// Entries keep the tiles' order within a workgroup's 256 tiles.
__global__ __launch_bounds__(256) void k_sp_list(SpGeom G, const int *visits, SpCount *cnt,
                                                 SpEntry *entries, SpMulti *multis) {
    __shared__ int wsum[3][4], base[3];
    const int t = blockIdx.x * 256 + threadIdx.x, block = blockIdx.y;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    SpCount &C = cnt[block];
    int level = 0;
    while (level < SP_LEVELS &&
           (C.need[level] > SP_SLOTS || (C.visits >> level) > SP_SHARE * SP_WAVES))
        ++level;
    const int n = t < G.ntile ? visits[(size_t)block * G.ntile + t] : -1;
    const int ch = level < SP_LEVELS ? SP_CH0 << level : 0x3fffffff;
    const int runs = n > 2 * ch ? (n + ch - 1) / ch : n >= 0 ? 1 : 0;
    // heavy, medium and light entries before this thread
    int inc[3] = {runs > 1 ? runs : 0, runs == 1 && n > ch / 2 ? 1 : 0,
                  runs == 1 && n <= ch / 2 ? 1 : 0};
    const unsigned long long split = __ballot(runs > 1);
#pragma unroll
    for (int h = 0; h < 3; ++h) {
        const int own = inc[h];
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int o = __shfl_up(inc[h], off, 64);
            if (lane >= off) inc[h] += o;
        }
        if (lane == 63) wsum[h][wave] = inc[h];
        inc[h] -= own;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        const int h = threadIdx.x;
        const int sum = wsum[h][0] + wsum[h][1] + wsum[h][2] + wsum[h][3];
        base[h] = atomicAdd(h == 0 ? &C.heavy : h == 1 ? &C.medium : &C.light, sum);
    }
    __syncthreads();
    SpEntry *E = entries + (size_t)block * G.entry_cap;
    const int tile = t < G.ntile ? tile_raster(G, t) : -1;
    const int cls = runs > 1 ? 0 : n > ch / 2 ? 1 : 2;
    int at = base[cls] + inc[cls];
    for (int w = 0; w < wave; ++w) at += wsum[cls][w];
    if (runs == 1) {
        // medium entries from the front of the whole tiles' part, light ones
        // from its end
        E[cls == 1 ? SP_SLOTS + at : G.entry_cap - 1 - at] = SpEntry{tile, 0, n, -1};
    } else if (runs > 1) {
        for (int r = 0; r < runs; ++r)
            E[at + r] = SpEntry{tile, r * ch, min(n, (r + 1) * ch), at + r};
        int m0 = 0;
        if (lane == __ffsll((unsigned long long)split) - 1)
            m0 = atomicAdd(&C.multis, __popcll(split));
        m0 = __shfl(m0, __ffsll((unsigned long long)split) - 1, 64) +
             __popcll(split & ((1ull << lane) - 1ull));
        multis[(size_t)block * SP_SLOTS + m0] = SpMulti{tile, at, runs, 0};
    }
}

typedef const __attribute__((address_space(4))) int *cint;

struct SpArgs {
    SpGeom G;
    int block;                 // row block
    int nt, ntp, nc;           // time terms, padded, coils
    int lc, ll;                // log2 of coil slots and time groups in a wave
    const int *start, *perm, *bx;
    const double *wx, *wy, *u;
    const double2 *wd;         // [sample][coil slot]
    const SpCount *cnt;
    const SpEntry *entries;
    const SpMulti *multis;
    double2 *part;             // [slot][NL * T][64]
    double2 *grid;             // [row in block][nfA][nt][nc]
};

template <int NL, int T>
__device__ __forceinline__ void sp_store(const SpArgs &P, int tile, int lane,
                                         const double2 (&acc)[NL][T]) {
    const int c = lane & ((1 << P.lc) - 1), lg = (lane >> P.lc) & ((1 << P.ll) - 1);
    const int yl = lane >> (P.lc + P.ll);
    const int row = (tile / P.G.ntx) * P.G.yg + yl, gx0 = (tile % P.G.ntx) * T;
    if (c >= P.nc || tile_row(P.G, P.block, tile / P.G.ntx) + yl >= P.G.nfB) return;
    double2 *out = P.grid + ((size_t)row * P.G.nfA + gx0) * P.nt * P.nc + c;
    const size_t sx = (size_t)P.nt * P.nc, sl = P.nc;
#pragma unroll
    for (int i = 0; i < T; ++i) {
#pragma unroll
        for (int k = 0; k < NL; ++k) {
            const int l = lg * NL + k;
            if (gx0 + i < P.G.nfA && l < P.nt) out[i * sx + l * sl] = acc[k][i];
        }
    }
}

// One wave sums one entry.  Lanes are (coil, time group, row); each holds NL
// time terms x T cells as complex FP64 sums in registers.  Visits go in
// batches of 64: lane v finds visit v's row and sample, the wave copies the
// visits' kernel weights and time factors to LDS, then runs over them with the
// next SP_PF sample weights on their way; a visit costs 2 NL (T + 1) FP64
// instructions against (T + NL) / 2 broadcast 16-byte LDS reads.
//
// The bound is the FP64 rate together with the latency of a visit's operands.
// Scalar loads for the factors instead (re and im in different lanes) took
// 528 us per launch on 512^2 x 32 coils; of its variants 588 us had the FP64
// work taken out and 387 us the loads (640 us with both).  With the factors in
// LDS: 577 us with one weight on its way, 526 with two, 500 with four; and
// 468 at a window of 11 cells instead of 12.  250 x 234 x 8 coils: 573 -> 377
// us; six slices of 128^2..384^2 x 8 coils: 3.26 -> 2.41 ms.  Larger tiles at
// two waves per SIMD: 628 us (512^2) and 486 (250 x 234).
constexpr int SP_BATCH = 64, SP_PF = 4;
template <int NL, int T, bool ROWS>
__global__ __launch_bounds__(64, NL * T > 24 ? 2 : 3) void k_spread(SpArgs P) {
    __shared__ double sx[SP_BATCH * T];
    extern __shared__ double dyn[];      // [SP_BATCH][ntp], then [SP_BATCH][yg] (ROWS)
    double *su = dyn, *sy = dyn + SP_BATCH * P.ntp;
    const int lane = threadIdx.x;
    // workgroups go round the 8 XCDs; each takes SP_RUN entries in a row, whose
    // samples then stay in that XCD's L2 (gridDim.x is a multiple of 8 SP_RUN)
    const int wave = (blockIdx.x / (8 * SP_RUN)) * 8 * SP_RUN + (blockIdx.x & 7) * SP_RUN +
                     ((blockIdx.x >> 3) & (SP_RUN - 1));
    const int nwaves = gridDim.x;
    const int c = lane & ((1 << P.lc) - 1), lg = (lane >> P.lc) & ((1 << P.ll) - 1);
    const int yl = ROWS ? lane >> (P.lc + P.ll) : 0;
    const int yg = ROWS ? P.G.yg : 1;
    const int nx = NW + 2 * (T - 1), ny = NW + 2 * (yg - 1);
    const int rows = NW + yg - 1;
    // long entries first, so that the launch ends on short ones: runs of split
    // tiles, then whole tiles by size class
    const cint pc = (cint)(const int *)&P.cnt[P.block];
    const int nh = pc[0], nm = nh + pc[1], ne = nm + pc[2];
    for (int e = wave; e < ne; e += nwaves) {
        const cint ep = (cint)(const int *)(P.entries + (size_t)P.block * P.G.entry_cap +
                                            (e < nh   ? e
                                             : e < nm ? SP_SLOTS + e - nh
                                                      : P.G.entry_cap - 1 - (e - nm)));
        const int tile = ep[0], v0 = ep[1], v1 = ep[2], slot = ep[3];
        const int gy0 = tile_row(P.G, P.block, tile / P.G.ntx), gx0 = (tile % P.G.ntx) * T;
        double2 acc[NL][T];
#pragma unroll
        for (int k = 0; k < NL; ++k)
#pragma unroll
            for (int i = 0; i < T; ++i) acc[k][i] = make_double2(0.0, 0.0);
        // lane r holds the sample range of row r (rows <= 64 - 1 + NW fits: at
        // most 64 rows per tile are split over the lanes twice)
        int rs = 0, rn = 0, rs2 = 0, rn2 = 0;
        if (lane < rows) rn = row_range(P.G, P.start, gy0, gx0, lane, &rs);
        if (ROWS && lane + 64 < rows) rn2 = row_range(P.G, P.start, gy0, gx0, lane + 64, &rs2);
        for (int vb = v0; vb < v1; vb += SP_BATCH) {
            const int nb = min(SP_BATCH, v1 - vb);
            // visit vb + lane: its row and sample
            int row = 0, smp = 0, base = 0;
            for (int r = 0; r < rows; ++r) {
                const int n = r < 64 ? __builtin_amdgcn_readlane(rn, r)
                                     : __builtin_amdgcn_readlane(rn2, r - 64);
                const int s = r < 64 ? __builtin_amdgcn_readlane(rs, r)
                                     : __builtin_amdgcn_readlane(rs2, r - 64);
                const int o = vb + lane - base;
                if (o >= 0 && o < n) {
                    row = r;
                    smp = s + o;
                }
                base += n;
            }
            int va = 0, vj = 0;
            if (lane < nb) {
                va = P.bx[smp];
                vj = P.perm[smp];
            }
            // offset of the tile's first cell in the sample's padded window;
            // row by = gy0 - (NW - 1) + r: tile row y takes weight gy0 + y - by
            const int ox = gx0 - va + T - 1, oy = NW - 1 - row + yg - 1;
            __syncthreads();
            // every lane takes part in the exchanges, also past the last
            // factor; the visits that pad the batch get factors of zero
            const int np = (nb + SP_PF - 1) / SP_PF * SP_PF;
            for (int i0 = 0; i0 < np * T; i0 += 64) {
                const int i = i0 + lane, v = min(i / T, SP_BATCH - 1), q = i % T;
                const size_t k = __shfl(smp, v, 64);
                const int x = __shfl(ox, v, 64), y = ROWS ? 0 : __shfl(oy, v, 64);
                if (i < np * T) {
                    double f = 0.0;
                    if (v < nb) {
                        f = P.wx[k * nx + x + q];
                        if (!ROWS) f *= P.wy[k * ny + y];
                    }
                    sx[i] = f;
                }
            }
            for (int i0 = 0; i0 < np * P.ntp; i0 += 64) {
                const int i = i0 + lane, v = min(i / P.ntp, SP_BATCH - 1);
                const size_t k = __shfl(smp, v, 64);
                if (i < np * P.ntp) su[i] = v < nb ? P.u[k * P.ntp + (i - v * P.ntp)] : 0.0;
            }
            if (ROWS)
                for (int i0 = 0; i0 < np * yg; i0 += 64) {
                    const int i = i0 + lane, v = min(i / yg, SP_BATCH - 1);
                    const size_t k = __shfl(smp, v, 64);
                    const int y = __shfl(oy, v, 64);
                    if (i < np * yg) sy[i] = v < nb ? P.wy[k * ny + y + (i - v * yg)] : 0.0;
                }
            __syncthreads();
            // SP_PF sample weights are on their way; visits past nb take zero
            auto weight = [&](int i) {
                return P.wd[((size_t)__builtin_amdgcn_readlane(vj, min(i, nb - 1)) << P.lc) + c];
            };
            double2 w[SP_PF];
#pragma unroll
            for (int h = 0; h < SP_PF; ++h) w[h] = weight(h);
            for (int i0 = 0; i0 < nb; i0 += SP_PF) {
#pragma unroll
                for (int h = 0; h < SP_PF; ++h) {
                    const int i = i0 + h;
                    double2 v = w[h];
                    if (i >= nb) v = make_double2(0.0, 0.0);
                    w[h] = weight(i + SP_PF);
                    if (ROWS) {
                        const double y = sy[i * yg + yl];
                        v.x *= y;
                        v.y *= y;
                    }
                    double wx[T];
#pragma unroll
                    for (int q = 0; q < T; ++q) wx[q] = sx[i * T + q];
                    const double *pu = su + i * P.ntp + lg * NL;
#pragma unroll
                    for (int k = 0; k < NL; ++k) {
                        const double u = pu[k], re = v.x * u, im = v.y * u;
#pragma unroll
                        for (int q = 0; q < T; ++q) {
                            acc[k][q].x = fma(re, wx[q], acc[k][q].x);
                            acc[k][q].y = fma(im, wx[q], acc[k][q].y);
                        }
                    }
                }
            }
        }
        if (slot < 0) {
            sp_store<NL, T>(P, tile, lane, acc);
        } else {
            double2 *o = P.part + (size_t)slot * NL * T * 64 + lane;
#pragma unroll
            for (int k = 0; k < NL; ++k)
#pragma unroll
                for (int i = 0; i < T; ++i) o[(k * T + i) * 64] = acc[k][i];
        }
    }
}

// tiles summed in several runs: one wave per (tile, time term) adds the runs
// in order
template <int NL, int T>
__global__ __launch_bounds__(256) void k_spread_multi(SpArgs P) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    const int c = lane & ((1 << P.lc) - 1), lg = (lane >> P.lc) & ((1 << P.ll) - 1);
    const int yl = lane >> (P.lc + P.ll);
    const int n = P.cnt[P.block].multis * NL;
    for (int e = wave; e < n; e += gridDim.x * 4) {
        const SpMulti M = P.multis[(size_t)P.block * SP_SLOTS + e / NL];
        const int k = e % NL;
        double2 acc[T];
#pragma unroll
        for (int i = 0; i < T; ++i) acc[i] = make_double2(0.0, 0.0);
        const double2 *o = P.part + ((size_t)M.slot * NL + k) * T * 64 + lane;
#pragma unroll 2
        for (int r = 0; r < M.n; ++r, o += NL * T * 64)
#pragma unroll
            for (int i = 0; i < T; ++i) {
                const double2 v = o[i * 64];
                acc[i].x += v.x;
                acc[i].y += v.y;
            }
        const int row = (M.tile / P.G.ntx) * P.G.yg + yl, gx0 = (M.tile % P.G.ntx) * T;
        const int l = lg * NL + k;
        if (c >= P.nc || tile_row(P.G, P.block, M.tile / P.G.ntx) + yl >= P.G.nfB || l >= P.nt)
            continue;
        double2 *g = P.grid + (((size_t)row * P.G.nfA + gx0) * P.nt + l) * P.nc + c;
#pragma unroll
        for (int i = 0; i < T; ++i)
            if (gx0 + i < P.G.nfA) g[(size_t)i * P.nt * P.nc] = acc[i];
    }
}

// cells per tile for nl time terms per lane: about 24 complex accumulators,
// which leave three waves per SIMD up to 12 time terms
constexpr int sp_cells(int nl) {
    return nl >= 9 ? 2 : nl >= 7 ? 3 : nl >= 5 ? 4 : nl == 4 ? 6 : nl == 3 ? 8 : nl == 2 ? 8 : 8;
}

using SpFn = void (*)(SpArgs);
template <int NL>
SpFn sp_pick1(bool rows) {
    return rows ? (SpFn)k_spread<NL, sp_cells(NL), true> : (SpFn)k_spread<NL, sp_cells(NL), false>;
}
template <int NL>
SpFn sp_multi1() { return (SpFn)k_spread_multi<NL, sp_cells(NL)>; }

template <class F>
auto sp_switch(int nl, F f) {
    switch (nl) {
        case 1: return f(std::integral_constant<int, 1>{});
        case 2: return f(std::integral_constant<int, 2>{});
        case 3: return f(std::integral_constant<int, 3>{});
        case 4: return f(std::integral_constant<int, 4>{});
        case 5: return f(std::integral_constant<int, 5>{});
        case 6: return f(std::integral_constant<int, 6>{});
        case 7: return f(std::integral_constant<int, 7>{});
        case 8: return f(std::integral_constant<int, 8>{});
        case 9: return f(std::integral_constant<int, 9>{});
        case 10: return f(std::integral_constant<int, 10>{});
        case 11: return f(std::integral_constant<int, 11>{});
        case 12: return f(std::integral_constant<int, 12>{});
        case 13: return f(std::integral_constant<int, 13>{});
        case 14: return f(std::integral_constant<int, 14>{});
        case 15: return f(std::integral_constant<int, 15>{});
        default: return f(std::integral_constant<int, 16>{});
    }
}
constexpr int SP_MAX_NL = 16;

// ---------------------------------------------------------- line transforms
// FP64 Stockham lines: E values per thread, lines interleaved in LDS
// [position][line] (columns q are contiguous in memory, so a wave's loads of
// one element cover LINES x 16 bytes), re and im exchanged in turn to halve
// the LDS.
namespace ln {
__host__ __device__ constexpr bool has3(int L) { return L % 3 == 0; }
__host__ __device__ constexpr int vals(int L) { return has3(L) ? 12 : 8; }
__host__ __device__ constexpr int threads(int L) { return L / vals(L); }
// lines of a workgroup of up to wg threads
__host__ __device__ constexpr int lines(int L, int wg) {
    int n = 64;
    while (n > 1 && n * threads(L) > wg) n /= 2;
    return n;
}
__host__ __device__ constexpr int bits(int n) { return n <= 1 ? 0 : 1 + bits(n / 2); }
// lengths 12 2^k and 144 2^k: radix-12 stages, then 4 and 2
__host__ __device__ constexpr int twelves(int L) { return L % 9 ? 1 : 2; }
__host__ __device__ constexpr int rest(int L) { return L / (L % 9 ? 12 : 144); }
__host__ __device__ constexpr int stages(int L) {
    return has3(L) ? twelves(L) + (bits(rest(L)) + 1) / 2 : (bits(L) + 2) / 3;
}
__host__ __device__ constexpr int radix(int L, int s) {
    return has3(L) ? (s < twelves(L) ? 12 : (bits(rest(L)) - 2 * (s - twelves(L)) >= 2 ? 4 : 2))
                   : (bits(L) - 3 * s >= 3 ? 8 : 1 << (bits(L) - 3 * s));
}
__host__ __device__ constexpr int span(int L, int s) {
    return s == 0 ? 1 : span(L, s - 1) * radix(L, s - 1);
}
__host__ __device__ constexpr int pad(int L, int i) { return i + i / vals(L); }
__host__ __device__ constexpr int words(int L, int P) { return (L + L / vals(L)) * P; }

// element index of register (b, r) before / after stage S
template <int L, int S>
__device__ __forceinline__ int in_idx(int t, int b, int r) {
    return t + threads(L) * b + r * (L / radix(L, S));
}
template <int L, int S>
__device__ __forceinline__ int out_idx(int t, int b, int r) {
    constexpr int R = radix(L, S), NS = span(L, S);
    const int j = t + threads(L) * b, k = NS > 1 ? j % NS : 0;
    return (j - k) * R + k + r * NS;
}

template <int L, int S>
__device__ __forceinline__ void butterflies(double2 (&v)[vals(L)], int t, const double2 *tw) {
    constexpr int R = radix(L, S), NS = span(L, S), NB = vals(L) / R;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if constexpr (NS > 1) {
            // one twiddle is loaded, the others are its powers (the combining
            // pass of 512^2 x 32 coils took 1.63 ms with table reads, 0.95
            // with none)
            const int k = (t + threads(L) * b) % NS, step = (L / (NS * R)) * k;
            double2 w[R];
            w[1] = tw[step];
#pragma unroll
            for (int r = 2; r < R; ++r) w[r] = cmul(w[r / 2], w[r - r / 2]);
#pragma unroll
            for (int r = 1; r < R; ++r) v[b * R + r] = cmul(v[b * R + r], w[r]);
        }
        fftc::dft<R, true>(&v[b * R]);
    }
}

template <int L, int S, int P>
__device__ __forceinline__ void exchange(double2 (&v)[vals(L)], int t, int c, double *buf) {
    constexpr int R = radix(L, S), NB = vals(L) / R;
    constexpr int R2 = radix(L, S + 1), NB2 = vals(L) / R2;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        __syncthreads();
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int r = 0; r < R; ++r)
                buf[pad(L, out_idx<L, S>(t, b, r)) * P + c] = h ? v[b * R + r].y : v[b * R + r].x;
        __syncthreads();
        double x[vals(L)];
#pragma unroll
        for (int b = 0; b < NB2; ++b)
#pragma unroll
            for (int r = 0; r < R2; ++r) x[b * R2 + r] = buf[pad(L, in_idx<L, S + 1>(t, b, r)) * P + c];
#pragma unroll
        for (int i = 0; i < vals(L); ++i) {
            if (h) v[i].y = x[i];
            else v[i].x = x[i];
        }
    }
}

// inverse DFT (e^{+i}) of a line held as in_idx<L, 0>; tw[m] = e^{+2 pi i m / L}
template <int L, int P, int S = 0>
__device__ __forceinline__ void transform(double2 (&v)[vals(L)], int t, int c, double *buf,
                                          const double2 *tw) {
    butterflies<L, S>(v, t, tw);
    if constexpr (S + 1 < stages(L)) {
        exchange<L, S, P>(v, t, c, buf);
        transform<L, P, S + 1>(v, t, c, buf, tw);
    }
}
}  // namespace ln

// One axis' tables: twiddles [L]; input scale [nf] (AX_FREE); output weights
// [n], followed by the points' offsets [n] from their bins in radians per cell
// (AX_NEAR), or [n][NW] with window starts base[n] (AX_FREE).
struct AxisTab {
    NuAxis X;
    const float *coord;
    int stride;
    double2 *tw;
    double *inw, *outw;
    int *base;
};

__global__ void k_nu_axis(AxisTab ta, AxisTab tb) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const AxisTab &P = blockIdx.y ? tb : ta;
    const NuAxis &X = P.X;
    if (i < X.L) {
        double s, c;
        sincospi(2.0 * i / X.L, &s, &c);
        P.tw[i] = make_double2(c, s);
    }
    if (X.kind == AX_FREE && i < X.nf) P.inw[i] = 1.0 / kb_hat((i - X.j0) / X.L);
    if (i >= X.n) return;
    // cycles per cell
    const double u0 = (double)(i - X.n / 2) / X.L;
    const double u = X.kind == AX_UNIFORM
                         ? u0 : ((double)P.coord[(size_t)i * P.stride] - X.xc) / X.inv_d;
    if (X.kind != AX_FREE) {
        P.outw[i] = 1.0 / kb_hat(u);
        if (X.kind == AX_NEAR) P.outw[X.n + i] = 2.0 * M_PI * (u - (X.flip ? -u0 : u0));
    } else {
        // the position in the transformed line
        const double p = u * X.L, h = kb_hat(u);
        const int b = (int)ceil(p - 0.5 * NW);
        P.base[i] = b;
        for (int k = 0; k < NW; ++k) P.outw[(size_t)i * NW + k] = kb(p - (b + k)) / h;
    }
}

// threads per workgroup: several share a CU, also in the combining pass, whose
// accumulators leave 2 to 3 waves per SIMD
constexpr int ST_WG = 256;

struct LineArgs {
    const double2 *in;          // element j of line x, column q: in[x in_line + j in_el + q]
    size_t in_line;
    unsigned in_el;
    int nq, nlines;             // columns, lines
    NuAxis X;
    const double2 *tw;
    const double *inw, *outw;
    const int *base;
};

// Loads the elements in_idx<L, 0> (mod L) of a line: grid points j = i + j0 mod
// L, folded unless the axis is AX_FREE (there the grid is L-periodic exactly),
// scaled on AX_FREE axes, times j - j0 for the first-order pass of AX_NEAR.
// base is wave-uniform and the lane offsets are 32 bits wide (a line's
// elements span far less than 4 GB): one address register per element.
// Every lane loads, from a clamped place, and selects afterwards: loads under
// a lane's condition are waited for one by one (384-point lines 93 -> 71 us).
template <int L, int KIND>
__device__ __forceinline__ void line_load(const LineArgs &P, const double2 *base, int t,
                                          unsigned q, bool ok, int order,
                                          double2 (&v)[ln::vals(L)]) {
    constexpr int E = ln::vals(L), R0 = ln::radix(L, 0);
    const unsigned cl = ok ? q : 0;
    const int last = P.X.nf - 1, j0 = (int)P.X.j0;
    auto at = [&](int i) {
        const int j = ln::in_idx<L, 0>(t, i / R0, i % R0) + P.X.shift;
        return j >= L ? j - L : j;
    };
#pragma unroll
    for (int i = 0; i < E; ++i) {
        const int j = at(i);
        const double2 x = base[(unsigned)min(j, last) * P.in_el + cl];
        v[i] = ok && j <= last ? x : make_double2(0.0, 0.0);
        if constexpr (KIND == AX_FREE) {
            const double w = P.inw[min(j, last)];
            v[i] = make_double2(v[i].x * w, v[i].y * w);
        }
        if (KIND == AX_NEAR && order) {
            const double w = j - j0;
            v[i] = make_double2(v[i].x * w, v[i].y * w);
        }
    }
    if constexpr (KIND != AX_FREE)
        for (int o = L; o <= last; o += L) {
#pragma unroll
            for (int i = 0; i < E; ++i) {
                const int j = at(i) + o;
                if (ok && j <= last) {
                    const double2 x = base[(unsigned)j * P.in_el + cl];
                    const double w = KIND == AX_NEAR && order ? j - j0 : 1;
                    v[i].x = fma(x.x, w, v[i].x);
                    v[i].y = fma(x.y, w, v[i].y);
                }
            }
        }
}

__device__ __forceinline__ double2 times_i(double2 v, double f) {
    return make_double2(-f * v.y, f * v.x);
}

// bin of an L-point transform -> image index, not on AX_FREE axes (or >= n)
__device__ __forceinline__ unsigned bin_index(const NuAxis &X, int L, int i) {
    const int f = i < L / 2 ? i : i - L;
    return (unsigned)((X.flip ? -f : f) + X.n / 2);
}

// Interpolated values of the thread's outputs o = t + T m (AX_FREE axes).
template <int L, int W>
__device__ __forceinline__ void line_interp(const LineArgs &P, double2 (&v)[ln::vals(L)], int t,
                                            int c, double *buf, double2 (&o)[ln::vals(L)]) {
    constexpr int E = ln::vals(L), T = ln::threads(L), S = ln::stages(L) - 1;
    constexpr int R = ln::radix(L, S), NB = E / R;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        __syncthreads();
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int r = 0; r < R; ++r)
                buf[ln::pad(L, ln::out_idx<L, S>(t, b, r)) * W + c] =
                    h ? v[b * R + r].y : v[b * R + r].x;
        __syncthreads();
#pragma unroll
        for (int m = 0; m < E; m += 2) {
            // two outputs' weights are loaded together; not more, and neither
            // they nor their places are kept from re to im (registers), nor are
            // the sums put off until the results are used
            int im = t + T * m;
            asm volatile("" : "+v"(im));
            double s[2] = {0.0, 0.0};
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                const int i = min(im + T * g, P.X.n - 1);
                const int b = P.base[i];
                const double *w = P.outw + (size_t)i * NW;
#pragma unroll
                for (int k = 0; k < NW; ++k) {
                    int p = b + k;
                    p += p < 0 ? L : 0;
                    s[g] = fma(w[k], buf[ln::pad(L, p) * W + c], s[g]);
                }
            }
            asm volatile("" : "+v"(s[0]), "+v"(s[1]));
            if (h) {
                o[m].y = s[0];
                o[m + 1].y = s[1];
            } else {
                o[m].x = s[0];
                o[m + 1].x = s[1];
            }
        }
    }
}

// One axis of a grid: out[i out_el + line out_line + q].
//
// AX_NEAR points lie e off their bins (radians per cell, e j < 6e-5: rounded
// coordinates): e^{i j (u + e)} = e^{i j u} (1 + i j e) to 2e-9, so a second
// transform, of j g[j], takes the place of interpolation from a line 1.5 times
// as long (384^2 x 8 coils, two slices: 1.47 -> 0.79 ms, of which 0.45 were LDS
// reads for the interpolation; 250 x 234 x 8 coils: 251 -> 136 us).
//
// Bound by memory: 512^2 x 32 coils, 768-point lines, 3.3 TB/s by the counters
// (reads alone 127 us, writes 87, the transforms 14 of 247 us per launch).
template <int L, int KIND>
__global__ __launch_bounds__(ln::threads(L) * ln::lines(L, ST_WG),
                             KIND == AX_NEAR ? 2 : 4) void k_line_store(
    LineArgs P, double2 *out, size_t out_line, size_t out_el) {
    constexpr int E = ln::vals(L), W = ln::lines(L, ST_WG), T = ln::threads(L);
    __shared__ double buf[ln::words(L, W)];
    const int c = threadIdx.x % W, t = threadIdx.x / W;
    const int np = (P.nq + W - 1) / W;
    // workgroups go round the 8 XCDs: b and b + 8 (one XCD) take adjacent
    // panels, which share 128-byte rows in that XCD's L2
    const int b = (blockIdx.x & ~15) | ((blockIdx.x & 7) << 1) | ((blockIdx.x >> 3) & 1);
    const int line = b / np, q = (b % np) * W + c;
    if (line >= P.nlines) return;
    const bool ok = q < P.nq;
    const double2 *base = P.in + (size_t)line * P.in_line;
    double2 *o = out + (size_t)line * out_line + q;
    constexpr int S = ln::stages(L) - 1, R = ln::radix(L, S);
    int tp = t;
    auto bin = [&](int i) { return bin_index(P.X, L, ln::out_idx<L, S>(tp, i / R, i % R)); };
    double2 v[E];
    if constexpr (KIND == AX_FREE) {
        line_load<L, KIND>(P, base, t, q, ok, 0, v);
        ln::transform<L, W>(v, t, c, buf, P.tw);
        double2 x[E];
        line_interp<L, W>(P, v, t, c, buf, x);
#pragma unroll
        for (int m = 0; m < E; ++m) {
            const int i = t + T * m;
            if (ok && i < P.X.n) o[i * out_el] = x[m];
        }
        return;
    }
    double2 d[E];
    if constexpr (KIND == AX_NEAR) {
        line_load<L, KIND>(P, base, t, q, ok, 1, d);
        ln::transform<L, W>(d, t, c, buf, P.tw);
#pragma unroll
        for (int i = 0; i < E; ++i)
            d[i] = times_i(d[i], P.outw[P.X.n + min(bin(i), (unsigned)P.X.n - 1)]);
    }
    if constexpr (KIND == AX_NEAR) asm volatile("" : "+v"(tp));   // indices anew: registers
    line_load<L, KIND>(P, base, tp, q, ok, 0, v);
    ln::transform<L, W>(v, tp, c, buf, P.tw);
#pragma unroll
    for (int i = 0; i < E; ++i) {
        const double w = P.outw[min(bin(i), (unsigned)P.X.n - 1)];
        if constexpr (KIND == AX_NEAR) v[i] = make_double2(v[i].x + d[i].x, v[i].y + d[i].y);
        v[i] = make_double2(v[i].x * w, v[i].y * w);
    }
#pragma unroll
    for (int i = 0; i < E; ++i)
        if (ok && bin(i) < (unsigned)P.X.n) o[bin(i) * out_el] = v[i];
}

// Last axis with the time and coil sums: line = ia, out over ib.
// partial[split][ia][ib] = sum over the split's coils and time terms of
// conj(S_c) i^(l mod 2) vt[l] P_(l,c).
//
// A workgroup's W columns are 2^lcw coils (up to W of them) times W >> lcw time
// terms; it steps through its time terms, keeps their sum per coil in
// registers, and applies conj(S) once at the end.  (One pass over all columns
// with conj(S) applied to each read the maps nt times, half the kernel's time.)
// A workgroup with several sets of coils adds them to its partial image.
//
// Bound by the latency of a step (load, three exchanges, factors) at three
// waves per SIMD, which the bounds above keep free of spills: 512^2 x 32 coils
// 1.62 -> 0.92 ms (2.6 TB/s of its input; the counters show twice the bytes, its
// columns being 64-byte pieces of 128-byte lines), 250 x 234 x 8 coils 290 -> 148
// us, two slices of 384^2 x 8 coils 1.12 -> 0.55 ms.
struct CombineArgs {
    int nc, nt;             // coils, time terms
    int lcw, ncs, nls;      // log2 of the coils side by side; splits of coils, of time terms
    const double *vt;
    const float2 *sens;
    unsigned nvox;
    double2 *partial;
};

template <int L, int KIND>
__global__ __launch_bounds__(ln::threads(L) * ln::lines(L, ST_WG), 3) void k_line_combine(
    LineArgs P, CombineArgs C) {
    constexpr int E = ln::vals(L), W = ln::lines(L, ST_WG), T = ln::threads(L);
    __shared__ double buf[ln::words(L, W)];
    const int c = threadIdx.x % W, t = threadIdx.x / W;
    const int splits = C.ncs * C.nls;
    const int line = blockIdx.x / splits, split = blockIdx.x % splits;
    const int cs = split / C.nls, ls = split % C.nls;
    const int cw = 1 << C.lcw, g = W >> C.lcw;
    const int ncp = (C.nc + cw - 1) >> C.lcw, nst = (C.nt + g - 1) / g;
    const int s0 = nst * ls / C.nls, s1 = nst * (ls + 1) / C.nls;
    constexpr int S = ln::stages(L) - 1, R = ln::radix(L, S);
    const double2 *base = P.in + (size_t)line * P.in_line;
    // element offsets within vt and sens are 32 bits wide: at most 48 terms or 32
    // coils x 4096 x 4096 points, below 2^30
    const double *vline = C.vt + (size_t)line * P.X.n;
    double2 *out = C.partial + (size_t)split * C.nvox + (size_t)line * P.X.n;
    const unsigned nmax = (unsigned)P.X.n - 1;
    auto index = [&](int tp, int i) -> unsigned {
        if constexpr (KIND == AX_FREE) return tp + T * i;
        else return bin_index(P.X, L, ln::out_idx<L, S>(tp, i / R, i % R));
    };
    for (int cp = ncp * cs / C.ncs; cp < ncp * (cs + 1) / C.ncs; ++cp) {
        const int cc = (cp << C.lcw) + (c & (cw - 1));
        double2 acc[E];
#pragma unroll
        for (int i = 0; i < E; ++i) acc[i] = make_double2(0.0, 0.0);
        // steps through the time terms, on AX_NEAR axes twice each (k_line_store)
        constexpr int ORD = KIND == AX_NEAR ? 2 : 1;
        for (int s = s0 * ORD; s < s1 * ORD; ++s) {
            // opaque to the optimizer: the LDS and element indices are recomputed
            // per step instead of being held in registers across them (spills)
            int tp = t;
            asm volatile("" : "+v"(tp));
            const int order = s % ORD, l = (s / ORD) * g + (c >> C.lcw);
            const bool ok = cc < C.nc && l < C.nt;
            double2 v[E];
            line_load<L, KIND>(P, base, tp, l * C.nc + cc, ok, order, v);
            ln::transform<L, W>(v, tp, c, buf, P.tw);
            if constexpr (KIND == AX_FREE) {
                double2 x[E];
                line_interp<L, W>(P, v, tp, c, buf, x);
#pragma unroll
                for (int i = 0; i < E; ++i) v[i] = x[i];
            }
            // columns past the last hold zeros; elements past the image are
            // summed but not stored
            const unsigned vo = (ok ? l : 0) * C.nvox;
            asm volatile("" : "+v"(tp));
#pragma unroll
            for (int i = 0; i < E; ++i) {
                const unsigned x = min(index(tp, i), nmax);
                double f = vline[vo + x];
                double2 p = l & 1 ? make_double2(-v[i].y, v[i].x) : v[i];
                if (KIND == AX_NEAR && order) p = times_i(p, P.outw[P.X.n + x]);
                acc[i].x = fma(f, p.x, acc[i].x);
                acc[i].y = fma(f, p.y, acc[i].y);
                if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
            }
        }
        int te = t;
        asm volatile("" : "+v"(te));
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const unsigned x = index(te, i), xl = min(x, nmax);
            double2 a = acc[i];
            if (C.sens) {
                const float2 s =
                    (C.sens + (size_t)line * P.X.n)[(cc < C.nc ? cc : 0) * C.nvox + xl];
                a = make_double2(a.x * s.x + a.y * s.y, a.y * s.x - a.x * s.y);
            }
#pragma unroll
            for (int off = W / 2; off > 0; off >>= 1) {
                a.x += __shfl_xor(a.x, off, 64);
                a.y += __shfl_xor(a.y, off, 64);
            }
            if (KIND != AX_FREE) {
                const double w = P.outw[xl];
                a = make_double2(a.x * w, a.y * w);
            }
            if (c == 0 && x <= nmax) {
                if (cp > ncp * cs / C.ncs) {
                    a.x += out[x].x;
                    a.y += out[x].y;
                }
                out[x] = a;
            }
        }
    }
}

// ------------------------------------------------------- forward (voxels -> k)
// The same separation read the other way round.  With conj(d) = sum conj(S rho)
// e^{+i(2pi k.r + w t)} every transform keeps the sign of the adjoint:
//   V_q(r) = conj(S_c rho) e^{i(2pi kc.r + w tc)} i^(l mod 2) vt[l],
// divided by the kernel's transform and summed onto the k grid one axis at a
// time; then each sample gathers its NW x NW window of every column.

// i-th output of a transformed line at grid points g = i + j0 mod L; d: the
// first-order part of AX_NEAR axes
template <int KIND>
__device__ __forceinline__ void fline_out(const LineArgs &P, double2 *base, unsigned el, unsigned c,
                                          int L, int i, double2 v, double2 d) {
    int g = i + P.X.shift;
    if (g >= L) g -= L;
    if constexpr (KIND != AX_FREE) {
        for (; g < P.X.nf; g += L) {
            double2 z = v;
            if constexpr (KIND == AX_NEAR) {
                const double2 r = times_i(d, g - (int)P.X.j0);
                z = make_double2(v.x + r.x, v.y + r.y);
            }
            base[(unsigned)g * el + c] = z;
        }
    } else if (g < P.X.nf) {
        const double w = P.inw[g];
        base[(unsigned)g * el + c] = make_double2(v.x * w, v.y * w);
    }
}

// One axis, image points -> grid.  FIRST: the points' values are formed here
// (line = ia, points ib) from img0 = conj(rho) e^{i(...)}, the maps and vt;
// else read from P.in as in k_line_store.  AX_NEAR points take a second
// transform, of their values times their offsets.  AX_FREE points are spread onto
// the line's L cells through LDS: cell p sums the points of its list
// (P.base[p] .. P.base[p + 1]; ascending, so the sum's order is fixed).
template <int L, int KIND, bool FIRST>
__global__ __launch_bounds__(ln::threads(L) * ln::lines(L, ST_WG),
                             KIND == AX_NEAR ? 2 : 3) void k_fline(
    LineArgs P, const int *list, const double *listw, int ncg, const double2 *img0,
    const float2 *sens, const double *vt, unsigned nvox, double2 *out, size_t out_line,
    unsigned out_el) {
    constexpr int E = ln::vals(L), W = ln::lines(L, ST_WG), T = ln::threads(L);
    constexpr int R0 = ln::radix(L, 0);
    __shared__ double buf[ln::words(L, W)];
    const int c = threadIdx.x % W, t = threadIdx.x / W;
    const int np = (P.nq + W - 1) / W;
    const int b = (blockIdx.x & ~15) | ((blockIdx.x & 7) << 1) | ((blockIdx.x >> 3) & 1);
    const int line = b / np, q = (b % np) * W + c;
    if (line >= P.nlines) return;
    const bool ok = q < P.nq;
    const int l = ok ? q / ncg : 0, cc = ok ? q - l * ncg : 0;
    auto point = [&](int i) {
        if constexpr (FIRST) {
            const size_t x = (size_t)line * P.X.n + i;
            double2 v = img0[x];
            if (sens) {
                const float2 s = sens[(size_t)cc * nvox + x];
                v = make_double2(v.x * s.x + v.y * s.y, v.y * s.x - v.x * s.y);
            }
            const double f = vt[(size_t)l * nvox + x];
            return (l & 1) ? make_double2(-f * v.y, f * v.x) : make_double2(f * v.x, f * v.y);
        } else {
            return P.in[(size_t)line * P.in_line + (size_t)i * P.in_el + (ok ? q : q - c)];
        }
    };
    double2 v[E], d[E];
    int tp = t;
    if constexpr (KIND != AX_FREE) {
        auto bins = [&](bool first_order, double2 (&o)[E]) {
#pragma unroll
            for (int i = 0; i < E; ++i) {
                const unsigned x = bin_index(P.X, L, ln::in_idx<L, 0>(tp, i / R0, i % R0));
                const unsigned xl = min(x, (unsigned)P.X.n - 1);
                const double2 z = point(xl);
                double w = P.outw[xl];
                if (first_order) w *= P.outw[P.X.n + xl];
                o[i] = ok && x < (unsigned)P.X.n ? make_double2(z.x * w, z.y * w)
                                                 : make_double2(0.0, 0.0);
            }
        };
        if constexpr (KIND == AX_NEAR) {
            bins(true, d);
            ln::transform<L, W>(d, tp, c, buf, P.tw);
            asm volatile("" : "+v"(tp));   // indices anew: registers
        }
        bins(false, v);
    } else {
        double2 z[E];
#pragma unroll
        for (int m = 0; m < E; ++m)
            z[m] = point(min(t + T * m, P.X.n - 1));
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            __syncthreads();
#pragma unroll
            for (int m = 0; m < E; ++m)
                if (t + T * m < P.X.n) buf[(t + T * m) * W + c] = h ? z[m].y : z[m].x;
            __syncthreads();
#pragma unroll
            for (int i = 0; i < E; ++i) {
                const int p = ln::in_idx<L, 0>(t, i / R0, i % R0);
                double s = 0.0;
                for (int e = P.base[p]; e < P.base[p + 1]; ++e)
                    s = fma(listw[e], buf[list[e] * W + c], s);
                if (h) v[i].y = s;
                else v[i].x = s;
            }
        }
    }
    ln::transform<L, W>(v, tp, c, buf, P.tw);
    if (!ok) return;
    constexpr int S = ln::stages(L) - 1, R = ln::radix(L, S);
    double2 *o = out + (size_t)line * out_line + (q - c);
#pragma unroll
    for (int i = 0; i < E; ++i)
        fline_out<KIND>(P, o, out_el, c, L, ln::out_idx<L, S>(tp, i / R, i % R), v[i],
                        KIND == AX_NEAR ? d[i] : v[i]);
}

// Lists of k_fline's AX_FREE axes: cell p of L takes the points within
// NW/2 cells of it (their positions wrap), weight kb / kb_hat.  One workgroup
// per axis counts, scans and fills; each cell visits the points in order.
struct FListTab {
    NuAxis X;
    const float *coord;
    int stride;
    int *first;       // [L + 1]
    int *list;        // [n (NW + 1)]
    double *w;
};
__global__ __launch_bounds__(1024) void k_nu_flists(FListTab ta, FListTab tb) {
    const FListTab &P = blockIdx.x ? tb : ta;
    const NuAxis &X = P.X;
    if (X.kind != AX_FREE) return;
    __shared__ double pos[4096];
    __shared__ int sm[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < X.n; i += 1024)
        pos[i] = ((double)P.coord[(size_t)i * P.stride] - X.xc) / X.inv_d * X.L;
    __syncthreads();
    // points of cell p: |pos - p| <= NW/2 as the windows of k_nu_axis take it
    auto visit = [&](int p, auto f) {
        for (int i = 0; i < X.n; ++i) {
            const int b = (int)ceil(pos[i] - 0.5 * NW);
            int k = (p - b) % X.L;
            if (k < 0) k += X.L;
            if (k < NW) f(i, b + k);
        }
    };
    int carry = 0;
    for (int p0 = 0; p0 < X.L; p0 += 1024) {
        const int p = p0 + threadIdx.x;
        int n = 0;
        if (p < X.L) visit(p, [&](int, int) { ++n; });
        int inc = n;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int o = __shfl_up(inc, off, 64);
            if (lane >= off) inc += o;
        }
        if (lane == 63) sm[wave] = inc;
        __syncthreads();
        int before = carry, total = 0;
        for (int w = 0; w < 16; ++w) {
            if (w < wave) before += sm[w];
            total += sm[w];
        }
        if (p < X.L) {
            int at = before + inc - n;
            P.first[p] = at;
            visit(p, [&](int i, int cell) {
                P.list[at] = i;
                P.w[at++] = kb(pos[i] - cell) / kb_hat(pos[i] / X.L);
            });
        }
        carry += total;
        __syncthreads();
    }
    if (threadIdx.x == 0) P.first[X.L] = carry;
}

// img0[ia][ib] = conj(rho) e^{i(2pi kc.r + w tc)}
__global__ __launch_bounds__(256) void k_nu_img0(int nA, int nB, const float *r_r,
                                                 const float *r_i, const float *cA,
                                                 const float *cB, const float *fm, double kcA,
                                                 double kcB, double tc_2pi, double2 *img0) {
    __shared__ double2 tile[16][17];
    const int a0 = blockIdx.x * 16, b0 = blockIdx.y * 16;
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    {
        const int ia = a0 + tx, ib = b0 + ty;
        if (ia < nA && ib < nB) {
            const size_t i = (size_t)ib * nA + ia;
            const double rev = kcA * cA[i] + kcB * cB[i] + (fm ? tc_2pi * fm[i] : 0.0);
            double s, c;
            sincospi(2.0 * (rev - rint(rev)), &s, &c);
            tile[tx][ty] = cmul(make_double2(r_r[i], -(double)r_i[i]), make_double2(c, s));
        }
    }
    __syncthreads();
    const int ia = a0 + ty, ib = b0 + tx;
    if (ia < nA && ib < nB) img0[(size_t)ia * nB + ib] = tile[ty][tx];
}

// Samples of a tile of TG x TG window starts gather together: GI_S samples
// per work entry.
constexpr int TG = 4, GI_S = 16, GI_W = 16;   // GI_W >= NW + TG - 1 cells per row
struct GiEntry {
    int tile, s0, n, pad;
};

__global__ __launch_bounds__(256) void k_gi_list(int m, int ntile, const int *key,
                                                 GiEntry *entries, int *count) {
    __shared__ int first[256 + 1];   // first sample of the block's tiles, and one more
    const int tile = blockIdx.x * 255 + threadIdx.x;
    int lo = 0, hi = m;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (key[mid] < tile) lo = mid + 1;
        else hi = mid;
    }
    first[threadIdx.x] = lo;
    __syncthreads();
    if (threadIdx.x == 255 || tile >= ntile) return;
    const int n = first[threadIdx.x + 1] - lo, runs = (n + GI_S - 1) / GI_S;
    if (!runs) return;
    const int e0 = atomicAdd(count, runs);
    for (int r = 0; r < runs; ++r)
        entries[e0 + r] = GiEntry{tile, lo + r * GI_S, min(GI_S, n - r * GI_S), 0};
}

typedef double dx4 __attribute__((ext_vector_type(4)));

struct GiArgs {
    int ntx, nfA, nfB, nt, nc, c0, m;
    const int *perm, *bx, *by;      // sorted
    const double *wx, *wy;          // [s][NW + 2 (TG - 1)], zeros around the window
    const double *u;                // [s][nt]
    const double2 *rot;             // [s] e^{i(wc (t - tc) + 2pi kappa.xc)}
    const int *count;
    const GiEntry *entries;
    const double *grid;             // [gB][gA][nt][nc][2]
    float *d_r, *d_i;
};

// One wave per entry: out[sample][column] = sum over the tile's NW + TG - 1 = 14
// rows x GI_W = 16 cells and nt terms of (wx wy u)[sample] grid[column], a
// product of a 16 x 224 nt by a 224 nt x 16 matrix on v_mfma_f64_16x16x4_f64
// (sample i = lane % 16 and cell k = lane / 16 of A, column j = lane % 16 of B,
// result row lane / 16 + 4 r); 121 of the 224 products are of a sample's own
// window.  FP64 MFMA runs at 37.7 TFLOP/s here against 57.6 of the FMAs, but
// needs the weights once per lane instead of 16 of them in scalar registers per
// value.
template <int CB>
__global__ __launch_bounds__(64) void k_gather(GiArgs P) {
    const int lane = threadIdx.x, i = lane & 15, k = lane >> 4;
    const int ne = *P.count;
    const int nq2 = P.nt * P.nc * 2;
    for (int e = blockIdx.x; e < ne; e += gridDim.x) {
        const GiEntry E = P.entries[e];
        const int ga = (E.tile % P.ntx) * TG, gb = (E.tile / P.ntx) * TG;
        const int s = E.s0 + min(i, E.n - 1);
        constexpr int NX = NW + 2 * (TG - 1);
        // cell offset of the tile inside the padded window of this sample
        const double *px = P.wx + (size_t)s * NX + (ga - P.bx[s] + TG - 1);
        const double *py = P.wy + (size_t)s * NX + (gb - P.by[s] + TG - 1);
        const double live = i < E.n ? 1.0 : 0.0;
        double wx[GI_W / 4];
#pragma unroll
        for (int h = 0; h < GI_W / 4; ++h)
            wx[h] = 4 * h + k < NW + TG - 1 ? live * px[4 * h + k] : 0.0;
        const double *pu = P.u + (size_t)s * P.nt;
        dx4 acc[CB];
#pragma unroll
        for (int b = 0; b < CB; ++b) acc[b] = dx4{0.0, 0.0, 0.0, 0.0};
        // columns of this lane: 16 values (8 coils, re and im) per block
        int col[CB];
#pragma unroll
        for (int b = 0; b < CB; ++b) col[b] = min(16 * b + i, 2 * P.nc - 1);
        for (int r = 0; r < NW + TG - 1 && gb + r < P.nfB; ++r) {
            const double wy = py[r];
            const double *row = P.grid + ((size_t)(gb + r) * P.nfA + ga) * nq2;
#pragma unroll
            for (int h = 0; h < GI_W / 4; ++h) {
                const double a = wx[h] * wy;
                // cells past the grid have weight zero: read the last one
                const int g = min(4 * h + k, P.nfA - 1 - ga);
                const double *cell = row + (size_t)g * nq2;
                for (int l = 0; l < P.nt; ++l) {
                    const double al = a * pu[l];
#pragma unroll
                    for (int b = 0; b < CB; ++b)
                        acc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                            al, cell[l * 2 * P.nc + col[b]], acc[b], 0, 0, 0);
                }
            }
        }
        // row lane / 16 + 4 r is sample r * 4 + k of the entry
#pragma unroll
        for (int b = 0; b < CB; ++b) {
            const int c = 8 * b + (i >> 1);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const double mine = acc[b][r], other = __shfl_xor(mine, 1, 64);
                const int n = 4 * r + k;
                if (n >= E.n || c >= P.nc) continue;
                const double2 z = P.rot[E.s0 + n];
                const size_t o = (size_t)(P.c0 + c) * P.m + P.perm[E.s0 + n];
                // conj((re + i im) rot)
                if (i & 1) P.d_i[o] = (float)-(other * z.y + mine * z.x);
                else P.d_r[o] = (float)(mine * z.x - other * z.y);
            }
        }
    }
}

// per sorted sample: window starts, both axes' weights (TG - 1 zeros around),
// time factors, rotation
__global__ __launch_bounds__(256) void k_gi_prep(int m, const int *perm, const float *kA,
                                                 const float *kB, const float *t, NuAxis A,
                                                 NuAxis B, double tc, double tinv, double wc_cyc,
                                                 const double *coef, const double *poly, int nt,
                                                 int nleg, int *bx, int *by, double *wx,
                                                 double *wy, double *u, double2 *rot) {
    __shared__ double px[PREP_S], py[PREP_S], pt[PREP_S], pl[KB_WORDS];
    const int s0 = blockIdx.x * PREP_S, ns = min(PREP_S, m - s0);
    for (int i = threadIdx.x; i < KB_WORDS; i += 256) pl[i] = poly[i];
    if ((int)threadIdx.x < ns) {
        const int i = threadIdx.x, j = perm[s0 + i];
        double p;
        const int a = window(A, kA[j], &p);
        px[i] = 2.0 * (p - a - (0.5 * NW - 1)) - 1.0;
        bx[s0 + i] = a;
        const int b = window(B, kB[j], &p);
        py[i] = 2.0 * (p - b - (0.5 * NW - 1)) - 1.0;
        by[s0 + i] = b;
        pt[i] = clamp1(((double)t[j] - tc) * tinv);
        const double rev = ((double)kA[j] - A.kc) * A.xc + ((double)kB[j] - B.kc) * B.xc +
                           ((double)t[j] - tc) * wc_cyc;
        double s, c;
        sincospi(2.0 * (rev - rint(rev)), &s, &c);
        rot[s0 + i] = make_double2(c, s);
    }
    __syncthreads();
    constexpr int NX = NW + 2 * (TG - 1);
    for (int e = threadIdx.x; e < ns * NX; e += 256) {
        const int s = e / NX, g = e - s * NX - (TG - 1);
        const bool in = g >= 0 && g < NW;
        wx[(size_t)s0 * NX + e] = in ? kb_cell(pl, g, px[s]) : 0.0;
        wy[(size_t)s0 * NX + e] = in ? kb_cell(pl, g, py[s]) : 0.0;
    }
    for (int e = threadIdx.x; e < ns * nt; e += 256) {
        const int s = e / nt, l = e - s * nt;
        u[(size_t)s0 * nt + e] =
            prolate(coef + (size_t)l * nleg, coef + (size_t)nt * nleg, nleg, l & 1, pt[s]);
    }
}

// tile of a sample's window start
__global__ void k_gi_keys(int m, const float *kA, const float *kB, NuAxis A, NuAxis B, int ntx,
                          int *key, int *val) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= m) return;
    double s;
    key[j] = (window(B, kB[j], &s) / TG) * ntx + window(A, kA[j], &s) / TG;
    val[j] = j;
}

// vt[l][ia][ib] = m_l psi_l(w), in (A, B) order; one thread per value
__global__ __launch_bounds__(256) void k_nu_vt(int nA, int nB, const float *fm, double wc,
                                               double winv, int nt, const double *coef,
                                               const double *mul, int nleg, double *vt) {
    const int x = blockIdx.x * 256 + threadIdx.x, l = blockIdx.y;
    if (x >= nA * nB) return;
    const int ia = x / nB, ib = x % nB;
    const double s = clamp1(((fm ? (double)fm[(size_t)ib * nA + ia] : 0.0) - wc) * winv);
    vt[(size_t)l * nA * nB + x] =
        mul[l] * prolate(coef + (size_t)l * nleg, coef + (size_t)nt * nleg, nleg, l & 1, s);
}

// S_c [ib][ia] split -> [ia][ib] pairs, 32 x 32 tiles
__global__ __launch_bounds__(256) void k_nu_sens(int nA, int nB, const float *s_r,
                                                 const float *s_i, float2 *out) {
    __shared__ float2 tile[32][33];
    const size_t o = (size_t)blockIdx.z * nA * nB;
    const int a0 = blockIdx.x * 32, b0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int r = ty; r < 32; r += 8) {
        const int ib = b0 + r, ia = a0 + tx;
        if (ib < nB && ia < nA) {
            const size_t i = o + (size_t)ib * nA + ia;
            tile[r][tx] = make_float2(s_r[i], s_i[i]);
        }
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
        const int ia = a0 + r, ib = b0 + tx;
        if (ib < nB && ia < nA) out[o + (size_t)ia * nB + ib] = tile[tx][r];
    }
}

// out[ib][ia] = e^{i(2pi kc.r + w tc)} sum_s partial[s][ia][ib]
__global__ __launch_bounds__(256) void k_nu_out(int nA, int nB, int splits,
                                                const double2 *partial, const float *cA,
                                                const float *cB, const float *fm, double kcA,
                                                double kcB, double tc_2pi, float *out_r,
                                                float *out_i) {
    __shared__ double2 tile[16][17];
    const int a0 = blockIdx.x * 16, b0 = blockIdx.y * 16;
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    {
        const int ia = a0 + ty, ib = b0 + tx;
        double2 s = make_double2(0.0, 0.0);
        if (ia < nA && ib < nB)
            for (int q = 0; q < splits; ++q) {
                const double2 v = partial[(size_t)q * nA * nB + (size_t)ia * nB + ib];
                s.x += v.x;
                s.y += v.y;
            }
        tile[ty][tx] = s;
    }
    __syncthreads();
    const int ia = a0 + tx, ib = b0 + ty;
    if (ia >= nA || ib >= nB) return;
    const size_t i = (size_t)ib * nA + ia;
    const double rev = kcA * cA[i] + kcB * cB[i] + (fm ? tc_2pi * fm[i] : 0.0);
    double s, c;
    sincospi(2.0 * (rev - rint(rev)), &s, &c);
    const double2 v = cmul(tile[tx][ty], make_double2(c, s));
    out_r[i] = (float)v.x;
    out_i[i] = (float)v.y;
}

// --------------------------------------------------------------- dispatching
constexpr int NU_LENGTHS[] = {96,  128, 144,  192,  256,  288,  384,  512, 576,
                              768, 1024, 1152, 1536, 2048, 2304, 3072, 4096};

int pick_length(double want) {
    for (int L : NU_LENGTHS)
        if (L >= want) return L;
    return 0;
}

template <class F>
int line_switch(int L, F f) {
    switch (L) {
        case 96: return f(std::integral_constant<int, 96>{});
        case 128: return f(std::integral_constant<int, 128>{});
        case 144: return f(std::integral_constant<int, 144>{});
        case 192: return f(std::integral_constant<int, 192>{});
        case 256: return f(std::integral_constant<int, 256>{});
        case 288: return f(std::integral_constant<int, 288>{});
        case 384: return f(std::integral_constant<int, 384>{});
        case 512: return f(std::integral_constant<int, 512>{});
        case 576: return f(std::integral_constant<int, 576>{});
        case 768: return f(std::integral_constant<int, 768>{});
        case 1024: return f(std::integral_constant<int, 1024>{});
        case 1152: return f(std::integral_constant<int, 1152>{});
        case 1536: return f(std::integral_constant<int, 1536>{});
        case 2048: return f(std::integral_constant<int, 2048>{});
        case 2304: return f(std::integral_constant<int, 2304>{});
        case 3072: return f(std::integral_constant<int, 3072>{});
        case 4096: return f(std::integral_constant<int, 4096>{});
        default: return fail(IMP_EINVAL, "NUDFT: line length %d", L);
    }
}

int line_store(imp_ctx *ctx, LineArgs P, int nlines, double2 *out, size_t out_line,
               size_t out_el) {
    P.nlines = nlines;
    return line_switch(P.X.L, [&](auto len) -> int {
        constexpr int L = decltype(len)::value;
        // a multiple of 16 for the panel order
        const long wgs = ((long)nlines * ceil_div(P.nq, ln::lines(L, ST_WG)) + 15) & ~15L;
        auto fn = P.X.kind == AX_UNIFORM ? k_line_store<L, AX_UNIFORM>
                  : P.X.kind == AX_NEAR  ? k_line_store<L, AX_NEAR>
                                         : k_line_store<L, AX_FREE>;
        hipLaunchKernelGGL(fn, dim3((unsigned)wgs),
                           dim3(ln::threads(L) * ln::lines(L, ST_WG)), 0, ctx->stream, P, out, out_line,
                           out_el);
        IMP_CHECK_LAUNCH();
        return IMP_OK;
    });
}

// Splits of the combining pass over coils, then over time terms: about 16
// workgroups per CU in all (4 waves each, 8 to 12 of them resident), at most
// `most` partial images.
int line_combine(imp_ctx *ctx, const LineArgs &P, int nlines, int most, CombineArgs C,
                 int *splits) {
    return line_switch(P.X.L, [&](auto len) -> int {
        constexpr int L = decltype(len)::value, W = ln::lines(L, ST_WG);
        C.lcw = std::min(ln::bits(W), C.nc > 1 ? 32 - __builtin_clz(C.nc - 1) : 0);
        const int want = std::max(1, std::min(most, 16 * ctx->num_cus / nlines));
        const int ncp = ceil_div(C.nc, 1 << C.lcw), nst = ceil_div(C.nt, W >> C.lcw);
        C.ncs = ceil_div(ncp, ceil_div(ncp, want));
        C.nls = std::min(nst, std::max(1, want / C.ncs));
        *splits = C.ncs * C.nls;
        auto fn = P.X.kind == AX_UNIFORM ? k_line_combine<L, AX_UNIFORM>
                  : P.X.kind == AX_NEAR  ? k_line_combine<L, AX_NEAR>
                                         : k_line_combine<L, AX_FREE>;
        hipLaunchKernelGGL(fn, dim3((unsigned)(nlines * *splits)), dim3(ln::threads(L) * W), 0,
                           ctx->stream, P, C);
        IMP_CHECK_LAUNCH();
        return IMP_OK;
    });
}

// Axis of n coordinates from c0 to c1 (dev: largest distance from uniform)
// against frequencies [klo, khi].  False: the transform lengths do not fit.
bool plan_axis(int n, float c0, float c1, float dev, float cmin, float cmax, float klo, float khi,
               NuAxis *X) {
    if (n < 2) return false;
    X->n = n;
    X->kc = 0.5 * ((double)klo + khi);
    const double Kh = 0.5 * ((double)khi - klo);
    const double d = ((double)c1 - c0) / (n - 1);
    // A coordinate off by dev turns the phase by at most 2 pi Kh dev: nothing
    // below 1e-10 turns, and to first order (2e-9 off) up to 1e-5, which takes
    // in coordinates rounded to FP32 up to about 1000 points.
    X->kind = d == 0.0 || !(Kh * dev < 1e-5) ? AX_FREE : Kh * dev < 1e-10 ? AX_UNIFORM : AX_NEAR;
    if (X->kind != AX_FREE) {
        X->L = pick_length(2.0 * NU_SIGMA * (n / 2));   // bins up to n / 2
        if (!X->L) return false;
        X->xc = c0 + (n / 2) * d;
        X->flip = d < 0.0;
        X->inv_d = X->L * std::fabs(d);
    } else {
        X->xc = 0.5 * ((double)cmin + cmax);
        const double Xh = 0.5 * ((double)cmax - cmin);
        if (!(Xh > 0.0)) return false;
        X->flip = 0;
        X->inv_d = 2.0 * NU_SIGMA * Xh;
    }
    const double cells = Kh * X->inv_d;
    if (!(cells < 4096.0)) return false;
    X->j0 = std::ceil(cells + 0.5 * NW) + 1;
    X->nf = 2 * (int)X->j0 + 1;
    if (X->kind == AX_FREE) {
        // at least n: every thread interpolates at most vals(L) outputs
        X->L = pick_length(std::max<double>(NU_SIGMA * X->nf, n));
        if (!X->L) return false;
    }
    X->shift = (int)X->j0 % X->L;
    return true;
}

}  // namespace

// Scan of the operands: value ranges, tensor structure of the voxels.  n = 0
// scans the samples alone.  geo: G_WORDS result words, part: block results.
// The last kernel writes the words to ctx->geo_host under this number (0: not).
static int geo_enqueue(imp_ctx *ctx, unsigned *geo, unsigned *part, int m, int n, const float *kx,
                       const float *ky, const float *t, const float *x, const float *y,
                       const float *z, const float *fm, unsigned seq) {
    unsigned *host = seq ? ctx->geo_host : nullptr;
    const hipStream_t st = ctx->stream;
    const int kb = std::min(256, ceil_div(m, 1024)), xb = std::min(256, ceil_div(n, 1024));
    hipLaunchKernelGGL(k_geo_scan, dim3(kb + xb), dim3(256), 0, st, m, kx, ky, t, n, x, y, fm, kb,
                       part);
    hipLaunchKernelGGL(k_geo_final, dim3(1), dim3(256), 0, st, kb, xb, (const unsigned *)part,
                       geo, n ? nullptr : host, seq);
    if (n) {
        hipLaunchKernelGGL(k_geo_check, dim3(std::min(4 * ctx->num_cus, ceil_div(n, 256))),
                           dim3(256), 0, st, n, x, y, z, geo);
        if (host)
            hipLaunchKernelGGL(k_geo_export, dim3(1), dim3(64), 0, st, (const unsigned *)geo, host,
                               seq);
    }
    IMP_CHECK_LAUNCH();
    return IMP_OK;
}

static int geo_buffers(imp_ctx *ctx, int scans, unsigned **geo, unsigned **part) {
    void *w = nullptr;
    IMP_TRY(workspace(ctx, WS_NU_GEO,
                      ((size_t)scans * G_WORDS + 512 * GB_WORDS) * sizeof(unsigned), &w));
    *geo = (unsigned *)w;
    *part = *geo + (size_t)scans * G_WORDS;
    return IMP_OK;
}

// results of `scans` scans on the host; waits for the stream
static int geo_read(imp_ctx *ctx, const unsigned *geo, int scans, unsigned *h) {
    IMP_HIP(hipMemcpyAsync(h, geo, (size_t)scans * G_WORDS * sizeof(unsigned),
                           hipMemcpyDeviceToHost, ctx->stream));
    IMP_HIP(hipStreamSynchronize(ctx->stream));
    ctx->table_slot = 0;   // no table upload is in flight
    return IMP_OK;
}

// One scan with its result exported: the words are here, and all that was
// queued before them has ended, once the host sees the scan's number.  Watched
// for about as long as a wake-up takes; then, or where the memory is not seen
// before the kernel ends, the stream is waited for.
static int geo_scan(imp_ctx *ctx, int m, int n, const float *kx, const float *ky, const float *t,
                    const float *x, const float *y, const float *z, const float *fm, unsigned *h) {
    unsigned *geo, *part;
    IMP_TRY(geo_buffers(ctx, 1, &geo, &part));
    if (++ctx->geo_seq == 0) ctx->geo_seq = 1;
    const unsigned seq = ctx->geo_seq;
    IMP_TRY(geo_enqueue(ctx, geo, part, m, n, kx, ky, t, x, y, z, fm, seq));
    const auto seen = [&] {
        return __atomic_load_n(&ctx->geo_host[G_WORDS], __ATOMIC_ACQUIRE) == seq;
    };
    const auto start = std::chrono::steady_clock::now();
    while (!seen()) {
        if (std::chrono::steady_clock::now() - start < std::chrono::microseconds(200)) continue;
        IMP_HIP(hipStreamSynchronize(ctx->stream));
        if (!seen()) return fail(IMP_EHIP, "NUDFT: the geometry scan left no result");
    }
    std::memcpy(h, ctx->geo_host, G_WORDS * sizeof(unsigned));
    ctx->table_slot = 0;   // no table upload is in flight
    return IMP_OK;
}

// Axes A and B and the ranges of t and w from a scan, or ok = false when the
// separable evaluation does not apply.
static void geo_image(const unsigned *h, int n, bool d3, bool fm, NuGeometry *G) {
    G->ok = false;
    int nA = 0, nz = 0;
    bool a_is_y = false;
    if (h[G_FLAGS] || h[G_KFLAG] || !geo_axes(h[G_FCX], h[G_FCY], n, d3, &a_is_y, &nA, &nz))
        return;
    const int nB = n / (nA * nz);
    auto lo = [&](int i) { return dec_f(h[G_MIN + i]); };
    auto hi = [&](int i) { return dec_f(h[G_MAX + i]); };
    const int a = a_is_y ? 1 : 0, b = 1 - a;
    if (!plan_axis(nA, bits_f(h[G_A0]), bits_f(h[G_A1]), bits_f(h[G_DEVA]), lo(3 + a), hi(3 + a),
                   lo(a), hi(a), &G->A) ||
        !plan_axis(nB, bits_f(h[G_B0]), bits_f(h[G_B1]), bits_f(h[G_DEVB]), lo(3 + b), hi(3 + b),
                   lo(b), hi(b), &G->B))
        return;
    const double tlo = lo(2), thi = hi(2), wlo = fm ? lo(5) : 0.0, whi = fm ? hi(5) : 0.0;
    G->nz = nz;
    G->tc = 0.5 * (tlo + thi);
    G->th = 0.5 * (thi - tlo);
    G->wc = 0.5 * (wlo + whi);
    G->wh = 0.5 * (whi - wlo);
    G->a_is_y = a_is_y;
    G->ok = G->wh * G->th <= NU_MAX_THETA;
}

// Geometry of an image problem (z null: 2D; else z fastest).  Synchronises
// (one small read-back).
int nufft_geometry(imp_ctx *ctx, int m, int n, const float *kx, const float *ky, const float *t,
                   const float *x, const float *y, const float *z, const float *fm,
                   NuGeometry *G) {
    unsigned h[G_WORDS];
    IMP_TRY(geo_scan(ctx, m, n, kx, ky, t, x, y, z, fm, h));
    geo_image(h, n, z != nullptr, fm != nullptr, G);
    return IMP_OK;
}

// The same for several 2D images with one read-back (jobs with scan[j] false
// are left out).
int nufft_geometry_batch(imp_ctx *ctx, int njobs, const imp_nudft_job *jobs,
                         const std::vector<char> &scan, std::vector<NuGeometry> *G) {
    unsigned *geo, *part;
    IMP_TRY(geo_buffers(ctx, njobs, &geo, &part));
    for (int j = 0; j < njobs; ++j) {
        const imp_nudft_job &b = jobs[j];
        if (scan[j])
            IMP_TRY(geo_enqueue(ctx, geo + (size_t)j * G_WORDS, part, b.num_k, b.num_x, b.kx, b.ky,
                                b.t, b.x, b.y, nullptr, b.fm, 0u));
    }
    std::vector<unsigned> h((size_t)njobs * G_WORDS);
    IMP_TRY(geo_read(ctx, geo, njobs, h.data()));
    for (int j = 0; j < njobs; ++j)
        if (scan[j])
            geo_image(&h[(size_t)j * G_WORDS], jobs[j].num_x, false, jobs[j].fm != nullptr,
                      &(*G)[j]);
    return IMP_OK;
}

namespace {

struct Carver {
    size_t off = 0;
    size_t take(size_t bytes) {
        const size_t o = off;
        off += (bytes + 255) & ~(size_t)255;
        return o;
    }
};

// largest spread-grid block and A-transformed grid (bytes): columns go in
// groups so the second stays below its limit, rows in blocks for the first
constexpr size_t NU_BLOCK_BYTES = (size_t)512 << 20;
constexpr size_t NU_MID_BYTES = (size_t)3 << 30;
// What a context keeps of the workspaces from call to call: 4.2 GB serve 512^2 x
// 32 coils, 12 GB the largest images at 32 coils.  Larger ones (samples far
// beyond the band, 10^7 samples and more) are freed when the call ends: making
// them anew took 0.4 ms for 1 to 32 GB in a bare process, and up to 27 ms per GB
// in others.
constexpr size_t NU_KEEP_BYTES = (size_t)16 << 30;

int log2i(int n) {
    int b = 0;
    while ((1 << b) < n) ++b;
    return b;
}

// time terms as the predicted times use them (within 1 of what prolate_expand
// finds from theta = 0.3 to 40, 2 below)
int terms_estimate(const NuGeometry &G) {
    const double th = G.wh * G.th;
    if (!(th > 0.0)) return 1;
    const double n = th > 1.0 ? 8.0 + 1.6 * std::pow(th - 1.0, 0.85) : 8.0 + 1.2 * std::log(th);
    return (int)std::lround(std::min<double>(NU_MAX_TERMS, std::max(2.0, n)));
}

// Coils (or other columns) of a group: the half-transformed grid within its
// limit, and column slots x time groups x rows = 64 lanes, so fewer columns
// when the time terms need more groups.
int column_group(const NuGeometry &G, int nt, int ncols) {
    int cg = std::min(32, 1 << log2i(ncols));
    while (cg > 1 && (size_t)G.A.n * G.B.nf * nt * cg * sizeof(double2) > NU_MID_BYTES) cg /= 2;
    while (cg > 1 && ceil_div(nt, 64 / cg) > SP_MAX_NL) cg /= 2;
    return cg;
}

// The split of the lanes beside 2^lc columns into time groups and rows with the
// fewest FP64 instructions per sample: visits x (2 NL (T + 1) + about 16 for
// the rest).
struct SpreadSplit {
    int ll = 0, nl = 1, yg = 1, T = 1;
    double cost = 0.0;
};
SpreadSplit spread_split(int nt, int lc) {
    SpreadSplit best;
    for (int l = 0; l <= std::min(6 - lc, log2i(nt)); ++l) {
        const int k = ceil_div(nt, 1 << l);
        if (k > SP_MAX_NL) continue;
        const int cells = sp_switch(k, [](auto n) { return sp_cells(decltype(n)::value); });
        const int rows = 1 << (6 - lc - l);
        const double cost = (double)(NW + rows - 1) / rows * (NW + cells - 1) / cells *
                            (2 * k * (cells + 1) + 16);
        if (best.cost == 0.0 || cost < best.cost) best = SpreadSplit{l, k, rows, cells, cost};
    }
    return best;
}

}  // namespace

// 8-bit digits of the cells' numbers 0..ncells - 1 (at least one: the sort
// also fills the sample order)
int nufft_sort_passes(int ncells) {
    int n = 1;
    while (n < 4 && (ncells - 1) >> (8 * n)) ++n;
    return n;
}

namespace {

// The stages shared by the separable operators: samples sorted by window,
// tables, work lists; then per group of columns, weights -> spread grid ->
// mid[ia][gB][q].
struct NuPass {
    imp_ctx *ctx;
    const NuGeometry &G;
    int m;                         // samples
    const float *kA, *kB, *t;
    int nt = 1, nleg = 1;          // time terms
    std::vector<double> tab;       // coefficients, recurrence, mul, KB polynomials
    size_t tab_mul = 0, tab_poly = 0;
    int cg = 1, groups = 1, lc = 0, ll = 0, nl = 1, yg = 1, T = 1, ntp = 1, blocks = 1;
    SpGeom S{};
    Carver W;
    size_t o_bx, o_wx, o_wy, o_u, o_wd, o_vis, o_cnt, o_ent, o_mul, o_part, o_tab, o_start,
        o_grid, o_mid, o_tw[2], o_in[2], o_ow[2], o_ob[2];
    char *ws = nullptr;
    const int *perm = nullptr, *key = nullptr;

    NuPass(imp_ctx *c, const NuGeometry &g, int m_, const float *kx, const float *ky,
           const float *t_)
        : ctx(c), G(g), m(m_), kA(g.a_is_y ? ky : kx), kB(g.a_is_y ? kx : ky), t(t_) {}

    // samples sorted by window start (or by the gather's tiles of starts;
    // launched before the time expansion is computed on the host)
    int sort(bool tiles = false) {
        const hipStream_t st = ctx->stream;
        const int gtx = ceil_div(G.A.nf - NW + 1, TG);
        const int ncells = tiles ? gtx * ceil_div(G.B.nf - NW + 1, TG)
                                 : (G.A.nf - NW + 1) * (G.B.nf - NW + 1);
        const int nblk = ceil_div(m, RX_BLOCK);
        Carver c;
        const size_t k0 = c.take((size_t)m * 4), k1 = c.take((size_t)m * 4);
        const size_t v0 = c.take((size_t)m * 4), v1 = c.take((size_t)m * 4);
        const size_t hi = c.take((size_t)RX_BINS * nblk * 4);
        void *p = nullptr;
        IMP_TRY(workspace(ctx, WS_NU_SORT, c.off, &p));
        char *b = (char *)p;
        int *key0 = (int *)(b + k0), *key1 = (int *)(b + k1);
        int *val0 = (int *)(b + v0), *val1 = (int *)(b + v1), *hist = (int *)(b + hi);
        if (tiles)
            hipLaunchKernelGGL(k_gi_keys, dim3(ceil_div(m, 256)), dim3(256), 0, st, m, kA, kB,
                               G.A, G.B, gtx, key0, val0);
        else
            hipLaunchKernelGGL(k_nu_keys, dim3(ceil_div(m, 256)), dim3(256), 0, st, m, kA, kB,
                               G.A, G.B, key0, val0);
        for (int pass = 0, shift = 0; pass < nufft_sort_passes(ncells); ++pass, shift += 8) {
            hipLaunchKernelGGL(k_rx_count, dim3(nblk), dim3(256), 0, st, (const int *)key0, m,
                               shift, hist);
            hipLaunchKernelGGL(k_rx_scatter, dim3(nblk), dim3(256), 0, st, (const int *)key0,
                               (const int *)val0, m, shift, nblk, (const int *)hist, key1, val1);
            std::swap(key0, key1);
            std::swap(val0, val1);
        }
        IMP_CHECK_LAUNCH();
        key = key0;
        perm = val0;
        return IMP_OK;
    }

    // sizes for ncols columns of coils (or other right-hand sides) and the
    // time expansion; the caller then takes its own regions from W
    int expand() {
        std::vector<double> mul;
        if (!prolate_expand(G.wh * G.th, tab, mul, &nt, &nleg))
            return fail(IMP_EINVAL, "NUDFT: time expansion of %g", G.wh * G.th);
        tab_mul = tab.size();
        tab.insert(tab.end(), mul.begin(), mul.end());
        tab_poly = tab.size();
        tab.insert(tab.end(), kb_poly_table(), kb_poly_table() + KB_WORDS);
        return IMP_OK;
    }
    void take_tables() {
        o_tab = W.take(tab.size() * 8);
        for (int a = 0; a < 2; ++a) {
            const NuAxis &X = a ? G.B : G.A;
            o_tw[a] = W.take((size_t)X.L * sizeof(double2));
            o_in[a] = W.take((size_t)X.nf * 8);
            o_ow[a] = W.take((size_t)X.n * (X.kind == AX_FREE ? NW : 2) * 8);
            o_ob[a] = W.take((size_t)X.n * 4);
        }
    }

    int layout(int ncols) {
        IMP_TRY(expand());
        const NuAxis &A = G.A, &B = G.B;
        cg = column_group(G, nt, ncols);
        groups = ceil_div(ncols, cg);
        lc = log2i(cg);
        const SpreadSplit split = spread_split(nt, lc);
        ll = split.ll;
        nl = split.nl;
        yg = split.yg;
        T = split.T;
        ntp = nl << ll;
        S.T = T;
        S.yg = yg;
        S.ncA = A.nf - NW + 1;
        S.ncB = B.nf - NW + 1;
        S.nfA = A.nf;
        S.nfB = B.nf;
        S.ntx = ceil_div(A.nf, T);
        const int nc0 = std::min(cg, ncols);
        const size_t row_bytes = (size_t)A.nf * nt * nc0 * sizeof(double2);
        int rb = (int)std::max<size_t>(1, NU_BLOCK_BYTES / row_bytes);
        rb = std::min(ceil_div(B.nf, yg) * yg, std::max(yg, rb / yg * yg));
        blocks = ceil_div(B.nf, rb);
        rb = ceil_div(ceil_div(B.nf, blocks), yg) * yg;   // even blocks
        blocks = ceil_div(B.nf, rb);
        S.rb = rb;
        S.nty = rb / yg;
        S.bw = T >= 6 ? 8 : 16;
        S.ntile = ceil_div(S.ntx, S.bw) * ceil_div(S.nty, SP_RUN / S.bw) * SP_RUN;
        S.entry_cap = S.ntile + SP_SLOTS;
        const int ncells = S.ncA * S.ncB;
        o_start = W.take(((size_t)ncells + 1) * 4);
        o_bx = W.take((size_t)m * 4);
        o_wx = W.take((size_t)m * (NW + 2 * (T - 1)) * 8);
        o_wy = W.take((size_t)m * (NW + 2 * (yg - 1)) * 8);
        o_u = W.take((size_t)m * ntp * 8);
        o_wd = W.take((size_t)m * (1 << lc) * sizeof(double2));
        o_vis = W.take((size_t)blocks * S.ntile * 4);
        o_cnt = W.take((size_t)blocks * sizeof(SpCount));
        o_ent = W.take((size_t)blocks * S.entry_cap * sizeof(SpEntry));
        o_mul = W.take((size_t)blocks * SP_SLOTS * sizeof(SpMulti));
        o_part = W.take((size_t)SP_SLOTS * nl * T * 64 * sizeof(double2));
        take_tables();
        o_grid = W.take((size_t)rb * row_bytes);
        o_mid = W.take((size_t)A.n * B.nf * nt * nc0 * sizeof(double2));
        return IMP_OK;
    }

    template <class P>
    P at(size_t o) const { return (P)(ws + o); }
    const double *coef() const { return at<const double *>(o_tab); }
    const double *mul() const { return coef() + tab_mul; }

    // Allocates everything taken from W, uploads the expansion and fills the
    // axis tables.  cA, cB: axis coordinates, sA and sB elements apart (read
    // on nonuniform axes).
    int alloc(const float *cA, int sA, const float *cB, int sB) {
        const hipStream_t st = ctx->stream;
        void *p = nullptr;
        IMP_TRY(workspace(ctx, WS_NU, W.off, &p));
        ws = (char *)p;
        // staged in a slot of the context's pinned memory that no upload reads
        if (tab.size() > HOST_TABLE_WORDS)
            return fail(IMP_EINVAL, "NUDFT: %zu table words", tab.size());
        if (ctx->table_slot >= HOST_TABLES) {
            IMP_HIP(hipStreamSynchronize(st));
            ctx->table_slot = 0;
        }
        double *slot = ctx->host_tables() + (size_t)ctx->table_slot++ * HOST_TABLE_WORDS;
        std::copy(tab.begin(), tab.end(), slot);
        IMP_HIP(hipMemcpyAsync(ws + o_tab, slot, tab.size() * 8, hipMemcpyHostToDevice, st));
        AxisTab ta[2];
        int len = 0;
        for (int a = 0; a < 2; ++a) {
            const NuAxis &X = a ? G.B : G.A;
            len = std::max(len, std::max(std::max(X.L, X.nf), X.n));
            ta[a] = AxisTab{X, a ? cB : cA, a ? sB : sA, at<double2 *>(o_tw[a]),
                            at<double *>(o_in[a]), at<double *>(o_ow[a]), at<int *>(o_ob[a])};
        }
        hipLaunchKernelGGL(k_nu_axis, dim3(ceil_div(len, 256), 2), dim3(256), 0, st, ta[0], ta[1]);
        IMP_CHECK_LAUNCH();
        return IMP_OK;
    }

    // the spread's tables and work lists
    int build(const float *cA, int sA, const float *cB, int sB) {
        IMP_TRY(alloc(cA, sA, cB, sB));
        const hipStream_t st = ctx->stream;
        const dim3 b256(256);
        const int ncells = S.ncA * S.ncB, ntile = S.ntile;
        SpCount *cnt = at<SpCount *>(o_cnt);
        hipLaunchKernelGGL(k_nu_starts, dim3(ceil_div(ncells + 1, 256)), b256, 0, st, m, key,
                           ncells, at<int *>(o_start), (int *)cnt,
                           (int)(blocks * sizeof(SpCount) / 4));
        hipLaunchKernelGGL(k_nu_prep, dim3(ceil_div(m, PREP_S)), b256, 0, st, m, perm, kA, kB, t,
                           G.A, G.B, G.tc, G.th > 0.0 ? 1.0 / G.th : 0.0, coef(),
                           coef() + tab_poly, nt, ntp, nleg, T - 1, yg - 1, at<int *>(o_bx),
                           at<double *>(o_wx), at<double *>(o_wy), at<double *>(o_u));
        hipLaunchKernelGGL(k_sp_count, dim3(ceil_div(ntile, 256), blocks), b256, 0, st, S,
                           at<const int *>(o_start), at<int *>(o_vis), cnt);
        hipLaunchKernelGGL(k_sp_list, dim3(ceil_div(ntile, 256), blocks), b256, 0, st, S,
                           at<const int *>(o_vis), cnt, at<SpEntry *>(o_ent),
                           at<SpMulti *>(o_mul));
        IMP_CHECK_LAUNCH();
        return IMP_OK;
    }

    LineArgs line(int axis, const void *in, size_t in_line, unsigned in_el, int nq) const {
        LineArgs P{};
        P.in = (const double2 *)in;
        P.in_line = in_line;
        P.in_el = in_el;
        P.nq = nq;
        P.X = axis ? G.B : G.A;
        P.tw = at<const double2 *>(o_tw[axis]);
        P.inw = at<const double *>(o_in[axis]);
        P.outw = at<const double *>(o_ow[axis]);
        P.base = at<const int *>(o_ob[axis]);
        return P;
    }

    // weights of nc columns (in wd) -> mid[ia][gB][l nc + c]
    int to_mid(int nc) {
        const hipStream_t st = ctx->stream;
        const int nq = nt * nc;
        SpFn spread = sp_switch(nl, [&](auto k) { return sp_pick1<decltype(k)::value>(yg > 1); });
        SpFn multi = sp_switch(nl, [](auto k) { return sp_multi1<decltype(k)::value>(); });
        SpArgs P{};
        P.G = S;
        P.nt = nt;
        P.ntp = ntp;
        P.nc = nc;
        P.lc = lc;
        P.ll = ll;
        P.start = at<const int *>(o_start);
        P.perm = perm;
        P.bx = at<const int *>(o_bx);
        P.wx = at<const double *>(o_wx);
        P.wy = at<const double *>(o_wy);
        P.u = at<const double *>(o_u);
        P.wd = at<const double2 *>(o_wd);
        P.cnt = at<const SpCount *>(o_cnt);
        P.entries = at<const SpEntry *>(o_ent);
        P.multis = at<const SpMulti *>(o_mul);
        P.part = at<double2 *>(o_part);
        P.grid = at<double2 *>(o_grid);
        LineArgs LA = line(0, ws + o_grid, (size_t)G.A.nf * nq, nq, nq);
        for (int b = 0; b < blocks; ++b) {
            P.block = b;
            // one-wave workgroups: a wave that ends makes room at once
            const int rec = prof_begin(ctx, "k_spread");
            const int wgs = ceil_div(std::min(S.entry_cap, 64 * ctx->num_cus), 8 * SP_RUN);
            hipLaunchKernelGGL(spread, dim3(wgs * 8 * SP_RUN), dim3(64),
                               SP_BATCH * (ntp + (yg > 1 ? yg : 0)) * sizeof(double), st, P);
            prof_end(ctx, rec);
            hipLaunchKernelGGL(multi, dim3(4 * ctx->num_cus), dim3(256), 0, st, P);
            IMP_CHECK_LAUNCH();
            IMP_TRY(line_store(ctx, LA, std::min(S.rb, G.B.nf - b * S.rb),
                               at<double2 *>(o_mid) + (size_t)b * S.rb * nq, nq,
                               (size_t)G.B.nf * nq));
        }
        return IMP_OK;
    }
    // the call's end: workspaces beyond what is kept are freed
    int finish() const {
        IMP_TRY(workspace_release(ctx, WS_NU_SORT, NU_KEEP_BYTES));
        return workspace_release(ctx, WS_NU, NU_KEEP_BYTES);
    }
    LineArgs lines_b(int nc) const {
        return line(1, ws + o_mid, (size_t)G.B.nf * nt * nc, nt * nc, nt * nc);
    }
};

}  // namespace

// kernel-timer record over a scope (closed on every return)
namespace {
struct ProfScope {
    imp_ctx *ctx;
    int rec;
    ProfScope(imp_ctx *c, const char *name) : ctx(c), rec(prof_begin(c, name)) {}
    ~ProfScope() { prof_end(ctx, rec); }
};
}  // namespace

// Predicted times.  Each form was timed on 1000 random single calls (12..900
// points per axis, 4e3..8e5 samples within 0.25 to 5 times the band, dense and
// even, 1 to 32 coils, 1 to 40 time terms, all axis kinds): the separable
// adjoint is within 15% rms (0.57 to 1.7 times) of the sum below, F within 13%,
// the direct sums within 6%.  Prices without the axis kinds, the columns that pad a
// workgroup and F's nearly empty tiles were 41% and 53% off and sent calls to
// the form that took up to 2.5 times as long.

// Lines of all columns along an axis, in transformed elements: whole
// workgroups' columns; AX_NEAR takes two transforms, AX_FREE an interpolation
// (about three).
static double line_work(const NuAxis &X, double nlines, double columns) {
    return nlines * columns * X.L * (X.kind == AX_UNIFORM ? 1 : X.kind == AX_NEAR ? 2 : 3);
}
static double padded(int columns, int L) {
    const int w = ln::lines(L, ST_WG);
    return (double)ceil_div(columns, w) * w;
}
// prolate functions of `points` points: every Legendre degree of each term
static double expansion_work(const NuGeometry &G, int nt, double points) {
    return points * nt * (0.75 * G.wh * G.th + 36.0);
}
// The sort's blocks each read every block's digit counts (about 5 TB/s).
static double sort_us(int m, double ncells) {
    const double nblk = ceil_div(m, RX_BLOCK);
    return nufft_sort_passes((int)ncells) * nblk * nblk * (RX_BINS * sizeof(int)) / 5e6;
}
static double cells(const NuAxis &A, const NuAxis &B) {
    return (double)(A.nf - NW + 1) * (B.nf - NW + 1);
}
// fixed part, samples and A transform of ncols columns
static double to_mid_us(const NuGeometry &G, int nt, int m, int ncols) {
    const int cg = column_group(G, nt, ncols), groups = ceil_div(ncols, cg);
    const SpreadSplit sp = spread_split(nt, log2i(cg));
    const double prep = 2 * NW + 2 * (sp.T - 1) + 2 * (sp.yg - 1) + nt +
                        2.0 * groups * (1 << log2i(cg));
    const double lines = groups * padded(nt * std::min(cg, ncols), G.A.L);
    // a group is half a dozen launches of some 8 us
    return 144.0 + 50.0 * (groups - 1) + sort_us(m, cells(G.A, G.B)) + m * (2.79e-6 * groups * sp.cost + 1.46e-5 * prep) +
           1.5e-6 * expansion_work(G, nt, m) + 9.74e-6 * G.A.nf * G.B.nf * (double)nt * ncols +
           4.16e-6 * line_work(G.A, G.B.nf, lines);
}

double nufft_adjoint_us(const NuGeometry &G, int m, int ncoils) {
    const int nt = terms_estimate(G);
    const int cg = column_group(G, nt, ncoils), groups = ceil_div(ncoils, cg);
    // the combining pass holds whole workgroups of coils x time terms
    const int nc = std::min(cg, ncoils), w = ln::lines(G.B.L, ST_WG);
    const int cw = std::min(w, 1 << log2i(nc));
    const double steps = (double)groups * ceil_div(nc, cw) * ceil_div(nt, w / cw) * w;
    return to_mid_us(G, nt, m, ncoils) + 4.16e-6 * line_work(G.B, G.A.n, steps) +
           8.7e-7 * expansion_work(G, nt, (double)G.A.n * G.B.n);
}

int nufft_adjoint(imp_ctx *ctx, const NuGeometry &G, int m, int ncoils, const float *kx,
                  const float *ky, const float *t, const float *x, const float *y,
                  const float *fm, const float *phi_r, const float *phi_i, const float *d_r,
                  const float *d_i, const float *s_r, const float *s_i, float *out_r,
                  float *out_i) {
    const hipStream_t st = ctx->stream;
    const dim3 b256(256);
    const float *cA = G.a_is_y ? y : x, *cB = G.a_is_y ? x : y;
    const int nA = G.A.n, nB = G.B.n;
    const size_t nvox = (size_t)nA * nB;
    const ProfScope prof(ctx, "nufft_adjoint");
    NuPass N(ctx, G, m, kx, ky, t);
    IMP_TRY(N.sort());
    IMP_TRY(N.layout(ncoils));
    constexpr int splits_max = 8;
    const size_t o_vt = N.W.take((size_t)N.nt * nvox * 8);
    const size_t o_sens = N.W.take(s_r ? (size_t)ncoils * nvox * sizeof(float2) : 0);
    const size_t o_img = N.W.take((size_t)N.groups * splits_max * nvox * sizeof(double2));
    IMP_TRY(N.build(cA, 1, cB, nA));
    hipLaunchKernelGGL(k_nu_vt, dim3(ceil_div((long)nvox, 256), N.nt), b256, 0, st, nA, nB, fm,
                       G.wc, G.wh > 0.0 ? 1.0 / G.wh : 0.0, N.nt, N.coef(), N.mul(), N.nleg,
                       N.at<double *>(o_vt));
    if (s_r)
        hipLaunchKernelGGL(k_nu_sens, dim3(ceil_div(nA, 32), ceil_div(nB, 32), ncoils), b256, 0,
                           st, nA, nB, s_r, s_i, N.at<float2 *>(o_sens));
    IMP_CHECK_LAUNCH();
    int parts = 0;
    for (int g = 0; g < N.groups; ++g) {
        const int c0 = g * N.cg, nc = std::min(N.cg, ncoils - c0);
        hipLaunchKernelGGL(k_nu_data, dim3(ceil_div(m, WD_S)), b256, 0, st, m, c0, nc, 1 << N.lc,
                           N.kA, N.kB, t, G.A, G.B, G.tc, G.wc / (2.0 * M_PI), phi_r, phi_i, d_r,
                           d_i, N.at<double2 *>(N.o_wd));
        IMP_TRY(N.to_mid(nc));
        const LineArgs LB = N.lines_b(nc);
        CombineArgs C{};
        C.nc = nc;
        C.nt = N.nt;
        C.vt = N.at<const double *>(o_vt);
        C.sens = s_r ? N.at<const float2 *>(o_sens) + (size_t)c0 * nvox : nullptr;
        C.nvox = (unsigned)nvox;
        C.partial = N.at<double2 *>(o_img) + (size_t)parts * nvox;
        int splits = 0;
        IMP_TRY(line_combine(ctx, LB, nA, splits_max, C, &splits));
        parts += splits;
    }
    hipLaunchKernelGGL(k_nu_out, dim3(ceil_div(nA, 16), ceil_div(nB, 16)), b256, 0, st, nA, nB,
                       parts, N.at<const double2 *>(o_img), cA, cB, fm, G.A.kc, G.B.kc,
                       G.tc / (2.0 * M_PI), out_r, out_i);
    IMP_CHECK_LAUNCH();
    return N.finish();
}

// ------------------------------------------------------------ stacks (3D F^H d)
// Samples in P partitions that repeat one 2D trajectory of K samples at kz_p:
//   out(x, y, z) = sum_l i^(l mod 2) vt[l](w(x, y, z)) sum_(c, p)
//                  conj(S_c(x, y, z)) e^{i 2pi kz_p z} P_(l, c, p)(x, y),
// P the separable 2D sums of the C P coil-partition columns over K samples.
namespace {

// vt[l][voxel] in the voxels' own order
__global__ __launch_bounds__(256) void k_nu_vt3(int n, const float *fm, double wc, double winv,
                                                int nt, const double *coef, const double *mul,
                                                int nleg, double *vt) {
    const int v = blockIdx.x * 256 + threadIdx.x, l = blockIdx.y;
    if (v >= n) return;
    const double s = clamp1(((fm ? (double)fm[v] : 0.0) - wc) * winv);
    vt[(size_t)l * n + v] =
        mul[l] * prolate(coef + (size_t)l * nleg, coef + (size_t)nt * nleg, nleg, l & 1, s);
}

// ez[p][iz] = e^{i 2pi kz_p z}
__global__ void k_nu_ez(int P, int K, int nz, const float *kz, const float *z, double2 *ez) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P * nz) return;
    const double rev = (double)kz[(size_t)(i / nz) * K] * z[i % nz];
    double s, c;
    sincospi(2.0 * (rev - rint(rev)), &s, &c);
    ez[i] = make_double2(c, s);
}

// The sum over a group's columns at every voxel (one thread each; the voxels
// of a column read the same P values), added to acc; the last group applies
// the centre's phase and stores.  ST_C columns' factors conj(S) ez stay in
// registers over the time terms.
constexpr int ST_C = 8;
__global__ __launch_bounds__(256) void k_nu_stack(int n, int nz, int P, int c0, int nc,
                                                  int nt, const double2 *grid, const double2 *ez,
                                                  const double *vt, const float *s_r,
                                                  const float *s_i, double2 *acc, int first,
                                                  int last, const float *cA, const float *cB,
                                                  const float *fm, double kcA, double kcB,
                                                  double tc_2pi, float *out_r, float *out_i) {
    const int v = blockIdx.x * 256 + threadIdx.x;
    if (v >= n) return;
    const int iz = v % nz;
    const double2 *col = grid + (size_t)(v / nz) * nt * nc;
    double2 sum = first ? make_double2(0.0, 0.0) : acc[v];
    for (int cb = 0; cb < nc; cb += ST_C) {
        double2 f[ST_C];
#pragma unroll
        for (int i = 0; i < ST_C; ++i) {
            const int q = c0 + min(cb + i, nc - 1);
            f[i] = ez[(q % P) * nz + iz];
            if (s_r) {
                const size_t o = (size_t)(q / P) * n + v;
                f[i] = cmul(f[i], make_double2(s_r[o], -(double)s_i[o]));
            }
            if (cb + i >= nc) f[i] = make_double2(0.0, 0.0);
        }
        for (int l = 0; l < nt; ++l) {
            const double2 *p = col + (size_t)l * nc + cb;
            double2 z = make_double2(0.0, 0.0);
#pragma unroll
            for (int i = 0; i < ST_C; ++i) {
                const double2 g = p[min(i, nc - 1 - cb)];
                z.x = fma(f[i].x, g.x, fma(-f[i].y, g.y, z.x));
                z.y = fma(f[i].x, g.y, fma(f[i].y, g.x, z.y));
            }
            const double w = vt[(size_t)l * n + v];
            sum.x = fma(w, (l & 1) ? -z.y : z.x, sum.x);
            sum.y = fma(w, (l & 1) ? z.x : z.y, sum.y);
        }
    }
    if (!last) {
        acc[v] = sum;
        return;
    }
    const double rev = kcA * cA[v] + kcB * cB[v] + (fm ? tc_2pi * fm[v] : 0.0);
    double s, c;
    sincospi(2.0 * (rev - rint(rev)), &s, &c);
    const double2 o = cmul(sum, make_double2(c, s));
    out_r[v] = (float)o.x;
    out_i[v] = (float)o.y;
}

}  // namespace

double nufft_stack_us(const NuGeometry &G, int K, int nrhs) {
    const int nt = terms_estimate(G);
    const int cg = column_group(G, nt, nrhs), groups = ceil_div(nrhs, cg);
    const double vox = (double)G.A.n * G.B.n * G.nz;
    const double lines = groups * padded(nt * std::min(cg, nrhs), G.B.L);
    return 50.0 + to_mid_us(G, nt, K, nrhs) + 4.16e-6 * line_work(G.B, G.A.n, lines) +
           8.7e-7 * expansion_work(G, nt, vox) + 4e-7 * vox * nt * nrhs;
}

int nufft_stack_adjoint(imp_ctx *ctx, const NuGeometry &G, int K, int P, int ncoils,
                        const float *kx, const float *ky, const float *kz, const float *t,
                        const float *x, const float *y, const float *z, const float *fm,
                        const float *phi_r, const float *phi_i, const float *d_r,
                        const float *d_i, const float *s_r, const float *s_i, float *out_r,
                        float *out_i) {
    const hipStream_t st = ctx->stream;
    const dim3 b256(256);
    const ProfScope prof(ctx, "nufft_stack");
    const float *cA = G.a_is_y ? y : x, *cB = G.a_is_y ? x : y;
    const int nA = G.A.n, nB = G.B.n, nz = G.nz, nrhs = ncoils * P;
    const int n = nA * nB * nz;
    NuPass N(ctx, G, K, kx, ky, t);
    IMP_TRY(N.sort());
    IMP_TRY(N.layout(nrhs));
    const size_t o_vt = N.W.take((size_t)N.nt * n * 8);
    const size_t o_ez = N.W.take((size_t)P * nz * sizeof(double2));
    const size_t o_acc = N.W.take((size_t)n * sizeof(double2));
    const size_t o_p = N.W.take((size_t)nA * nB * N.nt * std::min(N.cg, nrhs) * sizeof(double2));
    IMP_TRY(N.build(cA, nz, cB, nz * nA));
    hipLaunchKernelGGL(k_nu_vt3, dim3(ceil_div(n, 256), N.nt), b256, 0, st, n, fm, G.wc,
                       G.wh > 0.0 ? 1.0 / G.wh : 0.0, N.nt, N.coef(), N.mul(), N.nleg,
                       N.at<double *>(o_vt));
    hipLaunchKernelGGL(k_nu_ez, dim3(ceil_div(P * nz, 256)), b256, 0, st, P, K, nz, kz, z,
                       N.at<double2 *>(o_ez));
    IMP_CHECK_LAUNCH();
    for (int g = 0; g < N.groups; ++g) {
        const int c0 = g * N.cg, nc = std::min(N.cg, nrhs - c0), nq = N.nt * nc;
        hipLaunchKernelGGL(k_nu_data, dim3(ceil_div(K, WD_S)), b256, 0, st, K, c0, nc, 1 << N.lc,
                           N.kA, N.kB, t, G.A, G.B, G.tc, G.wc / (2.0 * M_PI), phi_r, phi_i, d_r,
                           d_i, N.at<double2 *>(N.o_wd));
        IMP_TRY(N.to_mid(nc));
        IMP_TRY(line_store(ctx, N.lines_b(nc), nA, N.at<double2 *>(o_p), nq, (size_t)nA * nq));
        hipLaunchKernelGGL(k_nu_stack, dim3(ceil_div(n, 256)), b256, 0, st, n, nz, P, c0, nc,
                           N.nt, N.at<const double2 *>(o_p), N.at<const double2 *>(o_ez),
                           N.at<const double *>(o_vt), s_r, s_i, N.at<double2 *>(o_acc), g == 0,
                           g + 1 == N.groups, cA, cB, fm, G.A.kc, G.B.kc, G.tc / (2.0 * M_PI),
                           out_r, out_i);
        IMP_CHECK_LAUNCH();
    }
    return N.finish();
}

// ---------------------------------------------------------------- forward host
namespace {

int line_forward(imp_ctx *ctx, LineArgs P, int nlines, bool first, const int *list,
                 const double *listw, int ncg, const double2 *img0, const float2 *sens,
                 const double *vt, unsigned nvox, double2 *out, size_t out_line,
                 unsigned out_el) {
    P.nlines = nlines;
    return line_switch(P.X.L, [&](auto len) -> int {
        constexpr int L = decltype(len)::value;
        const long wgs = ((long)nlines * ceil_div(P.nq, ln::lines(L, ST_WG)) + 15) & ~15L;
        auto fn = P.X.kind == AX_UNIFORM
                      ? (first ? k_fline<L, AX_UNIFORM, true> : k_fline<L, AX_UNIFORM, false>)
                  : P.X.kind == AX_NEAR
                      ? (first ? k_fline<L, AX_NEAR, true> : k_fline<L, AX_NEAR, false>)
                      : (first ? k_fline<L, AX_FREE, true> : k_fline<L, AX_FREE, false>);
        hipLaunchKernelGGL(fn, dim3((unsigned)wgs), dim3(ln::threads(L) * ln::lines(L, ST_WG)), 0,
                           ctx->stream, P, list, listw, ncg, img0, sens, vt, nvox, out, out_line,
                           out_el);
        IMP_CHECK_LAUNCH();
        return IMP_OK;
    });
}

// k grid of a coil group (bytes)
constexpr size_t NU_KGRID_BYTES = (size_t)2 << 30;

}  // namespace

// Coils that go through F together: the k grid (A.nf x B.nf) and the
// half-transformed grid (A.n x B.nf) of a group stay within their limits.  One
// is not enough: of 2730 x 2730 voxels and samples within +-20 cycles along A
// and the whole band along B, the half-transformed grid is 36 times the larger.
// k_fline's element offsets are 32 bits wide; a group within the limits has at
// most 2^28 elements, and a single coil 4096 x 8205 x 48 (plan_axis and
// prolate_expand admit no more), below 2^31.
int nufft_forward_group(size_t grid_bytes, size_t mid_bytes, int ncoils) {
    int cg = std::min(32, ncoils);
    while (cg > 1 && (grid_bytes * cg > NU_KGRID_BYTES || mid_bytes * cg > NU_MID_BYTES))
        cg = (cg + 1) / 2;
    return cg;
}

// The gather takes up to GI_S samples of a tile together, so where samples are
// few per tile it works on almost empty products; k_nu_flists visits every
// point of an AX_FREE axis for each 1024 cells, in one workgroup.
double nufft_forward_us(const NuGeometry &G, int m, int ncoils) {
    const int nt = terms_estimate(G);
    const NuAxis &A = G.A, &B = G.B;
    const double grid = (double)A.nf * B.nf * nt * sizeof(double2);
    const double mid = (double)A.n * B.nf * nt * sizeof(double2);
    const int cg = nufft_forward_group((size_t)grid, (size_t)mid, ncoils);
    const double tiles = (double)ceil_div(A.nf - NW + 1, TG) * ceil_div(B.nf - NW + 1, TG);
    const double entries = tiles * (1.0 - std::exp(-m / tiles)) + (double)m / GI_S;
    double blocks = 0.0, linesA = 0.0, linesB = 0.0, lists = 0.0;
    for (int c0 = 0; c0 < ncoils; c0 += cg) {
        const int nc = std::min(cg, ncoils - c0);
        blocks += ceil_div(nc, 8);
        linesA += padded(nt * nc, A.L);
        linesB += padded(nt * nc, B.L);
    }
    for (const NuAxis *X : {&A, &B})
        if (X->kind == AX_FREE) lists += (double)X->n * ceil_div(X->L, 1024);
    return 114.0 + sort_us(m, tiles) + 2.09e-3 * entries * nt * blocks + 3.6e-5 * (double)m * ncoils +
           5.35e-6 * expansion_work(G, nt, m) + 1.17e-5 * A.nf * B.nf * (double)nt * ncoils +
           0.48 * lists + 2.9e-6 * line_work(A, B.nf, linesA) +
           6.4e-6 * line_work(B, A.n, linesB) +
           8.0e-7 * expansion_work(G, nt, (double)A.n * B.n);
}

int nufft_forward(imp_ctx *ctx, const NuGeometry &G, int m, int ncoils, const float *kx,
                  const float *ky, const float *t, const float *x, const float *y,
                  const float *fm, const float *rho_r, const float *rho_i, const float *s_r,
                  const float *s_i, float *d_r, float *d_i) {
    const hipStream_t st = ctx->stream;
    const dim3 b256(256);
    const NuAxis &A = G.A, &B = G.B;
    const float *cA = G.a_is_y ? y : x, *cB = G.a_is_y ? x : y;
    const int nA = A.n, nB = B.n;
    const size_t nvox = (size_t)nA * nB;
    const ProfScope prof(ctx, "nufft_forward");
    NuPass N(ctx, G, m, kx, ky, t);
    IMP_TRY(N.sort(true));
    IMP_TRY(N.expand());
    N.take_tables();
    const size_t col_bytes = (size_t)A.nf * B.nf * N.nt * sizeof(double2);
    const size_t mid_bytes = (size_t)nA * B.nf * N.nt * sizeof(double2);
    const int cg = nufft_forward_group(col_bytes, mid_bytes, ncoils);
    Carver &W = N.W;
    constexpr int NX = NW + 2 * (TG - 1);
    const int ntx = ceil_div(A.nf - NW + 1, TG), ntile = ntx * ceil_div(B.nf - NW + 1, TG);
    const size_t o_bx = W.take((size_t)m * 4), o_by = W.take((size_t)m * 4);
    const size_t o_wx = W.take((size_t)m * NX * 8), o_wy = W.take((size_t)m * NX * 8);
    const size_t o_u = W.take((size_t)m * N.nt * 8), o_rot = W.take((size_t)m * sizeof(double2));
    const size_t o_cnt = W.take(256);
    const size_t o_ent = W.take(((size_t)ntile + m / GI_S + 1) * sizeof(GiEntry));
    size_t o_f[2], o_l[2], o_lw[2];
    for (int a = 0; a < 2; ++a) {
        const NuAxis &X = a ? B : A;
        o_f[a] = W.take(((size_t)X.L + 1) * 4);
        o_l[a] = W.take((size_t)X.n * (NW + 1) * 4);
        o_lw[a] = W.take((size_t)X.n * (NW + 1) * 8);
    }
    const size_t o_vt = W.take((size_t)N.nt * nvox * 8);
    const size_t o_sens = W.take(s_r ? (size_t)ncoils * nvox * sizeof(float2) : 0);
    const size_t o_img0 = W.take(nvox * sizeof(double2));
    const size_t o_mid = W.take(mid_bytes * cg);
    const size_t o_grid = W.take(col_bytes * cg);
    IMP_TRY(N.alloc(cA, 1, cB, nA));
    hipLaunchKernelGGL(k_nu_starts, dim3(1), b256, 0, st, m, N.key, -1, (int *)nullptr,
                       N.at<int *>(o_cnt), 1);
    hipLaunchKernelGGL(k_gi_list, dim3(ceil_div(ntile, 255)), b256, 0, st, m, ntile, N.key,
                       N.at<GiEntry *>(o_ent), N.at<int *>(o_cnt));
    hipLaunchKernelGGL(k_gi_prep, dim3(ceil_div(m, PREP_S)), b256, 0, st, m, N.perm, N.kA, N.kB,
                       t, A, B, G.tc, G.th > 0.0 ? 1.0 / G.th : 0.0, G.wc / (2.0 * M_PI),
                       N.coef(), N.coef() + N.tab_poly, N.nt, N.nleg, N.at<int *>(o_bx),
                       N.at<int *>(o_by), N.at<double *>(o_wx), N.at<double *>(o_wy),
                       N.at<double *>(o_u), N.at<double2 *>(o_rot));
    if (A.kind == AX_FREE || B.kind == AX_FREE) {
        FListTab ft[2];
        for (int a = 0; a < 2; ++a)
            ft[a] = FListTab{a ? B : A, a ? cB : cA, a ? nA : 1, N.at<int *>(o_f[a]),
                             N.at<int *>(o_l[a]), N.at<double *>(o_lw[a])};
        hipLaunchKernelGGL(k_nu_flists, dim3(2), dim3(1024), 0, st, ft[0], ft[1]);
    }
    hipLaunchKernelGGL(k_nu_vt, dim3(ceil_div((long)nvox, 256), N.nt), b256, 0, st, nA, nB, fm,
                       G.wc, G.wh > 0.0 ? 1.0 / G.wh : 0.0, N.nt, N.coef(), N.mul(), N.nleg,
                       N.at<double *>(o_vt));
    if (s_r)
        hipLaunchKernelGGL(k_nu_sens, dim3(ceil_div(nA, 32), ceil_div(nB, 32), ncoils), b256, 0,
                           st, nA, nB, s_r, s_i, N.at<float2 *>(o_sens));
    hipLaunchKernelGGL(k_nu_img0, dim3(ceil_div(nA, 16), ceil_div(nB, 16)), b256, 0, st, nA, nB,
                       rho_r, rho_i, cA, cB, fm, A.kc, B.kc, G.tc / (2.0 * M_PI),
                       N.at<double2 *>(o_img0));
    IMP_CHECK_LAUNCH();
    for (int c0 = 0; c0 < ncoils; c0 += cg) {
        const int nc = std::min(cg, ncoils - c0), nq = N.nt * nc;
        // B axis: lines ia -> mid[gB][ia][q]; A axis: lines gB -> grid[gB][gA][q]
        LineArgs LB = N.line(1, nullptr, 0, 0, nq);
        LB.base = N.at<const int *>(o_f[1]);
        IMP_TRY(line_forward(ctx, LB, nA, true, N.at<const int *>(o_l[1]),
                             N.at<const double *>(o_lw[1]), nc, N.at<const double2 *>(o_img0),
                             s_r ? N.at<const float2 *>(o_sens) + (size_t)c0 * nvox : nullptr,
                             N.at<const double *>(o_vt), (unsigned)nvox, N.at<double2 *>(o_mid),
                             nq, (unsigned)(nA * nq)));
        LineArgs LA = N.line(0, N.ws + o_mid, (size_t)nA * nq, nq, nq);
        LA.base = N.at<const int *>(o_f[0]);
        IMP_TRY(line_forward(ctx, LA, B.nf, false, N.at<const int *>(o_l[0]),
                             N.at<const double *>(o_lw[0]), nc, nullptr, nullptr, nullptr, 0u,
                             N.at<double2 *>(o_grid), (size_t)A.nf * nq, nq));
        GiArgs P{};
        P.ntx = ntx;
        P.nfA = A.nf;
        P.nfB = B.nf;
        P.nt = N.nt;
        P.nc = nc;
        P.c0 = c0;
        P.m = m;
        P.perm = N.perm;
        P.bx = N.at<const int *>(o_bx);
        P.by = N.at<const int *>(o_by);
        P.wx = N.at<const double *>(o_wx);
        P.wy = N.at<const double *>(o_wy);
        P.u = N.at<const double *>(o_u);
        P.rot = N.at<const double2 *>(o_rot);
        P.count = N.at<const int *>(o_cnt);
        P.entries = N.at<const GiEntry *>(o_ent);
        P.grid = N.at<const double *>(o_grid);
        P.d_r = d_r;
        P.d_i = d_i;
        const int cb = ceil_div(nc, 8);
        auto fn = cb == 1 ? k_gather<1> : cb == 2 ? k_gather<2> : cb == 3 ? k_gather<3>
                                                                           : k_gather<4>;
        const int rg = prof_begin(ctx, "k_gather");
        hipLaunchKernelGGL(fn, dim3(std::min(ntile + m / GI_S + 1, 64 * ctx->num_cus)), dim3(64),
                           0, st, P);
        prof_end(ctx, rg);
        IMP_CHECK_LAUNCH();
    }
    return N.finish();
}

// ------------------------------------------------------------------------ Q_l
// Q_l(r) = sum_k a_l(t_k) |phi_k|^2 e^{i 2pi k.r} on the standard grid
// r = (ix/Nx, iy/Ny), |ix| <= Nx, |iy| <= Ny.  The weights are real, so
// segments 2c and 2c + 1 share a column: with w = a_2c + i a_(2c+1) the
// column's sum is P = Q_2c + i Q_(2c+1), and Q_l(-r) = conj(Q_l(r)) gives
// Q_2c = (P(r) + conj(P(-r))) / 2, Q_(2c+1) = (P(r) - conj(P(-r))) / 2i, so
// Q_l comes out conjugate-symmetric bit for bit.
// Against the GEMM over phasor tables (toeplitz_q_sep) it is closer to 64 bits
// (2.6e-8 against 1.1e-7) and faster wherever samples are not few for the grid
// (16^2 x 500 samples, L = 10: 0.27 -> 0.16 ms; 512^2 x 393216, L = 10: 16 -> 1.07
// ms, and 255 in a process where the 9 GB of tables made on each call came
// slowly); the GEMM's time is in the samples: 700^2 x 500, L = 31: 0.75 ms
// against 3.9.  Price within 17% rms of 136 calls, 16^2 to 1300^2, 500 to 10^6
// samples, L = 3 to 31.
double nufft_q_us(const NuGeometry &G, int m, int nseg) {
    const int cols = (nseg + 1) / 2, cg = column_group(G, 1, cols);
    const SpreadSplit sp = spread_split(1, log2i(cg));
    const double prep = 2 * NW + 2 * (sp.T - 1) + 2 * (sp.yg - 1) + 1 + 2.0 * cg;
    return 151.0 + sort_us(m, cells(G.A, G.B)) + m * (2.17e-6 * sp.cost + 1.49e-5 * prep) +
           1.39e-5 * G.A.nf * G.B.nf * (double)cols +
           1.32e-5 * (line_work(G.A, G.B.nf, padded(cols, G.A.L)) +
                      line_work(G.B, G.A.n, padded(cols, G.B.L)));
}
namespace {

// [sample][slot] = (a_2c, a_(2c+1)) |phi|^2, a_l the Hanning interpolator of
// hanning_d (computeQ.cmem.cu:125-138); 2^lc slots, m of them may pass 2^31
__global__ void k_nu_qdata(int m, int nseg, int lc, const float *t, const float *phi_r,
                           const float *phi_i, float tau, float t0, double2 *wd) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)m << lc) return;
    const int j = (int)(i >> lc), c = (int)(i & ((1 << lc) - 1));
    double mag = 1.0;
    if (phi_r) {
        const double pr = phi_r[j], pi = phi_i[j];
        mag = pr * pr + pi * pi;
    }
    double w[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int l = 2 * c + h;
        const double arg = (double)t[j] - (double)tau * l - (double)t0;
        w[h] = l < nseg && fabs(arg) < (double)tau
                   ? (0.5 + 0.5 * cospi(arg / (double)tau)) * mag : 0.0;
    }
    wd[i] = make_double2(w[0], w[1]);
}

// P[ib][ia][c] (both edges of each axis kept) -> Q_l [iy][ix] without the far
// edges; cumulative: prefix sums over l
__global__ __launch_bounds__(256) void k_nu_qout(int Nx, int Ny, int nc, int nseg,
                                                 int cumulative, const double2 *P, double kcx,
                                                 double kcy, float *q_r, float *q_i) {
    const int ix = blockIdx.x * 256 + threadIdx.x, iy = blockIdx.y;
    if (ix >= 2 * Nx) return;
    const int nx = 2 * Nx + 1, ny = 2 * Ny + 1;
    const double2 *a = P + ((size_t)iy * nx + ix) * nc;
    const double2 *b = P + ((size_t)(ny - 1 - iy) * nx + (nx - 1 - ix)) * nc;
    const double rev = kcx * (ix - Nx) / Nx + kcy * (iy - Ny) / Ny;
    double s, c;
    sincospi(2.0 * (rev - rint(rev)), &s, &c);
    const double2 e = make_double2(0.5 * c, 0.5 * s);
    const size_t nq = (size_t)4 * Nx * Ny, o = (size_t)iy * 2 * Nx + ix;
    double2 run = make_double2(0.0, 0.0);
    for (int q = 0; q < nc; ++q) {
        const double2 p = a[q], r = b[q];
        const double2 v[2] = {cmul(make_double2(p.x + r.x, p.y - r.y), e),
                              cmul(make_double2(p.y + r.y, r.x - p.x), e)};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int l = 2 * q + h;
            if (l >= nseg) break;
            run = cumulative ? make_double2(run.x + v[h].x, run.y + v[h].y) : v[h];
            q_r[(size_t)l * nq + o] = (float)run.x;
            q_i[(size_t)l * nq + o] = (float)run.y;
        }
    }
}

}  // namespace

// Geometry of Q on the standard (Nx, Ny) grid; ok = false when it does not fit.
int nufft_q_geometry(imp_ctx *ctx, int m, const float *kx, const float *ky, const float *t, int Nx,
                     int Ny, int nseg, NuGeometry *G) {
    G->ok = false;
    unsigned h[G_WORDS];
    IMP_TRY(geo_scan(ctx, m, 0, kx, ky, t, nullptr, nullptr, nullptr, nullptr, h));
    if (h[G_KFLAG]) return IMP_OK;
    for (int a = 0; a < 2; ++a) {
        NuAxis &X = a ? G->B : G->A;
        const int N = a ? Ny : Nx;
        if (!plan_axis(2 * N + 1, -1.f, 1.f, 0.f, -1.f, 1.f, dec_f(h[G_MIN + a]),
                       dec_f(h[G_MAX + a]), &X))
            return IMP_OK;
        X.xc = 0.0;
        X.inv_d = (double)X.L / N;   // exactly, as the grid defines it
    }
    G->nz = 1;
    G->tc = dec_f(h[G_MIN + 2]);
    G->th = G->wc = G->wh = 0.0;
    G->a_is_y = false;
    // all columns in one group
    G->ok = ((size_t)G->A.n * G->B.nf * sizeof(double2) << log2i((nseg + 1) / 2)) <= NU_MID_BYTES;
    return IMP_OK;
}

int nufft_q(imp_ctx *ctx, const NuGeometry &G, int m, const float *kx, const float *ky,
            const float *t, const float *phi_r, const float *phi_i, int Nx, int Ny, int nseg,
            float tau, float t0, bool cumulative, float *q_r, float *q_i) {
    const hipStream_t st = ctx->stream;
    const ProfScope prof(ctx, "nufft_q");
    const int cols = (nseg + 1) / 2;
    NuPass N(ctx, G, m, kx, ky, t);
    IMP_TRY(N.sort());
    IMP_TRY(N.layout(cols));
    const size_t o_p = N.W.take((size_t)G.A.n * G.B.n * cols * sizeof(double2));
    IMP_TRY(N.build(nullptr, 1, nullptr, 1));
    if (N.groups != 1) return fail(IMP_EINVAL, "toeplitz_q: %d column groups", N.groups);
    hipLaunchKernelGGL(k_nu_qdata, dim3(ceil_div((long)m << N.lc, 256)), dim3(256), 0, st, m, nseg,
                       N.lc, t, phi_r, phi_i, tau, t0, N.at<double2 *>(N.o_wd));
    IMP_TRY(N.to_mid(cols));
    IMP_TRY(line_store(ctx, N.lines_b(cols), G.A.n, N.at<double2 *>(o_p), cols,
                       (size_t)G.A.n * cols));
    hipLaunchKernelGGL(k_nu_qout, dim3(ceil_div(2 * Nx, 256), 2 * Ny), dim3(256), 0, st, Nx, Ny,
                       cols, nseg, cumulative ? 1 : 0, N.at<const double2 *>(o_p), G.A.kc, G.B.kc,
                       q_r, q_i);
    IMP_CHECK_LAUNCH();
    return N.finish();
}

}  // namespace imp
