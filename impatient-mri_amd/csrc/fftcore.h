// Register-staged Stockham FFT building blocks for gfx950.
//
// A length-L line is transformed by T = L / E threads that each hold E = 16
// values (E = L for L < 16).  Stage s uses radix R_s from a fixed plan
// (16 first, then 16 / 8 / 4 / 2); every stage gives each thread
// Q / T = L / (R T) butterflies, so a thread always owns E values and the
// element sets it owns before and after a stage follow from (t, b, r)
// alone.  Between stages the values go through LDS; the first stage may read
// global memory directly and the last stage may write it directly.
//
// Stockham step with span NS (product of the earlier radices), Q = L / R:
//   for j in [0, Q): k = j mod NS
//     v[r] = x[j + r Q] * w^(r k L / (NS R)),  w = e^(-+2 pi i / L)
//     y[(j - k) R + k + r NS] = DFT_R(v)[r]
// After the last stage y is the DFT of x in natural order.
#pragma once

#include <hip/hip_runtime.h>

namespace imp {
namespace fftc {

// The butterflies are written once for float2 and double2 lines (the Toeplitz
// passes and the NUDFT's wide-kernel transforms).
template <class C2>
struct scalar_of;
template <>
struct scalar_of<float2> { using type = float; };
template <>
struct scalar_of<double2> { using type = double; };

template <class C2>
__device__ __forceinline__ C2 mk(typename scalar_of<C2>::type x, typename scalar_of<C2>::type y) {
    C2 r;
    r.x = x;
    r.y = y;
    return r;
}
template <class C2>
__device__ __forceinline__ C2 cmul(C2 a, C2 b) {
    return mk<C2>(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
template <class C2>
__device__ __forceinline__ C2 cadd(C2 a, C2 b) { return mk<C2>(a.x + b.x, a.y + b.y); }
template <class C2>
__device__ __forceinline__ C2 csub(C2 a, C2 b) { return mk<C2>(a.x - b.x, a.y - b.y); }
// multiply by -i (forward) or +i (inverse)
template <bool INV, class C2>
__device__ __forceinline__ C2 rot90(C2 a) {
    return INV ? mk<C2>(-a.y, a.x) : mk<C2>(a.y, -a.x);
}
// multiply by e^(-+ i pi / 4) (forward / inverse)
template <bool INV, class C2>
__device__ __forceinline__ C2 rot45(C2 a) {
    using F = typename scalar_of<C2>::type;
    constexpr F h = (F)0.70710678118654752440;
    return INV ? mk<C2>(h * (a.x - a.y), h * (a.x + a.y)) : mk<C2>(h * (a.x + a.y), h * (a.y - a.x));
}
template <bool INV, class C2>
__device__ __forceinline__ C2 rot135(C2 a) {  // e^(-+ 3 i pi / 4)
    using F = typename scalar_of<C2>::type;
    constexpr F h = (F)0.70710678118654752440;
    return INV ? mk<C2>(-h * (a.x + a.y), h * (a.x - a.y))
               : mk<C2>(h * (a.y - a.x), -h * (a.x + a.y));
}

template <bool INV, class C2>
__device__ __forceinline__ void dft2(C2 *v) {
    const C2 a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
}

template <bool INV, class C2>
__device__ __forceinline__ void dft4(C2 *v) {
    const C2 s02 = cadd(v[0], v[2]), d02 = csub(v[0], v[2]);
    const C2 s13 = cadd(v[1], v[3]), d13 = rot90<INV>(csub(v[1], v[3]));
    v[0] = cadd(s02, s13);
    v[2] = csub(s02, s13);
    v[1] = cadd(d02, d13);
    v[3] = csub(d02, d13);
}

// radix-2 decimation in time: X[k] = E[k] + w^k O[k], X[k + R/2] = E[k] - w^k O[k]
template <bool INV, class C2>
__device__ __forceinline__ void dft8(C2 *v) {
    C2 e[4] = {v[0], v[2], v[4], v[6]};
    C2 o[4] = {v[1], v[3], v[5], v[7]};
    dft4<INV>(e);
    dft4<INV>(o);
    o[1] = rot45<INV>(o[1]);
    o[2] = rot90<INV>(o[2]);
    o[3] = rot135<INV>(o[3]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        v[k] = cadd(e[k], o[k]);
        v[k + 4] = csub(e[k], o[k]);
    }
}

template <bool INV, class C2>
__device__ __forceinline__ void dft16(C2 *v) {
    using F = typename scalar_of<C2>::type;
    // 16 = 4 x 4: DFT-4 over n = a + 4 c (c), twiddle w16^(a k1), DFT-4 over a
    C2 x[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
#pragma unroll
        for (int c = 0; c < 4; ++c) x[a][c] = v[a + 4 * c];
        dft4<INV>(x[a]);  // x[a][k1]
    }
    // twiddles w16^(a k1) for a, k1 in 1..3 (exponents 1, 2, 3, 4, 6, 9);
    // w16^m = cos(pi m / 8) -+ i sin(pi m / 8)
    constexpr F c1 = (F)0.92387953251128675613, s1 = (F)0.38268343236508977173;
    constexpr F sg = INV ? (F)1 : (F)-1;
    const C2 w1 = mk<C2>(c1, sg * s1), w3 = mk<C2>(s1, sg * c1), w9 = mk<C2>(-c1, -sg * s1);
    x[1][1] = cmul(x[1][1], w1);
    x[1][2] = rot45<INV>(x[1][2]);
    x[1][3] = cmul(x[1][3], w3);
    x[2][1] = rot45<INV>(x[2][1]);
    x[2][2] = rot90<INV>(x[2][2]);
    x[2][3] = rot135<INV>(x[2][3]);
    x[3][1] = cmul(x[3][1], w3);
    x[3][2] = rot135<INV>(x[3][2]);
    x[3][3] = cmul(x[3][3], w9);
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
        C2 y[4] = {x[0][k1], x[1][k1], x[2][k1], x[3][k1]};
        dft4<INV>(y);
#pragma unroll
        for (int k2 = 0; k2 < 4; ++k2) v[k1 + 4 * k2] = y[k2];
    }
}

template <bool INV, class C2>
__device__ __forceinline__ void dft3(C2 *v) {
    using F = typename scalar_of<C2>::type;
    constexpr F r3 = (F)0.86602540378443864676;  // sqrt(3) / 2
    const C2 s = cadd(v[1], v[2]);
    const C2 d = rot90<INV>(csub(v[1], v[2]));
    const C2 t = mk<C2>(v[0].x - (F)0.5 * s.x, v[0].y - (F)0.5 * s.y);
    v[0] = cadd(v[0], s);
    v[1] = mk<C2>(t.x + r3 * d.x, t.y + r3 * d.y);
    v[2] = mk<C2>(t.x - r3 * d.x, t.y - r3 * d.y);
}

template <bool INV, class C2>
__device__ __forceinline__ void dft12(C2 *v) {
    using F = typename scalar_of<C2>::type;
    // 12 = 4 x 3: DFT-3 over n = a + 4 c (c), twiddle w12^(a k1), DFT-4 over a;
    // output k = k1 + 3 k2
    C2 x[4][3];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
#pragma unroll
        for (int c = 0; c < 3; ++c) x[a][c] = v[a + 4 * c];
        dft3<INV>(x[a]);
    }
    // w12^m = cos(pi m / 6) -+ i sin(pi m / 6), m = a k1 in {1, 2, 2, 4, 3, 6}
    constexpr F r3 = (F)0.86602540378443864676;
    constexpr F sg = INV ? (F)1 : (F)-1, hf = (F)0.5;
    const C2 w1 = mk<C2>(r3, sg * hf), w2 = mk<C2>(hf, sg * r3), w4 = mk<C2>(-hf, sg * r3);
    x[1][1] = cmul(x[1][1], w1);
    x[1][2] = cmul(x[1][2], w2);
    x[2][1] = cmul(x[2][1], w2);
    x[2][2] = cmul(x[2][2], w4);
    x[3][1] = rot90<INV>(x[3][1]);
    x[3][2] = mk<C2>(-x[3][2].x, -x[3][2].y);
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
        C2 y[4] = {x[0][k1], x[1][k1], x[2][k1], x[3][k1]};
        dft4<INV>(y);
#pragma unroll
        for (int k2 = 0; k2 < 4; ++k2) v[k1 + 3 * k2] = y[k2];
    }
}

// In-register DFT of size R in natural order: v[k] <- sum_n v[n] w^(nk),
// w = e^(-2 pi i / R) (forward) or e^(+2 pi i / R) (inverse).
template <int R, bool INV, class C2>
__device__ __forceinline__ void dft(C2 *v) {
    static_assert(R == 1 || R == 2 || R == 3 || R == 4 || R == 8 || R == 12 || R == 16, "radix");
    if constexpr (R == 2) dft2<INV>(v);
    if constexpr (R == 3) dft3<INV>(v);
    if constexpr (R == 4) dft4<INV>(v);
    if constexpr (R == 8) dft8<INV>(v);
    if constexpr (R == 12) dft12<INV>(v);
    if constexpr (R == 16) dft16<INV>(v);
}

// ------------------------------------------------------------------ plans
// Supported lengths: 2^k (2..4096) and 3 * 2^k (12..3072).
// Powers of two: E = 16 values per thread (E = L below 16), radix 16 while
// at least 4 bits remain, then the rest (2, 4, 8 or 16).
// Lengths 3 * 2^k: E = 12, a radix-12 stage first, then radix 4, and a
// final radix 2 when an odd power of two remains; every radix divides 12,
// so each stage gives each of the T = L / 12 threads whole butterflies.
__host__ __device__ constexpr int ilog2c(int n) { return n <= 1 ? 0 : 1 + ilog2c(n / 2); }
__host__ __device__ constexpr bool has3(int L) { return L % 3 == 0; }
__host__ __device__ constexpr int vals_per_thread(int L) {
    return has3(L) ? (L < 12 ? L : 12) : (L < 16 ? L : 16);
}
__host__ __device__ constexpr int threads_per_line(int L) { return L / vals_per_thread(L); }
// Threads per workgroup of the row-transform passes: 512 (8 lines of 1024
// points, whose LDS twiddle table then still leaves two workgroups per CU)
// from 512-point lines up, 256 below.
__host__ __device__ constexpr int row_threads(int L) { return L >= 512 ? 512 : 256; }
__host__ __device__ constexpr int num_stages(int L) {
    return has3(L) ? (L <= 12 ? 1 : 1 + (ilog2c(L / 12) + 1) / 2)
                   : (L <= 16 ? 1 : (ilog2c(L) + 3) / 4);
}
__host__ __device__ constexpr int stage_radix(int L, int s) {
    return has3(L) ? (L <= 12 ? L : (s == 0 ? 12 : (ilog2c(L / 12) - 2 * (s - 1) >= 2 ? 4 : 2)))
                   : (L <= 16 ? L : (s + 1 < num_stages(L) ? 16 : (1 << (ilog2c(L) - 4 * s))));
}
__host__ __device__ constexpr int stage_span(int L, int s) {  // NS: product of earlier radices
    return s == 0 ? 1 : stage_span(L, s - 1) * stage_radix(L, s - 1);
}
__host__ __device__ constexpr bool fft_length_supported(int L) {
    return L >= 2 && (has3(L) ? (L >= 12 && L <= 3072 && ((L / 3) & (L / 3 - 1)) == 0)
                              : (L <= 4096 && (L & (L - 1)) == 0));
}

// LDS index of element i of a line: one pad word every 16 elements keeps the
// strided stage writes within two-way bank conflicts.
__device__ __forceinline__ int lpad(int i) { return i + (i >> 4); }
__host__ __device__ constexpr int line_lds(int L) { return L + L / 16; }

// One Stockham stage for the thread with line-local index t.  LD(b, r, i)
// returns input element i (= j + r Q, j = t + T b); ST(b, r, i, v) stores
// output element i; b and r are compile-time after unrolling.  Twiddles come
// from tw[m] = exp(-2 pi i m / L).
//   FUSED = false: every load and butterfly of the thread, then MID() (a
//                  barrier when the stage reads and writes the same LDS
//                  lines), then every store.
//   FUSED = true:  MID() first, then load / butterfly / store one butterfly
//                  at a time (loads and stores must not alias); keeps fewer
//                  values live.
template <int L, int S, bool INV, bool FUSED, class LD, class MID, class ST>
__device__ __forceinline__ void stage(int t, const float2 *__restrict__ tw, LD ld, MID mid,
                                      ST st) {
    constexpr int R = stage_radix(L, S);
    constexpr int NS = stage_span(L, S);
    constexpr int T = threads_per_line(L);
    constexpr int Q = L / R;
    constexpr int NB = Q / T;
    static_assert(NB >= 1 && Q % T == 0, "radix plan does not fit the thread layout");
    auto butterfly = [&](int b, float2 *v) {
        const int j = t + T * b;
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = ld(b, r, j + r * Q);
        if constexpr (NS > 1) {
            const int k = j % NS;
            const int step = (L / (NS * R)) * k;
#pragma unroll
            for (int r = 1; r < R; ++r) {
                float2 w = tw[r * step];
                if (INV) w.y = -w.y;
                v[r] = cmul(v[r], w);
            }
        }
        dft<R, INV>(v);
    };
    auto store = [&](int b, const float2 *v) {
        const int j = t + T * b;
        const int k = NS > 1 ? j % NS : 0;
#pragma unroll
        for (int r = 0; r < R; ++r) st(b, r, (j - k) * R + k + r * NS, v[r]);
    };
    if constexpr (FUSED) {
        mid();
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            float2 v[R];
            butterfly(b, v);
            store(b, v);
        }
    } else {
        float2 v[NB][R];
#pragma unroll
        for (int b = 0; b < NB; ++b) butterfly(b, v[b]);
        mid();
#pragma unroll
        for (int b = 0; b < NB; ++b) store(b, v[b]);
    }
}

// Register index m of output element i after the last stage (i = t + T m).
template <int L>
__host__ __device__ constexpr int last_reg(int b, int r) {
    return b + (L / (stage_radix(L, num_stages(L) - 1) * threads_per_line(L))) * r;
}
// Register index m of input element i of the first stage (i = t + T m).
template <int L>
__host__ __device__ constexpr int first_reg(int b, int r) {
    return b + (L / (stage_radix(L, 0) * threads_per_line(L))) * r;
}

}  // namespace fftc
}  // namespace imp
