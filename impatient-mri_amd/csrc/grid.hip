// Gridding path of the Toeplitz method (-toeplitzGridding): Q_l and F^H d
// by Kaiser-Bessel gridding onto an oversampled Cartesian grid and a shifted,
// centre-cropped inverse DFT, as computeQ_GPU_Grid / computeFH_GPU_Grid do
// (toeplitz/computeQ.cmem.cu:401-754, computeFH.cmem.cu:470-802,
// 1032-1117; binning and gather in CUDA_interface.cu:26-400 and
// GPU_kernels.cu:68-581; crop, deapodization and shifts in
// gridding_utils.cu:6-290).
//
// The estimate per transform, for samples k_j (cycles of an n-point image
// axis) with weights v_j:
//   1. s_j = os (k_j + n/2) per axis; grid point g in [0, G) receives
//      v_j prod_axes KB(|s_j - g| / os) for |s_j - g| / os <= W/2 (W = 4),
//      KB(d) = I0(beta sqrt(1 - (2d/W)^2)) / W; the grid does not wrap;
//   2. out(i) = sum_g grid(g) e^{+i 2pi (g - G/2)(i - n/2) / G} per axis
//      (ifftshift, unnormalised inverse FFT, fftshift, centre crop);
//   3. out(i) /= os C(u_i) per axis, C the kernel's transform at
//      u_i = (i - n/2)/n.
//
// This build's structure:
//   - samples are sorted by grid cell (a stable radix sort, so each cell's
//     samples stay in index order), so each grid point gathers from
//     contiguous sample ranges with no atomics on the grid;
//   - one gather launch grids every coil of a segment at once (each sample's
//     kernel weight serves all coils); 2D grids of many coils in tiles of
//     points whose lanes are coils, with the coils innermost up to the sum over
//     them;
//   - the DFT of step 2 runs per axis on lines of length G = R P (P the
//     largest power of two dividing G): R radix-2 FFTs of length P in LDS,
//     then the R-term combination evaluated only at the n kept outputs, with
//     step 3 folded in; every pass writes its output with the transformed
//     axis outermost, so after one pass per axis the layout is the image's.
#include <algorithm>
#include <cmath>
#include <vector>

#include "common.h"
#include "fftcore.h"
#include "toeplitz.h"

namespace imp {

namespace {

constexpr float KB_WIDTH = 4.0f;
constexpr int GT = 256;

// I0(x), x >= 0, by the polynomial approximations of Abramowitz & Stegun,
// Handbook of Mathematical Functions, 9.8.1 (|err| < 1.6e-7 for x <= 3.75)
// and 9.8.2 (relative error < 1.9e-7 above).
__device__ __forceinline__ float bessel_i0(float x) {
    if (x < 3.75f) {
        float y = x * (1.0f / 3.75f);
        y *= y;
        return 1.0f + y * (3.5156229f + y * (3.0899424f + y * (1.2067492f + y * (0.2659732f +
                     y * (0.0360768f + y * 0.0045813f)))));
    }
    const float y = 3.75f / x;
    const float p = 0.39894228f + y * (0.01328592f + y * (0.00225319f + y * (-0.00157565f +
                    y * (0.00916281f + y * (-0.02057706f + y * (0.02635537f +
                    y * (-0.01647633f + y * 0.00392377f)))))));
    return p * expf(x) * rsqrtf(x);
}

// KB(d) = I0(beta sqrt(1 - (2d/W)^2)) / W for d = |s - g| / os <= W/2, else 0
__device__ __forceinline__ float kb_weight(float s, int g, float inv_os, float beta) {
    const float d = fabsf(s - (float)g) * inv_os;
    if (!(d <= 0.5f * KB_WIDTH)) return 0.f;
    const float u = 2.0f * d * (1.0f / KB_WIDTH);
    return bessel_i0(beta * sqrtf(fmaxf(1.0f - u * u, 0.0f))) * (1.0f / KB_WIDTH);
}

struct GridGeom {
    int G[3];        // grid size per axis (x, y, z); G[2] = 1 in 2D
    int n[3];        // image size per axis
    float os, inv_os, half, beta;
    int d3;
};

// shifted positions s = os (k + n/2) (float, as the reference computes them),
// and the sort key of every sample: its time bucket b (segment l weighs only
// buckets l and l + 1; b = floor((t - t0)/tau) + 1 clamped to [0, nseg]) and
// its grid cell ((cy Gx) + cx) Gz + cz, as b ncells + cell
__global__ void k_grid_cells(int m, const float *kx, const float *ky, const float *kz,
                             const float *t, float kscale, GridGeom g, float t0, float tau,
                             int nseg, float4 *pos, int *key, int *count) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= m) return;
    const float sx = g.os * (kscale * kx[j] + (float)g.n[0] / 2.0f);
    const float sy = g.os * (kscale * ky[j] + (float)g.n[1] / 2.0f);
    const float sz = g.d3 ? g.os * (kscale * kz[j] + (float)g.n[2] / 2.0f) : 0.f;
    const int cx = min(g.G[0] - 1, max(0, (int)floorf(sx)));
    const int cy = min(g.G[1] - 1, max(0, (int)floorf(sy)));
    const int cz = g.d3 ? min(g.G[2] - 1, max(0, (int)floorf(sz))) : 0;
    const int c = ((cy * g.G[0]) + cx) * g.G[2] + cz;
    int b = 0;
    if (tau > 0.f) {
        const double f = floor(((double)t[j] - (double)t0) / (double)tau);
        b = (int)fmin(fmax(f + 1.0, 0.0), (double)nseg);
    }
    const long ncells = (long)g.G[0] * g.G[1] * g.G[2];
    const int k = (int)(b * ncells + c);
    pos[j] = make_float4(sx, sy, sz, 0.f);
    key[j] = k;
    atomicAdd(&count[k], 1);
}

// exclusive scan of n ints in three launches: per-block scans with block
// totals, a scan of the totals by one workgroup, then the block offsets
__global__ __launch_bounds__(GT) void k_scan_blocks(const int *in, int n, int *out,
                                                    int *block_sum) {
    __shared__ int sm[GT];
    const int base = blockIdx.x * GT * 4;
    int v[4], s = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int i = base + threadIdx.x * 4 + e;
        v[e] = i < n ? in[i] : 0;
        s += v[e];
    }
    sm[threadIdx.x] = s;
    __syncthreads();
    for (int off = 1; off < GT; off <<= 1) {
        const int t = threadIdx.x >= off ? sm[threadIdx.x - off] : 0;
        __syncthreads();
        sm[threadIdx.x] += t;
        __syncthreads();
    }
    int run = sm[threadIdx.x] - s;   // exclusive prefix of this thread
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int i = base + threadIdx.x * 4 + e;
        if (i < n) out[i] = run;
        run += v[e];
    }
    if (threadIdx.x == GT - 1) block_sum[blockIdx.x] = sm[GT - 1];
}

__global__ __launch_bounds__(GT) void k_scan_totals(int *block_sum, int nb, int *total) {
    __shared__ int sm[GT];
    int carry = 0;
    for (int b0 = 0; b0 < nb; b0 += GT) {
        const int i = b0 + threadIdx.x;
        const int v = i < nb ? block_sum[i] : 0;
        sm[threadIdx.x] = v;
        __syncthreads();
        for (int off = 1; off < GT; off <<= 1) {
            const int t = threadIdx.x >= off ? sm[threadIdx.x - off] : 0;
            __syncthreads();
            sm[threadIdx.x] += t;
            __syncthreads();
        }
        if (i < nb) block_sum[i] = carry + sm[threadIdx.x] - v;
        const int tot = sm[GT - 1];
        __syncthreads();
        carry += tot;
    }
    if (threadIdx.x == 0) *total = carry;
}

__global__ void k_scan_add(int *out, int n, const int *block_sum, const int *total) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] += block_sum[i / (GT * 4)];
    if (i == n) out[n] = *total;
}

// Stable sort of the samples by cell (the gather then sums each cell's
// samples in index order, so every run gives the same bits): LSD radix sort
// of (cell, sample index) pairs, 4-bit digits, one element per thread and
// RS_BLOCK elements per workgroup.  Per pass:
//   k_rs_count    digit histogram of each block, stored digit-major
//                 hist[d * nblocks + block];
//   (exclusive scan of hist: every (digit, block) gets its output offset;
//   digits ascending, blocks in order)
//   k_rs_scatter  each element goes to its (digit, block) offset plus the
//                 number of earlier elements of its block with that digit
//                 (wave ballots within a wave, per-wave counts in LDS
//                 across waves), which keeps equal keys in input order.
constexpr int RS_BLOCK = 256;
constexpr int RS_WAVES = RS_BLOCK / 64;
constexpr int RS_BINS = 16;

__global__ __launch_bounds__(RS_BLOCK) void k_rs_count(const int *__restrict__ key, int m,
                                                       int shift, int nblocks,
                                                       int *__restrict__ hist) {
    __shared__ int cnt[RS_BINS];
    if (threadIdx.x < RS_BINS) cnt[threadIdx.x] = 0;
    __syncthreads();
    const int i = blockIdx.x * RS_BLOCK + threadIdx.x;
    if (i < m) atomicAdd(&cnt[(key[i] >> shift) & (RS_BINS - 1)], 1);
    __syncthreads();
    if (threadIdx.x < RS_BINS) hist[threadIdx.x * nblocks + blockIdx.x] = cnt[threadIdx.x];
}

__global__ __launch_bounds__(RS_BLOCK) void k_rs_scatter(const int *__restrict__ key_in,
                                                         const int *__restrict__ val_in, int m,
                                                         int shift, int nblocks,
                                                         const int *__restrict__ offs,
                                                         int *__restrict__ key_out,
                                                         int *__restrict__ val_out) {
    __shared__ int wcnt[RS_WAVES][RS_BINS];
    const int i = blockIdx.x * RS_BLOCK + threadIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool ok = i < m;
    const int k = ok ? key_in[i] : 0;
    const int d = ok ? (k >> shift) & (RS_BINS - 1) : RS_BINS;   // RS_BINS: no element
    const unsigned long long lt = (1ull << lane) - 1ull;
    int rank = 0;
#pragma unroll
    for (int bin = 0; bin < RS_BINS; ++bin) {
        const unsigned long long mk = __ballot(d == bin);
        if (d == bin) rank = __popcll(mk & lt);
        if (lane == 0) wcnt[wave][bin] = __popcll(mk);
    }
    __syncthreads();
    if (!ok) return;
    int before = 0;
    for (int w = 0; w < wave; ++w) before += wcnt[w][d];
    const int dst = offs[d * nblocks + blockIdx.x] + before + rank;
    key_out[dst] = k;
    val_out[dst] = val_in[i];
}

__global__ void k_iota(int m, int *v) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < m) v[i] = i;
}

// segment weights of every sample: a_l(t) is nonzero for at most two
// consecutive l; w.x = a_{l0}, w.y = a_{l0+1}, l0 in pos.w (as int bits).
// hanning_d of computeQ.cmem.cu:125-138 / GPU_kernels.cu:48-62 in FP64.
__global__ void k_grid_samples(int m, const int *perm, const float4 *pos_in, const float *t,
                               int nseg, float tau, float t0, float4 *pos, float2 *w) {
    const int ks = blockIdx.x * blockDim.x + threadIdx.x;
    if (ks >= m) return;
    const int j = perm[ks];
    float4 p = pos_in[j];
    const float tm = t[j];
    float wl[2] = {0.f, 0.f};
    int l0 = 0;
    if (tau > 0.f) {   // tau = 0 (one readout time): hanning_d is 0 everywhere
        l0 = (int)floor(((double)tm - (double)t0) / (double)tau);
        for (int q = 0; q < 2; ++q) {
            const int l = l0 + q;
            if (l < 0 || l >= nseg) continue;
            const float taul = tau * (float)l;
            const float x = tm - taul - t0;
            if (fabsf(x) < tau) wl[q] = (float)(0.5 + 0.5 * cospi((double)x / (double)tau));
        }
    }
    p.w = __int_as_float(l0);
    pos[ks] = p;
    w[ks] = make_float2(wl[0], wl[1]);
}

// coil data in sorted sample order, [ks][C] (unit data when d_r is null)
template <int C>
__global__ void k_grid_data(int m, int ncoils, const int *perm, const float *d_r,
                            const float *d_i, float2 *out) {
    const int ks = blockIdx.x * blockDim.x + threadIdx.x;
    if (ks >= m) return;
    const int j = perm[ks];
#pragma unroll
    for (int c = 0; c < C; ++c)
        out[(size_t)ks * C + c] = c < ncoils ? make_float2(d_r[(size_t)c * m + j],
                                                          d_i[(size_t)c * m + j])
                                             : make_float2(0.f, 0.f);
}

// coil data [m][C] in the samples' own order, 64 samples through LDS (393216
// samples x 32 coils: 41 us; k_grid_data, in sorted order, 275)
template <int C>
__global__ __launch_bounds__(GT) void k_grid_rows(int m, int ncoils, const float *d_r,
                                                  const float *d_i, float2 *out) {
    __shared__ float2 tile[C][65];
    const int j0 = blockIdx.x * 64, j = threadIdx.x & 63, q = threadIdx.x >> 6;
    for (int c = q; c < C; c += GT / 64)
        tile[c][j] = c < ncoils && j0 + j < m
                         ? make_float2(d_r[(size_t)c * m + j0 + j], d_i[(size_t)c * m + j0 + j])
                         : make_float2(0.f, 0.f);
    __syncthreads();
    for (int e = threadIdx.x; e < 64 * C && j0 + e / C < m; e += GT)
        out[(size_t)j0 * C + e] = tile[e % C][e / C];
}

// The window of grid point id ([gy][gx][gz], the innermost cell axis
// fastest): the cells whose samples can lie within W/2 of it.
struct Window {
    int gx, gy, gz, x0, x1, y0, y1, z0, z1;
};

__device__ __forceinline__ Window window_of(const GridGeom &g, long id) {
    Window W;
    if (g.d3) {
        W.gz = (int)(id % g.G[2]);
        W.gx = (int)((id / g.G[2]) % g.G[0]);
        W.gy = (int)(id / ((long)g.G[2] * g.G[0]));
    } else {
        W.gz = 0;
        W.gx = (int)(id % g.G[0]);
        W.gy = (int)(id / g.G[0]);
    }
    const int r_lo = (int)ceilf(g.half), r_hi = (int)floorf(g.half);
    W.y0 = max(0, W.gy - r_lo);
    W.y1 = min(g.G[1] - 1, W.gy + r_hi);
    W.x0 = max(0, W.gx - r_lo);
    W.x1 = min(g.G[0] - 1, W.gx + r_hi);
    W.z0 = g.d3 ? max(0, W.gz - r_lo) : 0;
    W.z1 = g.d3 ? min(g.G[2] - 1, W.gz + r_hi) : 0;
    return W;
}

// f(b, e) for each contiguous sample range [b, e) of the window: per time
// bucket l and l + 1 of segment l, per cell row (y, x) in 3D with z
// contiguous, per row y in 2D with x contiguous
template <class F>
__device__ __forceinline__ void for_ranges(const GridGeom &g, const int *start, int nbuck, int l,
                                           const Window &W, F f) {
    const long total = (long)g.G[0] * g.G[1] * g.G[2];
    const int o1 = g.d3 ? W.x0 : 0, o1e = g.d3 ? W.x1 : 0;
    const int b1 = min(l + 1, nbuck - 1);
    for (int bk = l; bk <= b1; ++bk) {
        const long bbase = (long)bk * total;
        for (int cy = W.y0; cy <= W.y1; ++cy) {
            for (int cx = o1; cx <= o1e; ++cx) {
                if (g.d3) {
                    const long row = bbase + ((long)cy * g.G[0] + cx) * g.G[2];
                    f(start[row + W.z0], start[row + W.z1 + 1]);
                } else {
                    const long row = bbase + (long)cy * g.G[0];
                    f(start[row + W.x0], start[row + W.x1 + 1]);
                }
            }
        }
    }
}

// samples b + off, b + off + stride, ... < e of segment l into the point's sums
template <int C>
__device__ __forceinline__ void accumulate(const GridGeom &g, const Window &W,
                                           const float4 *__restrict__ pos,
                                           const float2 *__restrict__ w,
                                           const float2 *__restrict__ data, int l, int b, int e,
                                           int off, int stride, float *acc_r, float *acc_i) {
    constexpr int NC = C > 0 ? C : 1;
    for (int ks = b + off; ks < e; ks += stride) {
        const float4 p = pos[ks];
        const float2 ww = w[ks];
        const int l0 = __float_as_int(p.w);
        const float a = l == l0 ? ww.x : (l == l0 + 1 ? ww.y : 0.f);
        if (a == 0.f) continue;
        float kw = kb_weight(p.x, W.gx, g.inv_os, g.beta);
        if (kw == 0.f) continue;
        kw *= kb_weight(p.y, W.gy, g.inv_os, g.beta);
        if (g.d3) kw *= kb_weight(p.z, W.gz, g.inv_os, g.beta);
        const float s = kw * a;
        if (C == 0) {
            acc_r[0] += s;
        } else {
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const float2 v = data[(size_t)ks * NC + c];
                acc_r[c] = fmaf(s, v.x, acc_r[c]);
                acc_i[c] = fmaf(s, v.y, acc_i[c]);
            }
        }
    }
}

// a point whose window holds more samples than this is summed by a whole
// wave (k_grid_gather_heavy): near the centre of a variable-density
// trajectory a window holds thousands of samples, and one lane per point
// would leave its wave waiting on that lane
constexpr int GATHER_HEAVY = 64;

// One thread per grid point: sum over the samples within the kernel window
// of segment l (weight a_l), for C coils (C = 0: unit data, one plane).
// Grid layout per coil: [gy][gx][gz], written at grid + c * plane.  Points
// with more than GATHER_HEAVY samples are listed in heavy[] (in any order)
// and left to k_grid_gather_heavy.
template <int C>
__global__ __launch_bounds__(GT) void k_grid_gather(GridGeom g, const int *start, int nbuck,
                                                    const float4 *pos, const float2 *w,
                                                    const float2 *data, int l, float2 *grid,
                                                    size_t plane, int *heavy, int *nheavy) {
    constexpr int NC = C > 0 ? C : 1;
    const long id = (long)blockIdx.x * GT + threadIdx.x;
    const long total = (long)g.G[0] * g.G[1] * g.G[2];
    if (id >= total) return;
    const Window W = window_of(g, id);
    int count = 0;
    for_ranges(g, start, nbuck, l, W, [&](int b, int e) { count += e - b; });
    if (count > GATHER_HEAVY) {
        heavy[atomicAdd(nheavy, 1)] = (int)id;
        return;
    }
    float acc_r[NC], acc_i[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) acc_r[c] = acc_i[c] = 0.f;
    for_ranges(g, start, nbuck, l, W, [&](int b, int e) {
        accumulate<C>(g, W, pos, w, data, l, b, e, 0, 1, acc_r, acc_i);
    });
#pragma unroll
    for (int c = 0; c < NC; ++c) grid[c * plane + id] = make_float2(acc_r[c], acc_i[c]);
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// The listed points, one wave each: lane k sums the window's samples
// k, k + 64, ... of every range, then a fixed butterfly adds the lanes, so
// the result does not depend on which wave takes the point.  Waves stride
// over the list; every wave reads the same count and ends.
template <int C>
__global__ __launch_bounds__(GT) void k_grid_gather_heavy(GridGeom g, const int *start, int nbuck,
                                                          const float4 *pos, const float2 *w,
                                                          const float2 *data, int l,
                                                          float2 *grid, size_t plane,
                                                          const int *heavy,
                                                          const int *nheavy) {
    constexpr int NC = C > 0 ? C : 1;
    const int lane = threadIdx.x & 63;
    const int wave = (int)((blockIdx.x * GT + threadIdx.x) >> 6);
    const int nwaves = (int)(gridDim.x * (GT / 64));
    const int n = *nheavy;
    for (int it = wave; it < n; it += nwaves) {
        const long id = heavy[it];
        const Window W = window_of(g, id);
        float acc_r[NC], acc_i[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) acc_r[c] = acc_i[c] = 0.f;
        for_ranges(g, start, nbuck, l, W, [&](int b, int e) {
            accumulate<C>(g, W, pos, w, data, l, b, e, lane, 64, acc_r, acc_i);
        });
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            acc_r[c] = wave_sum(acc_r[c]);
            acc_i[c] = wave_sum(acc_i[c]);
        }
        if (lane == 0) {
#pragma unroll
            for (int c = 0; c < NC; ++c) grid[c * plane + id] = make_float2(acc_r[c], acc_i[c]);
        }
    }
}

// Tiles of 2D grid points, C coils side by side, grid[gy][gx][coil].  Lanes are
// coils x sub-tiles of 4 x 4 points, whose sums stay in registers.  The samples
// of the cells around the tile (few contiguous ranges) go in batches of 64: lane
// v computes the kernel weights of sample v at the tile's columns and rows, all
// lanes then run over the samples with the next TL_PF samples' data on their
// way.  A tile of more than H.heavy samples is listed (by the first launch, of
// one wave per tile) and summed by TL_WAVES waves, added in a fixed order; one of
// more than TL_PART (the centre of a variable-density trajectory) by several
// such workgroups, whose sums k_grid_tiles_sum adds.
//
// One thread per point, as below, evaluates a weight for each pair of point and
// sample and waits on the sample's 32 coils each time.  512^2 x 32 coils, grid
// 704^2, 11 segments of 393216 samples: gathers 4.31 ms -> 1.27 ms.  TL_WAVES 4, 8,
// 16: 2.99, 1.67, 1.33 ms for the listed tiles (before they were parted);
// TL_HEAVY 128, 256, 512, 1024: 0.64, 0.87, 1.15, 1.54 ms for the others.
//
// Few samples leave few tiles that are long, and the launch waits for the waves
// that sum 200 of them: up to TL_FEW samples a tile is listed above TL_LOW. Whole
// calls of 3 coils, 16000 samples, os 1.5, one thread per point / 256 / 64: 64^2
// 662 / 739 / 530 us, 96^2 682 / 767 / 580. At 64 from 160000 samples on: 0.9 to
// 1.8 times the time at 256.
constexpr int TL_PF = 4, TL_HEAVY = 256, TL_LOW = 64, TL_FEW = 40000, TL_WAVES = 16,
              TL_PART = 2048;
struct TileList {
    int4 *entries;    // tile, part, parts, slot
    int4 *multis;     // tile, parts, first slot
    int *count;       // entries, slots, multis
    float2 *slots;    // [slot][16][64]
    int heavy;        // samples above which a tile is listed
};
template <int C>
struct Tile {
    static constexpr int SUB = 64 / C, SX = SUB >= 8 ? 4 : 2, SY = SUB / SX;
    static constexpr int TX = 4 * SX, TY = 4 * SY;
};

template <int C>
__device__ __forceinline__ void tile_store(const GridGeom &g, int gx0, int gy0, int lane,
                                           const float2 (&v)[4][4], float2 *grid) {
    const int c = lane & (C - 1), sub = lane / C;
    gx0 += (sub % Tile<C>::SX) * 4;
    gy0 += (sub / Tile<C>::SX) * 4;
#pragma unroll
    for (int y = 0; y < 4; ++y)
#pragma unroll
        for (int x = 0; x < 4; ++x)
            if (gy0 + y < g.G[1] && gx0 + x < g.G[0])
                grid[((size_t)(gy0 + y) * g.G[0] + gx0 + x) * C + c] = v[y][x];
}

template <int C, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void k_grid_tiles(GridGeom g, const int *start,
                                                           int nbuck, const float4 *pos,
                                                           const float2 *w, const int *perm,
                                                           const float2 *data, int l,
                                                           float2 *grid, int ntx,
                                                           TileList H) {
    using TS = Tile<C>;
    constexpr int TX = TS::TX, TY = TS::TY;
    constexpr int FACT = WAVES * 64 * (TX + TY), RED = WAVES > 1 ? WAVES / 2 * 16 * 64 * 2 : 0;
    __shared__ float4 smem[(FACT > RED ? FACT : RED) / 4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float *wx = (float *)smem + wave * 64 * (TX + TY), *wy = wx + 64 * TX;
    const int c = lane & (C - 1), sub = lane / C, px = (sub % TS::SX) * 4, py = (sub / TS::SX) * 4;
    const int r_lo = (int)ceilf(g.half), r_hi = (int)floorf(g.half);
    const int nrow = TY + r_lo + r_hi, nb = min(l + 1, nbuck - 1) - l + 1;
    const int count = WAVES > 1 ? H.count[0] : (int)gridDim.x;
    for (int it = blockIdx.x; it < count; it += gridDim.x) {
        const int4 E = WAVES > 1 ? H.entries[it] : make_int4(it, 0, 1, 0);
        const int tile = E.x;
        const int gx0 = (tile % ntx) * TX, gy0 = (tile / ntx) * TY;
        // lane r: sample range of cell row r of a time bucket (2 nrow <= 64)
        int rs = 0, rn = 0;
        const int cy = gy0 - r_lo + lane % nrow;
        if (lane < nb * nrow && cy >= 0 && cy < g.G[1]) {
            const long row = ((long)(l + lane / nrow) * g.G[1] + cy) * g.G[0];
            rs = start[row + max(0, gx0 - r_lo)];
            rn = start[row + min(g.G[0] - 1, gx0 + TX - 1 + r_hi) + 1] - rs;
        }
        int total = rn;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) total += __shfl_xor(total, off, 64);
        if (WAVES == 1 && total > H.heavy) {
            if (lane == 0) {
                const int parts = (total + TL_PART - 1) / TL_PART;
                const int e0 = atomicAdd(&H.count[0], parts);
                const int s0 = parts > 1 ? atomicAdd(&H.count[1], parts) : 0;
                for (int k = 0; k < parts; ++k) H.entries[e0 + k] = make_int4(tile, k, parts, s0 + k);
                if (parts > 1) H.multis[atomicAdd(&H.count[2], 1)] = make_int4(tile, parts, s0, 0);
            }
            return;
        }
        // each batch is summed by itself: no chain of FP32 sums is longer than 64
        float2 tot[4][4];
#pragma unroll
        for (int y = 0; y < 4; ++y)
#pragma unroll
            for (int x = 0; x < 4; ++x) tot[y][x] = make_float2(0.f, 0.f);
        for (int vb = (E.y * WAVES + wave) * 64; vb < total; vb += 64 * WAVES * E.z) {
            const int n = min(64, total - vb);
            int smp = 0, base = 0;
            for (int r = 0; r < nb * nrow; ++r) {
                const int k = __builtin_amdgcn_readlane(rn, r), o = vb + lane - base;
                if (o >= 0 && o < k) smp = __builtin_amdgcn_readlane(rs, r) + o;
                base += k;
            }
            // this lane's sample; lanes past the batch hold weights of zero
            float a = 0.f;
            int row = 0;
            if (lane < n) {
                row = perm[smp];
                const float4 p = pos[smp];
                const float2 ww = w[smp];
                const int l0 = __float_as_int(p.w);
                a = l == l0 ? ww.x : (l == l0 + 1 ? ww.y : 0.f);
#pragma unroll
                for (int q = 0; q < TX; ++q)
                    wx[lane * TX + q] = kb_weight(p.x, gx0 + q, g.inv_os, g.beta);
#pragma unroll
                for (int q = 0; q < TY; ++q)
                    wy[lane * TY + q] = a * kb_weight(p.y, gy0 + q, g.inv_os, g.beta);
            } else {
                for (int q = 0; q < TX; ++q) wx[lane * TX + q] = 0.f;
                for (int q = 0; q < TY; ++q) wy[lane * TY + q] = 0.f;
            }
            // the wave reads its own LDS words only
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            auto load = [&](int i) {
                return data[(size_t)__builtin_amdgcn_readlane(row, min(i, n - 1)) * C + c];
            };
            float2 acc[4][4];
#pragma unroll
            for (int y = 0; y < 4; ++y)
#pragma unroll
                for (int x = 0; x < 4; ++x) acc[y][x] = make_float2(0.f, 0.f);
            float2 d[TL_PF];
#pragma unroll
            for (int h = 0; h < TL_PF; ++h) d[h] = load(h);
            for (int i0 = 0; i0 < n; i0 += TL_PF) {
#pragma unroll
                for (int h = 0; h < TL_PF; ++h) {
                    const int i = i0 + h;
                    // samples of weight zero in time are left out (not finite)
                    const float at = __int_as_float(
                        __builtin_amdgcn_readlane(__float_as_int(a), min(i, 63)));
                    float2 v = at != 0.f ? d[h] : make_float2(0.f, 0.f);
                    d[h] = load(i + TL_PF);
                    const float4 x4 = *(const float4 *)&wx[i * TX + px];
                    const float4 y4 = *(const float4 *)&wy[i * TY + py];
                    const float xs[4] = {x4.x, x4.y, x4.z, x4.w};
                    const float ys[4] = {y4.x, y4.y, y4.z, y4.w};
#pragma unroll
                    for (int y = 0; y < 4; ++y) {
                        const float vr = v.x * ys[y], vi = v.y * ys[y];
#pragma unroll
                        for (int x = 0; x < 4; ++x) {
                            acc[y][x].x = fmaf(vr, xs[x], acc[y][x].x);
                            acc[y][x].y = fmaf(vi, xs[x], acc[y][x].y);
                        }
                    }
                }
            }
#pragma unroll
            for (int y = 0; y < 4; ++y)
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    tot[y][x].x += acc[y][x].x;
                    tot[y][x].y += acc[y][x].y;
                }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        if constexpr (WAVES > 1) {
            float2 *red = (float2 *)smem;
            for (int h = WAVES / 2; h > 0; h >>= 1) {
                __syncthreads();
                if (wave >= h && wave < 2 * h)
#pragma unroll
                    for (int k = 0; k < 16; ++k)
                        red[((wave - h) * 16 + k) * 64 + lane] = tot[k / 4][k % 4];
                __syncthreads();
                if (wave < h)
#pragma unroll
                    for (int k = 0; k < 16; ++k) {
                        const float2 v = red[(wave * 16 + k) * 64 + lane];
                        tot[k / 4][k % 4].x += v.x;
                        tot[k / 4][k % 4].y += v.y;
                    }
            }
            __syncthreads();
        }
        if (wave) continue;
        if (WAVES > 1 && E.z > 1) {
#pragma unroll
            for (int k = 0; k < 16; ++k) H.slots[((size_t)E.w * 16 + k) * 64 + lane] = tot[k / 4][k % 4];
            continue;
        }
        tile_store<C>(g, gx0, gy0, lane, tot, grid);
    }
}

// one wave per parted tile: the parts in order
template <int C>
__global__ __launch_bounds__(64) void k_grid_tiles_sum(GridGeom g, float2 *grid, int ntx,
                                                       TileList H) {
    const int lane = threadIdx.x, n = H.count[2];
    for (int it = blockIdx.x; it < n; it += gridDim.x) {
        const int4 M = H.multis[it];
        float2 tot[4][4];
#pragma unroll
        for (int k = 0; k < 16; ++k) tot[k / 4][k % 4] = make_float2(0.f, 0.f);
        for (int p = 0; p < M.y; ++p)
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const float2 v = H.slots[((size_t)(M.z + p) * 16 + k) * 64 + lane];
                tot[k / 4][k % 4].x += v.x;
                tot[k / 4][k % 4].y += v.y;
            }
        tile_store<C>(g, (M.x % ntx) * Tile<C>::TX, (M.x / ntx) * Tile<C>::TY, lane, tot, grid);
    }
}

// ---- steps 2 and 3 on grids with the coils innermost
// Lines of G = R 2^LOGP points, R odd: a radix-R stage, then radix 8 with a last
// 4 or 2 (Stockham: input j + r G/RAD, output (j - k) RAD + k + r NS with k = j
// mod NS).  The first stage reads global memory, the last writes it, those
// between exchange through LDS [element][coil].  Bound by memory: 704 x 704 x 32
// coils, 41 us per axis (5.3 TB/s); k_line_dft, which reads and writes its LDS
// once per radix-2 stage, 147.
template <int R>
struct OddTab {   // cos and sin of 2 pi m / R
    float c[R] = {}, s[R] = {};
    constexpr OddTab() {
        for (int m = 0; m < R; ++m) {
            const double x = 2.0 * 3.14159265358979323846 * m / R;
            double tc = 1.0, ts = x, sc = 0.0, ss = 0.0;
            for (int i = 1; i < 40; ++i) {   // the Taylor series
                sc += tc;
                ss += ts;
                tc *= -x * x / ((2 * i - 1) * (2 * i));
                ts *= -x * x / ((2 * i) * (2 * i + 1));
            }
            c[m] = (float)sc;
            s[m] = (float)ss;
        }
    }
};

// v[k] <- sum_n v[n] e^{+2 pi i n k / R}, R odd, from the sums and differences
// of v[m] and v[R - m]
template <int R>
__device__ __forceinline__ void dft_odd(float2 *v) {
    constexpr OddTab<R> tab;
    constexpr int H = (R - 1) / 2;
    float2 p[H], d[H];
#pragma unroll
    for (int m = 0; m < H; ++m) {
        const float2 a = v[m + 1], b = v[R - 1 - m];
        p[m] = make_float2(a.x + b.x, a.y + b.y);
        d[m] = make_float2(a.x - b.x, a.y - b.y);
    }
    const float2 v0 = v[0];
#pragma unroll
    for (int m = 0; m < H; ++m) {
        v[0].x += p[m].x;
        v[0].y += p[m].y;
    }
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        float2 e = v0, o = make_float2(0.f, 0.f);
#pragma unroll
        for (int m = 0; m < H; ++m) {
            const int i = (m + 1) * k % R;
            e.x = fmaf(tab.c[i], p[m].x, e.x);
            e.y = fmaf(tab.c[i], p[m].y, e.y);
            o.x = fmaf(tab.s[i], d[m].x, o.x);
            o.y = fmaf(tab.s[i], d[m].y, o.y);
        }
        v[k] = make_float2(e.x - o.y, e.y + o.x);
        v[R - k] = make_float2(e.x + o.y, e.y - o.x);
    }
}

template <int R, int LOGP>
struct GridLine {
    static constexpr int G = R << LOGP, T = G / 8;
    static constexpr int cols() {   // coils of a workgroup
        int n = 32;
        while (n > 1 && (n * T > 1024 || (long)n * G * 8 > 65536)) n /= 2;
        return n;
    }
    static constexpr int C = cols();
};

template <int G, int T, int RAD, int NS, class LD, class MID, class ST>
__device__ __forceinline__ void grid_stage(int t, const float2 *tw, LD ld, MID mid, ST st) {
    constexpr int NB = G / RAD, IT = (NB + T - 1) / T;
    float2 v[IT][RAD];
#pragma unroll
    for (int b = 0; b < IT; ++b) {
        const int j = t + T * b;
        if (NB % T && j >= NB) break;
#pragma unroll
        for (int r = 0; r < RAD; ++r) v[b][r] = ld(j + r * NB);
        if constexpr (NS > 1) {
            const int step = G / (NS * RAD) * (j % NS);
#pragma unroll
            for (int r = 1; r < RAD; ++r) v[b][r] = fftc::cmul(v[b][r], tw[r * step]);
        }
        if constexpr (RAD == 2 || RAD == 4 || RAD == 8) fftc::dft<RAD, true>(v[b]);
        else dft_odd<RAD>(v[b]);
    }
    mid();
#pragma unroll
    for (int b = 0; b < IT; ++b) {
        const int j = t + T * b, k = NS > 1 ? j % NS : 0;
        if (NB % T && j >= NB) break;
#pragma unroll
        for (int r = 0; r < RAD; ++r) st((j - k) * RAD + k + r * NS, v[b][r]);
    }
}

// the power-of-two stages, NS points done
template <int G, int T, int NS, class LLD, class LST, class GST>
__device__ __forceinline__ void grid_stages(int t, const float2 *tw, LLD lld, LST lst, GST gst) {
    constexpr int LEFT = G / NS, RAD = LEFT >= 8 ? 8 : LEFT;
    if constexpr (RAD == LEFT) {
        grid_stage<G, T, RAD, NS>(t, tw, lld, [] {}, gst);
    } else {
        grid_stage<G, T, RAD, NS>(t, tw, lld, [] { __syncthreads(); }, lst);
        __syncthreads();
        grid_stages<G, T, NS * RAD>(t, tw, lld, lst, gst);
    }
}

// Element j of line b, coil c at in[(b G + j) cs + c]; kept output i at
// out[i out_el + b cs + c].
template <int R, int LOGP>
__global__ __launch_bounds__((GridLine<R, LOGP>::T * GridLine<R, LOGP>::C)) void k_grid_lines(
    const float2 *__restrict__ in, float2 *__restrict__ out, int nlines, int nc, int cs,
    size_t out_el, int n, const float2 *__restrict__ tw, const float *__restrict__ dp) {
    using GL = GridLine<R, LOGP>;
    constexpr int G = GL::G, T = GL::T, P = GL::C;
    __shared__ float2 buf[G * P];
    __shared__ float2 twl[G];
    __shared__ float dpl[G];
    for (int i = threadIdx.x; i < G; i += T * P) {
        twl[i] = tw[i];
        dpl[i] = i < n ? dp[i] : 0.f;
    }
    const int q = threadIdx.x % P, t = threadIdx.x / P;
    const int np = (nc + P - 1) / P;
    // workgroups go round the 8 XCDs: b and b + 8 (one XCD) take adjacent coils
    const int blk = (blockIdx.x & ~15) | ((blockIdx.x & 7) << 1) | ((blockIdx.x >> 3) & 1);
    const int line = blk / np, c = (blk % np) * P + q;
    if (line >= nlines) return;
    const bool ok = c < nc;
    const float2 *col = in + (size_t)line * G * cs + (ok ? c : 0);
    float2 *o = out + (size_t)line * cs + c;
    auto gld = [&](int i) {
        const float2 v = col[(unsigned)i * cs];
        return ok ? v : make_float2(0.f, 0.f);
    };
    auto gst = [&](int i, float2 v) {
        const int x = (i < G / 2 ? i : i - G) + n / 2;
        if (ok && (unsigned)x < (unsigned)n) {
            const float f = dpl[x];
            o[x * out_el] = make_float2(v.x * f, v.y * f);
        }
    };
    auto lld = [&](int i) { return buf[i * P + q]; };
    auto lst = [&](int i, float2 v) { buf[i * P + q] = v; };
    constexpr int R0 = R > 1 ? R : 8;
    grid_stage<G, T, R0, 1>(t, tw, gld, [] {}, lst);
    __syncthreads();
    grid_stages<G, T, R0>(t, twl, lld, lst, gst);
}

// f(R, LOGP) for the line lengths of k_grid_lines; false: another length
template <class F>
bool grid_line_switch(int G, F f) {
    auto pow2 = [&](auto r) {
        constexpr int R = decltype(r)::value;
        switch (G / R) {
            case 8:
                if constexpr (R > 1) f(r, std::integral_constant<int, 3>{});
                return R > 1;
            case 16: f(r, std::integral_constant<int, 4>{}); return true;
            case 32: f(r, std::integral_constant<int, 5>{}); return true;
            case 64: f(r, std::integral_constant<int, 6>{}); return true;
            case 128: f(r, std::integral_constant<int, 7>{}); return true;
            case 256: f(r, std::integral_constant<int, 8>{}); return true;
            default: return false;
        }
    };
    if (G % 8 || G > 4096) return false;
    int r = G;
    while (r % 2 == 0) r /= 2;
    switch (r) {
        case 3: return pow2(std::integral_constant<int, 3>{});
        case 5: return pow2(std::integral_constant<int, 5>{});
        case 7: return pow2(std::integral_constant<int, 7>{});
        case 9: return pow2(std::integral_constant<int, 9>{});
        case 11: return pow2(std::integral_constant<int, 11>{});
        case 1:
            if (G == 512) return f(std::integral_constant<int, 1>{}, std::integral_constant<int, 9>{}), true;
            if (G == 1024) return f(std::integral_constant<int, 1>{}, std::integral_constant<int, 10>{}), true;
            return pow2(std::integral_constant<int, 1>{});
        default: return false;
    }
}

// Cropped, shifted inverse DFT along the contiguous axis of every line:
//   out[b][i][a] = dp[i] sum_{g<G} in[b][a][g] e^{+i 2pi g (i - n/2) / G}
// (dp carries (-1)^(i - n/2) of the shift and 1 / (os C(u_i))), for lines
// a < A of batch item b.  G = R P: R radix-2 FFTs of length P in LDS over
// the subsequences g = R q + j, then the R-term combination at each kept i,
//   out(nn) = sum_j Y_j[nn mod P] e^{+i 2pi j nn / G},  nn = i - n/2,
// with the twiddle index j nn mod G stepped by additions.  tw[k] =
// e^{+i 2pi k / G}.  2^logLPW lines per workgroup; every index is 32-bit
// and every division by a power of two is a shift (q = g / R by a float
// reciprocal and one correction step).
__global__ __launch_bounds__(GT) void k_line_dft(const float2 *__restrict__ in,
                                                 float2 *__restrict__ out, int G, int R, int P,
                                                 int logP, int n, int A, int nlines, int logLPW,
                                                 float rcpR, const float2 *__restrict__ tw,
                                                 const float *__restrict__ dp) {
    extern __shared__ float2 lds[];
    const int LPW = 1 << logLPW;
    const int line0 = blockIdx.x * LPW;
    const int nl = min(LPW, nlines - line0);
    // load: each line in natural order (coalesced), scattered to the
    // bit-reversed position of its subsequence
    for (int li = 0; li < nl; ++li) {
        const float2 *__restrict__ src = in + (size_t)(line0 + li) * G;
        float2 *dst = lds + li * G;
        for (int g = threadIdx.x; g < G; g += GT) {
            int q = (int)((float)g * rcpR);
            int j = g - q * R;
            if (j < 0) {
                --q;
                j += R;
            } else if (j >= R) {
                ++q;
                j -= R;
            }
            const int qr = logP ? (int)(__brev((unsigned)q) >> (32 - logP)) : 0;
            dst[j * P + qr] = src[g];
        }
    }
    __syncthreads();
    // radix-2 stages: butterfly span h = 2^lh = 1, 2, ..., P/2
    if (logP > 0) {
        const int nb = (nl * R) << (logP - 1);
        for (int lh = 0; lh < logP; ++lh) {
            const int h = 1 << lh;
            const int tstride = G >> (lh + 1);                 // G / (2h), exact
            const int gmask = (P >> (lh + 1)) - 1;             // P / (2h) - 1
            for (int bi = threadIdx.x; bi < nb; bi += GT) {
                const int k = bi & (h - 1);
                const int grp = (bi >> lh) & gmask;
                const int sub = bi >> (logP - 1);              // (line, j)
                const int base = sub * P + grp * 2 * h + k;
                const float2 wv = tw[k * tstride];
                const float2 u = lds[base], v = lds[base + h];
                const float2 tv = make_float2(v.x * wv.x - v.y * wv.y, v.x * wv.y + v.y * wv.x);
                lds[base] = make_float2(u.x + tv.x, u.y + tv.y);
                lds[base + h] = make_float2(u.x - tv.x, u.y - tv.y);
            }
            __syncthreads();
        }
    }
    // combination at the kept outputs, written with the axis outermost:
    // consecutive threads take consecutive lines of one output index
    const int b0 = line0 / A, a0 = line0 - b0 * A;
    for (int e = threadIdx.x; e < (n << logLPW); e += GT) {
        const int li = e & (LPW - 1), i = e >> logLPW;
        if (li >= nl) continue;
        const int nn = i - n / 2;
        const int m = nn & (P - 1);                            // nn mod P (P a power of two)
        int step = nn % G;
        if (step < 0) step += G;
        const float2 *y = lds + li * G + m;
        float sr = 0.f, si = 0.f;
        int kk = 0;
        for (int j = 0; j < R; ++j) {
            const float2 yv = y[j * P];
            const float2 wv = tw[kk];
            sr += yv.x * wv.x - yv.y * wv.y;
            si += yv.x * wv.y + yv.y * wv.x;
            kk += step;
            if (kk >= G) kk -= G;
        }
        int a = a0 + li, b = b0;
        while (a >= A) {
            a -= A;
            ++b;
        }
        const float f = dp[i];
        out[((size_t)b * n + i) * A + a] = make_float2(sr * f, si * f);
    }
}

__global__ void k_twiddle_g(int G, float2 *tw) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < G) {
        double s, c;
        sincospi(2.0 * (double)k / (double)G, &s, &c);
        tw[k] = make_float2((float)c, (float)s);
    }
}

// dp[i] = (-1)^(i - n/2) / (os C(u_i)), C(u) = sin(sqrt(pi^2 W^2 u^2 -
// beta^2)) / sqrt(...) (sinh below zero), u_i = (i - n/2) / n, in FP64
__global__ void k_deapod(int n, double os, double beta, float *dp) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int nn = i - n / 2;
    const double u = (double)nn / (double)n;
    const double e = M_PI * M_PI * (double)KB_WIDTH * (double)KB_WIDTH * u * u - beta * beta;
    double c;
    if (e > 0.0) {
        const double r = sqrt(e);
        c = sin(r) / r;
    } else if (e < 0.0) {
        const double r = sqrt(-e);
        c = sinh(r) / r;
    } else {
        c = 1.0;
    }
    dp[i] = (float)(((nn & 1) ? -1.0 : 1.0) / (os * c));
}

// F^H d epilogue of segment l: acc += e^{+i w (t0 + l tau)} sum_c conj(S_c) y_c
__global__ void k_grid_fhd_accum(long nv, int ncoils, const float2 *y, size_t plane,
                                 const float *s_r, const float *s_i, const float *fm,
                                 float tl, double2 *acc) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nv) return;
    double vr = 0.0, vi = 0.0;
    for (int c = 0; c < ncoils; ++c) {
        const float2 v = y[c * plane + i];
        const double sr = s_r ? s_r[(size_t)c * nv + i] : 1.0;
        const double si = s_r ? s_i[(size_t)c * nv + i] : 0.0;
        vr += sr * v.x + si * v.y;
        vi += sr * v.y - si * v.x;
    }
    // the reference's expfm: cos / sin of the float product fm (tau l + t0)
    const float arg = fm ? fm[i] * tl : 0.f;
    double sn, cs;
    sincos((double)arg, &sn, &cs);
    double2 a = acc[i];
    a.x += cs * vr - sn * vi;
    a.y += cs * vi + sn * vr;
    acc[i] = a;
}

// The same with the coils innermost, y[i][C]: 64 voxels through LDS, four
// groups of coils (512^2 x 32 coils: 44 us, 3.0 TB/s; one thread per voxel
// reading its 256 bytes: 85).
template <int C>
__global__ __launch_bounds__(GT) void k_grid_accum_rows(long nv, int ncoils, const float2 *y,
                                                        const float *s_r, const float *s_i,
                                                        const float *fm, float tl, double2 *acc) {
    __shared__ float2 tile[64][C + 1];
    __shared__ double2 part[4][64];
    const long i0 = (long)blockIdx.x * 64;
    for (int e = threadIdx.x; e < 64 * C; e += GT)
        if (i0 + e / C < nv) tile[e / C][e % C] = y[i0 * C + e];
    __syncthreads();
    const int j = threadIdx.x & 63, q = threadIdx.x >> 6;
    const long i = i0 + j;
    double vr = 0.0, vi = 0.0;
    if (i < nv) {
#pragma unroll
        for (int k = 0; k < C / 4; ++k) {
            const int c = q * (C / 4) + k;
            if (c >= ncoils) break;
            const float2 v = tile[j][c];
            const double sr = s_r ? s_r[(size_t)c * nv + i] : 1.0;
            const double si = s_r ? s_i[(size_t)c * nv + i] : 0.0;
            vr += sr * v.x + si * v.y;
            vi += sr * v.y - si * v.x;
        }
    }
    part[q][j] = make_double2(vr, vi);
    __syncthreads();
    if (q || i >= nv) return;
    for (int k = 1; k < 4; ++k) {
        vr += part[k][j].x;
        vi += part[k][j].y;
    }
    const float arg = fm ? fm[i] * tl : 0.f;
    double sn, cs;
    sincos((double)arg, &sn, &cs);
    double2 a = acc[i];
    a.x += cs * vr - sn * vi;
    a.y += cs * vi + sn * vr;
    acc[i] = a;
}

__global__ void k_grid_fhd_out(long nv, const double2 *acc, float *out_r, float *out_i) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nv) {
        out_r[i] = (float)acc[i].x;
        out_i[i] = (float)acc[i].y;
    }
}

__global__ void k_grid_q_out(long nq, const float2 *y, float *q_r, float *q_i) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nq) {
        q_r[i] = y[i].x;
        q_i[i] = y[i].y;
    }
}

__global__ void k_zero_i(int *p, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

__global__ void k_zero_d2(double2 *p, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = make_double2(0.0, 0.0);
}

// grid set-up of computeQ_GPU_Grid / computeFH_GPU_Grid for an image of
// n[0] x n[1] x n[2] (computeQ.cmem.cu:433-498, computeFH.cmem.cu:495-543):
// gridOS rounded in float so x/y grids are even (2D) or z a multiple of 4
// (3D), Beatty's beta, G = ceil(os n) with x and y bumped to even
GridGeom grid_geometry(const int n[3], float gridOS) {
    GridGeom g{};
    for (int a = 0; a < 3; ++a) g.n[a] = n[a];
    g.d3 = n[2] > 1;
    float os = gridOS;
    if (!g.d3)
        os = 2.0f * std::ceil((os * (float)n[0]) / 2.0f) / (float)n[0];
    else
        os = 4.0f * std::ceil((os * (float)n[2]) / 4.0f) / (float)n[2];
    g.os = os;
    g.inv_os = 1.0f / os;
    g.half = KB_WIDTH * os / 2.0f;
    const double o = (double)os, W = KB_WIDTH;
    g.beta = (float)(M_PI * std::sqrt((o - 0.5) * (o - 0.5) * (W * W * 4.0) / (o * o) - 0.8));
    g.G[0] = (int)std::ceil(os * (float)n[0]);
    g.G[1] = (int)std::ceil(os * (float)n[1]);
    g.G[0] += g.G[0] % 2;
    g.G[1] += g.G[1] % 2;
    g.G[2] = g.d3 ? (int)std::ceil(os * (float)n[2]) : 1;
    return g;
}

// pointers carved from one workspace slot
struct Carve {
    char *p;
    template <class T>
    T *take(size_t count) {
        T *r = (T *)p;
        p += (count * sizeof(T) + 255) & ~(size_t)255;
        return r;
    }
};

// Sorted samples of one trajectory on one grid: cell ranges, positions and
// segment weights.
struct Binned {
    int nbuck;        // time buckets (segments + 1)
    int *start;       // [nbuck * ncells + 1]
    int *perm;        // [m] sample index of sorted position
    float4 *pos;      // [m] sorted
    float2 *w;        // [m] sorted segment weights
};

// the radix sort's histogram of m elements, and the block sums of an
// exclusive scan of n ints
long rs_blocks(int m) { return (m + RS_BLOCK - 1) / RS_BLOCK; }
long scan_blocks(long n) { return (n + GT * 4 - 1) / (GT * 4); }

// keys: time bucket x grid cell; nseg + 1 buckets
long key_range(long ncells, int nseg) { return ncells * (nseg + 1); }

size_t binned_bytes(int m, long ncells, int nseg) {
    auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
    const long nk = key_range(ncells, nseg);
    const long nh = (long)RS_BINS * rs_blocks(m);
    const long nb = std::max(scan_blocks(nk), scan_blocks(nh));
    return al((nk + 1) * 4) * 2 + al(nb * 4) + al(16) + al((size_t)m * 4) * 4 +
           al((size_t)(nh + 1) * 4) * 2 + al((size_t)m * 16) * 2 + al((size_t)m * 8);
}

// exclusive scan of n ints in three launches (out has n + 1 entries: the
// total last); bsum holds scan_blocks(n) ints
void scan_ints(hipStream_t st, const int *in, int *out, long n, int *bsum, int *total) {
    const long nb = scan_blocks(n);
    hipLaunchKernelGGL(k_scan_blocks, dim3((unsigned)nb), dim3(GT), 0, st, in, (int)n, out, bsum);
    hipLaunchKernelGGL(k_scan_totals, dim3(1), dim3(GT), 0, st, bsum, (int)nb, total);
    hipLaunchKernelGGL(k_scan_add, dim3(ceil_div(n + 1, 256)), dim3(256), 0, st, out, (int)n, bsum,
                       total);
}

int bin_samples(imp_ctx *ctx, Carve &cv, const GridGeom &g, int m, const float *kx,
                const float *ky, const float *kz, float kscale, const float *t, int nseg,
                float tau, float t0, Binned &B) {
    const hipStream_t st = ctx->stream;
    const long ncells = (long)g.G[0] * g.G[1] * g.G[2];
    const long nk = key_range(ncells, nseg);
    if (nk >= (1L << 30))
        return fail(IMP_EUNSUPPORTED, "gridding: %ld time buckets x grid cells (at most 2^30)", nk);
    const long nrb = rs_blocks(m), nh = (long)RS_BINS * nrb;
    const long nb = std::max(scan_blocks(nk), scan_blocks(nh));
    int *count = cv.take<int>(nk + 1);
    B.start = cv.take<int>(nk + 1);
    int *bsum = cv.take<int>(nb);
    int *total = cv.take<int>(4);
    int *key[2] = {cv.take<int>(m), cv.take<int>(m)};
    int *val[2] = {cv.take<int>(m), cv.take<int>(m)};
    int *hist = cv.take<int>(nh + 1);
    int *offs = cv.take<int>(nh + 1);
    float4 *pos_raw = cv.take<float4>(m);
    B.pos = cv.take<float4>(m);
    B.w = cv.take<float2>(m);
    hipLaunchKernelGGL(k_zero_i, dim3(ceil_div(nk + 1, 256)), dim3(256), 0, st, count, nk + 1);
    hipLaunchKernelGGL(k_grid_cells, dim3(ceil_div(m, 256)), dim3(256), 0, st, m, kx, ky, kz, t,
                       kscale, g, t0, tau, nseg, pos_raw, key[0], count);
    scan_ints(st, count, B.start, nk, bsum, total);
    hipLaunchKernelGGL(k_iota, dim3(ceil_div(m, 256)), dim3(256), 0, st, m, val[0]);
    IMP_CHECK_LAUNCH();
    // keys are < nk: sort on the bits that can be set
    B.nbuck = nseg + 1;
    int bits = 1;
    while (bits < 31 && (1L << bits) < nk) ++bits;
    int cur = 0;
    for (int shift = 0; shift < bits; shift += 4, cur ^= 1) {
        hipLaunchKernelGGL(k_rs_count, dim3((unsigned)nrb), dim3(RS_BLOCK), 0, st, key[cur], m,
                           shift, (int)nrb, hist);
        scan_ints(st, hist, offs, nh, bsum, total);
        hipLaunchKernelGGL(k_rs_scatter, dim3((unsigned)nrb), dim3(RS_BLOCK), 0, st, key[cur],
                           val[cur], m, shift, (int)nrb, offs, key[cur ^ 1], val[cur ^ 1]);
        IMP_CHECK_LAUNCH();
    }
    B.perm = val[cur];
    hipLaunchKernelGGL(k_grid_samples, dim3(ceil_div(m, 256)), dim3(256), 0, st, m, B.perm,
                       pos_raw, t, nseg, tau, t0, B.pos, B.w);
    IMP_CHECK_LAUNCH();
    return IMP_OK;
}

// line-transform schedule of one axis
struct AxisPlan {
    int G, R, P, logP, n, logLPW;
    float2 *tw;
    float *dp;
};

size_t axis_bytes(int G, int n) {
    return (((size_t)G * 8 + 255) & ~(size_t)255) + (((size_t)n * 4 + 255) & ~(size_t)255);
}

int plan_axis(imp_ctx *ctx, Carve &cv, const GridGeom &g, int a, AxisPlan &ap) {
    ap.G = g.G[a];
    ap.n = g.n[a];
    int P = 1, logP = 0;
    while (ap.G % (2 * P) == 0) {
        P *= 2;
        ++logP;
    }
    ap.P = P;
    ap.logP = logP;
    ap.R = ap.G / P;
    // lines per workgroup: a power of two, at most 16 and 64 KB of LDS
    ap.logLPW = 0;
    while (ap.logLPW < 4 && (2L << ap.logLPW) * ap.G * (long)sizeof(float2) <= 65536) ++ap.logLPW;
    ap.tw = cv.take<float2>(ap.G);
    ap.dp = cv.take<float>(ap.n);
    hipLaunchKernelGGL(k_twiddle_g, dim3(ceil_div(ap.G, 256)), dim3(256), 0, ctx->stream, ap.G,
                       ap.tw);
    hipLaunchKernelGGL(k_deapod, dim3(ceil_div(ap.n, 256)), dim3(256), 0, ctx->stream, ap.n,
                       (double)g.os, (double)g.beta, ap.dp);
    IMP_CHECK_LAUNCH();
    return IMP_OK;
}

int run_axis(imp_ctx *ctx, const AxisPlan &ap, const float2 *in, float2 *out, long nlines,
             long A) {
    if (nlines > INT32_MAX / 2 || A > INT32_MAX / 2 || (long)ap.n * A > INT32_MAX)
        return fail(IMP_EUNSUPPORTED, "gridding: %ld lines of %ld too many", nlines, A);
    const int lpw = 1 << ap.logLPW;
    const unsigned wgs = (unsigned)((nlines + lpw - 1) / lpw);
    const size_t lds = (size_t)lpw * ap.G * sizeof(float2);
    hipLaunchKernelGGL(k_line_dft, dim3(wgs), dim3(GT), lds, ctx->stream, in, out, ap.G, ap.R,
                       ap.P, ap.logP, ap.n, (int)A, (int)nlines, ap.logLPW,
                       1.0f / (float)ap.R, ap.tw, ap.dp);
    IMP_CHECK_LAUNCH();
    return IMP_OK;
}

// every axis of `planes` grids [gy][gx][gz] -> images [ny][nx][nz]; the
// result ends in *res (one of a / b)
int transform_planes(imp_ctx *ctx, const GridGeom &g, AxisPlan ax[3], int planes, float2 *a,
                     float2 *b, float2 **res) {
    // current layout dims, outermost first; the contiguous axis is last
    const int nd = g.d3 ? 3 : 2;
    // axis order of the passes: contiguous axis first (z in 3D, x in 2D)
    const int order3[3] = {2, 0, 1}, order2[2] = {0, 1};
    const int *order = g.d3 ? order3 : order2;
    // sizes of the current layout (all axes), starting from the grid
    int cur[3] = {g.G[0], g.G[1], g.G[2]};
    float2 *src = a, *dst = b;
    for (int p = 0; p < nd; ++p) {
        const int axis = order[p];
        long per_plane = 1;
        for (int q = 0; q < 3; ++q) per_plane *= cur[q];
        const long A = per_plane / cur[axis];
        IMP_TRY(run_axis(ctx, ax[axis], src, dst, (long)planes * A, A));
        cur[axis] = g.n[axis];
        std::swap(src, dst);
    }
    *res = src;
    return IMP_OK;
}

int check_traj(const GridGeom &g) {
    for (int a = 0; a < (g.d3 ? 3 : 2); ++a)
        if (g.G[a] > 4096 || g.G[a] < 2)
            return fail(IMP_EUNSUPPORTED, "gridding: grid of %d points along axis %d (2..4096)",
                        g.G[a], a);
    return IMP_OK;
}

void host_t_ends(imp_ctx *ctx, const float *t, int m, float *tt, int *st) {
    *st = IMP_OK;
    if (hipMemcpyAsync(&tt[0], t, sizeof(float), hipMemcpyDeviceToHost, ctx->stream) != hipSuccess ||
        hipMemcpyAsync(&tt[1], t + (m - 1), sizeof(float), hipMemcpyDeviceToHost, ctx->stream) !=
            hipSuccess ||
        hipStreamSynchronize(ctx->stream) != hipSuccess)
        *st = fail(IMP_EHIP, "gridding: %s", hipGetErrorString(hipGetLastError()));
}

// gather of segment l: light points one per lane, then the listed heavy
// points one per wave (heavy holds ncells ints, nheavy one)
template <int C>
void launch_gather(imp_ctx *ctx, const GridGeom &g, const Binned &B, const float2 *data, int l,
                   float2 *grid, size_t plane, int *heavy, int *nheavy) {
    const long total = (long)g.G[0] * g.G[1] * g.G[2];
    hipLaunchKernelGGL(k_zero_i, dim3(1), dim3(256), 0, ctx->stream, nheavy, 1L);
    hipLaunchKernelGGL(k_grid_gather<C>, dim3((unsigned)ceil_div(total, GT)), dim3(GT), 0,
                       ctx->stream, g, B.start, B.nbuck, B.pos, B.w, data, l, grid, plane, heavy,
                       nheavy);
    hipLaunchKernelGGL(k_grid_gather_heavy<C>, dim3(4 * (unsigned)ctx->num_cus), dim3(GT), 0,
                       ctx->stream, g, B.start, B.nbuck, B.pos, B.w, data, l, grid, plane, heavy,
                       nheavy);
}

bool grid_line_ok(int G) {
    return grid_line_switch(G, [](auto, auto) {});
}

// f(CP) for the coil lanes of the tiled form of 2D F^H d.  Whole calls before
// and after: 64^2 x 4 coils 1.49 -> 1.12 ms, 128^2 x 8 1.57 -> 1.03, 256^2 x 4
// 1.80 -> 1.18, 256^2 x 16 2.27 -> 1.08, 512^2 x 32 8.60 -> 2.98.  With 2 coils
// a tile would span more cell rows than there are lanes to hold their ranges.
template <class F>
bool tile_switch(int CP, F f) {
    switch (CP) {
        case 4: return f(std::integral_constant<int, 4>{});
        case 8: return f(std::integral_constant<int, 8>{});
        case 16: return f(std::integral_constant<int, 16>{});
        case 32: return f(std::integral_constant<int, 32>{});
        default: return false;
    }
}

// Most slots that the parted tiles of C coils can take: a sample lies in the
// windows of at most `per` tiles, and a parted tile has parts <= 2 total / TL_PART.
template <int C>
long tile_slots(const GridGeom &g, int m) {
    const int w = (int)std::ceil(g.half) + (int)std::floor(g.half);
    const long per = (long)(1 + ceil_div(w, Tile<C>::TX)) * (1 + ceil_div(w, Tile<C>::TY));
    return 2 * per * m / TL_PART + 1;
}
template <int C>
long tile_count(const GridGeom &g) {
    return (long)ceil_div(g.G[0], Tile<C>::TX) * ceil_div(g.G[1], Tile<C>::TY);
}
size_t tile_list_bytes(long tiles, long slots) {
    return (size_t)(tiles + 2 * slots) * sizeof(int4) + (size_t)slots * 16 * 64 * sizeof(float2) +
           2048;
}
TileList tile_list(Carve &cv, long tiles, long slots, int m) {
    TileList H;
    H.heavy = m <= TL_FEW ? TL_LOW : TL_HEAVY;
    H.entries = cv.take<int4>(tiles + slots);
    H.multis = cv.take<int4>(slots);
    H.count = cv.take<int>(4);
    H.slots = cv.take<float2>((size_t)slots * 16 * 64);
    return H;
}

// tiles of segment l: one wave each, then the listed ones
template <int C>
void launch_tiles(imp_ctx *ctx, const GridGeom &g, const Binned &B, const float2 *data, int l,
                  float2 *grid, const TileList &H) {
    const int ntx = ceil_div(g.G[0], Tile<C>::TX);
    hipLaunchKernelGGL(k_zero_i, dim3(1), dim3(256), 0, ctx->stream, H.count, 4L);
    hipLaunchKernelGGL((k_grid_tiles<C, 1>), dim3((unsigned)tile_count<C>(g)), dim3(64), 0,
                       ctx->stream, g, B.start, B.nbuck, B.pos, B.w, B.perm, data, l, grid, ntx, H);
    hipLaunchKernelGGL((k_grid_tiles<C, TL_WAVES>), dim3(2 * ctx->num_cus), dim3(64 * TL_WAVES), 0,
                       ctx->stream, g, B.start, B.nbuck, B.pos, B.w, B.perm, data, l, grid, ntx, H);
    hipLaunchKernelGGL(k_grid_tiles_sum<C>, dim3(ctx->num_cus), dim3(64), 0, ctx->stream, g, grid,
                       ntx, H);
}

// coils-innermost grids in and out, along axis 0 (x) of G[1] lines, then y
int lines_tiled(imp_ctx *ctx, const GridGeom &g, const AxisPlan ax[3], int nc, int cs, float2 *a,
                float2 *b) {
    for (int q = 0; q < 2; ++q) {
        const int nlines = q ? g.n[0] : g.G[1];
        // axis x: b[ix][gy][c]; axis y: a[iy][ix][c]
        grid_line_switch(g.G[q], [&](auto r, auto lp) {
            constexpr int R = decltype(r)::value, LP = decltype(lp)::value;
            using GL = GridLine<R, LP>;
            const unsigned wgs = ((unsigned)nlines * ceil_div(nc, GL::C) + 15) & ~15u;
            hipLaunchKernelGGL((k_grid_lines<R, LP>), dim3(wgs), dim3(GL::T * GL::C), 0,
                               ctx->stream, q ? b : a, q ? a : b, nlines, nc, cs,
                               (size_t)nlines * cs, g.n[q], ax[q].tw, ax[q].dp);
        });
        IMP_CHECK_LAUNCH();
    }
    return IMP_OK;
}

template <int C>
void launch_data(imp_ctx *ctx, int m, int ncoils, const int *perm, const float *d_r,
                 const float *d_i, float2 *out) {
    hipLaunchKernelGGL(k_grid_data<C>, dim3(ceil_div(m, 256)), dim3(256), 0, ctx->stream, m,
                       ncoils, perm, d_r, d_i, out);
}

}  // namespace

int gridding_q(imp_ctx *ctx, int num_k, const float *kx, const float *ky, const float *kz,
               const float *t, int Nx, int Ny, int Nz, int ntime_segs, float gridOS, float *q_r,
               float *q_i) {
    if (!ctx || num_k <= 0 || !kx || !ky || !t || !q_r || !q_i || Nx <= 0 || Ny <= 0 ||
        Nz <= 0 || ntime_segs < 0 || !(gridOS >= 1.0f) || (Nz > 1 && !kz))
        return fail(IMP_EINVAL, "imp_toeplitz_q_gridding: bad arguments");
    const int nseg = ntime_segs + 1;
    const int n[3] = {2 * Nx, 2 * Ny, Nz > 1 ? 2 * Nz : 1};
    const GridGeom g = grid_geometry(n, gridOS);
    IMP_TRY(check_traj(g));
    float tt[2];
    int st = IMP_OK;
    host_t_ends(ctx, t, num_k, tt, &st);
    IMP_TRY(st);
    const float tau = ntime_segs > 0 ? (tt[1] - tt[0]) / (float)ntime_segs : (tt[1] - tt[0]);
    const long ncells = (long)g.G[0] * g.G[1] * g.G[2];
    const long nq = (long)n[0] * n[1] * n[2];
    const size_t gbytes = (size_t)nseg * ncells * sizeof(float2);
    size_t bytes = binned_bytes(num_k, ncells, nseg) + 2 * (((gbytes + 255) & ~(size_t)255)) + 4096 +
                   (((size_t)ncells * 4 + 255) & ~(size_t)255) + 256 +
                   axis_bytes(g.G[0], n[0]) + axis_bytes(g.G[1], n[1]) + axis_bytes(g.G[2], n[2]);
    void *ws = nullptr;
    IMP_TRY(workspace(ctx, WS_GRID, bytes, &ws));
    Carve cv{(char *)ws};
    Binned B{};
    // Q samples sit at 2k on the 2N grid, with unit data (computeQ.cmem.cu:515-525)
    IMP_TRY(bin_samples(ctx, cv, g, num_k, kx, ky, kz, 2.0f, t, nseg, tau, tt[0], B));
    float2 *bufA = cv.take<float2>((size_t)nseg * ncells);
    float2 *bufB = cv.take<float2>((size_t)nseg * ncells);
    int *heavy = cv.take<int>(ncells);
    int *nheavy = cv.take<int>(1);
    AxisPlan ax[3];
    for (int a = 0; a < (g.d3 ? 3 : 2); ++a) IMP_TRY(plan_axis(ctx, cv, g, a, ax[a]));
    const int rec = prof_begin(ctx, "k_grid_gather");
    for (int l = 0; l < nseg; ++l)
        launch_gather<0>(ctx, g, B, nullptr, l, bufA + (size_t)l * ncells, 0, heavy, nheavy);
    prof_end(ctx, rec);
    IMP_CHECK_LAUNCH();
    float2 *res = nullptr;
    const int rec2 = prof_begin(ctx, "k_line_dft");
    IMP_TRY(transform_planes(ctx, g, ax, nseg, bufA, bufB, &res));
    prof_end(ctx, rec2);
    hipLaunchKernelGGL(k_grid_q_out, dim3(ceil_div((long)nseg * nq, 256)), dim3(256), 0,
                       ctx->stream, (long)nseg * nq, res, q_r, q_i);
    IMP_CHECK_LAUNCH();
    IMP_TRY(workspace_release(ctx, WS_GRID, 1ull << 30));
    return IMP_OK;
}

int gridding_fhd(imp_ctx *ctx, int num_k, int ncoils, const float *kx, const float *ky,
                 const float *kz, const float *t, int Nx, int Ny, int Nz, const float *fm,
                 const float *d_r, const float *d_i, const float *s_r, const float *s_i,
                 int ntime_segs, float gridOS, float *out_r, float *out_i) {
    if (!ctx || num_k <= 0 || ncoils <= 0 || !kx || !ky || !t || !d_r || !d_i || !out_r ||
        !out_i || Nx <= 0 || Ny <= 0 || Nz <= 0 || ntime_segs < 0 || !(gridOS >= 1.0f) ||
        (Nz > 1 && !kz) || (s_r == nullptr) != (s_i == nullptr))
        return fail(IMP_EINVAL, "imp_fhd_gridding: bad arguments");
    const int nseg = ntime_segs + 1;
    const int n[3] = {Nx, Ny, Nz};
    const GridGeom g = grid_geometry(n, gridOS);
    IMP_TRY(check_traj(g));
    float tt[2];
    int st = IMP_OK;
    host_t_ends(ctx, t, num_k, tt, &st);
    IMP_TRY(st);
    const float tau = ntime_segs > 0 ? (tt[1] - tt[0]) / (float)ntime_segs : (tt[1] - tt[0]);
    const long ncells = (long)g.G[0] * g.G[1] * g.G[2];
    const long nv = (long)Nx * Ny * Nz;
    const int CP = ncoils <= 1 ? 1 : ncoils <= 2 ? 2 : ncoils <= 4 ? 4 : ncoils <= 8 ? 8
                 : ncoils <= 16 ? 16 : 32;
    const int groups = ceil_div(ncoils, CP);
    const size_t gbytes = (size_t)CP * ncells * sizeof(float2);
    bool tiled = !g.d3 && grid_line_ok(g.G[0]) && grid_line_ok(g.G[1]) && nv * CP < INT32_MAX;
    long tiles = 0, slots = 0;
    tiled = tiled && tile_switch(CP, [&](auto cp) {
        constexpr int C = decltype(cp)::value;
        tiles = tile_count<C>(g);
        slots = tile_slots<C>(g, num_k);
        // a lane per cell row of two time buckets
        return 2 * (Tile<C>::TY + std::ceil(g.half) + std::floor(g.half)) <= 64;
    });
    if (!tiled) tiles = slots = 0;
    size_t bytes = binned_bytes(num_k, ncells, nseg) + tile_list_bytes(tiles, slots) +
                   2 * ((gbytes + 255) & ~(size_t)255) +
                   (((size_t)ncells * 4 + 255) & ~(size_t)255) + 256 +
                   (((size_t)num_k * CP * 8 + 255) & ~(size_t)255) + nv * 16 + 8192 +
                   axis_bytes(g.G[0], n[0]) + axis_bytes(g.G[1], n[1]) + axis_bytes(g.G[2], n[2]);
    void *ws = nullptr;
    IMP_TRY(workspace(ctx, WS_GRID, bytes, &ws));
    Carve cv{(char *)ws};
    Binned B{};
    IMP_TRY(bin_samples(ctx, cv, g, num_k, kx, ky, kz, 1.0f, t, nseg, tau, tt[0], B));
    float2 *bufA = cv.take<float2>((size_t)CP * ncells);
    float2 *bufB = cv.take<float2>((size_t)CP * ncells);
    int *heavy = cv.take<int>(ncells);
    int *nheavy = cv.take<int>(1);
    const TileList H = tile_list(cv, tiles, slots, num_k);
    float2 *data = cv.take<float2>((size_t)num_k * CP);
    double2 *acc = cv.take<double2>(nv);
    AxisPlan ax[3];
    for (int a = 0; a < (g.d3 ? 3 : 2); ++a) IMP_TRY(plan_axis(ctx, cv, g, a, ax[a]));
    hipLaunchKernelGGL(k_zero_d2, dim3(ceil_div(nv, 256)), dim3(256), 0, ctx->stream, acc, nv);
    for (int grp = 0; grp < groups; ++grp) {
        const int c0 = grp * CP, cn = std::min(CP, ncoils - c0);
        const float *dr = d_r + (size_t)c0 * num_k, *di = d_i + (size_t)c0 * num_k;
        if (tiled) {
            tile_switch(CP, [&](auto cp) {
                hipLaunchKernelGGL(k_grid_rows<decltype(cp)::value>, dim3(ceil_div(num_k, 64)),
                                   dim3(GT), 0, ctx->stream, num_k, cn, dr, di, data);
                return true;
            });
        } else switch (CP) {
            case 1: launch_data<1>(ctx, num_k, cn, B.perm, dr, di, data); break;
            case 2: launch_data<2>(ctx, num_k, cn, B.perm, dr, di, data); break;
            case 4: launch_data<4>(ctx, num_k, cn, B.perm, dr, di, data); break;
            case 8: launch_data<8>(ctx, num_k, cn, B.perm, dr, di, data); break;
            case 16: launch_data<16>(ctx, num_k, cn, B.perm, dr, di, data); break;
            default: launch_data<32>(ctx, num_k, cn, B.perm, dr, di, data); break;
        }
        IMP_CHECK_LAUNCH();
        for (int l = 0; l < nseg; ++l) {
            const int rec = prof_begin(ctx, "k_grid_gather");
            if (tiled) {
                tile_switch(CP, [&](auto cp) {
                    launch_tiles<decltype(cp)::value>(ctx, g, B, data, l, bufA, H);
                    return true;
                });
            } else switch (CP) {
                case 1: launch_gather<1>(ctx, g, B, data, l, bufA, ncells, heavy, nheavy); break;
                case 2: launch_gather<2>(ctx, g, B, data, l, bufA, ncells, heavy, nheavy); break;
                case 4: launch_gather<4>(ctx, g, B, data, l, bufA, ncells, heavy, nheavy); break;
                case 8: launch_gather<8>(ctx, g, B, data, l, bufA, ncells, heavy, nheavy); break;
                case 16: launch_gather<16>(ctx, g, B, data, l, bufA, ncells, heavy, nheavy); break;
                default: launch_gather<32>(ctx, g, B, data, l, bufA, ncells, heavy, nheavy); break;
            }
            prof_end(ctx, rec);
            IMP_CHECK_LAUNCH();
            float2 *res = nullptr;
            const int rec2 = prof_begin(ctx, "k_line_dft");
            if (tiled) {
                IMP_TRY(lines_tiled(ctx, g, ax, cn, CP, bufA, bufB));
                res = bufA;
            } else {
                IMP_TRY(transform_planes(ctx, g, ax, cn, bufA, bufB, &res));
            }
            prof_end(ctx, rec2);
            // expfm argument fm (tau l + t0) in float (recon.cu:1281-1285)
            const float tl = tau * (float)l + tt[0];
            const float *sr = s_r ? s_r + (size_t)c0 * nv : nullptr;
            const float *si = s_i ? s_i + (size_t)c0 * nv : nullptr;
            if (tiled) {
                tile_switch(CP, [&](auto cp) {
                    hipLaunchKernelGGL(k_grid_accum_rows<decltype(cp)::value>,
                                       dim3(ceil_div(nv, 64)), dim3(GT), 0, ctx->stream, nv, cn,
                                       res, sr, si, fm, tl, acc);
                    return true;
                });
            } else {
                hipLaunchKernelGGL(k_grid_fhd_accum, dim3(ceil_div(nv, 256)), dim3(256), 0,
                                   ctx->stream, nv, cn, res, (size_t)nv, sr, si, fm, tl, acc);
            }
            IMP_CHECK_LAUNCH();
        }
    }
    hipLaunchKernelGGL(k_grid_fhd_out, dim3(ceil_div(nv, 256)), dim3(256), 0, ctx->stream, nv,
                       acc, out_r, out_i);
    IMP_CHECK_LAUNCH();
    IMP_TRY(workspace_release(ctx, WS_GRID, 1ull << 30));
    return IMP_OK;
}

}  // namespace imp

extern "C" int imp_toeplitz_q_gridding(imp_ctx *ctx, int num_k, const float *kx, const float *ky,
                                       const float *kz, const float *t, int Nx, int Ny, int Nz,
                                       int ntime_segs, float gridOS, float *q_r, float *q_i) {
    return imp::gridding_q(ctx, num_k, kx, ky, kz, t, Nx, Ny, Nz, ntime_segs, gridOS, q_r, q_i);
}

extern "C" int imp_fhd_gridding(imp_ctx *ctx, int num_k, int ncoils, const float *kx,
                                const float *ky, const float *kz, const float *t, int Nx, int Ny,
                                int Nz, const float *fm, const float *d_r, const float *d_i,
                                const float *s_r, const float *s_i, int ntime_segs, float gridOS,
                                float *out_r, float *out_i) {
    return imp::gridding_fhd(ctx, num_k, ncoils, kx, ky, kz, t, Nx, Ny, Nz, fm, d_r, d_i, s_r,
                             s_i, ntime_segs, gridOS, out_r, out_i);
}
