// Separable evaluation of the NUDFT on image grids (nufft.hip).
#pragma once

#include "common.h"

#include <vector>

namespace imp {

// Every operator below returns IMP_ENOMEM before it has written a result when
// its workspace cannot be had; callers then take the direct path.

// Points c0 + i d: read the transform's bins; nearly so: a first-order step
// from the bins; any other: interpolate.
enum { AX_UNIFORM, AX_NEAR, AX_FREE };

// One image axis against the sample coordinate k it pairs with.
struct NuAxis {
    int n;            // image points
    int L;            // transform length
    int nf;           // spread-grid points (every sample's window fits)
    int kind;         // AX_*
    int flip;         // d < 0
    int shift;        // grid point of bin 0, mod L
    double kc;        // centre of k
    double xc;        // centre of the points
    double inv_d;     // grid cells per unit of k
    double j0;        // grid point of kc
};

struct NuGeometry {
    bool ok = false;
    bool a_is_y = false;      // axis A (fastest in the voxel index after z) is y
    NuAxis A{}, B{};
    int nz = 1;               // z planes (z fastest)
    double tc = 0, th = 0;    // centre and half width of t, and of w
    double wc = 0, wh = 0;
};

bool prolate_expand(double theta, std::vector<double> &coef, std::vector<double> &mul, int *nt,
                    int *nleg);

// radix passes of the sort by cell
int nufft_sort_passes(int ncells);
int nufft_geometry(imp_ctx *ctx, int m, int n, const float *kx, const float *ky, const float *t,
                   const float *x, const float *y, const float *z, const float *fm,
                   NuGeometry *G);
int nufft_geometry_batch(imp_ctx *ctx, int njobs, const imp_nudft_job *jobs,
                         const std::vector<char> &scan, std::vector<NuGeometry> *G);
// Predicted time of nufft_adjoint in microseconds (for the choice against
// the direct kernels).
double nufft_adjoint_us(const NuGeometry &G, int m, int ncoils);
int nufft_adjoint(imp_ctx *ctx, const NuGeometry &G, int m, int ncoils, const float *kx,
                  const float *ky, const float *t, const float *x, const float *y,
                  const float *fm, const float *phi_r, const float *phi_i, const float *d_r,
                  const float *d_i, const float *s_r, const float *s_i, float *out_r,
                  float *out_i);

// F^H d of a stack: samples [p K, (p + 1) K) repeat kx, ky, t of the first K
// at their own kz; G from the first K samples.
double nufft_stack_us(const NuGeometry &G, int K, int nrhs);
int nufft_stack_adjoint(imp_ctx *ctx, const NuGeometry &G, int K, int P, int ncoils,
                        const float *kx, const float *ky, const float *kz, const float *t,
                        const float *x, const float *y, const float *z, const float *fm,
                        const float *phi_r, const float *phi_i, const float *d_r,
                        const float *d_i, const float *s_r, const float *s_i, float *out_r,
                        float *out_i);
// coils of a group of F from the bytes per coil of its k grid and
// half-transformed grid
int nufft_forward_group(size_t grid_bytes, size_t mid_bytes, int ncoils);
double nufft_forward_us(const NuGeometry &G, int m, int ncoils);
int nufft_forward(imp_ctx *ctx, const NuGeometry &G, int m, int ncoils, const float *kx,
                  const float *ky, const float *t, const float *x, const float *y,
                  const float *fm, const float *rho_r, const float *rho_i, const float *s_r,
                  const float *s_i, float *d_r, float *d_i);

int nufft_q_geometry(imp_ctx *ctx, int m, const float *kx, const float *ky, const float *t, int Nx,
                     int Ny, int nseg, NuGeometry *G);
double nufft_q_us(const NuGeometry &G, int m, int nseg);
int nufft_q(imp_ctx *ctx, const NuGeometry &G, int m, const float *kx, const float *ky,
            const float *t, const float *phi_r, const float *phi_i, int Nx, int Ny, int nseg,
            float tau, float t0, bool cumulative, float *q_r, float *q_i);

}  // namespace imp
