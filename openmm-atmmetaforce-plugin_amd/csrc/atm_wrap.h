// Periodic images of one position: wrapping into the box, the lattice images of a box pair
// and the z-bins of a cutoff (FP32), cells and grid points (FP64), for the kernels of
// atm_kernels.hip and atm_pme.hip (and for the host program that tests them).  Positions may be any float: what is made from a
// wrapped position (cell and bin indices, cluster boxes, image counts) relies on
// 0 <= w <= L, so a coordinate too large for one FP32 step to bring home is folded again
// and, past that, put on the edge.
#pragma once
#include <hip/hip_runtime.h>
#include <cmath>

namespace atm {

__host__ __device__ inline float fold_coord(float x, float L, float invL) {
    // x - L floor(x/L) is exact on the 2^-20 grid (single rounding of an
    // exactly representable result); one correction step fixes floor() misses.
    float w = fmaf(-L, floorf(x * invL), x);
    if (w < 0.0f) w += L;
    if (w >= L) w -= L;
    return w;
}

__host__ __device__ inline float clamp_coord(float w, float L) { return w < 0.0f ? 0.0f : (w > L ? L : w); }  // (NaN stays)

__host__ __device__ inline float wrap_coord(float x, float L, float invL) {
    float w = fold_coord(x, L, invL);
    if (w < 0.0f || w > L) w = clamp_coord(fold_coord(w, L, invL), L);  // floor() missed by more than one (x beyond 4e6 L)
    return w;
}

// Triclinic box in OpenMM's reduced form (a = (L0, 0, 0), b = (tilt0, L1, 0),
// c = (tilt1, tilt2, L2)): wrap a position into the brick [0, L0) x [0, L1) x
// [0, L2), which tiles space under the lattice -- by c to 0 <= z < L2, then by b
// to 0 <= y < L1, then by a.  Each step is exact on the 2^-20 grid below 16 nm.
__host__ __device__ inline void fold_tri(const float* L, const float* invL, const float* tilt, float& px, float& py,
                                         float& pz) {
    float n = floorf(pz * invL[2]);
    const float z = fmaf(-L[2], n, pz);
    n += z < 0.f ? -1.f : (z >= L[2] ? 1.f : 0.f);
    pz = fmaf(-L[2], n, pz);
    py = fmaf(-tilt[2], n, py);
    px = fmaf(-tilt[1], n, px);
    n = floorf(py * invL[1]);
    const float y = fmaf(-L[1], n, py);
    n += y < 0.f ? -1.f : (y >= L[1] ? 1.f : 0.f);
    py = fmaf(-L[1], n, py);
    px = fmaf(-tilt[0], n, px);
    px = fold_coord(px, L[0], invL[0]);
}

__host__ __device__ inline void wrap_tri(const float* L, const float* invL, const float* tilt, float& px, float& py,
                                         float& pz) {
    fold_tri(L, invL, tilt, px, py, pz);
    if (px < 0.f || px > L[0] || py < 0.f || py > L[1] || pz < 0.f || pz > L[2]) {
        fold_tri(L, invL, tilt, px, py, pz);
        px = clamp_coord(px, L[0]);
        py = clamp_coord(py, L[1]);
        pz = clamp_coord(pz, L[2]);
    }
}

// The images n of one lattice direction (edge 1 / invL) under which |d - n L| - h < r can hold
// (reach = h + r): [n0, n1], often empty or one.  1e-4 of the edge of slack covers the rounding
// here; the caller's test of each image decides.  Boxes of wrapped positions reach at most 5
// edges over (the tilts add half an edge per image of the direction before): bounds past 8 come
// from no position, and a walk over them would not end.
constexpr float kMaxImages = 8.f;
__host__ __device__ inline void image_range(float d, float reach, float invL, int& n0, int& n1) {
    // (NaN: none)
    n0 = (int)ceilf(fmaxf(fminf(fmaf(d - reach, invL, -1e-4f), kMaxImages), -kMaxImages));
    n1 = (int)floorf(fminf(fmaxf(fmaf(d + reach, invL, 1e-4f), -kMaxImages), kMaxImages));
}

// The same for the FP64 positions of the PME evaluation.
//
// x wrapped into [0, L) and its cell of m.  Past some 4e15 L the step to the box leaves more than
// it can take off, and x has no place in the box: 0 (grid points are made from w).
__host__ __device__ inline int wrap_cell(double x, double L, double invL, int m, double* w) {
    double v = x - L * floor(x * invL);
    if (v < 0.0) v += L;
    if (v >= L) v -= L;
    if (!(v >= 0.0 && v < L)) v = 0.0;
    *w = v;
    int c = (int)(v * invL * m);
    return c < 0 ? 0 : (c >= m ? m - 1 : c);
}

// x / L without its whole part, in [0, 1] but for the rounding: the fused step keeps the half unit
// that the product lost, 1e-16 either way for a position in the box and 64 for one at 1e18 L.  Up
// to 1/2048 past either end (x of some 1e12 L) the grid point, times K <= 1024, stays in [-1, K];
// further out x has no place on the grid: 0.
__host__ __device__ inline double grid_fraction(double x, double invL) {
    const double f = fma(x, invL, -floor(x * invL));
    return f > -1.0 / 2048 && f < 1.0 + 1.0 / 2048 ? f : 0.0;
}

// The z-bins (nz of them, 1 / invZe wide, over [0, Lz]) within hz of z and one more on each
// side, as [za0, za1] and, where they wrap, [zb0, zb1] (empty: zb0 > zb1): every bin at most
// once, every index in [0, nz), whatever z, for 0 <= hz <= Lz.
__host__ __device__ inline void z_bins(float z, float hz, float invZe, float Lz, int nz, int& za0, int& za1, int& zb0,
                                       int& zb1) {
    z = fminf(fmaxf(z, 0.f), Lz);  // (NaN: 0)
    za0 = (int)floorf((z - hz) * invZe) - 1;
    za1 = (int)floorf((z + hz) * invZe) + 1;
    zb0 = 1;
    zb1 = 0;
    if (za1 - za0 + 1 >= nz) { za0 = 0; za1 = nz - 1; }
    else if (za0 < 0) { zb0 = za0 + nz; zb1 = nz - 1; za0 = 0; }
    else if (za1 >= nz) { zb0 = 0; zb1 = za1 - nz; za1 = nz - 1; }
}

}  // namespace atm
