// Rejection of whole runs of samples of a ray: bounds of their points against the box and the coarse occupancy level.
// Shared by the culling kernels; the decisions equal those of the per-sample tests in lm_common.h.
#pragma once
#include <limits.h>

#include "lm_common.h"

namespace {

// Bounds of the points of samples s0 .. s0 + n - 1 of one ray: they lie between the first and the last one (the depth
// tables are monotone, and so is o + d * z in z), widened by a margin a hundred times the rounding of the operations
// involved.  lo[k] <= pt[k] <= hi[k] for every sample of the run.  fminf / fmaxf drop NaNs; with FLAG_NAN a NaN anywhere
// on the way makes the bounds NaN (for the cell test, which must make no statement then; the box test needs no flag:
// what its bounds miss fails the per-sample test as well).
template <bool FLAG_NAN>
__device__ __forceinline__ void run_bounds(const lm_geom &g, const float *ray, float rp, int s0, int n, float *lo, float *hi) {
    const float za = lm_sample_z(g, rp, s0), zb = lm_sample_z(g, rp, s0 + n - 1);
    const float zlo = fminf(za, zb), zhi = fmaxf(za, zb);
    // the depth is a sum of two terms bounded by |near| and the ray's parameter (or by the depth itself)
    const float zm = 1e-5f * (fmaxf(fabsf(zlo), fabsf(zhi)) + fabsf(rp) + fabsf(g.near_));
    const bool z_nan = FLAG_NAN && (!(za == za) || !(zb == zb));
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float o = ray[k], d = ray[3 + k];
        const float e0 = d * (zlo - zm), e1 = d * (zhi + zm), e2 = d * (zlo + zm), e3 = d * (zhi - zm);
        const float l = o + fminf(fminf(e0, e1), fminf(e2, e3)), h = o + fmaxf(fmaxf(e0, e1), fmaxf(e2, e3));
        const float m = 1e-5f * (fabsf(o) + fmaxf(fabsf(l), fabsf(h))) + 1e-30f;
        const bool bad = FLAG_NAN && (z_nan || !(e0 == e0) || !(e1 == e1) || !(e2 == e2) || !(e3 == e3));
        lo[k] = bad ? NAN : l - m;
        hi[k] = bad ? NAN : h + m;
    }
}

// 1: every point within the bounds fails the box test (it stays on the outer side of one face).  Anything doubtful
// (NaN included) is 0.
__device__ __forceinline__ bool bounds_outside(const lm_geom &g, const float *lo, const float *hi) {
    bool outside = false;
#pragma unroll
    for (int k = 0; k < 3; ++k) outside |= (hi[k] < g.aabb[k]) | (lo[k] > g.aabb[3 + k]);
    return outside;
}

// The coarse level of a cell table (lm_pack_occupancy_coarse): blocks of 8 x 8 x 8 cells, entry b set when a cell of
// blocks b .. b + 1 (per axis) has a bit set.
constexpr int kCoarseShift = 3;
__host__ __device__ inline int coarse_dim(int cells) { return (cells + (1 << kCoarseShift) - 1) >> kCoarseShift; }

// Cell index range of the points within the bounds, per axis, with lm_cells_positive's own float operations: each of
// them is monotone (weakly, rounding included) in the coordinate when vol_inv > 0, so the floor of a point's cell
// coordinate lies between the floors of the bounds'.  Returns 0 when the bounds hold a NaN or the volume is degenerate
// (no statement), 1 with the block range [b0, b1] per axis otherwise; `none` = every index is outside the table
// (all samples are rejected by the lookup itself).
__device__ __forceinline__ bool coarse_range(const lm_geom &g, const float *lo, const float *hi, int *b0, int *b1, bool &none) {
    const int dims[3] = {g.vw, g.vh, g.vd};
    none = false;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        if (!(lo[k] <= hi[k]) || !(g.vol_inv[k] > 0.0f) || dims[k] < 2) return false;
        const float s = (float)(dims[k] - 1);
        float il = (((lo[k] - g.vol_aabb_min[k]) * g.vol_inv[k] - 1.0f) + 1.0f) / 2.0f * s;
        float ih = (((hi[k] - g.vol_aabb_min[k]) * g.vol_inv[k] - 1.0f) + 1.0f) / 2.0f * s;
        if (!(il <= ih)) return false;
        il = fminf(fmaxf(floorf(il), -2.0f), (float)dims[k]);
        ih = fminf(fmaxf(floorf(ih), -2.0f), (float)dims[k]);
        // cell index = floor + 1; indices outside 0 .. dims fail the lookup's range test
        int c0 = (int)il + 1, c1 = (int)ih + 1;
        if (c1 < 0 || c0 > dims[k]) none = true;
        c0 = max(c0, 0);
        c1 = min(c1, dims[k]);
        b0[k] = c0 >> kCoarseShift;
        b1[k] = c1 >> kCoarseShift;
    }
    return true;
}

// 1: no sample of the run can pass the cell lookup (every cell it can fall into is empty, or lies outside the table)
__device__ __forceinline__ bool coarse_empty(const lm_geom &g, const float *lo, const float *hi, int &span) {
    int b0[3], b1[3];
    bool none;
    span = INT_MAX;
    if (!coarse_range(g, lo, hi, b0, b1, none)) return false;
    if (none) return true;
    span = max(max(b1[0] - b0[0], b1[1] - b0[1]), b1[2] - b0[2]);
    if (span > 1) return false;
    const int nx = coarse_dim(g.vw + 1), ny = coarse_dim(g.vh + 1);
    return g.vol_coarse[((size_t)b0[2] * ny + b0[1]) * nx + b0[0]] == 0;
}

}  // namespace
