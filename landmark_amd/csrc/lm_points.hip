// Density features of many given points: the points are put in order of where they lie, then every part of a plane is read
// once.
//
// Points in no order read four texels each from anywhere in tables far larger than the caches: 2^24 points on three planes
// of 2048^2 x 64 channels move 51 GB for 3.2 GB of table.  Here:
//   k_bin_decide   looks at a sample: points that come in some order, or crowd in parts of a plane, meet in the caches by
//                  themselves and go to k_density_xyz, as before (the kernels below return at once, and it does otherwise);
//   k_bin_count, k_bin_scan, k_bin_scatter  records (x, y, z, number of the point) sorted by cubic block of the volume, about
//                  kBinPoints points each; a block is one or more units of up to kUnit points;
//   k_bin_order    the points of a unit by sub-tile of each plane, as 16-bit positions within the unit, and where each
//                  sub-tile's points start;
//   k_bin_density  per plane: a workgroup per sub-tile of a column (the blocks over one another as the plane sees them): its
//                  texels into LDS once, then all its points from there, C / 4 lanes to a point.
// Sums stay with the records until the last plane writes them by point number.  The blocks of a column are worked on by one
// XCD at about the same time and stay in its L2, so that records are read from memory once per plane whatever the order
// within a unit.  A block of too many points becomes several units, a column of many units several groups, and a sub-tile
// with few points is not staged, its points read the table directly.
// 2^24 points, three planes of 2048^2 x 64 channels: 8.8 -> 3.2 ms (kernel trace: sorting 0.58, planes 0.77 + 0.84 + 1.12; the last
// writes 4 bytes per point anywhere in 64 MB).  What bounds a plane: 2 KB of LDS reads and 512 bytes of line texels per point, 45
// vector instructions per four points, each 0.25 - 0.4 ms by itself, and the round trip task -> units -> order -> record -> line
// of a task that takes 15 us, three workgroups to a compute unit.  Measured on the way: records sorted again per orientation instead
// of 16-bit positions 3.6 ms (moving 20 bytes per point cost more than the planes' locality gained); texels through registers
// in a loop over tasks 3.8 (spills); two texel halves per lane (8 lanes per point) 3.7; line texels two points ahead 3.3.
#include <algorithm>

#include "lm_common.h"
#include "lm_gather.h"

namespace {

constexpr int kScatter = 1024;           // threads of the sorting kernels
constexpr int kPer = 16;                 // points per thread of a sorting workgroup
constexpr int kUnit = kScatter * kPer;   // points of a unit, at most
constexpr int kBinPoints = 10000;        // points of a block, on average
constexpr int kMaxSide = 12;             // blocks per axis
constexpr int kMaxBins = kMaxSide * kMaxSide * kMaxSide;
constexpr int kSubMax = 1024;            // sub-tiles of a column
constexpr int kGroup = 16;               // units of a group, at most
constexpr int kTaskThreads = 512;
constexpr int kTileFloats = 144 * 64;    // a sub-tile with its right and lower neighbours' texels
static_assert(kTileFloats / 4 % LM_WAVE == 0, "whole transfers");
constexpr int64_t kSlice = (int64_t)1 << 24;  // points per pass over the tables

typedef float f4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) const void *gptr;
typedef __attribute__((address_space(3))) void *lptr;
// element at a 32-bit byte offset from a uniform base: one address register per load
template <typename V> __device__ __forceinline__ V at_bytes(const void *base, uint32_t offset) {
    return *reinterpret_cast<const V *>(static_cast<const char *>(base) + offset);
}

// strip of an axis a normalised coordinate falls into; everything outside (and NaN) goes to an edge strip
__device__ __forceinline__ int strip_of(float c, int n) {
    return (int)fminf(fmaxf((c + 1.0f) * (0.5f * (float)n), 0.0f), (float)(n - 1));
}
__device__ __forceinline__ uint32_t block_of(int side, float x, float y, float z) {
    return (uint32_t)((strip_of(x, side) * side + strip_of(y, side)) * side + strip_of(z, side));
}

__device__ __forceinline__ int pick_step(const int *v, int ax) { return ax == 0 ? v[0] : ax == 1 ? v[1] : v[2]; }

struct Axes {
    int n;
    int8_t ax0[LM_MAX_PLANES], ax1[LM_MAX_PLANES];
    int W[LM_MAX_PLANES], H[LM_MAX_PLANES];
};

// One workgroup looks at kSample points and their successors: *flag = 1 if fewer than one in eight shares its 1 / 64 x 1 / 64 of
// the first plane with its successor, and no such part of a plane holds more than kCrowd points of the sample (one on average:
// of 4096 evenly spread points some part on one of three orientations gets more than 16 once in 7e10 calls, ten or more once in
// 700).  It also clears the counters.
constexpr int kSample = 4096, kCells = 64, kCrowd = 16;
__global__ __launch_bounds__(kScatter) void k_bin_decide(Axes axes, const float *__restrict__ xyz, uint32_t M, uint32_t *__restrict__ counts,
                                                         int n_counts, uint32_t *__restrict__ queue, uint32_t *__restrict__ flag) {
    __shared__ uint32_t s_cell[kCells * kCells], s_same, s_crowded;
    uint32_t same = 0, most = 0;
    constexpr int kEach = kSample / kScatter;
    for (int i = threadIdx.x; i < n_counts; i += kScatter) counts[i] = 0u;
    if ((int)threadIdx.x < axes.n * LM_XCDS) queue[threadIdx.x] = 0u;
    if (threadIdx.x == 0) s_same = s_crowded = 0u;
    float q[kEach][3], next[kEach][3];
    const uint32_t stride = M / kSample;
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
        const uint32_t k = i * kScatter + threadIdx.x;
        const size_t p = min(k * stride + (stride ? (k * 2654435761u >> 8) % stride : 0u), M - 2u);  // somewhere in the k-th part
#pragma unroll
        for (int d = 0; d < 3; ++d) { q[i][d] = xyz[3 * p + d]; next[i][d] = xyz[3 * p + 3 + d]; }
    }
    for (int k = 0; k < axes.n; ++k) {
        const int ax0 = axes.ax0[k], ax1 = axes.ax1[k];
        if (k && axes.ax0[k - 1] == ax0 && axes.ax1[k - 1] == ax1) continue;
        __syncthreads();
        for (int i = threadIdx.x; i < kCells * kCells; i += kScatter) s_cell[i] = 0u;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kEach; ++i) {
            const int cell = strip_of(pick(q[i], ax0), kCells) * kCells + strip_of(pick(q[i], ax1), kCells);
            atomicAdd(&s_cell[cell], 1u);
            if (k == 0) same += cell == strip_of(pick(next[i], ax0), kCells) * kCells + strip_of(pick(next[i], ax1), kCells);
        }
        __syncthreads();
        for (int i = threadIdx.x; i < kCells * kCells; i += kScatter) most = max(most, s_cell[i]);
    }
    if (most > (uint32_t)kCrowd) atomicAdd(&s_crowded, 1u);
    if (same) atomicAdd(&s_same, same);
    __syncthreads();
    if (threadIdx.x == 0) *flag = s_same < kSample / 8 && s_crowded == 0u;
}

// counts[block] += points
__global__ __launch_bounds__(kScatter) void k_bin_count(const uint32_t *__restrict__ flag, int side, const float *__restrict__ xyz, uint32_t M,
                                                        uint32_t *__restrict__ counts) {
    if (*flag == 0u) return;
    __shared__ uint32_t s_count[kMaxBins];
    const int n = side * side * side;
    for (int i = threadIdx.x; i < n; i += kScatter) s_count[i] = 0u;
    __syncthreads();
    for (uint32_t p = blockIdx.x * kScatter + threadIdx.x; p < M; p += gridDim.x * kScatter)
        atomicAdd(&s_count[block_of(side, xyz[3 * (size_t)p], xyz[3 * (size_t)p + 1], xyz[3 * (size_t)p + 2])], 1u);
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += kScatter)
        if (s_count[i]) atomicAdd(counts + i, s_count[i]);
}

// first texel a column's strip can reach: one before its own, for the roundings
__device__ __forceinline__ int strip_texel(int strip, int side, int size) {
    return max(0, strip * (size - 1) / side - 1);
}
// The columns of a plane and their units, kGroup units to a group (~0u past the last), with the column's first texel.
struct Group {
    int x, y;
    uint32_t unit[kGroup];
};

// One workgroup: counts -> first position of every block (in place, the scatter's cursors), the units, {first position,
// points, block} each, and the groups of every plane.
__global__ __launch_bounds__(kScatter) void k_bin_scan(const uint32_t *__restrict__ flag, int side, Axes axes, uint32_t *__restrict__ count,
                                                       uint4 *__restrict__ units, uint32_t *__restrict__ n_units, Group *__restrict__ groups,
                                                       uint32_t max_groups, uint32_t *__restrict__ n_groups) {
    __shared__ uint2 s_sum[kScatter];
    __shared__ uint32_t s_unit[kMaxBins + 1];  // first unit of a block
    constexpr int kEach = (kMaxBins + kScatter - 1) / kScatter;
    if (*flag == 0u) return;
    const int bins = side * side * side, t = (int)threadIdx.x;
    uint32_t n[kEach];
    uint2 mine = {0u, 0u};  // points, units
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
        const int at = t * kEach + i;
        n[i] = at < bins ? count[at] : 0u;
        mine.x += n[i];
        mine.y += (n[i] + kUnit - 1) / kUnit;
    }
    s_sum[t] = mine;
    __syncthreads();
    for (int d = 1; d < kScatter; d <<= 1) {
        const uint2 before = t >= d ? s_sum[t - d] : make_uint2(0u, 0u);
        __syncthreads();
        s_sum[t].x += before.x;
        s_sum[t].y += before.y;
        __syncthreads();
    }
    if (t == kScatter - 1) *n_units = s_unit[bins] = s_sum[t].y;
    uint32_t first = s_sum[t].x - mine.x, u = s_sum[t].y - mine.y;
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
        const int at = t * kEach + i;
        if (at >= bins) break;
        count[at] = first;
        s_unit[at] = u;
        const uint32_t parts = (n[i] + kUnit - 1) / kUnit, each = parts ? (n[i] + parts - 1) / parts : 0u;
        for (uint32_t k = 0; k < parts; ++k, ++u) units[u] = make_uint4(first + k * each, min(each, n[i] - k * each), (uint32_t)at, 0u);
        first += n[i];
    }
    __syncthreads();
    const int step[3] = {side * side, side, 1};
    for (int k = 0; k < axes.n; ++k) {
        const int ax0 = axes.ax0[k], ax1 = axes.ax1[k], axl = 3 - ax0 - ax1;
        const int base = (t / side) * pick_step(step, ax0) + (t % side) * pick_step(step, ax1), along = pick_step(step, axl);
        uint32_t units_here = 0;
        if (t < side * side)
            for (int i = 0; i < side; ++i) units_here += s_unit[base + i * along + 1] - s_unit[base + i * along];
        const uint32_t parts = (units_here + kGroup - 1) / kGroup;
        __syncthreads();
        s_sum[t].x = parts;
        __syncthreads();
        for (int d = 1; d < 256; d <<= 1) {  // (side * side <= 256)
            const uint32_t before = t >= d && t < 256 ? s_sum[t - d].x : 0u;
            __syncthreads();
            if (t < 256) s_sum[t].x += before;
            __syncthreads();
        }
        if (t == 255) n_groups[k] = s_sum[t].x;
        if (t < side * side) {
            Group *g = groups + (size_t)k * max_groups + (s_sum[t].x - parts);
            const int x = strip_texel(t / side, side, axes.W[k]), y = strip_texel(t % side, side, axes.H[k]);
            uint32_t j = 0;
            for (int i = 0; i < side; ++i)
                for (uint32_t v = s_unit[base + i * along]; v < s_unit[base + i * along + 1]; ++v, ++j) {
                    g[j / kGroup].x = x;
                    g[j / kGroup].y = y;
                    g[j / kGroup].unit[j % kGroup] = v;
                }
            for (; j % kGroup; ++j) g[j / kGroup].unit[j % kGroup] = ~0u;
        }
    }
}

__global__ __launch_bounds__(kScatter) void k_bin_scatter(const uint32_t *__restrict__ flag, int side, const float *__restrict__ xyz, uint32_t M,
                                                          uint32_t *__restrict__ cursor, float4 *__restrict__ rec) {
    __shared__ uint32_t s_at[kMaxBins];
    if (*flag == 0u) return;
    const int bins = side * side * side;
    for (int i = threadIdx.x; i < bins; i += kScatter) s_at[i] = 0u;
    __syncthreads();
    float x[kPer], y[kPer], z[kPer];
    uint32_t where[kPer];  // block, and rank among the workgroup's points of that block
    const uint32_t p0 = blockIdx.x * kUnit + threadIdx.x;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const size_t p = min(p0 + i * kScatter, M - 1u);
        x[i] = xyz[3 * p]; y[i] = xyz[3 * p + 1]; z[i] = xyz[3 * p + 2];
    }
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const uint32_t b = block_of(side, x[i], y[i], z[i]);
        if (p0 + i * kScatter < M) where[i] = (b << 16) + atomicAdd(&s_at[b], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < bins; i += kScatter) {
        const uint32_t n = s_at[i];
        if (n) s_at[i] = atomicAdd(cursor + i, n);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const uint32_t p = p0 + i * kScatter;
        if (p >= M) break;
        rec[s_at[where[i] >> 16] + (where[i] & 0xffffu)] = make_float4(x[i], y[i], z[i], __uint_as_float(p));
    }
}

// first corner of a point along an axis, as plane_taps clamps it
__device__ __forceinline__ int first_texel(float c, int size) {
    const int i = (int)fminf(fmaxf(floorf(unnorm(c, size)), -2.0f), (float)size);
    return min(max(i, 0), size - 1);
}

// How a plane's part over a column is cut into sub-tiles: tx x ty texels each, nx x ny of them, counted from the column's
// first texel.  v / tx = v * mx >> 16 for the texels of a column.
struct Cut {
    int tx, ty, nx, ny;
    uint32_t mx, my, mt, mn;  // of tx, ty, tx + 1 and nx
};
// strip of a block along an axis
__device__ __forceinline__ int strip_along(int block, int side, int axis) {
    return axis == 2 ? block % side : axis == 1 ? block / side % side : block / (side * side);
}

struct Cuts {
    Cut of[LM_MAX_PLANES];
};

// Per plane (blockIdx.y): order[unit's positions] = the unit's points by sub-tile, as positions within the unit; tab[unit][s] = first of sub-tile s
__global__ __launch_bounds__(kScatter) void k_bin_order(const uint32_t *__restrict__ flag, PlaneSet ps, int side, Cuts cuts,
                                                        const uint4 *__restrict__ units, const uint32_t *__restrict__ n_units,
                                                        const float4 *__restrict__ rec, size_t order_step, size_t tab_step,
                                                        uint16_t *__restrict__ order, uint16_t *__restrict__ tab) {
    __shared__ uint32_t s_next[kSubMax];
    __shared__ __align__(16) uint16_t s_order[kUnit];
    if (*flag == 0u) return;
    const lm_plane pl = ps.p[blockIdx.y];
    const Cut cut = cuts.of[blockIdx.y];
    const unsigned lane = lm_lane();
    const int ns = cut.nx * cut.ny;
    const uint32_t total = *n_units;
    order += blockIdx.y * order_step;
    tab += blockIdx.y * tab_step;
    for (uint32_t u = blockIdx.x; u < total; u += gridDim.x) {
        const uint4 unit = units[u];
        const uint32_t n = unit.y;
        const float4 *my = rec + unit.x;
        __syncthreads();
        const int ox = strip_texel(strip_along((int)unit.z, side, pl.ax0), side, pl.W), oy = strip_texel(strip_along((int)unit.z, side, pl.ax1), side, pl.H);
        for (int i = threadIdx.x; i < ns; i += kScatter) s_next[i] = 0u;
        __syncthreads();
        uint32_t where[kPer];
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const uint32_t byte = 16u * min(threadIdx.x + i * kScatter, n - 1u);
            const uint32_t x = (uint32_t)max(first_texel(at_bytes<float>(my, byte + 4u * pl.ax0), pl.W) - ox, 0),
                           y = (uint32_t)max(first_texel(at_bytes<float>(my, byte + 4u * pl.ax1), pl.H) - oy, 0);
            where[i] = min((y * cut.my) >> 16, (uint32_t)cut.ny - 1u) * (uint32_t)cut.nx + min((x * cut.mx) >> 16, (uint32_t)cut.nx - 1u);
        }
#pragma unroll
        for (int i = 0; i < kPer; ++i)
            if (threadIdx.x + i * kScatter < n) where[i] = (where[i] << 16) + atomicAdd(&s_next[where[i]], 1u);
        __syncthreads();
        if (threadIdx.x < LM_WAVE) {
            uint16_t *my_tab = tab + (size_t)u * (ns + 1);
            uint32_t before = 0;
            for (int base = 0; base < ns; base += LM_WAVE) {
                const int i = base + (int)lane;
                const uint32_t mine = i < ns ? s_next[i] : 0u;
                uint32_t incl = mine;
#pragma unroll
                for (int d = 1; d < LM_WAVE; d <<= 1) {
                    const uint32_t v = __shfl_up(incl, d);
                    if ((int)lane >= d) incl += v;
                }
                if (i < ns) {
                    s_next[i] = before + incl - mine;
                    my_tab[i] = (uint16_t)(before + incl - mine);
                }
                before += __shfl(incl, LM_WAVE - 1);
            }
            if (lane == 0) my_tab[ns] = (uint16_t)n;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kPer; ++i)
            if (threadIdx.x + i * kScatter < n) s_order[s_next[where[i] >> 16] + (where[i] & 0xffffu)] = (uint16_t)(threadIdx.x + i * kScatter);
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < n; i += kScatter) order[unit.x + i] = s_order[i];
    }
}

// a point's footprint as the lanes of its group read it
struct __align__(16) Item {
    uint32_t corner;  // byte of the first corner in the staged sub-tile; or column | row << 8, 1 << 16: the next column counts, 1 << 17: the next row
    float w00, w01, w10, w11;
    uint32_t line;    // byte of the line's lower texel, + 1: the upper one is the same texel
    float l0, l1;
};

// A workgroup per sub-tile and group: the sub-tile's texels into LDS, then its points from there.
// mode: 1 = the points' first plane (no sum yet), 2 = their last (write by point number)
template <int C, bool NONLINEAR>
__global__ __launch_bounds__(kTaskThreads) __attribute__((amdgpu_waves_per_eu(6))) void k_bin_density(
    const uint32_t *__restrict__ flag, lm_plane plane, Cut cut, const float *__restrict__ den_w, const Group *__restrict__ groups, const uint32_t *__restrict__ n_groups, uint32_t *__restrict__ queue,
    const uint4 *__restrict__ units, const uint16_t *__restrict__ tab, const uint16_t *__restrict__ order, const float4 *__restrict__ rec,
    float *__restrict__ sum, int mode, float *__restrict__ out) {
    constexpr int LPP = C / 4;  // lanes per point
    constexpr int kWaves = kTaskThreads / LM_WAVE;
    constexpr int kStage = (kTileFloats / 4 + kTaskThreads - 1) / kTaskThreads;
    __shared__ __align__(16) float s_tile[kTileFloats];
    __shared__ Item s_item[kWaves][LM_WAVE];
    // a task's units: points up to and with the unit's, its records, its first in order; this task's and the next one's
    __shared__ uint32_t s_ends[2][kGroup], s_units[2][kGroup], s_firsts[2][kGroup], s_task[2];
    auto uniform = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };
    if (*flag == 0u) return;
    // Neighbouring tasks on one XCD at a time (workgroup b runs on XCD b % 8), handed out one by one: with a fixed share per
    // workgroup the launch took 937 instead of 836 us (first plane of 2^24 points and 2048^2 x 64 channels)
    const uint32_t ns = (uint32_t)(cut.nx * cut.ny), total = *n_groups * ns, each = (total + LM_XCDS - 1) / LM_XCDS;
    const uint32_t xcd = blockIdx.x % LM_XCDS, xcd_end = min((xcd + 1u) * each, total);
    auto look_up = [&](uint32_t buf, unsigned lane) {  // the next task and its units, by one wave
        uint32_t task = 0;
        if (lane == 0) task = s_task[buf] = xcd * each + atomicAdd(queue + xcd, 1u);
        task = uniform(task);
        if (task >= xcd_end) return;
        const uint32_t g = task / ns, s = task - g * ns;
        uint32_t n = 0, first = 0, start = 0;
        if (lane < kGroup) {
            const uint32_t u = groups[g].unit[lane];
            if (u != ~0u) {
                const uint16_t *t = tab + (size_t)u * (ns + 1) + s;
                start = units[u].x;
                first = start + t[0];
                n = (uint32_t)t[1] - t[0];
            }
        }
#pragma unroll
        for (int d = 1; d < kGroup; d <<= 1) {
            const uint32_t v = __shfl_up(n, d);
            if ((int)lane >= d) n += v;
        }
        if (lane < kGroup) { s_ends[buf][lane] = n; s_units[buf][lane] = start; s_firsts[buf][lane] = first; }
    };
    if (threadIdx.x < LM_WAVE) look_up(0u, lm_lane());
    for (uint32_t buf = 0;; buf ^= 1u) {
        // Nothing below that depends on the lane or the plane alone is to be kept in registers from task to task
        uint32_t tid = threadIdx.x;
        lm_plane pl = plane;
        asm volatile("" : "+v"(tid), "+s"(pl.W), "+s"(pl.H), "+s"(pl.Len));
        const unsigned lane = tid % LM_WAVE, wave = uniform(tid / LM_WAVE), group = lane / LPP, in = lane % LPP;
        // A group's items lie in an order of its own, so that the groups of a wave, reading their k-th at once, meet in different
        // banks: with one order for all, 28 % of the LDS cycles were conflicts, now 4 % (0.67 -> 0.50 M busy cycles per CU in the first
        // of three planes); 2^24 points, 3 x 2048^2 x 64 channels: 3211 -> 3185 us, 16 M points, 3 x 1000^2 x 32: 2320 -> 2273 us
        const unsigned twist = group % LPP;
        __syncthreads();  // the task before has left LDS, this one's units are there
        const uint32_t task = uniform(s_task[buf]);
        if (task >= xcd_end) break;
        const uint32_t g = task / ns, s = task - g * ns;
        const uint32_t *s_end = s_ends[buf], *s_unit = s_units[buf], *s_first = s_firsts[buf];
        const int row = (int)((s * cut.mn) >> 16), x0 = groups[g].x + ((int)s - row * cut.nx) * cut.tx, y0 = groups[g].y + row * cut.ty;
        const int cols = min(cut.tx + 1, pl.W - x0), rows = min(cut.ty + 1, pl.H - y0);
        const float *Ln = reinterpret_cast<const float *>(pl.line);
        const float *origin = reinterpret_cast<const float *>(pl.plane) + ((size_t)y0 * pl.W + x0) * C;
        const uint32_t tile_pitch = (uint32_t)(cut.tx + 1) * C;
        const uint32_t count = uniform(s_end[kGroup - 1]);
        const uint32_t share = (count + kWaves - 1) / kWaves, p_end = min((wave + 1) * share, count);
        // few points: reading the sub-tile would move more than their footprints
        const bool staged = count && 2u * count >= (uint32_t)(cols * rows);
        if (staged) {
            // straight into LDS: a wave's 64 transfers of 16 bytes lie behind one another there
#pragma unroll
            for (int i = 0; i < kStage; ++i) {
                const uint32_t k0 = wave * LM_WAVE + i * kTaskThreads, k = k0 + lane, t = k / (C / 4), y = (t * cut.mt) >> 16, x = t - y * (uint32_t)(cut.tx + 1);
                // (past the sub-tile: its last texel once more)
                const uint32_t byte = (min(y, (uint32_t)rows - 1u) * (uint32_t)pl.W + min(x, (uint32_t)cols - 1u)) * (C * 4u) + 16u * (k % (C / 4));
                if (k0 < kTileFloats / 4) __builtin_amdgcn_global_load_lds((gptr)((const char *)origin + byte), (lptr)(s_tile + 4 * k0), 16, 0, 0);
            }
        }
        // lanes g * LPP + t hold point g * per + t of a batch of m points, t < per
        auto batch_of = [&](uint32_t p) { return p < p_end ? min(p_end - p, (uint32_t)LM_WAVE) : 0u; };
        auto per_of = [&](uint32_t m) { return (m + LM_WAVE / LPP - 1) / (LM_WAVE / LPP); };
        uint32_t m = batch_of(wave * share), at = 0;
        float cx = 0.0f, cy = 0.0f, cl = 0.0f;  // the point's coordinates on the plane and on the line
        float before = 0.0f;
        auto fetch_points = [&](uint32_t p) {
            const uint32_t i = p + min(group * per_of(m) + in, m - 1u);
            uint32_t k = 0;  // the unit point i is in: the first with s_end > i
#pragma unroll
            for (uint32_t d = kGroup / 2; d; d >>= 1)
                if (s_end[k + d - 1] <= i) k += d;
            at = s_unit[k] + order[s_first[k] + (i - (k ? s_end[k - 1] : 0u))];
            cx = at_bytes<float>(rec, at * 16u + 4u * pl.ax0);
            cy = at_bytes<float>(rec, at * 16u + 4u * pl.ax1);
            cl = at_bytes<float>(rec, at * 16u + 4u * pl.axl);
            if (!(mode & 1)) before = at_bytes<float>(sum, at * 4u);
        };
        if (m) fetch_points(wave * share);
        if (wave == kWaves - 1) look_up(buf ^ 1u, lane);  // (the wave with the fewest points)
        if (staged) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the transfers have landed
            __syncthreads();
        }
        for (uint32_t p = wave * share; m; p += m, m = batch_of(p)) {
            const uint32_t per = per_of(m);
            if (p != wave * share) fetch_points(p);
            // Footprints the lanes of a group read from LDS.  Where all of the batch lie inside the table, in a staged
            // sub-tile, corners and line texels are fixed steps apart; else (a clamped corner, a table read directly) the steps
            // are in the item.
            bool fast;
            {
                const Taps2 t2 = plane_taps(pl, cx, cy);
                const Taps1 t1 = line_taps(pl, cl);
                const int x = first_texel(cx, pl.W) - x0, y = first_texel(cy, pl.H) - y0;
                const bool right = t2.o01 != t2.o00, below = t2.o10 != t2.o00, upper = t1.o1 != t1.o0;
                fast = staged && __all(right && below && upper && x >= 0 && x < cut.tx && y >= 0 && y < cut.ty);
                Item it;
                it.w00 = t2.w00; it.w01 = t2.w01; it.w10 = t2.w10; it.w11 = t2.w11;
                it.l0 = t1.w0; it.l1 = t1.w1;
                it.line = 4u * (uint32_t)t1.o0 + (fast || upper ? 0u : 1u);
                if (fast) it.corner = 4u * (uint32_t)(y * (int)tile_pitch + x * C);
                else it.corner = (uint32_t)min(max(x, 0), cols - 1) | ((uint32_t)min(max(y, 0), rows - 1) << 8) | (right ? 1u << 16 : 0u) | (below ? 1u << 17 : 0u);
                s_item[wave][group * LPP + (in ^ twist)] = it;
            }
            lm_wave_lds_fence();
            float mine = 0.0f;  // the value of this lane's point
            const Item *items = s_item[wave] + group * LPP;  // point k of the group: items[k ^ twist]
            const uint32_t channel = 16u * in;
            auto value = [&](const Item &it, const f4 &a, const f4 &bb, const f4 &cc, const f4 &d, const f4 &la, const f4 &lb) {
                float v = 0.0f;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float pv = a[i] * it.w00;
                    pv = fmaf(bb[i], it.w01, pv);
                    pv = fmaf(cc[i], it.w10, pv);
                    pv = fmaf(d[i], it.w11, pv);
                    const float lv = fmaf(lb[i], it.l1, la[i] * it.l0);
                    if constexpr (NONLINEAR) v = fmaf(at_bytes<float>(den_w, channel + 4u * i), pv * lv, v);
                    else v = fmaf(pv, lv, v);
                }
                return v;
            };
            auto group_sum = [](float v) {  // over the point's lanes, on all of them
                v = quad_sum(v);
                if constexpr (LPP >= 8) v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, false));   // mirrored within 8 lanes
                if constexpr (LPP >= 16) v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xf, 0xf, false));  // within 16
                return v;
            };
            if (fast) {
                f4 l0, l1;
                auto request = [&](uint32_t k) {  // the line texels of the group's next point
                    const uint32_t line = items[k ^ twist].line;
                    l0 = at_bytes<f4>(Ln, line + channel);
                    l1 = at_bytes<f4>(Ln, line + channel + 4u * C);
                };
                request(0u);
                for (uint32_t k = 0; k < per; ++k) {
                    __builtin_amdgcn_sched_barrier(0);
                    const Item it = items[k ^ twist];
                    const float *c = s_tile + (it.corner + channel) / 4u;
                    const float v = group_sum(value(it, *reinterpret_cast<const f4 *>(c), *reinterpret_cast<const f4 *>(c + C), *reinterpret_cast<const f4 *>(c + tile_pitch),
                                                    *reinterpret_cast<const f4 *>(c + tile_pitch + C), l0, l1));
                    if (in == k) mine = v;
                    __builtin_amdgcn_sched_barrier(0);
                    if (k + 1 < per) request(k + 1);
                }
            } else {
                for (uint32_t k = 0; k < per; ++k) {
                    const Item it = items[k ^ twist];
                    const uint32_t cn = it.corner, line = (it.line & ~3u) + channel, up = it.line & 1u ? 0u : 4u * C;
                    const uint32_t o00 = (((cn >> 8) & 255u) * (uint32_t)pl.W + (cn & 255u)) * (4u * C) + channel, dx = (cn >> 16) & 1u ? 4u * C : 0u,
                                   dy = cn >> 17 ? (uint32_t)pl.W * (4u * C) : 0u;
                    const float v = group_sum(value(it, at_bytes<f4>(origin, o00), at_bytes<f4>(origin, o00 + dx), at_bytes<f4>(origin, o00 + dy),
                                                    at_bytes<f4>(origin, o00 + dy + dx), at_bytes<f4>(Ln, line), at_bytes<f4>(Ln, line + up)));
                    if (in == k) mine = v;
                }
            }
            if (in < per && group * per + in < m) {
                mine += mode & 1 ? 0.0f : before;
                if (!(mode & 2)) sum[at] = mine;
                else out[at_bytes<uint32_t>(rec, at * 16u + 12u)] = NONLINEAR ? fmaxf(mine, 0.0f) : mine;
            }
            lm_wave_lds_fence();
        }
    }
}

struct Plan {
    int side;               // blocks per axis
    Cuts cuts;
    Axes axes;
    int64_t slice;          // points per pass
    uint32_t max_units, max_groups, max_subs;
    size_t o_counts, o_queue, o_flag, o_n_units, o_n_groups, o_units, o_groups, o_tab, o_order, o_rec, o_sum, total;
};

// The cut with the fewest texels to read, neighbours included
bool cut_plane(const lm_plane &p, int side, Cut &best) {
    // texels of a column: its own, rounded up, and the margins
    const int w = std::min(p.W, (p.W - 1) / side + 4), h = std::min(p.H, (p.H - 1) / side + 4), room = kTileFloats / p.C;
    int64_t cost = INT64_MAX;
    auto magic = [](int d) { return 65536u / (uint32_t)d + 1u; };
    for (int nx = 1; nx <= std::min(w, kSubMax); ++nx) {
        const int tx = (w + nx - 1) / nx;
        if (2 * (tx + 1) > room || tx > 250) continue;
        int ty = std::min(std::min(room / (tx + 1) - 1, h), 250);
        const int ny = (h + ty - 1) / ty;
        ty = (h + ny - 1) / ny;
        // v * magic >> 16 is exact while v * divisor < 65536
        if ((int64_t)p.W * side >= 1 << 30 || (int64_t)p.H * side >= 1 << 30) return false;
        if (w * tx >= 65536 || h * ty >= 65536 || (kTileFloats / p.C + kTaskThreads) * (tx + 1) >= 65536 || kSubMax * nx >= 65536) continue;
        const int64_t c = (int64_t)nx * ny * (tx + 1) * (ty + 1);
        if ((int64_t)nx * ny <= kSubMax && c < cost) {
            cost = c;
            best = {tx, ty, nx, ny, magic(tx), magic(ty), magic(tx + 1), magic(nx)};
        }
    }
    return cost != INT64_MAX;
}

bool plan_density(const lm_plane *planes, int n, int64_t M, Plan &pn) {
    if (M < kSample || planes[0].dtype != LM_F32) return false;
    const int64_t slices = (M + kSlice - 1) / kSlice;
    pn.slice = (M + slices - 1) / slices;
    pn.side = 1;
    while (pn.side < kMaxSide && (int64_t)pn.side * pn.side * pn.side * kBinPoints < pn.slice) ++pn.side;
    pn.max_subs = 0;
    pn.axes.n = n;
    for (int k = 0; k < n; ++k) {
        const lm_plane &p = planes[k];
        if (p.C != 16 && p.C != 32 && p.C != 64) return false;
        if (p.ax0 == p.ax1 || p.axl == p.ax0 || p.axl == p.ax1) return false;
        if ((int64_t)p.Len * p.C >= 1 << 30 || (int64_t)p.W * p.C >= 1 << 22) return false;  // 32-bit byte offsets into a line, into 251 rows of a plane
        pn.axes.ax0[k] = (int8_t)p.ax0;
        pn.axes.ax1[k] = (int8_t)p.ax1;
        pn.axes.W[k] = p.W;
        pn.axes.H[k] = p.H;
        if (!cut_plane(p, pn.side, pn.cuts.of[k])) return false;
        pn.max_subs = std::max(pn.max_subs, (uint32_t)(pn.cuts.of[k].nx * pn.cuts.of[k].ny));
    }
    const int bins = pn.side * pn.side * pn.side;
    pn.max_units = (uint32_t)(bins + pn.slice / kUnit + 1);
    pn.max_groups = (uint32_t)(pn.side * pn.side + pn.max_units / kGroup + 1);
    pn.total = 0;
    auto carve = [&](size_t bytes) {
        const size_t at = pn.total;
        pn.total = (pn.total + bytes + 255) & ~(size_t)255;
        return at;
    };
    pn.o_counts = carve((size_t)bins * 4);
    pn.o_queue = carve((size_t)n * LM_XCDS * 4);
    pn.o_flag = carve(4);
    pn.o_n_units = carve(4);
    pn.o_n_groups = carve((size_t)n * 4);
    pn.o_units = carve((size_t)pn.max_units * 16);
    pn.o_groups = carve((size_t)n * pn.max_groups * sizeof(Group));
    pn.o_tab = carve((size_t)n * pn.max_units * (pn.max_subs + 1) * 2);
    pn.o_order = carve((size_t)n * pn.slice * 2);
    pn.o_rec = carve((size_t)pn.slice * 16);
    pn.o_sum = carve((size_t)pn.slice * 4);
    return true;
}

}  // namespace

int lm_check_planes(const lm_plane *planes, int32_t n, int *dtype_out, int *K_out);

// Where it pays.  Whole calls with k_density_xyz / here, three planes, evenly spread points in no order: 2048^2 x 64 channels,
// 2^24 points 8800 / 3200 us, 6 million 3310 / 1740, 3 million (fewer than texels) 1690 / 1560; 1000^2 x 32, 2^24 points 4870 /
// 2240; 512^2 x 64, 2^24 points 6940 / 2710.  Points that k_bin_decide sends back cost 40 - 60 us more than without a look:
// 2^24 points in a twentieth of the box 4037 / 4077, all at one place 2146 / 2207, on a lattice in its order 4244 / 4290.  The line
// at 1.2e9 channels (6 million points of 192) keeps that to a fifteenth of the shortest call that gains nothing (0.8 ms; others take
// up to 3.3 ms); below it evenly spread points would still gain (2 million points of 512^2 x 64 860 / 430).
static bool density_pays(const lm_plane *planes, int n, int64_t M) {
    int64_t channels = 0, bytes = 0, texels = 0;
    for (int k = 0; k < n; ++k) {
        channels += planes[k].C;
        bytes += (int64_t)planes[k].H * planes[k].W * planes[k].C * 4;
        texels = std::max(texels, (int64_t)planes[k].H * planes[k].W);
    }
    return M >= texels && M * channels >= 1200000000ll && bytes >= (int64_t)64 << 20;
}

extern "C" size_t lm_gather_density_workspace_bytes(const lm_plane *planes, int32_t n_planes, int64_t M) {
    int dtype;
    Plan pn;
    if (lm_check_planes(planes, n_planes, &dtype, nullptr) || !density_pays(planes, n_planes, M)) return 0;
    return plan_density(planes, n_planes, M, pn) ? pn.total : 0;
}

extern "C" int lm_gather_density_binned(const lm_plane *planes, int32_t n_planes, const float *density_basis, const float *xyz,
                                        int64_t M, float *out, void *workspace, size_t workspace_bytes, void *stream) {
    int dtype;
    if (int rc = lm_check_planes(planes, n_planes, &dtype, nullptr)) return rc;
    LM_REQUIRE(M >= 0, "negative count");
    if (M == 0) return LM_OK;
    LM_REQUIRE(xyz && out && workspace && lm_aligned16(workspace), "null or misaligned buffer");
    Plan pn;
    if (!plan_density(planes, n_planes, M, pn)) LM_FAIL(LM_ERR_UNSUPPORTED, "binned density covers fp32 planes of 16, 32 or 64 channels and %d points or more", kSample);
    if (workspace_bytes < pn.total) LM_FAIL(LM_ERR_WORKSPACE, "workspace of %zu bytes, %zu needed", workspace_bytes, pn.total);
    hipStream_t st = (hipStream_t)stream;
    char *ws = (char *)workspace;
    uint32_t *counts = (uint32_t *)(ws + pn.o_counts), *flag = (uint32_t *)(ws + pn.o_flag), *n_units = (uint32_t *)(ws + pn.o_n_units),
             *n_groups = (uint32_t *)(ws + pn.o_n_groups);
    uint4 *units = (uint4 *)(ws + pn.o_units);
    uint32_t *queue = (uint32_t *)(ws + pn.o_queue);
    Group *groups = (Group *)(ws + pn.o_groups);
    uint16_t *tab = (uint16_t *)(ws + pn.o_tab), *order = (uint16_t *)(ws + pn.o_order);
    float4 *rec = (float4 *)(ws + pn.o_rec);
    float *sum = (float *)(ws + pn.o_sum);
    const int side = pn.side, bins = side * side * side;
    const size_t order_step = (size_t)pn.slice, tab_step = (size_t)pn.max_units * (pn.max_subs + 1);
    const PlaneSet ps = make_set(planes, n_planes);
    const unsigned grid = (unsigned)(lm_persistent_blocks(3) / LM_XCDS * LM_XCDS);  // as many as LDS lets live at once
    const bool all64 = planes_all_64(planes, n_planes);
#define LM_DX(C_)                                                                                                            \
    hipLaunchKernelGGL((k_density_xyz<float, C_, true>), dim3(density_xyz_grid(m)), dim3(kBlock), 0, st, ps, density_basis, pts, \
                       (uint64_t)m, out + at, flag)
    for (int64_t at = 0; at < M; at += pn.slice) {
        const uint32_t m = (uint32_t)std::min(pn.slice, M - at);
        const float *pts = xyz + 3 * at;
        const unsigned wgs = (m + kUnit - 1) / kUnit;
        hipLaunchKernelGGL(k_bin_decide, dim3(1), dim3(kScatter), 0, st, pn.axes, pts, m, counts, bins, queue, flag);
        if (all64) LM_DX(64); else LM_DX(0);
        hipLaunchKernelGGL(k_bin_count, dim3(std::min(wgs, (unsigned)lm_persistent_blocks(1))), dim3(kScatter), 0, st, flag, side, pts, m, counts);
        hipLaunchKernelGGL(k_bin_scan, dim3(1), dim3(kScatter), 0, st, flag, side, pn.axes, counts, units, n_units, groups, pn.max_groups, n_groups);
        hipLaunchKernelGGL(k_bin_scatter, dim3(wgs), dim3(kScatter), 0, st, flag, side, pts, m, counts, rec);
        hipLaunchKernelGGL(k_bin_order, dim3(std::min(pn.max_units, (unsigned)lm_persistent_blocks(2)), n_planes), dim3(kScatter), 0, st, flag, ps, side, pn.cuts, units, n_units, rec, order_step,
                           tab_step, order, tab);
        int col = 0;
        for (int k = 0; k < n_planes; ++k) {
            const lm_plane &p = planes[k];
            const int mode = (k == 0 ? 1 : 0) | (k == n_planes - 1 ? 2 : 0);
            const float *w = density_basis ? density_basis + col : nullptr;
#define LM_BD(C_, NL_)                                                                                                             \
    hipLaunchKernelGGL((k_bin_density<C_, NL_>), dim3(grid), dim3(kTaskThreads), 0, st, flag, p, pn.cuts.of[k], w,           \
                       groups + (size_t)k * pn.max_groups, n_groups + k, queue + k * LM_XCDS, units, tab + k * tab_step, order + k * order_step, rec, sum, mode, out + at)
#define LM_BD_C(NL_)                    \
    switch (p.C) {                      \
        case 16: LM_BD(16, NL_); break; \
        case 32: LM_BD(32, NL_); break; \
        default: LM_BD(64, NL_); break; \
    }
            if (w) { LM_BD_C(true) } else { LM_BD_C(false) }
#undef LM_BD_C
#undef LM_BD
            col += p.C;
        }
    }
#undef LM_DX
    LM_CHECK_LAUNCH("k_bin_density");
    return LM_OK;
}
