// Device side of the feature lookup shared by the kernels that gather: table access by storage type, bilinear and
// linear footprints, plane x line products and the per-sample density sums.  See lm_gather.hip for the lane layout.
#pragma once
#include <hip/hip_fp16.h>

#include <algorithm>
#include <type_traits>

#include "lm_common.h"

// Chunks of up to this many rays are small: a kernel from rays to appearance entries, or a wave per ray (lm_ray.hip).  The
// line lies below where the first stops paying.  Whole calls with it / with the kernels per stage: 16384 rays of nine planes
// 359 / 453 us, three small planes 325 / 315, 886 samples per ray 780 / 1187, 2 x 3 blocks 249 / 307, city tables 253 / 320;
// 32768 rays 616 / 549, 509 / 427, 1469 / 1629, 430 / 396, 405 / 437; at the line itself 234 / 331, 203 / 245, 625 / 1112,
// 148 / 227 (first four).
#ifndef LM_RAYS_LIMIT
#define LM_RAYS_LIMIT 12288
#endif

namespace {

constexpr int kBlock = 256;
constexpr int kQuad = 4;
constexpr int kTile = kBlock / kQuad;  // samples per workgroup iteration

struct PlaneSet {
    lm_plane p[LM_MAX_PLANES];
    int n;
    int nblk;  // > 0: block-stacked tables, planes [nblk][H][W][C], lines [Len][nblk][C]
};

// A lane's share of one texel: loaded as it is stored (fetch), converted to float where it is
// used (unpack), so that loads in flight hold the stored width in registers and no conversion
// waits for a load that other work could run under.
template <typename T> struct Vec;
template <> struct Vec<float> {
    using elem = float;
    using raw = float4;
    static constexpr int V = 4;
    __device__ static __forceinline__ raw fetch(const float *p) { return *reinterpret_cast<const float4 *>(p); }
    __device__ static __forceinline__ void unpack(const raw &v, float *o) { o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w; }
};
template <> struct Vec<__half> {
    using elem = __half;
    using raw = uint4;
    static constexpr int V = 8;
    __device__ static __forceinline__ raw fetch(const __half *p) { return *reinterpret_cast<const uint4 *>(p); }
    __device__ static __forceinline__ void unpack(const raw &v, float *o) {
        const __half2 *h = reinterpret_cast<const __half2 *>(&v);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float2 f = __half22float2(h[i]);
            o[2 * i] = f.x; o[2 * i + 1] = f.y;
        }
    }
};
// fp16 tables read four channels (8 bytes) per lane: for 16- and 48-channel planes, where
// 16-byte loads would leave half of a quad idle on the last 16 channels
struct Half4 {};
template <> struct Vec<Half4> {
    using elem = __half;
    using raw = uint2;
    static constexpr int V = 4;
    __device__ static __forceinline__ raw fetch(const __half *p) { return *reinterpret_cast<const uint2 *>(p); }
    __device__ static __forceinline__ void unpack(const raw &v, float *o) {
        const __half2 *h = reinterpret_cast<const __half2 *>(&v);
        const float2 a = __half22float2(h[0]), b = __half22float2(h[1]);
        o[0] = a.x; o[1] = a.y; o[2] = b.x; o[3] = b.y;
    }
};

// fp16 planes of 48 channels (96-byte texels) in the fused appearance gather: six channels (12 bytes) per lane, two load
// instructions per texel and quad instead of three.  The kernel keeps its texture addresser busy 82 % of the time at a
// cost per instruction that depends on the lines touched, not on the bytes (4K city block: 26.7 -> 24.5 ms per frame).
struct Half6 {};
struct __attribute__((aligned(4))) Raw12 {
    uint32_t x, y, z;
};
template <> struct Vec<Half6> {
    using elem = __half;
    using raw = Raw12;
    static constexpr int V = 6;
    __device__ static __forceinline__ raw fetch(const __half *p) { return *reinterpret_cast<const Raw12 *>(p); }
    __device__ static __forceinline__ void unpack(const raw &v, float *o) {
        const __half2 *h = reinterpret_cast<const __half2 *>(&v);
        const float2 a = __half22float2(h[0]), b = __half22float2(h[1]), c = __half22float2(h[2]);
        o[0] = a.x; o[1] = a.y; o[2] = b.x; o[3] = b.y; o[4] = c.x; o[5] = c.y;
    }
};

// (unused entries repeat the first plane)
inline PlaneSet make_set(const lm_plane *planes, int n, const lm_geom *g = nullptr) {
    PlaneSet ps;
    for (int k = 0; k < LM_MAX_PLANES; ++k) ps.p[k] = planes[k < n ? k : 0];
    ps.n = n;
    ps.nblk = g && g->div0 > 0 ? g->div0 * g->div1 : 0;
    return ps;
}

struct Taps2 {  // bilinear footprint: element offsets of the 4 corners and their weights
    int64_t o00, o01, o10, o11;
    float w00, w01, w10, w11;
};
struct Taps1 {
    int o0, o1;
    float w0, w1;
};

__device__ __forceinline__ float unnorm(float c, int size) { return ((c + 1.0f) / 2.0f) * (float)(size - 1); }

// Corner (y, x) outside the table has weight zero (grid_sample's zeros padding) and is read from
// the nearest texel inside.  A row of the table has fewer than 2^31 elements (checked on the host).
__device__ __forceinline__ Taps2 plane_taps(const lm_plane &pl, float cx, float cy) {
    const float ix = unnorm(cx, pl.W), iy = unnorm(cy, pl.H);
    const float fx = floorf(ix), fy = floorf(iy);
    float wx1 = ix - fx, wx0 = (fx + 1.0f) - ix, wy1 = iy - fy, wy0 = (fy + 1.0f) - iy;
    // clamp in float first: coordinates far outside the table must not overflow the int cast
    const int x0 = (int)fminf(fmaxf(fx, -2.0f), (float)pl.W), y0 = (int)fminf(fmaxf(fy, -2.0f), (float)pl.H);
    const int x1 = x0 + 1, y1 = y0 + 1;
    if ((unsigned)x0 >= (unsigned)pl.W) wx0 = 0.0f;
    if ((unsigned)x1 >= (unsigned)pl.W) wx1 = 0.0f;
    if ((unsigned)y0 >= (unsigned)pl.H) wy0 = 0.0f;
    if ((unsigned)y1 >= (unsigned)pl.H) wy1 = 0.0f;
    const int x0c = min(max(x0, 0), pl.W - 1), x1c = min(max(x1, 0), pl.W - 1);
    const int y0c = min(max(y0, 0), pl.H - 1), y1c = min(max(y1, 0), pl.H - 1);
    const int row = pl.W * pl.C;
    Taps2 t;
    const int dx = x1c != x0c ? pl.C : 0, dy = y1c != y0c ? row : 0;
    t.o00 = (int64_t)y0c * row + x0c * pl.C;
    t.o01 = t.o00 + dx;
    t.o10 = t.o00 + dy;
    t.o11 = t.o10 + dx;
    t.w00 = wx0 * wy0; t.w01 = wx1 * wy0; t.w10 = wx0 * wy1; t.w11 = wx1 * wy1;
    return t;
}

__device__ __forceinline__ Taps1 line_taps(const lm_plane &pl, float c) {
    const float i = unnorm(c, pl.Len);
    const float f = floorf(i);
    float w1 = i - f, w0 = (f + 1.0f) - i;
    int i0 = (int)fminf(fmaxf(f, -2.0f), (float)pl.Len), i1 = i0 + 1;
    if (i0 < 0 || i0 >= pl.Len) w0 = 0.0f;
    if (i1 < 0 || i1 >= pl.Len) w1 = 0.0f;
    i0 = min(max(i0, 0), pl.Len - 1); i1 = min(max(i1, 0), pl.Len - 1);
    Taps1 t;
    t.o0 = i0 * pl.C; t.o1 = i1 * pl.C;
    t.w0 = w0; t.w1 = w1;
    return t;
}

// Queries are float[4]: normalised x, y, z and, for block-stacked tables, the block index as
// integer bits in q[3].  Moves the taps to the block; a block outside the table reads as zero.
__device__ __forceinline__ void block_taps(const lm_plane &pl, int nblk, const float *q, Taps2 &t2, Taps1 &t1) {
    if (nblk <= 0) return;
    const int blk = __float_as_int(q[3]);
    if (blk < 0 || blk >= nblk) {
        t2.w00 = t2.w01 = t2.w10 = t2.w11 = 0.0f;
        t1.w0 = t1.w1 = 0.0f;
        return;
    }
    const int64_t base = (int64_t)blk * pl.H * pl.W * pl.C;
    t2.o00 += base; t2.o01 += base; t2.o10 += base; t2.o11 += base;
    t1.o0 = t1.o0 * nblk + blk * pl.C;
    t1.o1 = t1.o1 * nblk + blk * pl.C;
}

// Sum over the four lanes of a quad, on all four (DPP moves: partner 1 away, then 2 away).
__device__ __forceinline__ float quad_sum(float v) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xb1, 0xf, 0xf, false));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4e, 0xf, 0xf, false));
    return v;
}

__device__ __forceinline__ float pick(const float *q, int ax) { return ax == 0 ? q[0] : (ax == 1 ? q[1] : q[2]); }

// products of one plane for the V channels starting at c (lane-private)
template <typename T>
__device__ __forceinline__ void plane_products(const lm_plane &pl, const Taps2 &t2, const Taps1 &t1, int c, float *prod) {
    constexpr int V = Vec<T>::V;
    using E = typename Vec<T>::elem;
    const E *P = reinterpret_cast<const E *>(pl.plane);
    const E *Ln = reinterpret_cast<const E *>(pl.line);
    float a[V], b[V], cc[V], d[V], l0[V], l1[V];
    const typename Vec<T>::raw ra = Vec<T>::fetch(P + t2.o00 + c), rb = Vec<T>::fetch(P + t2.o01 + c),
                               rc = Vec<T>::fetch(P + t2.o10 + c), rd = Vec<T>::fetch(P + t2.o11 + c),
                               r0 = Vec<T>::fetch(Ln + t1.o0 + c), r1 = Vec<T>::fetch(Ln + t1.o1 + c);
    Vec<T>::unpack(ra, a); Vec<T>::unpack(rb, b); Vec<T>::unpack(rc, cc); Vec<T>::unpack(rd, d);
    Vec<T>::unpack(r0, l0); Vec<T>::unpack(r1, l1);
#pragma unroll
    for (int i = 0; i < V; ++i) {
        float pv = a[i] * t2.w00;
        pv = fmaf(b[i], t2.w01, pv);
        pv = fmaf(cc[i], t2.w10, pv);
        pv = fmaf(d[i], t2.w11, pv);
        float lv = fmaf(l1[i], t1.w1, l0[i] * t1.w0);
        prod[i] = pv * lv;
    }
}

// den_w == NULL: plain sum over planes and channels.  Otherwise the reference's
// nonlinear_density: relu(sum of den_w[plane*C + channel] * product) (gridnerf_sequential.py:819-822)
template <typename T>
__device__ __forceinline__ float density_sum(const PlaneSet &ps, const float *q, unsigned qlane,
                                             const float *__restrict__ den_w) {
    constexpr int V = Vec<T>::V;
    float sum = 0.0f;
    int col = 0;
    for (int k = 0; k < ps.n; ++k) {
        const lm_plane pl = ps.p[k];
        Taps2 t2 = plane_taps(pl, pick(q, pl.ax0), pick(q, pl.ax1));
        Taps1 t1 = line_taps(pl, pick(q, pl.axl));
        block_taps(pl, ps.nblk, q, t2, t1);
        for (int c = V * qlane; c < pl.C; c += V * kQuad) {
            float prod[V];
            plane_products<T>(pl, t2, t1, c, prod);
            if (den_w) {
#pragma unroll
                for (int i = 0; i < V; ++i) sum = fmaf(den_w[col + c + i], prod[i], sum);
            } else {
#pragma unroll
                for (int i = 0; i < V; ++i) sum += prod[i];
            }
        }
        col += pl.C;
    }
    sum = quad_sum(sum);
    return den_w ? fmaxf(sum, 0.0f) : sum;
}

// The loads of plane_products and the arithmetic on what they return, as two steps, for callers
// that want several footprints' loads in flight before the first use.
template <typename T> struct Footprint {
    typename Vec<T>::raw a, b, c, d, l0, l1;
};
template <typename T>
__device__ __forceinline__ void footprint_load(const lm_plane &pl, const Taps2 &t2, const Taps1 &t1, int c, Footprint<T> &f) {
    using E = typename Vec<T>::elem;
    const E *P = reinterpret_cast<const E *>(pl.plane);
    const E *Ln = reinterpret_cast<const E *>(pl.line);
    f.a = Vec<T>::fetch(P + t2.o00 + c);
    f.b = Vec<T>::fetch(P + t2.o01 + c);
    f.c = Vec<T>::fetch(P + t2.o10 + c);
    f.d = Vec<T>::fetch(P + t2.o11 + c);
    f.l0 = Vec<T>::fetch(Ln + t1.o0 + c);
    f.l1 = Vec<T>::fetch(Ln + t1.o1 + c);
}
template <typename T>
__device__ __forceinline__ void footprint_products(const Footprint<T> &f, const Taps2 &t2, const Taps1 &t1, float *prod) {
    constexpr int V = Vec<T>::V;
    float a[V], b[V], c[V], d[V], l0[V], l1[V];
    Vec<T>::unpack(f.a, a); Vec<T>::unpack(f.b, b); Vec<T>::unpack(f.c, c); Vec<T>::unpack(f.d, d);
    Vec<T>::unpack(f.l0, l0); Vec<T>::unpack(f.l1, l1);
#pragma unroll
    for (int i = 0; i < V; ++i) {
        float pv = a[i] * t2.w00;
        pv = fmaf(b[i], t2.w01, pv);
        pv = fmaf(c[i], t2.w10, pv);
        pv = fmaf(d[i], t2.w11, pv);
        const float lv = fmaf(l1[i], t1.w1, l0[i] * t1.w0);
        prod[i] = pv * lv;
    }
}

// Value of v on lane n of this lane's quad (n is a constant after unrolling): one DPP move.
__device__ __forceinline__ int quad_lane(int v, int n) {
    switch (n & 3) {
        case 0: return __builtin_amdgcn_update_dpp(0, v, 0x00, 0xf, 0xf, false);
        case 1: return __builtin_amdgcn_update_dpp(0, v, 0x55, 0xf, 0xf, false);
        case 2: return __builtin_amdgcn_update_dpp(0, v, 0xaa, 0xf, 0xf, false);
        default: return __builtin_amdgcn_update_dpp(0, v, 0xff, 0xf, 0xf, false);
    }
}
__device__ __forceinline__ float quad_lane(float v, int n) { return __int_as_float(quad_lane(__float_as_int(v), n)); }
__device__ __forceinline__ int64_t quad_lane(int64_t v, int n) {
    const uint32_t lo = (uint32_t)quad_lane((int)(uint32_t)v, n), hi = (uint32_t)quad_lane((int)(uint32_t)((uint64_t)v >> 32), n);
    return (int64_t)(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ Taps2 quad_lane(const Taps2 &t, int n) {
    Taps2 r;
    // the corners are less than 2^31 elements apart: one 64-bit offset and two 32-bit steps go round
    const int dx = quad_lane((int)(t.o01 - t.o00), n), dy = quad_lane((int)(t.o10 - t.o00), n);
    r.o00 = quad_lane(t.o00, n);
    r.o01 = r.o00 + dx;
    r.o10 = r.o00 + dy;
    r.o11 = r.o10 + dx;
    r.w00 = quad_lane(t.w00, n); r.w01 = quad_lane(t.w01, n); r.w10 = quad_lane(t.w10, n); r.w11 = quad_lane(t.w11, n);
    return r;
}
__device__ __forceinline__ Taps1 quad_lane(const Taps1 &t, int n) {
    Taps1 r;
    r.o0 = quad_lane(t.o0, n); r.o1 = quad_lane(t.o1, n); r.w0 = quad_lane(t.w0, n); r.w1 = quad_lane(t.w1, n);
    return r;
}

// NS samples of a quad at once (the marching kernel's look-ahead).  Lane n of the quad brings
// the coordinates of sample n (lanes NS.. repeat) and works out that sample's footprints, one
// sample per lane instead of every sample on every lane; the footprints then go round the quad
// and each lane loads its quarter of the channels of all NS samples, every load issued before
// the first use, so a ray's chain of dependent memory round trips is NS times shorter.  Same
// operations per sample as density_sum, hence the same bits.  out[n] is valid on all four lanes.
template <typename T, int NS>
__device__ __forceinline__ void density_sum_n(const PlaneSet &ps, const float *q_mine, unsigned qlane,
                                              const float *__restrict__ den_w, float *out) {
    constexpr int V = Vec<T>::V;
    float sum[NS];
#pragma unroll
    for (int n = 0; n < NS; ++n) sum[n] = 0.0f;
    int col = 0;
    for (int k = 0; k < ps.n; ++k) {
        const lm_plane pl = ps.p[k];
        Taps2 m2 = plane_taps(pl, pick(q_mine, pl.ax0), pick(q_mine, pl.ax1));
        Taps1 m1 = line_taps(pl, pick(q_mine, pl.axl));
        block_taps(pl, ps.nblk, q_mine, m2, m1);
        Taps2 t2[NS];
        Taps1 t1[NS];
#pragma unroll
        for (int n = 0; n < NS; ++n) {
            t2[n] = quad_lane(m2, n);
            t1[n] = quad_lane(m1, n);
        }
        for (int c = V * qlane; c < pl.C; c += V * kQuad) {
            Footprint<T> f[NS];
#pragma unroll
            for (int n = 0; n < NS; ++n) footprint_load<T>(pl, t2[n], t1[n], c, f[n]);
            // keep the 6 * NS loads ahead of the first use
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int n = 0; n < NS; ++n) {
                float prod[V];
                footprint_products<T>(f[n], t2[n], t1[n], prod);
                if (den_w) {
#pragma unroll
                    for (int i = 0; i < V; ++i) sum[n] = fmaf(den_w[col + c + i], prod[i], sum[n]);
                } else {
#pragma unroll
                    for (int i = 0; i < V; ++i) sum[n] += prod[i];
                }
            }
        }
        col += pl.C;
    }
#pragma unroll
    for (int n = 0; n < NS; ++n) {
        float v = sum[n];
        v = quad_sum(v);
        out[n] = den_w ? fmaxf(v, 0.0f) : v;
    }
}

// density_sum_n of four samples for planes of one channel group per lane and tables below 4 GB (density_rolls): the next plane's
// footprints are worked out while this one's loads travel, and its loads are issued as soon as products have left the
// registers (all four samples' at once with 16-byte loads, two at a time with 8-byte ones).  Offsets are 32-bit bytes from the plane's (scalar) address:
// a seventh of the march's vector instructions less (3.54 -> 3.03 G on the frame below, its loads 170 -> 152 M) and 202 instead of
// 231 registers.  Same operations per sample, hence the same bits.
// 960 x 540 rays of 3544 samples, three fp32 planes with a projection, one view: frame 26.1 -> 22.5 ms (march 13.2 -> 10.1; over the
// views of an orbit 29.5 -> 25.3); 4K city (fp16) 39.7 -> 39.0 ms; frames bound by bytes the same within 0.5 %
// (a tenth more lines fetched, at a higher rate).  Two samples at a time in fp32 too 23.0, one
// 23.5; the same without work on the next plane 24.5.  The projection's weights are loaded once per plane: once per sample is
// what the compiler made of the plain form, and that took 30.0.
struct RollTaps {
    uint32_t o00, l0;  // first corner and lower line texel
    uint32_t dx, dy, dl;
    float w00, w01, w10, w11, lw0, lw1;
};
template <typename E> __device__ __forceinline__ RollTaps roll_taps(const lm_plane &pl, int nblk, const float *q) {
    const float cx = pick(q, pl.ax0), cy = pick(q, pl.ax1), cl = pick(q, pl.axl);
    RollTaps t;
    {
        // plane_taps with byte offsets
        const float ix = unnorm(cx, pl.W), iy = unnorm(cy, pl.H);
        const float fx = floorf(ix), fy = floorf(iy);
        float wx1 = ix - fx, wx0 = (fx + 1.0f) - ix, wy1 = iy - fy, wy0 = (fy + 1.0f) - iy;
        const int x0 = (int)fminf(fmaxf(fx, -2.0f), (float)pl.W), y0 = (int)fminf(fmaxf(fy, -2.0f), (float)pl.H);
        const int x1 = x0 + 1, y1 = y0 + 1;
        if ((unsigned)x0 >= (unsigned)pl.W) wx0 = 0.0f;
        if ((unsigned)x1 >= (unsigned)pl.W) wx1 = 0.0f;
        if ((unsigned)y0 >= (unsigned)pl.H) wy0 = 0.0f;
        if ((unsigned)y1 >= (unsigned)pl.H) wy1 = 0.0f;
        const int x0c = min(max(x0, 0), pl.W - 1), x1c = min(max(x1, 0), pl.W - 1);
        const int y0c = min(max(y0, 0), pl.H - 1), y1c = min(max(y1, 0), pl.H - 1);
        const uint32_t texel = (uint32_t)(pl.C * (int)sizeof(E)), row = (uint32_t)pl.W * texel;
        t.o00 = (uint32_t)y0c * row + (uint32_t)x0c * texel;
        t.dx = x1c != x0c ? texel : 0u;
        t.dy = y1c != y0c ? row : 0u;
        t.w00 = wx0 * wy0; t.w01 = wx1 * wy0; t.w10 = wx0 * wy1; t.w11 = wx1 * wy1;
        const Taps1 l = line_taps(pl, cl);
        t.l0 = (uint32_t)l.o0 * (uint32_t)sizeof(E);
        t.dl = (uint32_t)(l.o1 - l.o0) * (uint32_t)sizeof(E);
        t.lw0 = l.w0; t.lw1 = l.w1;
        if (nblk > 0) {  // block_taps
            const int blk = __float_as_int(q[3]);
            if (blk < 0 || blk >= nblk) {
                t.w00 = t.w01 = t.w10 = t.w11 = t.lw0 = t.lw1 = 0.0f;
            } else {
                t.o00 += (uint32_t)blk * (uint32_t)pl.H * row;
                t.l0 = t.l0 * (uint32_t)nblk + (uint32_t)blk * texel;
                t.dl *= (uint32_t)nblk;
            }
        }
    }
    return t;
}
template <typename T> __device__ __forceinline__ typename Vec<T>::raw fetch_at(const void *base, uint32_t byte) {
    return Vec<T>::fetch(reinterpret_cast<const typename Vec<T>::elem *>(static_cast<const char *>(base) + byte));
}
// the host's side: tables the rolling sum covers (planes of up to four lanes' channels, every offset below 4 GB)
template <typename T> inline bool density_rolls(const lm_plane *planes, int n, int nblk) {
    for (int k = 0; k < n; ++k) {
        const lm_plane &p = planes[k];
        const int64_t texel = (int64_t)p.C * (int64_t)sizeof(typename Vec<T>::elem) * (nblk > 0 ? nblk : 1);
        if (p.C > Vec<T>::V * kQuad || (int64_t)p.H * p.W * texel >= (int64_t)1 << 32 || (int64_t)p.Len * texel >= (int64_t)1 << 32) return false;
    }
    return true;
}
// NS samples of a quad: lane n brings sample n's taps (NS = 1: every lane its own sample's).  A lane beyond a narrow plane's
// channels reads its last ones and adds nothing.
template <typename T> __device__ __forceinline__ int roll_channel(const lm_plane &pl, unsigned qlane) { return min(Vec<T>::V * (int)qlane, pl.C - Vec<T>::V); }
template <typename T, int NS>
__device__ __forceinline__ void roll_load(const lm_plane &pl, const RollTaps &m, int n, unsigned qlane, Footprint<T> &f) {
    auto of = [&](uint32_t v) { return NS == 1 ? v : (uint32_t)quad_lane((int)v, n); };
    const uint32_t c = (uint32_t)(roll_channel<T>(pl, qlane) * (int)sizeof(typename Vec<T>::elem));
    const uint32_t o00 = of(m.o00) + c, dx = of(m.dx), dy = of(m.dy), l0 = of(m.l0) + c, dl = of(m.dl), o10 = o00 + dy;
    f.a = fetch_at<T>(pl.plane, o00);
    f.b = fetch_at<T>(pl.plane, o00 + dx);
    f.c = fetch_at<T>(pl.plane, o10);
    f.d = fetch_at<T>(pl.plane, o10 + dx);
    f.l0 = fetch_at<T>(pl.line, l0);
    f.l1 = fetch_at<T>(pl.line, l0 + dl);
}
template <typename T> __device__ __forceinline__ void roll_weights(const lm_plane &pl, const float *__restrict__ den_w, int col, unsigned qlane, float *w) {
    if (!den_w) return;
#pragma unroll
    for (int i = 0; i < Vec<T>::V; ++i) w[i] = den_w[col + roll_channel<T>(pl, qlane) + i];
}
template <typename T, int NS>
__device__ __forceinline__ void roll_use(const lm_plane &pl, const RollTaps &m, int n, unsigned qlane, const Footprint<T> &f, bool weighted, const float *w,
                                         float &sum) {
    constexpr int V = Vec<T>::V;
    auto of = [&](float v) { return NS == 1 ? v : quad_lane(v, n); };
    Taps2 t2;
    Taps1 t1;
    t2.w00 = of(m.w00); t2.w01 = of(m.w01); t2.w10 = of(m.w10); t2.w11 = of(m.w11);
    t1.w0 = of(m.lw0); t1.w1 = of(m.lw1);
    float prod[V];
    footprint_products<T>(f, t2, t1, prod);
    if (V * (int)qlane >= pl.C) return;
#pragma unroll
    for (int i = 0; i < V; ++i) sum = weighted ? fmaf(w[i], prod[i], sum) : sum + prod[i];
}
template <typename T>
__device__ __forceinline__ void density_sum_rolling(const PlaneSet &ps, const float *q_mine, unsigned qlane, const float *__restrict__ den_w,
                                                    float *out) {
    constexpr int V = Vec<T>::V, NS = 4, HALF = sizeof(typename Vec<T>::raw) == 16 ? 4 : 2;
    using E = typename Vec<T>::elem;
    float sum[NS];
#pragma unroll
    for (int n = 0; n < NS; ++n) sum[n] = 0.0f;
    Footprint<T> f[NS];
    lm_plane pl = ps.p[0];
    RollTaps now = roll_taps<E>(pl, ps.nblk, q_mine);
    float w[V] = {}, w_next[V] = {};
    roll_weights<T>(pl, den_w, 0, qlane, w);
#pragma unroll
    for (int n = 0; n < NS; ++n) roll_load<T, NS>(pl, now, n, qlane, f[n]);
    int col = 0;
    for (int k = 0;;) {
        const bool last = k + 1 == ps.n;
        const lm_plane pn = ps.p[last ? k : k + 1];
        __builtin_amdgcn_sched_barrier(0);
        RollTaps next;
        if (!last) next = roll_taps<E>(pn, ps.nblk, q_mine);
#pragma unroll
        for (int h = 0; h < NS; h += HALF) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int n = h; n < h + HALF; ++n) roll_use<T, NS>(pl, now, n, qlane, f[n], den_w != nullptr, w, sum[n]);
            __builtin_amdgcn_sched_barrier(0);
            if (!last) {
                if (h == 0) roll_weights<T>(pn, den_w, col + pl.C, qlane, w_next);
#pragma unroll
                for (int n = h; n < h + HALF; ++n) roll_load<T, NS>(pn, next, n, qlane, f[n]);
            }
        }
        if (last) break;
        col += pl.C;
        now = next;
        pl = pn;
#pragma unroll
        for (int i = 0; i < V; ++i) w[i] = w_next[i];
        ++k;
    }
#pragma unroll
    for (int n = 0; n < NS; ++n) {
        const float v = quad_sum(sum[n]);
        out[n] = den_w ? fmaxf(v, 0.0f) : v;
    }
}

// Same sum with a compile-time channel count shared by all planes: the channel groups of a
// plane are unrolled, so a lane has 6 * C / (4 V) independent loads in flight per plane
// instead of 6 (wide planes, e.g. the 64-channel isolated-gather configuration).
template <typename T, int C>
__device__ __forceinline__ float density_sum_fixed(const PlaneSet &ps, const float *q, unsigned qlane,
                                                   const float *__restrict__ den_w) {
    constexpr int V = Vec<T>::V;
    constexpr int NG = (C + V * kQuad - 1) / (V * kQuad);
    float sum = 0.0f;
    for (int k = 0; k < ps.n; ++k) {
        const lm_plane pl = ps.p[k];
        Taps2 t2 = plane_taps(pl, pick(q, pl.ax0), pick(q, pl.ax1));
        Taps1 t1 = line_taps(pl, pick(q, pl.axl));
        block_taps(pl, ps.nblk, q, t2, t1);
        float prod[NG][V];
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) {
            const int c = V * (int)qlane + gi * V * kQuad;
            plane_products<T>(pl, t2, t1, c < C ? c : C - V, prod[gi]);
        }
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) {
            const int c = V * (int)qlane + gi * V * kQuad;
            if (c < C) {
#pragma unroll
                for (int i = 0; i < V; ++i) sum = den_w ? fmaf(den_w[k * C + c + i], prod[gi][i], sum) : sum + prod[gi][i];
            }
        }
    }
    sum = quad_sum(sum);
    return den_w ? fmaxf(sum, 0.0f) : sum;
}

// Plane x line products of the sixteen samples of a wave (four lanes each), written in whole lines: a quad's own stores
// are 64-byte pieces of sixteen different rows per instruction, which reach the memory as partial lines (measured on
// 2^24 random queries of 3 x 64 channels: 16.3 GB written and 86.8 GB read for 12.9 GB of products and 51.5 GB of texels).
// Each plane's products go through a tile in LDS (sixteen rows of C + 4 floats per wave) and leave as runs of C floats
// per sample, a lane storing 16 bytes of a run.  Samples p0 .. p0 + 15 belong to the wave; those at or beyond M are
// computed (from a clamped query) and not stored.  Planes of more than kStageC channels take the direct form.
constexpr int kStageC = 64;
constexpr int kStageRow = kStageC + 4;
template <typename T>
__device__ __forceinline__ void app_store_wave(const PlaneSet &ps, const float *q, uint64_t p0, uint64_t M, int K,
                                               float *__restrict__ out, float *tile) {
    constexpr int V = Vec<T>::V;
    const unsigned lane = lm_lane(), qlane = lane & 3u, qs = lane >> 2;
    int col = 0;
    for (int k = 0; k < ps.n; ++k) {
        const lm_plane pl = ps.p[k];
        Taps2 t2 = plane_taps(pl, pick(q, pl.ax0), pick(q, pl.ax1));
        Taps1 t1 = line_taps(pl, pick(q, pl.axl));
        block_taps(pl, ps.nblk, q, t2, t1);
        const bool staged = pl.C <= kStageC;
        if (staged) {
            // every load of the plane's footprint is issued before the first use: one memory round trip per plane
            constexpr int NG = kStageC / (V * kQuad);
            Footprint<T> fp[NG];
#pragma unroll
            for (int gi = 0; gi < NG; ++gi) {
                const int c = V * (int)qlane + gi * V * kQuad;
                if (c < pl.C) footprint_load<T>(pl, t2, t1, c, fp[gi]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int gi = 0; gi < NG; ++gi) {
                const int c = V * (int)qlane + gi * V * kQuad;
                if (c >= pl.C) continue;
                float prod[V];
                footprint_products<T>(fp[gi], t2, t1, prod);
#pragma unroll
                for (int i = 0; i < V; i += 4)
                    *reinterpret_cast<float4 *>(tile + qs * kStageRow + c + i) = make_float4(prod[i], prod[i + 1], prod[i + 2], prod[i + 3]);
            }
        } else {
            for (int c = V * qlane; c < pl.C; c += V * kQuad) {
                float prod[V];
                plane_products<T>(pl, t2, t1, c, prod);
#pragma unroll
                for (int i = 0; i < V; i += 4)
                    if (p0 + qs < M)
                        *reinterpret_cast<float4 *>(out + (p0 + qs) * (uint64_t)K + col + c + i) =
                            make_float4(prod[i], prod[i + 1], prod[i + 2], prod[i + 3]);
            }
        }
        if (staged) {
            // LDS operations of one wave complete in order; the fences only pin the compiler
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const unsigned c4 = (unsigned)pl.C / 4u;  // 16-byte pieces per sample
            for (unsigned idx = lane; idx < 16u * c4; idx += LM_WAVE) {
                const unsigned s_i = idx / c4, f = idx - s_i * c4;
                if (p0 + s_i < M)
                    *reinterpret_cast<float4 *>(out + (p0 + s_i) * (uint64_t)K + col + 4 * f) =
                        *reinterpret_cast<const float4 *>(tile + s_i * kStageRow + 4 * f);
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        col += pl.C;
    }
}

// coordinates of list entry `flat` (= ray*S + s): same operations as the sampler
__device__ __forceinline__ void list_coords(const lm_geom &g, const float *__restrict__ rays, uint32_t flat, float *q) {
    const uint32_t r = flat / (uint32_t)g.S;
    const int s = (int)(flat - r * (uint32_t)g.S);
    float ray[6];
    const float2 *rp = reinterpret_cast<const float2 *>(rays + 6 * (size_t)r);
    float2 a = rp[0], b = rp[1], c = rp[2];
    ray[0] = a.x; ray[1] = a.y; ray[2] = b.x; ray[3] = b.y; ray[4] = c.x; ray[5] = c.y;
    const float z = lm_sample_z(g, lm_ray_param(g, ray), s);
    float pt[3];
    lm_point(ray, z, pt);
    lm_normalise(g, pt, q);
    q[3] = __int_as_float(g.div0 > 0 ? lm_block_coords(g, q) : 0);
}

__device__ __forceinline__ float activate(float f, int act, float shift) {
    if (act == LM_ACT_SOFTPLUS) {
        const float x = f + shift;
        return x > 20.0f ? x : log1pf(expf(x));
    }
    return fmaxf(f, 0.0f);
}

// ---- density features of points given by their coordinates ------------------------------------------------------
// SKIP: nothing to do where *skip is not zero (sorted points; built in lm_points.hip).  A form of its own: with a test of the pointer
// in the plain one, calls without it were 0.1 % slower (3 million points, 3 x 1000^2 x 32 channels 876.7 -> 878.0 us, now 873.2 against 873.1
// before the test).  Built next to the plain one it moves k_march in its code object, and 20 000 rays on nine planes take 494
// instead of 428 us.
template <typename T, int CFIX, bool SKIP>  // CFIX > 0: every plane has CFIX channels
__global__ __launch_bounds__(kBlock) void k_density_xyz(PlaneSet ps, const float *__restrict__ den_w,
                                                        const float *__restrict__ xyz, uint64_t M,
                                                        float *__restrict__ out, const uint32_t *__restrict__ skip) {
    if (SKIP && *skip) return;
    const unsigned qlane = threadIdx.x & 3u, slot = threadIdx.x >> 2;
    const uint64_t n_tiles = (M + kTile - 1) / kTile;
    for (uint64_t tile = lm_xcd_swizzle(blockIdx.x, gridDim.x); tile < n_tiles; tile += gridDim.x) {
        const uint64_t p = tile * kTile + slot;
        if (p >= M) continue;
        float q[4] = {xyz[3 * p], xyz[3 * p + 1], xyz[3 * p + 2], 0.0f};
        const float s = CFIX > 0 ? density_sum_fixed<T, (CFIX > 0 ? CFIX : 16)>(ps, q, qlane, den_w)
                                 : density_sum<T>(ps, q, qlane, den_w);
        if (qlane == 0) out[p] = s;
    }
}
inline unsigned density_xyz_grid(int64_t M) {
    return (unsigned)std::min<uint64_t>(((uint64_t)M + kTile - 1) / kTile, (uint64_t)lm_persistent_blocks(8));
}
inline bool planes_all_64(const lm_plane *planes, int n) {
    bool all = true;
    for (int k = 0; k < n; ++k) all &= planes[k].C == 64;
    return all;
}

}  // namespace
