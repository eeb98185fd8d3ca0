// Part 2: bilinear plane x linear line feature gather over channel-last tables.
//
// Four lanes share one sample.  Lane q of the quad owns channels [V*q, V*q+V) of every
// group of 4V channels (V = 4 floats or 8 halves = one 16-byte load), so the quad reads
// 64 contiguous bytes per load instruction and a corner of a 16-channel fp32 plane is one
// such read.  All planes of all resolution levels are walked inside one launch; the
// per-plane partial sums stay in registers.  Work is a grid-stride loop over tiles of 64
// samples so the launch shape does not depend on counts that only exist on the device.
//
// Interpolation follows F.grid_sample(align_corners=True, zeros padding) as the reference
// calls it (app/models/gridnerf_sequential.py:803-812, 851-862): unnormalise
// ((c+1)/2)*(size-1), corners floor/floor+1, out-of-range corners contribute zero.
#include <algorithm>

#include "lm_common.h"
#include "lm_gather.h"
#include "lm_mma.h"

namespace {

// ---- explicit coordinates (density: lm_gather.h) ------------------------------------------
template <typename T>
__global__ __launch_bounds__(kBlock) void k_app_xyz(PlaneSet ps, int K, const float *__restrict__ xyz, uint64_t M,
                                                    float *__restrict__ out) {
    __shared__ __align__(16) float s_tile[kBlock / LM_WAVE][16 * kStageRow];
    const unsigned slot = threadIdx.x >> 2, wave = threadIdx.x / LM_WAVE;
    const uint64_t n_tiles = (M + kTile - 1) / kTile;
    for (uint64_t tile = lm_xcd_swizzle(blockIdx.x, gridDim.x); tile < n_tiles; tile += gridDim.x) {
        const uint64_t p0 = tile * kTile + wave * 16;  // whole waves stay or leave
        if (p0 >= M) continue;
        const uint64_t p = tile * kTile + slot, pc = p < M ? p : M - 1;
        float q[4] = {xyz[3 * pc], xyz[3 * pc + 1], xyz[3 * pc + 2], 0.0f};
        app_store_wave<T>(ps, q, p0, M, K, out, s_tile[wave]);
    }
}

// ---- alpha on a lattice over the AABB (getDenseAlpha / compute_alpha) ------------------------
// Point (i, j, k) = aabb0 * (1 - s) + aabb1 * s with s from three host tables, every product and
// sum rounded on its own like the reference's tensor expression.  A point the existing occupancy
// volume does not see (lookup not > 0) keeps sigma 0.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_dense_alpha(lm_geom g, PlaneSet ps, const float *__restrict__ den_w,
                                                        const float *__restrict__ lin_x,
                                                        const float *__restrict__ lin_y,
                                                        const float *__restrict__ lin_z, int gx, int gy, int gz,
                                                        int act, float shift, float length, float *__restrict__ alpha) {
    const unsigned qlane = threadIdx.x & 3u, slot = threadIdx.x >> 2;
    const uint64_t M = (uint64_t)gx * gy * gz;
    const uint64_t n_tiles = (M + kTile - 1) / kTile;
    for (uint64_t tile = lm_xcd_swizzle(blockIdx.x, gridDim.x); tile < n_tiles; tile += gridDim.x) {
        const uint64_t p = tile * kTile + slot;
        if (p >= M) continue;
        const int k = (int)(p % (uint64_t)gz), j = (int)((p / (uint64_t)gz) % (uint64_t)gy);
        const int i = (int)(p / ((uint64_t)gz * gy));
        const float s[3] = {lin_x[i], lin_y[j], lin_z[k]};
        float pt[3], q[4];
        q[3] = 0.0f;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const float a = g.aabb[d] * (1.0f - s[d]);
            const float b = g.aabb[3 + d] * s[d];
            pt[d] = a + b;
        }
        float sigma = 0.0f;
        if (!g.vol || lm_alpha_lookup(g, pt) > 0.0f) {
            lm_normalise(g, pt, q);
            sigma = activate(density_sum<T>(ps, q, qlane, den_w), act, shift);
        }
        if (qlane == 0) alpha[p] = 1.0f - expf((-sigma) * length);
    }
}

// ---- list driven (inside the render) -------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(kBlock) void k_density_list(lm_geom g, PlaneSet ps, const float *__restrict__ den_w,
                                                         const float *__restrict__ rays,
                                                         const uint32_t *__restrict__ list,
                                                         const uint32_t *__restrict__ count, int act, float shift,
                                                         float *__restrict__ sigma) {
    const unsigned qlane = threadIdx.x & 3u, slot = threadIdx.x >> 2;
    const uint64_t M = *count;
    const uint64_t n_tiles = (M + kTile - 1) / kTile;
    for (uint64_t tile = lm_xcd_swizzle(blockIdx.x, gridDim.x); tile < n_tiles; tile += gridDim.x) {
        const uint64_t p = tile * kTile + slot;
        if (p >= M) continue;
        float q[4];
        list_coords(g, rays, list[p], q);
        const float s = density_sum<T>(ps, q, qlane, den_w);
        if (qlane == 0) sigma[p] = activate(s, act, shift);
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_app_list(lm_geom g, PlaneSet ps, int K, const float *__restrict__ rays,
                                                     const uint32_t *__restrict__ list,
                                                     const uint32_t *__restrict__ count, uint32_t cap,
                                                     float *__restrict__ out) {
    __shared__ __align__(16) float s_tile[kBlock / LM_WAVE][16 * kStageRow];
    const unsigned slot = threadIdx.x >> 2, wave = threadIdx.x / LM_WAVE;
    const uint64_t M = min(*count, cap);  // the counter keeps counting past the list's capacity
    const uint64_t n_tiles = (M + kTile - 1) / kTile;
    for (uint64_t tile = lm_xcd_swizzle(blockIdx.x, gridDim.x); tile < n_tiles; tile += gridDim.x) {
        const uint64_t p0 = tile * kTile + wave * 16;  // whole waves stay or leave
        if (p0 >= M) continue;
        const uint64_t p = tile * kTile + slot;
        float q[4];
        list_coords(g, rays, list[p < M ? p : M - 1], q);
        app_store_wave<T>(ps, q, p0, M, K, out, s_tile[wave]);
    }
}


// ---- density gather fused with the transmittance march ------------------------------------
// Four lanes (a quad) own one ray at a time and walk its valid samples in order: gather the
// density of the next sample (each lane a quarter of the channels), turn it into alpha and a
// weight, carry the transmittance along.  Quads take rays from a queue of the rays that have
// valid samples and fetch a new one as soon as theirs ends, so the sixteen quads of a wave
// stay busy whatever the rays' lengths.  Two things follow from walking rays in lock step:
// neighbouring rays are at similar depths in the same load instruction, so their corner
// texels share cache lines; and a ray can stop once its transmittance is below term_eps,
// before the density of the samples behind is ever fetched, or (skip_lost) once nothing behind can change its results
// (155.8 -> 129.2 million samples gathered for 518400 rays of 3544 steps, 8.4 -> 5.9 million for 160000 rays of 128).  With term_eps = 0 the weights
// are those of the separate density + weights kernels, bit for bit (same operations, and the
// transmittance is the same sequential product torch.cumprod forms, app/tools/utils.py:51-64).
template <typename T, int NS, bool ROLL>  // NS samples of a ray per round
__global__ __launch_bounds__(kBlock) void k_march(lm_geom g, PlaneSet ps, const float *__restrict__ den_w,
                                                  const float *__restrict__ rays, const uint64_t *__restrict__ bitmap,
                                                  const uint32_t *__restrict__ p_first,
                                                  const uint64_t *__restrict__ word_mask,
                                                  const uint32_t *__restrict__ ray_list,
                                                  const uint32_t *__restrict__ bins, uint32_t n_rays,
                                                  uint32_t *__restrict__ queue,
                                                  int act, float shift, float distance_scale, float weight_thres,
                                                  float stop, float *__restrict__ w_valid,
                                                  float *__restrict__ acc_out, float *__restrict__ depth_out,
                                                  uint32_t *__restrict__ app_cnt, uint32_t *__restrict__ p_end_out,
                                                  uint32_t *__restrict__ n_marched) {
    const unsigned lane = lm_lane(), qlane = lane & 3u, leader = lane & ~3u;
    // One cursor per XCD (workgroups go to the XCDs round robin): an XCD takes every n_queues-th
    // granule of consecutive queue entries, so rays that are neighbours on screen march on the
    // same XCD at the same time and meet in its L2.  Granules of 1024 rays when there are many,
    // smaller ones for short queues so that every XCD still gets its share.
    const uint32_t n_queues = gridDim.x < (unsigned)LM_XCDS ? gridDim.x : (unsigned)LM_XCDS;
    const uint32_t my_q = blockIdx.x % n_queues;
    uint32_t *my_queue = queue + my_q;
    uint32_t marched = 0;  // samples whose density this lane's quad gathered (statistics)
    // cumulative sizes of the four ray lists (long rays first)
    const uint32_t end0 = bins[0], end1 = end0 + bins[1], end2 = end1 + bins[2], n_active = end2 + bins[3];
    const int log_n = 31 - __clz((int)(n_active | 1u));
    const uint32_t granule_shift = (uint32_t)(log_n >= 16 ? 10 : log_n >= 10 ? log_n - 6 : 4);
    const int S = g.S;
    bool have = false, done = false;
    uint32_t r = 0, p = 0, cnt = 0;
    uint64_t flat0 = 0;
    float ray[6] = {0, 0, 0, 0, 0, 0}, rp = 0.0f, Tr = 1.0f, acc = 0.0f, depth = 0.0f, z_last = 0.0f;
    BitWalk it;
    it.bits = 0; it.w = it.w0 = it.w_last = 0; it.flat1 = 0; it.pos = 0; it.bitmap = bitmap; it.prefix = nullptr;
    it.todo = it.ahead = 0; it.masked = false;
    while (true) {
        // quads without a ray take the next ones from the queue: one atomic per wave and round
        const bool need = !have && !done;
        const uint64_t need_mask = __ballot(need && qlane == 0);
        if (need_mask) {
            const int first = __ffsll((unsigned long long)need_mask) - 1;
            uint32_t base = 0;
            if ((int)lane == first) base = atomicAdd(my_queue, (uint32_t)__popcll(need_mask));
            base = __shfl(base, first);
            if (need) {
                const uint32_t local = base + (uint32_t)__popcll(need_mask & ((1ull << leader) - 1ull));
                const uint32_t idx = ((((local >> granule_shift) * n_queues + my_q)) << granule_shift) + (local & ((1u << granule_shift) - 1u));
                if (idx >= n_active) {
                    done = true;
                } else {
                    r = idx < end0   ? ray_list[idx]
                        : idx < end1 ? ray_list[(size_t)n_rays + (idx - end0)]
                        : idx < end2 ? ray_list[2 * (size_t)n_rays + (idx - end1)]
                                     : ray_list[3 * (size_t)n_rays + (idx - end2)];
                    const float2 *rp2 = reinterpret_cast<const float2 *>(rays + 6 * (size_t)r);
                    const float2 a = rp2[0], b = rp2[1], c = rp2[2];
                    ray[0] = a.x; ray[1] = a.y; ray[2] = b.x; ray[3] = b.y; ray[4] = c.x; ray[5] = c.y;
                    rp = lm_ray_param(g, ray);
                    flat0 = (uint64_t)r * (uint64_t)S;
                    it.start_at(bitmap, flat0, flat0 + S, p_first[r], word_mask ? word_mask[r] : ~0ull);
                    p = it.pos;
                    z_last = lm_sample_z(g, rp, S - 1);
                    Tr = 1.0f; acc = 0.0f; depth = 0.0f; cnt = 0;
                    have = true;
                }
            }
        }
        if (!__any(have)) break;
        if (have) {
            // up to NS samples per round: their densities are gathered together, the weights follow in order
            uint64_t flat[NS];
            int n_have = 0;
#pragma unroll
            for (int n = 0; n < NS; ++n) {
                flat[n] = n ? flat[n - 1] : 0;
                if (n_have == n && it.next(flat[n])) n_have = n + 1;
            }
            bool finish = n_have == 0;
            if (!finish) {
                // lane n of the quad prepares sample n: coordinates, footprints, and after the
                // gather its alpha (missing samples repeat the first; their results are unused)
                const int mine = (int)(qlane & (unsigned)(NS - 1));
                uint64_t flat_m = flat[0];
#pragma unroll
                for (int n = 1; n < NS; ++n)
                    if (mine == n && n < n_have) flat_m = flat[n];
                const int s_m = (int)(flat_m - flat0);
                const float z_m = lm_sample_z(g, rp, s_m);
                float q_m[4], f[NS];
                {
                    float pt[3];
                    lm_point(ray, z_m, pt);
                    lm_normalise(g, pt, q_m);
                    q_m[3] = __int_as_float(g.div0 > 0 ? lm_block_coords(g, q_m) : 0);
                }
                if constexpr (ROLL) density_sum_rolling<T>(ps, q_m, qlane, den_w, f);
                else density_sum_n<T, NS>(ps, q_m, qlane, den_w, f);
                marched += (uint32_t)n_have;
                float f_m = f[0];
#pragma unroll
                for (int n = 1; n < NS; ++n)
                    if (mine == n) f_m = f[n];
                const float sig = activate(f_m, act, shift);
                const float dist = (s_m + 1 < S) ? lm_sample_z(g, rp, s_m + 1) - z_m : 0.0f;
                const float d2 = dist * distance_scale;
                const float alpha_m = 1.0f - expf(-sig * d2);
                float alpha_n[NS], z_n[NS];
#pragma unroll
                for (int n = 0; n < NS; ++n) {
                    alpha_n[n] = quad_lane(alpha_m, n);
                    z_n[n] = quad_lane(z_m, n);
                }
#pragma unroll
                for (int n = 0; n < NS; ++n) {
                    if (n >= n_have || finish) break;
                    const float alpha = alpha_n[n];
                    const float wgt = alpha * Tr;
                    Tr = Tr * ((1.0f - alpha) + 1e-10f);
                    if (qlane == 0) w_valid[p] = wgt;
                    acc += wgt;
                    depth += wgt * z_n[n];
                    cnt += wgt > weight_thres;
                    ++p;
                    finish = stop > 0.0f && Tr < stop;
                }
                if (n_have < NS) finish = true;  // the ray's last samples
                else if (stop < 0.0f && !finish)
                    finish = lm_rest_is_lost(Tr, acc, depth, quad_lane(dist, NS - 1), z_last, weight_thres);
            }
            if (finish) {
                if (qlane == 0) {
                    acc_out[r] = acc; depth_out[r] = depth; app_cnt[r] = cnt; p_end_out[r] = p;
                }
                have = false;
            }
        }
    }
    if (qlane != 0) marched = 0;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) marched += __shfl_xor(marched, d);
    if (lane == 0 && marched) atomicAdd(n_marched, marched);
}

// ---- appearance gather fused with basis_mat --------------------------------------------------
// One wave owns 32 appearance samples; lane (j, h) gathers, for sample j, CW consecutive
// channels of every group of 2*CW (the lane pair of a sample covers the group), multiplies
// plane by line and feeds the products straight into the matrix cores as the B operand of
// basis_mat (A = the packed basis fragments, resident in LDS).  The [n, P*L*C] product
// matrix never exists in memory; the kernel writes the 27 projected features per sample.
template <int PREC> struct AppFeatBlock { static constexpr int N = 512; };

// LDS: [basis fragments | one product tile per wave].  A tile is 32 samples x (C + 4) floats.
__host__ __device__ inline size_t app_feat_tile_bytes(int C) { return (size_t)32 * (C + 4) * sizeof(float); }

// XYZ: the samples are M_host points given by their normalised coordinates (`rays` = xyz[M][3]) instead of list entries.
// Products through memory and a second kernel for basis_mat instead (k_app_xyz + k_basis) take 2.56 ms for 1 000 003 random
// points of nine 48-channel planes, 1.7 GB of products written and read again; this kernel takes 1.46 ms.
template <int PREC, typename T, int NU, bool XYZ>  // NU = groups of 16 channels per plane (C = 16 * NU)
__global__ __launch_bounds__(AppFeatBlock<PREC>::N) void k_app_feat(lm_geom g, PlaneSet ps, int K,
                                                                   const char *__restrict__ packed, lm_mma::PackLayout L,
                                                                   const float *__restrict__ rays, uint64_t M_host,
                                                                   const uint32_t *__restrict__ list,
                                                                   const uint32_t *__restrict__ count, uint32_t cap,
                                                                   float *__restrict__ feat) {
    using namespace lm_mma;
    using Mm = Mma<PREC>;
    using frag = typename Mm::frag;
    constexpr int NP = Mm::NP;
    constexpr int V = Vec<T>::V;
    constexpr int C = 16 * NU, ROW = C + 4;
    constexpr int NG = (C + V * kQuad - 1) / (V * kQuad);  // 16-byte loads per lane, corner and plane
    constexpr int G = Mm::G, CW = Mm::CW;
    extern __shared__ __align__(16) char lds[];
    const size_t basis_bytes = (size_t)32 * K * sizeof(typename Mm::elem) * NP;  // K MFMA K-slots x 32 rows
    {
        const uint4 *src = reinterpret_cast<const uint4 *>(packed + L.basis);
        uint4 *dst = reinterpret_cast<uint4 *>(lds);
        for (size_t i = threadIdx.x; i < basis_bytes / 16; i += blockDim.x) dst[i] = src[i];
        __syncthreads();
    }
    const frag *A = reinterpret_cast<const frag *>(lds);
    const unsigned lane = lm_lane(), j = lane & 31u, h = lane >> 5;
    const unsigned qlane = lane & 3u, gs = lane >> 2;  // gather role: 4 lanes per sample, 16 samples per pass
    float *tile = reinterpret_cast<float *>(lds + basis_bytes + (threadIdx.x / LM_WAVE) * app_feat_tile_bytes(C));
    const uint64_t M = XYZ ? M_host : (uint64_t)min(*count, cap);  // the counter keeps counting past the list's capacity
    const uint64_t n_tiles = (M + 31) / 32;
    constexpr unsigned kWaves = AppFeatBlock<PREC>::N / LM_WAVE;
    const uint64_t wave_id = (uint64_t)lm_xcd_swizzle(blockIdx.x, gridDim.x) * kWaves + threadIdx.x / LM_WAVE;
    const uint64_t n_waves = (uint64_t)gridDim.x * kWaves;
    for (uint64_t tile_id = wave_id; tile_id < n_tiles; tile_id += n_waves) {
        // the two samples this lane gathers for (pass 0: tile row gs, pass 1: row 16 + gs)
        float q0[4], q1[4];
        {
            const uint64_t p0 = tile_id * 32 + gs, p1 = p0 + 16, c0 = p0 < M ? p0 : M - 1, c1 = p1 < M ? p1 : M - 1;
            if constexpr (XYZ) {
#pragma unroll
                for (int i = 0; i < 3; ++i) { q0[i] = rays[3 * c0 + i]; q1[i] = rays[3 * c1 + i]; }
                q0[3] = q1[3] = 0.0f;
            } else {
                list_coords(g, rays, list[c0], q0);
                list_coords(g, rays, list[c1], q1);
            }
        }
        floatx16 acc;
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
        int t = 0;  // running MFMA step over the concatenated channels
        // Both samples' footprints of a plane are loaded with every load issued before the first use
        // (one memory round trip per plane), and the loads of plane k + 1 are issued before the
        // matrix step of plane k, which then runs under their latency.  Where that many loads in
        // flight would not fit the registers (wide planes), one sample's loads at a time.
        constexpr bool kAhead = 2 * NG * 6 * V <= 144;
        Taps2 t2[2];
        Taps1 t1[2];
        Footprint<T> fp[2][NG];
        auto taps_pass = [&](int k, int pass) {
            const lm_plane &pl = ps.p[k];
            const float *q = pass ? q1 : q0;
            t2[pass] = plane_taps(pl, pick(q, pl.ax0), pick(q, pl.ax1));
            t1[pass] = line_taps(pl, pick(q, pl.axl));
            block_taps(pl, ps.nblk, q, t2[pass], t1[pass]);
        };
        auto load_pass = [&](int k, int pass) {
            const lm_plane &pl = ps.p[k];
#pragma unroll
            for (int gi = 0; gi < NG; ++gi) {
                const int c = V * (int)qlane + gi * V * kQuad;
                if (c < C) footprint_load<T>(pl, t2[pass], t1[pass], c, fp[pass][gi]);
            }
        };
        auto emit_pass = [&](int pass) {
            float *row = tile + (pass * 16 + gs) * ROW;
#pragma unroll
            for (int gi = 0; gi < NG; ++gi) {
                const int c = V * (int)qlane + gi * V * kQuad;
                if (c >= C) continue;
                float prod[V];
                footprint_products<T>(fp[pass][gi], t2[pass], t1[pass], prod);
                if constexpr (V % 4 == 0) {
#pragma unroll
                    for (int i = 0; i < V; i += 4)
                        *reinterpret_cast<float4 *>(row + c + i) = make_float4(prod[i], prod[i + 1], prod[i + 2], prod[i + 3]);
                } else {
#pragma unroll
                    for (int i = 0; i < V; i += 2) *reinterpret_cast<float2 *>(row + c + i) = make_float2(prod[i], prod[i + 1]);
                }
            }
        };
        if (kAhead) { taps_pass(0, 0); taps_pass(0, 1); load_pass(0, 0); load_pass(0, 1); }
        for (int k = 0; k < ps.n; ++k) {
            if (kAhead) {
                __builtin_amdgcn_sched_barrier(0);
                emit_pass(0);
                emit_pass(1);
                __builtin_amdgcn_sched_barrier(0);
                if (k + 1 < ps.n) { taps_pass(k + 1, 0); taps_pass(k + 1, 1); load_pass(k + 1, 0); load_pass(k + 1, 1); }
            } else {
#pragma unroll
                for (int pass = 0; pass < 2; ++pass) {
                    taps_pass(k, pass);
                    load_pass(k, pass);
                    __builtin_amdgcn_sched_barrier(0);
                    emit_pass(pass);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            // LDS operations of one wave complete in order; the fence only pins the compiler
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            // a lane-half reads CW consecutive channels of every 2*CW and feeds them G at a time
            // (the order lm_mlp_pack lays the basis fragments out in)
#pragma unroll
            for (int it = 0; it < C / (2 * CW); ++it) {
                float cw[CW];
                const float4 *src = reinterpret_cast<const float4 *>(tile + j * ROW + 2 * CW * it + CW * (int)h);
#pragma unroll
                for (int i = 0; i < CW / 4; ++i) {
                    const float4 x = src[i];
                    cw[4 * i] = x.x; cw[4 * i + 1] = x.y; cw[4 * i + 2] = x.z; cw[4 * i + 3] = x.w;
                }
#pragma unroll
                for (int u = 0; u < CW / G; ++u, ++t) {
                    frag bf[NP];
                    Mm::pack(cw + u * G, bf);
                    const frag a0 = A[(t * NP) * 64 + lane];
                    acc = Mm::mma(a0, bf[0], acc);
                    if constexpr (NP == 2) {
                        const frag a1 = A[(t * NP + 1) * 64 + lane];
                        acc = Mm::mma(a1, bf[0], acc);
                        acc = Mm::mma(a0, bf[1], acc);
                    }
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        const uint64_t p = tile_id * 32 + j;
        if (p < M) {
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int r = row_of(v, (int)h);
                if (r < kAppDim) feat[p * kAppDim + r] = acc[v];
            }
        }
    }
}

size_t app_feat_lds(int prec, int K, int C) {
    using namespace lm_mma;
    const size_t elem = prec == LM_MLP_F32 || prec == LM_MLP_F16X2 ? 4 : 2;  // F16X2: two parts
    return (size_t)32 * K * elem + (AppFeatBlock<LM_MLP_F16>::N / LM_WAVE) * app_feat_tile_bytes(C);
}

template <int PREC, typename T, bool XYZ>
int launch_app_feat(int nu, const lm_geom &geom, const void *packed, const PlaneSet &ps, int K, const float *rays, uint64_t M,
                    const uint32_t *list, const uint32_t *count, uint32_t cap, float *feat, hipStream_t st) {
    using namespace lm_mma;
    const PackLayout L = pack_layout(PREC, K);
    constexpr int kThreads = AppFeatBlock<PREC>::N;
    const size_t lds = app_feat_lds(PREC, K, 16 * nu);
    if (lds > 160 * 1024) LM_FAIL(LM_ERR_UNSUPPORTED, "basis_mat fragments + tiles (%zu bytes) do not fit LDS", lds);
    const unsigned per_cu = (unsigned)std::max<size_t>(1, std::min<size_t>(2, (size_t)(160 * 1024) / lds));
    unsigned grid = (unsigned)lm_persistent_blocks((int)per_cu);
    if (XYZ) grid = (unsigned)std::min<uint64_t>(grid, (M + 31) / 32);  // few points: a tile per workgroup
#define LM_AF_CASE(NU_)                                                                                            \
    case NU_: {                                                                                                    \
        auto kern = &k_app_feat<PREC, T, NU_, XYZ>;                                                                \
        static thread_local size_t reserved_on[LM_MAX_DEVICES] = {}; /* set once per thread, device, kernel, size */ \
        size_t &reserved = reserved_on[lm_current_device()];                                                       \
        if (reserved != lds) {                                                                                     \
            hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),                               \
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);              \
            if (e != hipSuccess)                                                                                   \
                LM_FAIL(LM_ERR_LAUNCH, "k_app_feat: LDS reservation failed: %s", hipGetErrorString(e));            \
            reserved = lds;                                                                                        \
        }                                                                                                          \
        hipLaunchKernelGGL(kern, dim3(grid), dim3(kThreads), lds, st, geom, ps, K, (const char *)packed, L, rays, M, \
                           list, count, cap, feat);                                                                \
        break;                                                                                                     \
    }
    if constexpr (std::is_same<T, Half6>::value) {  // six channels per lane divide 48-channel planes only
        switch (nu) {
            LM_AF_CASE(3)
            default: LM_FAIL(LM_ERR_UNSUPPORTED, "unsupported channel grouping %d", nu);
        }
    } else {
        switch (nu) {
            LM_AF_CASE(1)
            LM_AF_CASE(2)
            LM_AF_CASE(3)
            LM_AF_CASE(4)
            default: LM_FAIL(LM_ERR_UNSUPPORTED, "unsupported channel grouping %d", nu);
        }
    }
#undef LM_AF_CASE
    LM_CHECK_LAUNCH("k_app_feat");
    return LM_OK;
}

}  // namespace

// -------------------------------------------------------------------------------------------
int lm_check_planes(const lm_plane *planes, int32_t n, int *dtype_out, int *K_out) {
    LM_REQUIRE(planes != nullptr, "planes is null");
    LM_REQUIRE(n >= 1 && n <= LM_MAX_PLANES, "n_planes %d out of range 1..%d", n, LM_MAX_PLANES);
    int K = 0;
    for (int k = 0; k < n; ++k) {
        const lm_plane &p = planes[k];
        LM_REQUIRE(p.plane && p.line, "plane %d: null table", k);
        LM_REQUIRE(lm_aligned16(p.plane) && lm_aligned16(p.line), "plane %d: tables must be 16-byte aligned", k);
        LM_REQUIRE(p.H > 0 && p.W > 0 && p.Len > 0, "plane %d: empty table", k);
        LM_REQUIRE(p.C > 0 && (int64_t)p.W * p.C < ((int64_t)1 << 31), "plane %d: a row of more than 2^31 elements", k);
        LM_REQUIRE(p.dtype == planes[0].dtype, "planes must share one storage type");
        LM_REQUIRE(p.dtype == LM_F32 || p.dtype == LM_F16, "plane %d: unknown dtype %d", k, p.dtype);
        const int V = p.dtype == LM_F32 ? 4 : 8;
        LM_REQUIRE(p.C > 0 && p.C % V == 0, "plane %d: channel count %d must be a multiple of %d", k, p.C, V);
        LM_REQUIRE(p.ax0 >= 0 && p.ax0 < 3 && p.ax1 >= 0 && p.ax1 < 3 && p.axl >= 0 && p.axl < 3, "plane %d: bad axis", k);
        K += p.C;
    }
    *dtype_out = planes[0].dtype;
    if (K_out) *K_out = K;
    return LM_OK;
}

extern "C" int lm_gather_density_xyz(const lm_plane *planes, int32_t n_planes, const float *density_basis,
                                     const float *xyz, int64_t M, float *out, void *stream) {
    int dtype;
    if (int rc = lm_check_planes(planes, n_planes, &dtype, nullptr)) return rc;
    LM_REQUIRE(M >= 0, "negative count");
    if (M == 0) return LM_OK;
    LM_REQUIRE(xyz && out, "null buffer");
    const PlaneSet ps = make_set(planes, n_planes);
    const unsigned grid = density_xyz_grid(M);
    const bool all64 = planes_all_64(planes, n_planes);
#define LM_DX(T_, C_)                                                                                                    \
    hipLaunchKernelGGL((k_density_xyz<T_, C_, false>), dim3(grid), dim3(kBlock), 0, (hipStream_t)stream, ps, density_basis, xyz, \
                       (uint64_t)M, out, nullptr)
    if (dtype == LM_F32) {
        if (all64) LM_DX(float, 64); else LM_DX(float, 0);
    } else {
        if (all64) LM_DX(__half, 64); else LM_DX(__half, 0);
    }
#undef LM_DX
    LM_CHECK_LAUNCH("k_density_xyz");
    return LM_OK;
}

extern "C" int lm_gather_app_xyz(const lm_plane *planes, int32_t n_planes, const float *xyz, int64_t M, float *out,
                                 void *stream) {
    int dtype, K;
    if (int rc = lm_check_planes(planes, n_planes, &dtype, &K)) return rc;
    LM_REQUIRE(M >= 0, "negative count");
    if (M == 0) return LM_OK;
    LM_REQUIRE(xyz && out && lm_aligned16(out), "null or misaligned buffer");
    const PlaneSet ps = make_set(planes, n_planes);
    const uint64_t tiles = ((uint64_t)M + kTile - 1) / kTile;
    const unsigned grid = (unsigned)std::min<uint64_t>(tiles, (uint64_t)lm_persistent_blocks(8));
    if (dtype == LM_F32)
        hipLaunchKernelGGL(k_app_xyz<float>, dim3(grid), dim3(kBlock), 0, (hipStream_t)stream, ps, K, xyz, (uint64_t)M, out);
    else
        hipLaunchKernelGGL(k_app_xyz<__half>, dim3(grid), dim3(kBlock), 0, (hipStream_t)stream, ps, K, xyz, (uint64_t)M, out);
    LM_CHECK_LAUNCH("k_app_xyz");
    return LM_OK;
}

int lm_check_geom(const lm_geom *g);

extern "C" int lm_density_valid(const lm_model *m, const float *rays, const uint32_t *valid_idx,
                                const uint32_t *counters, float *sigma, void *stream) {
    LM_REQUIRE(m != nullptr, "model is null");
    if (int rc = lm_check_geom(&m->geom)) return rc;
    int dtype;
    if (int rc = lm_check_planes(m->density, m->n_planes, &dtype, nullptr)) return rc;
    LM_REQUIRE(rays && valid_idx && counters && sigma, "null buffer");
    LM_REQUIRE(m->act == LM_ACT_SOFTPLUS || m->act == LM_ACT_RELU, "unknown activation %d", m->act);
    const PlaneSet ps = make_set(m->density, m->n_planes, &m->geom);
    const unsigned grid = (unsigned)lm_persistent_blocks(8);
    if (dtype == LM_F32)
        hipLaunchKernelGGL(k_density_list<float>, dim3(grid), dim3(kBlock), 0, (hipStream_t)stream, m->geom, ps,
                           m->density_basis, rays, valid_idx, counters + LM_STAT_N_VALID, m->act, m->density_shift, sigma);
    else
        hipLaunchKernelGGL(k_density_list<__half>, dim3(grid), dim3(kBlock), 0, (hipStream_t)stream, m->geom, ps,
                           m->density_basis, rays, valid_idx, counters + LM_STAT_N_VALID, m->act, m->density_shift, sigma);
    LM_CHECK_LAUNCH("k_density_list");
    return LM_OK;
}

extern "C" int lm_dense_alpha(const lm_model *m, const float *lin_x, const float *lin_y, const float *lin_z,
                              int32_t gx, int32_t gy, int32_t gz, float length, float *alpha, void *stream) {
    LM_REQUIRE(m != nullptr, "model is null");
    const lm_geom &g = m->geom;
    if (g.vol) {
        LM_REQUIRE(g.vd > 0 && g.vh > 0 && g.vw > 0, "occupancy volume has an empty dimension");
        LM_REQUIRE(g.vol_dtype == LM_F32 || g.vol_dtype == LM_U8 || g.vol_dtype == LM_CELLS, "occupancy volume dtype %d",
                   g.vol_dtype);
    }
    int dtype;
    if (int rc = lm_check_planes(m->density, m->n_planes, &dtype, nullptr)) return rc;
    LM_REQUIRE(gx > 0 && gy > 0 && gz > 0, "empty lattice %d x %d x %d", gx, gy, gz);
    LM_REQUIRE(lin_x && lin_y && lin_z && alpha, "null buffer");
    if (g.div0 > 0)
        LM_FAIL(LM_ERR_UNSUPPORTED, "dense alpha of a block-stacked model: the reference evaluates it per block during "
                                    "training only");
    LM_REQUIRE(m->act == LM_ACT_SOFTPLUS || m->act == LM_ACT_RELU, "unknown activation %d", m->act);
    const PlaneSet ps = make_set(m->density, m->n_planes, &m->geom);
    const uint64_t tiles = ((uint64_t)gx * gy * gz + kTile - 1) / kTile;
    const unsigned grid = (unsigned)std::min<uint64_t>(tiles, (uint64_t)lm_persistent_blocks(8));
    if (dtype == LM_F32)
        hipLaunchKernelGGL(k_dense_alpha<float>, dim3(grid), dim3(kBlock), 0, (hipStream_t)stream, g, ps, m->density_basis,
                           lin_x, lin_y, lin_z, gx, gy, gz, m->act, m->density_shift, length, alpha);
    else
        hipLaunchKernelGGL(k_dense_alpha<__half>, dim3(grid), dim3(kBlock), 0, (hipStream_t)stream, g, ps, m->density_basis,
                           lin_x, lin_y, lin_z, gx, gy, gz, m->act, m->density_shift, length, alpha);
    LM_CHECK_LAUNCH("k_dense_alpha");
    return LM_OK;
}

// `count` entries of the list (at most `cap`, the list's capacity) -> products [count, K]
int lm_launch_app_products(const lm_model *m, const float *rays, const uint32_t *app_idx, const uint32_t *count, uint32_t cap,
                           float *products, hipStream_t st) {
    LM_REQUIRE(m != nullptr, "model is null");
    if (int rc = lm_check_geom(&m->geom)) return rc;
    int dtype, K;
    if (int rc = lm_check_planes(m->app, m->n_planes, &dtype, &K)) return rc;
    LM_REQUIRE(rays && app_idx && count && products && lm_aligned16(products), "null or misaligned buffer");
    const PlaneSet ps = make_set(m->app, m->n_planes, &m->geom);
    const unsigned grid = (unsigned)lm_persistent_blocks(8);
    if (dtype == LM_F32)
        hipLaunchKernelGGL(k_app_list<float>, dim3(grid), dim3(kBlock), 0, st, m->geom, ps, K, rays, app_idx, count, cap, products);
    else
        hipLaunchKernelGGL(k_app_list<__half>, dim3(grid), dim3(kBlock), 0, st, m->geom, ps, K, rays, app_idx, count, cap, products);
    LM_CHECK_LAUNCH("k_app_list");
    return LM_OK;
}

extern "C" int lm_app_products(const lm_model *m, const float *rays, const uint32_t *app_idx, const uint32_t *counters,
                               float *products, void *stream) {
    LM_REQUIRE(counters != nullptr, "counters is null");
    return lm_launch_app_products(m, rays, app_idx, counters + LM_STAT_N_APP, UINT32_MAX, products, (hipStream_t)stream);
}

// True when the fused gather + basis_mat kernel covers these appearance planes.
static int app_feat_covers(const lm_plane *planes, int n) {
    const int C = planes[0].C;
    for (int k = 0; k < n; ++k)
        if (planes[k].C != C) return 0;
    return C % 16 == 0 && C >= 16 && C <= 64;
}
int lm_app_feat_supported(const lm_model *m) { return app_feat_covers(m->app, m->n_planes); }

int lm_check_prec(int prec);
int lm_check_K(int K);
int lm_launch_app_features(const lm_model *m, const float *rays, const uint32_t *app_idx, const uint32_t *cnt, uint32_t cap,
                           float *feat, hipStream_t st);

// appearance samples (list order) -> feat [n_app, 27] = basis_mat(plane * line products)
extern "C" int lm_app_features(const lm_model *m, const float *rays, const uint32_t *app_idx, const uint32_t *counters,
                               float *feat, void *stream) {
    LM_REQUIRE(counters != nullptr, "counters is null");
    return lm_launch_app_features(m, rays, app_idx, counters + LM_STAT_N_APP, UINT32_MAX, feat, (hipStream_t)stream);
}

template <bool XYZ>
static int app_features(int prec, int dtype, int nu, const lm_geom &geom, const void *packed, const PlaneSet &ps, int K,
                        const float *rays, uint64_t M, const uint32_t *app_idx, const uint32_t *cnt, uint32_t cap, float *feat,
                        hipStream_t st) {
#define LM_AF_ONE(PREC_, T_) launch_app_feat<PREC_, T_, XYZ>(nu, geom, packed, ps, K, rays, M, app_idx, cnt, cap, feat, st)
#define LM_AF_GO(PREC_)                                                                                         \
    return dtype == LM_F32 ? LM_AF_ONE(PREC_, float)                                                            \
           : nu == 3       ? LM_AF_ONE(PREC_, Half6)                                                            \
           : (nu & 1)      ? LM_AF_ONE(PREC_, Half4)                                                            \
                           : LM_AF_ONE(PREC_, __half)
    switch (prec) {
        case LM_MLP_F32: LM_AF_GO(LM_MLP_F32);
        case LM_MLP_F16: LM_AF_GO(LM_MLP_F16);
        case LM_MLP_BF16: LM_AF_GO(LM_MLP_BF16);
        default: LM_AF_GO(LM_MLP_F16X2);
    }
#undef LM_AF_GO
#undef LM_AF_ONE
}

int lm_launch_app_features(const lm_model *m, const float *rays, const uint32_t *app_idx, const uint32_t *cnt, uint32_t cap,
                           float *feat, hipStream_t st) {
    LM_REQUIRE(m != nullptr, "model is null");
    if (int rc = lm_check_geom(&m->geom)) return rc;
    int dtype, K;
    if (int rc = lm_check_planes(m->app, m->n_planes, &dtype, &K)) return rc;
    if (int rc = lm_check_prec(m->mlp_prec)) return rc;
    if (int rc = lm_check_K(K)) return rc;
    LM_REQUIRE(rays && app_idx && cnt && feat, "null buffer");
    LM_REQUIRE(m->mlp_packed && lm_aligned16(m->mlp_packed), "packed colour-network weights are null or misaligned");
    if (!lm_app_feat_supported(m))
        LM_FAIL(LM_ERR_UNSUPPORTED, "fused appearance gather needs equal channel counts of 16..64 in steps of 16");
    const PlaneSet ps = make_set(m->app, m->n_planes, &m->geom);
    return app_features<false>(m->mlp_prec, dtype, m->app[0].C / 16, m->geom, m->mlp_packed, ps, K, rays, 0, app_idx, cnt, cap,
                               feat, st);
}

bool lm_few_points_take(int prec, int K, int64_t M);
int lm_launch_few_points(const lm_plane *planes, int n, int prec, int dtype, int K, const void *packed, const float *xyz, uint32_t M,
                         float *feat, hipStream_t st);

extern "C" int lm_app_features_xyz_supported(const lm_plane *planes, int32_t n_planes, int32_t prec) {
    int dtype, K;
    if (lm_check_planes(planes, n_planes, &dtype, &K) || lm_check_prec(prec) || lm_check_K(K)) return 0;
    return app_feat_covers(planes, n_planes) && app_feat_lds(prec, K, planes[0].C) <= 160 * 1024;
}

extern "C" int lm_app_features_xyz(const lm_plane *planes, int32_t n_planes, int32_t prec, const void *packed, const float *xyz,
                                   int64_t M, float *feat, void *stream) {
    int dtype, K;
    if (int rc = lm_check_planes(planes, n_planes, &dtype, &K)) return rc;
    if (int rc = lm_check_prec(prec)) return rc;
    if (int rc = lm_check_K(K)) return rc;
    LM_REQUIRE(M >= 0, "negative count");
    if (M == 0) return LM_OK;
    LM_REQUIRE(packed && xyz && feat && lm_aligned16(packed), "null or misaligned buffer");
    if (!lm_app_features_xyz_supported(planes, n_planes, prec))
        LM_FAIL(LM_ERR_UNSUPPORTED, "needs equal channel counts of 16..64 in steps of 16 and a basis_mat that fits LDS (K %d)", K);
    if (lm_few_points_take(prec, K, M)) return lm_launch_few_points(planes, n_planes, prec, dtype, K, packed, xyz, (uint32_t)M, feat, (hipStream_t)stream);
    return app_features<true>(prec, dtype, planes[0].C / 16, lm_geom{}, packed, make_set(planes, n_planes), K, xyz, (uint64_t)M,
                              nullptr, nullptr, 0u, feat, (hipStream_t)stream);
}

int lm_launch_march_wave(const lm_model *m, const float *rays, const uint64_t *bitmap, const uint32_t *p_first, const uint64_t *word_mask,
                         const uint32_t *ray_list, const uint32_t *bins, uint32_t n_rays, float *w_valid, float *acc, float *depth,
                         uint32_t *app_cnt, uint32_t *p_end, uint32_t *n_marched, hipStream_t st);

// Density + transmittance march over the rays listed in ray_list (those with valid samples).
int lm_launch_march(const lm_model *m, const float *rays, const uint64_t *bitmap, const uint32_t *p_first,
                    const uint64_t *word_mask, const uint32_t *ray_list, const uint32_t *bins, uint32_t n_rays, uint32_t *queue, float *w_valid,
                    float *acc,
                    float *depth, uint32_t *app_cnt, uint32_t *p_end, uint32_t *n_marched, hipStream_t st) {
    int dtype;
    if (int rc = lm_check_planes(m->density, m->n_planes, &dtype, nullptr)) return rc;
    LM_REQUIRE(m->act == LM_ACT_SOFTPLUS || m->act == LM_ACT_RELU, "unknown activation %d", m->act);
    const PlaneSet ps = make_set(m->density, m->n_planes, &m->geom);
    // as many workgroups as are resident at once (the kernel's register count decides), at most four per CU
    auto resident_grid = [](const void *kernel) {
        // asked once per thread and kernel: the answer depends on the kernel's registers only
        static thread_local const void *known_on[LM_MAX_DEVICES][6] = {};
        static thread_local unsigned grid_on[LM_MAX_DEVICES][6] = {};
        const int dev = lm_current_device();
        const void **known = known_on[dev];
        unsigned *grid = grid_on[dev];
        for (int i = 0; i < 6; ++i)
            if (known[i] == kernel) return grid[i];
        int per_cu = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kBlock, 0) != hipSuccess || per_cu < 1) per_cu = 2;
        const unsigned g = (unsigned)lm_persistent_blocks(std::min(per_cu, 4));
        for (int i = 0; i < 6; ++i)
            if (!known[i]) { known[i] = kernel; grid[i] = g; break; }
        return g;
    };
    int c_max = 0;
    for (int k = 0; k < m->n_planes; ++k) c_max = std::max(c_max, (int)m->density[k].C);
    // few rays: a wave per ray, one launch-wide round trip per 64-sample word instead of one per four samples
    if (n_rays <= LM_RAYS_LIMIT)
        return lm_launch_march_wave(m, rays, bitmap, p_first, word_mask, ray_list, bins, n_rays, w_valid, acc, depth, app_cnt, p_end, n_marched, st);
    // Up to four rays per quad of two workgroups per CU: no third workgroup, where the registers would allow one (fp16 tables of
    // 16 channels and fewer, 153 registers).  With few rays it adds none in flight at the end, when only long ones are left, and
    // shares the CU with them.  Whole calls, two / three per CU (and the plain sum, two per CU), us: city block of 256 samples per
    // ray and 4096^2 planes 13 000 rays 377 / 387 (382), 60 000 710 / 735 (712), 120 000 1115 / 1140 (1121), 250 000 2100 / 2115 (2109);
    // three 256^2 planes 13 000 226 / 237 (229), 60 000 569 / 584 (577), 120 000 948 / 948 (962), 250 000 1799 / 1768 (1833), 1 000 000
    // 6759 / 6471 (6912); nine planes 13 000 279 / 292 (292), 60 000 597 / 610 (620), 120 000 943 / 933 (957); block-stacked 13 000
    // 199 / 211, 120 000 627 / 655.  With a density projection the wait for its weights wants the third from earlier on
    // (60 000 rays of 886 samples 1602 / 1618, 120 000 3080 / 2908): always three there.
    const unsigned two = (unsigned)lm_persistent_blocks(2);
    const unsigned most = !m->density_basis && n_rays <= two * (unsigned)kTile * 4u ? two : ~0u;
#define LM_MARCH_ONE(T_, ROLL_)                                                                                            \
    hipLaunchKernelGGL((k_march<T_, 4, ROLL_>), dim3(std::min(most, resident_grid(reinterpret_cast<const void *>(&k_march<T_, 4, ROLL_>)))), \
                       dim3(kBlock), 0, st, m->geom, ps, m->density_basis, rays, bitmap,   \
                       p_first, word_mask, ray_list, bins, n_rays, queue, m->act, m->density_shift, m->distance_scale,            \
                       m->weight_thres, lm_stop_value(*m), w_valid, acc, depth, app_cnt, p_end, n_marched)
#define LM_MARCH(T_)                                                                   \
    if (density_rolls<T_>(m->density, m->n_planes, ps.nblk)) LM_MARCH_ONE(T_, true);   \
    else LM_MARCH_ONE(T_, false)
    // Four samples per round: one per lane of the quad for the footprint arithmetic, 24 loads per lane and plane
    // in flight, half as many dependent round trips per ray as with two (1080p frame, nine fp32 planes: 2.70 ->
    // 2.50 ms although the kernel then holds two waves per SIMD instead of three).  The rolling sum forced into three waves
    // (168 registers) spills: 22.9 -> 25.6 ms on the frame of 3544 samples per ray.
    if (dtype == LM_F32) {
        LM_MARCH(float);
    } else if (c_max <= 16) {  // 16-byte loads would leave half of every quad idle
        LM_MARCH(Half4);
    } else {
        LM_MARCH(__half);
    }
#undef LM_MARCH
#undef LM_MARCH_ONE
    LM_CHECK_LAUNCH("k_march");
    return LM_OK;
}
