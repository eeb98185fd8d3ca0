// The front half of a small chunk in one kernel: sampling, culling, density gather, transmittance and appearance
// entries, a workgroup of four waves for four rays.
//
// A chunk of a few thousand rays is a chain of dependent memory round trips, not bytes: with a kernel per stage
// (zeroed bitmap, cull, march with a wave per ray, list) each stage waits for the one before, a ray's words are marched
// one after the other, and most lanes of a word have no valid sample.  Here a workgroup takes its rays through all of it:
//   1. a wave owns a ray.  Lane = bitmap word: which runs of 64 samples can hold a valid one (box, coarse occupancy
//      level).  Lane = sample: the decisions of those words, four words' lookups in flight, kept in LDS;
//   2. rounds: every ray contributes its next (up to) 64 valid samples, ascending.  The round's samples are dealt evenly
//      to the four waves and gathered four lanes to a sample.  Up to 16 samples per wave give every quad one sample and
//      three planes at a time, up to 32 two samples and two planes, more four samples and one plane: about 24 loads per
//      lane in flight either way, and nine planes are three round trips instead of nine for the rays with a dozen valid
//      samples that are usual at 128 samples per ray;
//   3. the transmittance runs through a ray's samples of the round in order (the product torch.cumprod forms); the
//      round's appearance entries are appended to the ray's list in LDS;
//   4. one reservation per workgroup in the appearance list.  It is the only addition every workgroup makes to the counter
//      block (dropped rays, and valid samples where they are checked against a capacity, are added too): the counts per ray
//      go to memory and the composite kernel sums them, 64 rays at a time.  Additions of thousands of workgroups to one line
//      take 6.5 ns each: 12288 rays on three small planes, whole call, 232 us with valid and gathered samples added here too,
//      204 this way.
// Four rays per workgroup: with eight the rays that see something crowd into fewer workgroups, with two or one the
// samples of a round do not fill the waves (4096 rays of 128 samples on nine planes: 82 / 58 / 80 / 133 us with 8 / 4 / 2 /
// 1 rays before the transmittance was spread over the lanes).
// Measured against zeroed bitmap + cull + march with a wave per ray + list: 4096 rays as above 93 -> 45 us, 8192 rays of
// 886 samples on three planes 393 -> 310 us, 1024 rays on three 256^2 planes 51 -> 23 us.  With skip_lost (rays
// stop after the round behind which nothing can change their results) the second takes 230 us, the third 18.
// What bounds it (counters of the first / second): 3.1 / 3.8 TB/s past the L2, texture addressers 30 / 41 % busy, vector
// ALU 28 %, 1.1 / 1.5 waves per SIMD in flight on average: latency and the longest ray of a workgroup, not bytes.
// With 32-bit offsets and only the weights of the taps kept (density_sum_lean, tables below 4 GB) the fp32 kernel holds 210 registers
// instead of 256 and five spilled: 1024 rays 51.0 -> 48.4 us, 4096 rays 108.4 -> 104.2, 8192 rays of 886 samples 454 -> 419 (whole
// calls).  Forced into three waves per SIMD (168 registers, 30 spilled) 4096 rays take 126.
// Operations and order per ray are those of the kernels for large chunks, hence the same bits.
#include <algorithm>

#include "lm_common.h"
#include "lm_cull.h"
#include "lm_gather.h"

namespace {

constexpr int kRays = kBlock / LM_WAVE;  // rays per workgroup: a wave owns one
constexpr int kWordsMax = 64;            // a ray's decisions: up to 64 words of 64 samples
constexpr int kEntriesMax = 1024;        // appearance entries of a ray: at most S and 1 / weight threshold
constexpr int kRound = 64;               // samples a ray contributes to a round

// density_sum_n with G planes' loads in flight; planes of one channel group per lane only (G > 1)
template <typename T, int NS, int G>
__device__ __forceinline__ void density_sum_planes(const PlaneSet &ps, const float *q_mine, unsigned qlane,
                                                   const float *__restrict__ den_w, float *out) {
    constexpr int V = Vec<T>::V;
    float sum[NS];
#pragma unroll
    for (int n = 0; n < NS; ++n) sum[n] = 0.0f;
    const int c = V * (int)qlane;
    int col = 0;
    for (int k0 = 0; k0 < ps.n; k0 += G) {
        Taps2 t2[G][NS];
        Taps1 t1[G][NS];
        Footprint<T> f[G][NS];
#pragma unroll
        for (int i = 0; i < G; ++i) {
            if (k0 + i >= ps.n) break;
            const lm_plane pl = ps.p[k0 + i];
            Taps2 m2 = plane_taps(pl, pick(q_mine, pl.ax0), pick(q_mine, pl.ax1));
            Taps1 m1 = line_taps(pl, pick(q_mine, pl.axl));
            block_taps(pl, ps.nblk, q_mine, m2, m1);
#pragma unroll
            for (int n = 0; n < NS; ++n) {
                t2[i][n] = NS == 1 ? m2 : quad_lane(m2, n);
                t1[i][n] = NS == 1 ? m1 : quad_lane(m1, n);
                if (c < pl.C) footprint_load<T>(pl, t2[i][n], t1[i][n], c, f[i][n]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < G; ++i) {
            if (k0 + i >= ps.n) break;
            const int C = ps.p[k0 + i].C;
            if (c < C) {
#pragma unroll
                for (int n = 0; n < NS; ++n) {
                    float prod[V];
                    footprint_products<T>(f[i][n], t2[i][n], t1[i][n], prod);
#pragma unroll
                    for (int j = 0; j < V; ++j) sum[n] = den_w ? fmaf(den_w[col + c + j], prod[j], sum[n]) : sum[n] + prod[j];
                }
            }
            col += C;
        }
    }
#pragma unroll
    for (int n = 0; n < NS; ++n) {
        const float v = quad_sum(sum[n]);
        out[n] = den_w ? fmaxf(v, 0.0f) : v;
    }
}

// The same for tables density_sum_rolling takes: 32-bit offsets that are used up by the loads, and of the taps only the weights
// kept (on the lane that worked them out).  Same operations per sample, hence the same bits.
template <typename T, int NS, int G>
__device__ __forceinline__ void density_sum_lean(const PlaneSet &ps, const float *q_mine, unsigned qlane, const float *__restrict__ den_w, float *out) {
    float sum[NS];
#pragma unroll
    for (int n = 0; n < NS; ++n) sum[n] = 0.0f;
    int col = 0;
    for (int k0 = 0; k0 < ps.n; k0 += G) {
        RollTaps m[G];
        Footprint<T> f[G][NS];
        float w[G][Vec<T>::V] = {};
        int at = col;
#pragma unroll
        for (int i = 0; i < G; ++i) {
            if (k0 + i >= ps.n) break;
            const lm_plane pl = ps.p[k0 + i];
            m[i] = roll_taps<typename Vec<T>::elem>(pl, ps.nblk, q_mine);
            roll_weights<T>(pl, den_w, at, qlane, w[i]);
            at += pl.C;
#pragma unroll
            for (int n = 0; n < NS; ++n) roll_load<T, NS>(pl, m[i], n, qlane, f[i][n]);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < G; ++i) {
            if (k0 + i >= ps.n) break;
            const lm_plane pl = ps.p[k0 + i];
#pragma unroll
            for (int n = 0; n < NS; ++n) roll_use<T, NS>(pl, m[i], n, qlane, f[i][n], den_w != nullptr, w[i], sum[n]);
        }
        col = at;
    }
#pragma unroll
    for (int n = 0; n < NS; ++n) {
        const float v = quad_sum(sum[n]);
        out[n] = den_w ? fmaxf(v, 0.0f) : v;
    }
}

template <typename T, bool ROLL>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2))) void k_rays(
    lm_geom g, PlaneSet ps, int narrow, const float *__restrict__ den_w, const float *__restrict__ rays, uint32_t N, uint32_t row,
    int ent, int act, float shift, float distance_scale, float weight_thres, float stop, uint32_t cap_valid,
    uint32_t *__restrict__ app_first, uint32_t *__restrict__ app_cnt, uint32_t *__restrict__ app_idx, float *__restrict__ app_w,
    uint32_t cap_app, float *__restrict__ acc_out, float *__restrict__ depth_out, uint32_t *__restrict__ ray_valid,
    uint32_t *__restrict__ ray_marched, uint32_t *__restrict__ counters) {
    __shared__ float s_ray[kRays][8];                 // origin, direction, ray parameter
    __shared__ uint64_t s_word[kRays][kWordsMax];     // decisions
    __shared__ uint16_t s_item[kRays][kRound];        // the round's samples
    // their alphas, then transmittance factors, transmittances, weights; their depths, then weight x depth
    __shared__ __align__(16) float s_val[kRays][kRound + 4], s_z[kRays][kRound + 4];
    __shared__ uint32_t s_n[kRays], s_cnt[kRays], s_done[kRays], s_first[kRays];
    extern __shared__ __align__(16) char s_entries[];  // [kRays][ent] weights, [kRays][ent] sample indices
    const unsigned lane = lm_lane(), qlane = lane & 3u, quad = lane >> 2, wave = threadIdx.x / LM_WAVE;
    float *e_w = reinterpret_cast<float *>(s_entries) + wave * (unsigned)ent;
    uint16_t *e_s = reinterpret_cast<uint16_t *>(reinterpret_cast<float *>(s_entries) + kRays * ent) + wave * (unsigned)ent;
    const int S = g.S;
    // Workgroup b runs on XCD b % 8: granules of 16 neighbouring rays stay on one XCD and share its L2
    uint32_t b = blockIdx.x;
    if (b < gridDim.x / 32u * 32u) b = (b & ~31u) + (b & 7u) * 4u + ((b & 31u) >> 3);
    const uint32_t o = b * kRays + wave;  // this wave's ray, as a position of the visiting order
    const bool have = o < N;
    const uint32_t r = have ? lm_ray_order(o, N, row) : 0u;
    const bool cells0 = g.vol && g.vol_dtype == LM_CELLS && g.vol_thre == 0.0f;
    const bool coarse = cells0 && g.vol_coarse;
    auto uniform = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };

    // ---- decisions
    uint32_t n_ray = 0;
    if (have) {
        float ray[6];
        lm_load_ray(rays, r, ray);
        const float rp = lm_ray_param(g, ray);
        if (lane == 0) {
#pragma unroll
            for (int j = 0; j < 6; ++j) s_ray[wave][j] = ray[j];
            s_ray[wave][6] = rp;
        }
        bool visit = false;
        const int w0 = (int)lane * 64;
        if (w0 < S) {
            const int n = min(64, S - w0);
            float lo[3], hi[3];
            int span;
            if (coarse) run_bounds<true>(g, ray, rp, w0, n, lo, hi);
            else run_bounds<false>(g, ray, rp, w0, n, lo, hi);
            visit = !bounds_outside(g, lo, hi) && !(coarse && coarse_empty(g, lo, hi, span));
        }
        uint64_t todo = __ballot(visit), word = 0;  // word: lane i keeps the decisions of samples 64 i .. 64 i + 63
        while (todo) {
            constexpr int kAhead = 4;
            int at[kAhead];
            bool ok[kAhead];
            unsigned live[kAhead];
            uint8_t cell[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                at[u] = -1; ok[u] = false; live[u] = 0u; cell[u] = 0;
                if (todo == 0) continue;
                at[u] = __ffsll((unsigned long long)todo) - 1;
                todo &= todo - 1;
                const int s = at[u] * 64 + (int)lane;
                float pt[3];
                lm_point(ray, lm_sample_z(g, rp, min(s, S - 1)), pt);
                if (cells0) {
                    ok[u] = s < S && lm_inside(g, pt);
                    cell[u] = reinterpret_cast<const uint8_t *>(g.vol)[lm_cells_find(g, pt, live[u])];
                } else {
                    ok[u] = s < S && lm_sample_valid(g, pt);
                    live[u] = cell[u] = 1;
                }
            }
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const uint64_t bits = __ballot(ok[u] && (cell[u] & live[u]) != 0u);
                if ((int)lane == at[u]) word = bits;
                n_ray += (uint32_t)__popcll(bits);
            }
        }
        s_word[wave][lane] = word;
        lm_wave_lds_fence();
    }
    if (lane == 0) { s_n[wave] = n_ray; s_cnt[wave] = 0u; s_done[wave] = 0u; }
    const bool limited = (uint64_t)cap_valid < (uint64_t)N * (uint64_t)S;  // the caller gave less than the worst case
    if (limited) {
        // room is handed out ray by ray; a ray that gets none is rendered as one without valid samples, and counted
        __syncthreads();
        if (threadIdx.x == 0) {
            const uint32_t n_valid = s_n[0] + s_n[1] + s_n[2] + s_n[3];
            uint32_t first = n_valid ? atomicAdd(counters + LM_STAT_N_VALID, n_valid) : 0u, over = 0;
            for (int i = 0; i < kRays; ++i) {
                s_first[i] = first;
                over += s_n[i] != 0u && (uint64_t)first + s_n[i] > (uint64_t)cap_valid;
                first += s_n[i];
            }
            if (over) atomicAdd(counters + LM_STAT_OVERFLOW, over);
        }
        __syncthreads();
        if ((uint64_t)s_first[wave] + n_ray > (uint64_t)cap_valid) n_ray = 0;
    }

    // ---- rounds
    float Tr = 1.0f, sum = 0.0f;                 // transmittance (lane 0); opacity (lane 0) and depth (lane 1)
    uint32_t left = uniform(n_ray), at = 0;      // valid samples still to gather, current word
    uint64_t rest = left ? s_word[wave][0] : 0;  // samples of the current word still to gather
    while (true) {
        const uint32_t want = min(left, (uint32_t)kRound);
        for (uint32_t got = 0; got < want;) {
            if (rest == 0ull) {
                rest = s_word[wave][++at];
                continue;
            }
            const uint32_t rank = got + lm_mbcnt(rest);
            const bool take = ((rest >> lane) & 1ull) && rank < want;
            if (take) s_item[wave][rank] = (uint16_t)(at * 64u + lane);
            const uint64_t taken = __ballot(take);
            rest &= ~taken;
            got += (uint32_t)__popcll(taken);
        }
        left -= want;
        __syncthreads();  // every wave has read s_n
        if (lane == 0) s_n[wave] = want;
        if (!__syncthreads_or(want != 0u)) break;
        // the round's samples, ray after ray, dealt to the waves
        const uint32_t end0 = uniform(s_n[0]), end1 = end0 + uniform(s_n[1]), end2 = end1 + uniform(s_n[2]),
                       total = end2 + uniform(s_n[3]);
        const uint32_t share = (total + kRays - 1) / kRays, f0 = min(uniform(wave) * share, total), f1 = min(f0 + share, total);
        auto batch = [&](auto nsc, auto gc) {
            constexpr int NS = decltype(nsc)::value, G = decltype(gc)::value;
            if (f0 + quad * NS >= f1) return;
            const uint32_t sub = qlane & (unsigned)(NS - 1), f = f0 + quad * NS + sub, fc = min(f, f1 - 1u);
            const int i = (fc >= end0) + (fc >= end1) + (fc >= end2);
            const uint32_t k = fc - (i == 0 ? 0u : i == 1 ? end0 : i == 2 ? end1 : end2);
            float ray[6];
#pragma unroll
            for (int j = 0; j < 6; ++j) ray[j] = s_ray[i][j];
            const float rp = s_ray[i][6];
            const int s_m = (int)s_item[i][k];
            const float z_m = lm_sample_z(g, rp, s_m);
            float q_m[4], d[NS], pt[3];
            lm_point(ray, z_m, pt);
            lm_normalise(g, pt, q_m);
            q_m[3] = __int_as_float(g.div0 > 0 ? lm_block_coords(g, q_m) : 0);
            if constexpr (ROLL) density_sum_lean<T, NS, G>(ps, q_m, qlane, den_w, d);
            else if constexpr (G > 1) density_sum_planes<T, NS, G>(ps, q_m, qlane, den_w, d);
            else density_sum_n<T, NS>(ps, q_m, qlane, den_w, d);
            float d_m = d[0];
#pragma unroll
            for (int n = 1; n < NS; ++n)
                if ((int)sub == n) d_m = d[n];
            const float sig = activate(d_m, act, shift);
            const float dist = (s_m + 1 < S) ? lm_sample_z(g, rp, s_m + 1) - z_m : 0.0f;
            const float d2 = dist * distance_scale;
            const float alpha = 1.0f - expf(-sig * d2);
            if (qlane < (unsigned)NS && f < f1) {
                s_val[i][k] = alpha;
                s_z[i][k] = z_m;
            }
        };
        using std::integral_constant;
        if ((ROLL || narrow) && share <= 16u) batch(integral_constant<int, 1>{}, integral_constant<int, 3>{});
        else if ((ROLL || narrow) && share <= 32u) batch(integral_constant<int, 2>{}, integral_constant<int, 2>{});
        else batch(integral_constant<int, 4>{}, integral_constant<int, 1>{});
        __syncthreads();
        // Transmittance of the wave's own ray.  Only the three running values are a chain: lane 0 multiplies its way
        // through the factors, the weights are formed by all lanes, lane 0 adds up the weights and lane 1 weight x depth.
        // Walked sample by sample on one lane a full round took 5.7 us, this takes under one.
        uint32_t used = want;
        if (want) {
            const bool mine = lane < want;
            const float a_m = mine ? s_val[wave][lane] : 0.0f, z_m = mine ? s_z[wave][lane] : 0.0f;
            s_val[wave][lane] = (1.0f - a_m) + 1e-10f;
            lm_wave_lds_fence();
            if (lane == 0) {
                for (uint32_t t = 0; t < want; t += 4) {  // factors past the round's end are 1
                    const float4 f = *reinterpret_cast<const float4 *>(&s_val[wave][t]);
                    const float4 before = {Tr, Tr * f.x, (Tr * f.x) * f.y, ((Tr * f.x) * f.y) * f.z};
                    Tr = (((Tr * f.x) * f.y) * f.z) * f.w;
                    *reinterpret_cast<float4 *>(&s_val[wave][t]) = before;
                }
                s_val[wave][(want + 3u) & ~3u] = Tr;
                s_done[wave] += want;
            }
            lm_wave_lds_fence();
            float w_m = a_m * s_val[wave][lane];
            const uint64_t over = __ballot(mine && stop > 0.0f && s_val[wave][lane + 1] < stop);
            if (over) used = (uint32_t)__ffsll((unsigned long long)over);
            w_m = lane < used ? w_m : 0.0f;
            s_val[wave][lane] = w_m;
            s_z[wave][lane] = lane < used ? w_m * z_m : 0.0f;
            lm_wave_lds_fence();
            if (lane < 2) {
                const float *src = lane == 0 ? s_val[wave] : s_z[wave];
                for (uint32_t t = 0; t < used; t += 4) {
                    const float4 v = *reinterpret_cast<const float4 *>(&src[t]);
                    sum = (((sum + v.x) + v.y) + v.z) + v.w;
                }
            }
            if (over) left = 0u;
            else if (stop < 0.0f && left) {
                auto of = [](float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); };
                const float z_last = lm_sample_z(g, s_ray[wave][6], S - 1), dist = z_last - of(z_m, 0);
                if (lm_rest_is_lost(of(Tr, 0), of(sum, 0), of(sum, 1), dist / (float)S, z_last, weight_thres)) left = 0u;
            }
            const bool take = w_m > weight_thres && lane < used;
            const uint64_t bits = __ballot(take);
            const uint32_t cnt = s_cnt[wave], slot = cnt + lm_mbcnt(bits);
            if (take && slot < (uint32_t)ent) {
                e_w[slot] = w_m;
                e_s[slot] = s_item[wave][lane];
            }
            if (lane == 0) s_cnt[wave] = cnt + (uint32_t)__popcll(bits);
        }
    }

    // ---- results and appearance entries: a contiguous range of slots per ray, in sample order
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t total = 0, over = 0;
        for (int i = 0; i < kRays; ++i) {
            s_first[i] = total;
            total += s_cnt[i];
        }
        const uint32_t base = total ? atomicAdd(counters + LM_STAT_N_APP, total) : 0u;
        for (int i = 0; i < kRays; ++i) {
            s_first[i] += base;
            // s_n: slots the ray may fill (0: no room, it keeps the background colour and is counted)
            const bool room = s_cnt[i] <= (uint32_t)ent && (uint64_t)s_first[i] + s_cnt[i] <= (uint64_t)cap_app;
            s_n[i] = room ? s_cnt[i] : 0u;
            over += !room;
        }
        if (over) atomicAdd(counters + LM_STAT_OVERFLOW, over);
    }
    __syncthreads();
    if (!have) return;
    const uint32_t first = s_first[wave], n = s_n[wave], cnt = s_cnt[wave], flat0 = r * (uint32_t)S;
    if (lane == 0) { acc_out[r] = sum; app_first[r] = first; app_cnt[r] = n; ray_valid[r] = n_ray; ray_marched[r] = s_done[wave]; }
    if (lane == 1) depth_out[r] = sum;
    for (uint32_t j = lane; j < n; j += LM_WAVE) {
        app_idx[first + j] = flat0 + e_s[j];
        app_w[first + j] = e_w[j];
    }
    // slots below the capacity that a ray without room covers still get a sample index of this chunk and weight zero
    if (n == 0u)
        for (uint32_t j = lane; j < cnt && first + j < cap_app; j += LM_WAVE) { app_idx[first + j] = flat0; app_w[first + j] = 0.0f; }
}

// ---- the march of the kernels per stage with a whole wave per ray ------------------------------------------------
// For chunks with too few rays to fill the GPU with one quad each that k_rays does not take (more than 64 words per ray, or
// more than 1024 samples with a threshold below 1e-3): a launch of k_march lasts as long as the longest
// chain of dependent gathers, four samples per round.  Here a wave owns a ray and takes one 64-sample word of
// its bitmap per round: lane j prepares sample j of the word, quad i gathers samples 4i .. 4i+3 (the same
// density_sum_n, quads without a valid sample sit the round out), so a round's 64 densities come back in one
// memory round trip.  The transmittance then runs through the word's valid samples in order, every lane
// computing the same scalars from values read off the owning lanes: the same operations in the same order as
// the quad march, hence the same bits (weights, sums, counts, the sample at which a ray stops), whichever of
// the two kernels a chunk's size selects.  It does not stop at lost samples.
// Whole calls, quad per ray / wave per ray: 4096 rays of 4726 samples 3570 / 1510 us, 4096 rays of 7088 5000 / 1990,
// 1024 rays of 7088 2430 / 950, 12288 rays of 7088 5700 / 3750, 4096 rays of 3544 at threshold 1e-4 2950 / 1790.
// It lives here and not beside k_march: with it in that file k_march's code, unchanged, lay elsewhere in the code object and
// took a quarter longer on short queues (20000 rays, nine planes: 185 -> 232 us).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_march_wave(lm_geom g, PlaneSet ps, const float *__restrict__ den_w,
                                                       const float *__restrict__ rays, const uint64_t *__restrict__ bitmap,
                                                       const uint32_t *__restrict__ p_first,
                                                       const uint64_t *__restrict__ word_mask,
                                                       const uint32_t *__restrict__ ray_list,
                                                       const uint32_t *__restrict__ bins, uint32_t n_rays, int act,
                                                       float shift, float distance_scale, float weight_thres, float term_eps,
                                                       float *__restrict__ w_valid, float *__restrict__ acc_out,
                                                       float *__restrict__ depth_out, uint32_t *__restrict__ app_cnt,
                                                       uint32_t *__restrict__ p_end_out, uint32_t *__restrict__ n_marched) {
    const unsigned lane = lm_lane(), qlane = lane & 3u;
    const uint32_t end0 = bins[0], end1 = end0 + bins[1], end2 = end1 + bins[2], n_active = end2 + bins[3];
    const uint32_t n_waves = gridDim.x * (kBlock / LM_WAVE);
    const int S = g.S;
    uint32_t marched = 0;
    // everything that steers a wave is the same on all of its lanes: kept in scalar registers
    auto uniform = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };
    auto uniform64 = [&](uint64_t v) { return ((uint64_t)uniform((uint32_t)(v >> 32)) << 32) | uniform((uint32_t)v); };
    for (uint32_t idx = uniform(blockIdx.x * (kBlock / LM_WAVE) + threadIdx.x / LM_WAVE); idx < n_active; idx += n_waves) {
        const uint32_t r = idx < end0   ? ray_list[idx]
                           : idx < end1 ? ray_list[(size_t)n_rays + (idx - end0)]
                           : idx < end2 ? ray_list[2 * (size_t)n_rays + (idx - end1)]
                                        : ray_list[3 * (size_t)n_rays + (idx - end2)];
        float ray[6];
        {
            const float2 *rp2 = reinterpret_cast<const float2 *>(rays + 6 * (size_t)r);
            const float2 a = rp2[0], b = rp2[1], c = rp2[2];
            ray[0] = a.x; ray[1] = a.y; ray[2] = b.x; ray[3] = b.y; ray[4] = c.x; ray[5] = c.y;
        }
        const float rp = lm_ray_param(g, ray);
        const uint64_t flat0 = (uint64_t)r * (uint64_t)S, flat1 = flat0 + (uint64_t)S;
        const uint64_t w0 = flat0 >> 6, w_last = (flat1 - 1) >> 6;
        uint64_t todo = word_mask ? uniform64(word_mask[r]) : ~0ull;  // the ray's non-empty words; all ones: every word
        const bool masked = todo != ~0ull && w_last - w0 < 64;
        uint32_t p = uniform(p_first[r]), cnt = 0;
        float Tr = 1.0f, acc = 0.0f, depth = 0.0f;
        bool finish = false;
        for (uint64_t w = w0; !finish;) {
            if (masked) {
                if (todo == 0) break;
                w = w0 + (uint64_t)(__ffsll((unsigned long long)todo) - 1);
                todo &= todo - 1;
            } else if (w > w_last) {
                break;
            }
            uint64_t bits = uniform64(bitmap[w]);
            if (w == w0 && (flat0 & 63)) bits &= ~((1ull << (flat0 & 63)) - 1ull);  // a neighbouring ray's samples share the word
            if (w == w_last && (flat1 & 63)) bits &= (1ull << (flat1 & 63)) - 1ull;
            if (bits) {
                // lane j prepares sample j of the word; samples that are not valid get the coordinates of the word's
                // first valid one (in range for the tables, results unused)
                const bool mine = (bits >> lane) & 1ull;
                const int j_m = mine ? (int)lane : __ffsll((unsigned long long)bits) - 1;
                const int s_m = (int)(w * 64 + (uint64_t)j_m - flat0);
                const float z_m = lm_sample_z(g, rp, s_m);
                float alpha_m = 0.0f;
                if ((bits >> (lane & ~3u)) & 0xFull) {  // the quad has a valid sample
                    float q_m[4], f[4];
                    {
                        float pt[3];
                        lm_point(ray, z_m, pt);
                        lm_normalise(g, pt, q_m);
                        q_m[3] = __int_as_float(g.div0 > 0 ? lm_block_coords(g, q_m) : 0);
                    }
                    density_sum_n<T, 4>(ps, q_m, qlane, den_w, f);
                    float f_m = f[0];
#pragma unroll
                    for (int n = 1; n < 4; ++n)
                        if ((int)qlane == n) f_m = f[n];
                    const float sig = activate(f_m, act, shift);
                    const float dist = (s_m + 1 < S) ? lm_sample_z(g, rp, s_m + 1) - z_m : 0.0f;
                    const float d2 = dist * distance_scale;
                    alpha_m = 1.0f - expf(-sig * d2);
                }
                marched += (uint32_t)__popcll(bits);
                // the word's valid samples in order; every lane carries the same transmittance and sums
                float w_mine = 0.0f;
                uint32_t done = 0;
                for (uint64_t rem = bits; rem;) {
                    const int j = __ffsll((unsigned long long)rem) - 1;
                    rem &= rem - 1;
                    const float alpha = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(alpha_m), j));
                    const float z = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(z_m), j));
                    const float wgt = alpha * Tr;
                    Tr = Tr * ((1.0f - alpha) + 1e-10f);
                    if ((int)lane == j) w_mine = wgt;
                    acc += wgt;
                    depth += wgt * z;
                    cnt += wgt > weight_thres;
                    ++done;
                    if (term_eps > 0.0f && Tr < term_eps) { finish = true; break; }
                }
                const uint32_t rank = lm_mbcnt(bits);
                if (mine && rank < done) w_valid[p + rank] = w_mine;
                p += done;
            }
            ++w;
        }
        if (lane == 0) {
            acc_out[r] = acc; depth_out[r] = depth; app_cnt[r] = cnt; p_end_out[r] = p;
        }
    }
    if (lane == 0 && marched) atomicAdd(n_marched, marched);
}

}  // namespace

int lm_check_planes(const lm_plane *planes, int32_t n, int *dtype_out, int *K_out);

// Chunks of up to LM_RAYS_LIMIT rays whose decisions fit 64 words per ray and whose appearance entries fit LDS: one per
// sample, or as many as weights above the threshold can be (they sum to at most 1).
bool lm_rays_kernel_takes(const lm_model *m, int64_t N) {
    const bool entries_fit = m->geom.S <= kEntriesMax || m->weight_thres * (float)(kEntriesMax - 2) >= 1.001f;
    return N <= LM_RAYS_LIMIT && m->geom.S <= 64 * kWordsMax && entries_fit;
}

// Everything up to the appearance list for a small chunk; leaves acc, depth, the list and its counter behind like
// lm_launch_cull_setup + lm_launch_march + lm_launch_app_slots, and per ray how many samples were valid and gathered, for
// lm_launch_composite to sum.
int lm_launch_rays(const lm_model *m, const float *rays, uint32_t N, uint32_t row, uint32_t cap_valid, uint32_t *app_first,
                   uint32_t *app_cnt, uint32_t *app_idx, float *app_w, uint32_t cap_app, float *acc, float *depth,
                   uint32_t *ray_valid, uint32_t *ray_marched, uint32_t *counters, hipStream_t st) {
    int dtype;
    if (int rc = lm_check_planes(m->density, m->n_planes, &dtype, nullptr)) return rc;
    LM_REQUIRE(m->act == LM_ACT_SOFTPLUS || m->act == LM_ACT_RELU, "unknown activation %d", m->act);
    LM_REQUIRE((reinterpret_cast<uintptr_t>(rays) & 7u) == 0, "rays must be 8-byte aligned");
    const PlaneSet ps = make_set(m->density, m->n_planes, &m->geom);
    int c_max = 0;
    for (int k = 0; k < m->n_planes; ++k) c_max = std::max(c_max, (int)m->density[k].C);
    const int ent = std::min(m->geom.S, kEntriesMax);
    const size_t lds = (size_t)kRays * ent * (sizeof(float) + sizeof(uint16_t));
#define LM_RAYS_ONE(T_, ROLL_)                                                                                                \
    hipLaunchKernelGGL((k_rays<T_, ROLL_>), dim3((N + kRays - 1) / kRays), dim3(kBlock), lds, st, m->geom, ps, c_max <= Vec<T_>::V * kQuad ? 1 : 0, \
                       m->density_basis, rays, N, row, ent, m->act, m->density_shift, m->distance_scale, m->weight_thres,    \
                       lm_stop_value(*m), cap_valid, app_first, app_cnt, app_idx, app_w, cap_app, acc, depth, ray_valid,       \
                       ray_marched, counters)
#define LM_RAYS(T_)                                                                  \
    if (density_rolls<T_>(m->density, m->n_planes, ps.nblk)) LM_RAYS_ONE(T_, true);  \
    else LM_RAYS_ONE(T_, false)
    if (dtype == LM_F32) {
        LM_RAYS(float);
    } else if (c_max <= 16) {
        LM_RAYS(Half4);
    } else {
        LM_RAYS(__half);
    }
#undef LM_RAYS
#undef LM_RAYS_ONE
    LM_CHECK_LAUNCH("k_rays");
    return LM_OK;
}

// The march over the rays in ray_list (those with valid samples) for few rays; the caller has checked the arguments.
int lm_launch_march_wave(const lm_model *m, const float *rays, const uint64_t *bitmap, const uint32_t *p_first, const uint64_t *word_mask,
                         const uint32_t *ray_list, const uint32_t *bins, uint32_t n_rays, float *w_valid, float *acc, float *depth,
                         uint32_t *app_cnt, uint32_t *p_end, uint32_t *n_marched, hipStream_t st) {
    int dtype;
    if (int rc = lm_check_planes(m->density, m->n_planes, &dtype, nullptr)) return rc;
    const PlaneSet ps = make_set(m->density, m->n_planes, &m->geom);
    int c_max = 0;
    for (int k = 0; k < m->n_planes; ++k) c_max = std::max(c_max, (int)m->density[k].C);
    const unsigned grid = std::min<unsigned>((n_rays + kBlock / LM_WAVE - 1) / (kBlock / LM_WAVE), (unsigned)lm_persistent_blocks(8));
#define LM_MARCH_WAVE(T_)                                                                                                    \
    hipLaunchKernelGGL((k_march_wave<T_>), dim3(grid), dim3(kBlock), 0, st, m->geom, ps, m->density_basis, rays, bitmap, p_first, \
                       word_mask, ray_list, bins, n_rays, m->act, m->density_shift, m->distance_scale, m->weight_thres,       \
                       m->term_eps, w_valid, acc, depth, app_cnt, p_end, n_marched)
    if (dtype == LM_F32) LM_MARCH_WAVE(float);
    else if (c_max <= 16) LM_MARCH_WAVE(Half4);
    else LM_MARCH_WAVE(__half);
#undef LM_MARCH_WAVE
    LM_CHECK_LAUNCH("k_march_wave");
    return LM_OK;
}
