// Part 4: volume compositing as a per-ray segmented scan over the valid samples only.
//
// k_weights: one lane per ray.  The ray's valid samples are the set bits of its slice of
// the sample bitmap; their densities sit contiguously in the compacted sigma array.  The
// lane walks those bits in sample order and carries the transmittance along, which is
// exactly the sequential product torch.cumprod forms; culled samples have sigma = 0 in the
// reference, i.e. alpha = 0 and a factor (1 - 0 + 1e-10) that rounds to 1.0f, so skipping
// them changes nothing.  Two passes: the first stores the weights of the valid samples and
// counts those above the threshold, a wave-wide prefix sum plus one atomic per wave reserves
// a contiguous slot range per ray in the appearance list, the second pass fills the slots.
// A ray's slots are therefore contiguous and in sample order.
// k_composite: a quad per ray sums weight * rgb over its slots, adds the white
// background and clamps.
// In the whole-chunk render the weights come from the marching kernel (density gather fused with
// the transmittance walk); k_app_slots then builds the appearance list from the stored weights the
// way k_weights' second pass does.  k_weights remains the stage-level form.
//
// Reference: raw2alpha (app/tools/utils.py:51-64), dists with a zero last interval
// (app/models/gridnerf_sequential.py:457, 531-534), weight threshold (:479, :553) and the
// sums / white background / clamp / depth of :493-504 and :565-576.
#include "lm_common.h"

namespace {

constexpr int kBlock = 256;
#ifndef LM_SLOTS_STAGE
#define LM_SLOTS_STAGE 4096
#endif
// list entries a wave of k_app_slots moves through LDS at once
constexpr int kSlotsStage = LM_SLOTS_STAGE;

__global__ __launch_bounds__(kBlock) void k_weights(lm_geom g, const float *__restrict__ rays, uint64_t N,
                                                    const uint64_t *__restrict__ bitmap,
                                                    const uint32_t *__restrict__ word_prefix,
                                                    const float *__restrict__ sigma, float distance_scale,
                                                    float weight_thres, float term_eps, float *__restrict__ w_valid,
                                                    float *__restrict__ weight_out, uint32_t *__restrict__ app_first,
                                                    uint32_t *__restrict__ app_cnt, uint32_t *__restrict__ app_idx,
                                                    float *__restrict__ app_w, float *__restrict__ acc_out,
                                                    float *__restrict__ depth_out, uint32_t *__restrict__ app_count) {
    const unsigned lane = lm_lane();
    const uint64_t r = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    const bool active = r < N;
    const int S = g.S;
    float acc = 0.0f, depth = 0.0f;
    uint32_t cnt = 0, p_first = 0, p_end = 0;
    float rp = 0.0f;
    const uint64_t flat0 = r * (uint64_t)S;
    if (active) {
        float ray[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) ray[k] = rays[6 * r + k];
        rp = lm_ray_param(g, ray);
        BitWalk it;
        it.start(bitmap, word_prefix, flat0, flat0 + S);
        p_first = it.pos;
        uint32_t p = p_first;
        float T = 1.0f;
        uint64_t flat;
        while (it.next(flat)) {
            const int s = (int)(flat - flat0);
            const float z = lm_sample_z(g, rp, s);
            const float dist = (s + 1 < S) ? lm_sample_z(g, rp, s + 1) - z : 0.0f;
            const float d2 = dist * distance_scale;
            const float alpha = 1.0f - expf(-sigma[p] * d2);
            const float wgt = alpha * T;
            T = T * ((1.0f - alpha) + 1e-10f);
            w_valid[p] = wgt;
            if (weight_out) weight_out[flat] = wgt;
            acc += wgt;
            depth += wgt * z;
            cnt += wgt > weight_thres;
            ++p;
            if (term_eps > 0.0f && T < term_eps) break;
        }
        p_end = p;
    }
    // slot range per ray: exclusive prefix over the wave + one atomic
    uint32_t incl = cnt;
#pragma unroll
    for (int d = 1; d < LM_WAVE; d <<= 1) {
        const uint32_t y = __shfl_up(incl, d);
        if (lane >= (unsigned)d) incl += y;
    }
    const uint32_t total = __shfl(incl, LM_WAVE - 1);
    uint32_t base = 0;
    if (total) {
        if (lane == 0) base = atomicAdd(app_count, total);
        base = __shfl(base, 0);
    }
    if (!active) return;
    uint32_t slot = base + incl - cnt;
    app_first[r] = slot;
    app_cnt[r] = cnt;
    acc_out[r] = acc;
    depth_out[r] = depth;
    if (cnt) {
        BitWalk it;
        it.start(bitmap, word_prefix, flat0, flat0 + S);
        uint64_t flat;
        for (uint32_t p = p_first; p < p_end; ++p) {
            it.next(flat);
            const float wgt = w_valid[p];
            if (wgt > weight_thres) {
                app_idx[slot] = (uint32_t)flat;
                app_w[slot] = wgt;
                ++slot;
            }
        }
    }
}

// Samples per ray (any order) and where their sums go; count_valid: whether the valid ones are not counted there already
struct RayStats {
    const uint32_t *valid, *marched;
    uint32_t *counters;
    int count_valid;
};

// A quad per ray, a lane per colour channel: a quad's loads fall into one run of the list whatever the order the rays'
// ranges lie in, sixteen entries in flight.  A lane per ray, with the wave's range of the list staged through LDS in
// windows, waits for each window and does badly where neighbouring rays' ranges lie apart (k_rays reserves four rays at a
// time): 8192 rays of 30 entries 13 - 75 -> 5.8 us, 4096 rays of 5 entries 13 -> 5 us, 518400 rays of 57 entries 390 -> 223 us,
// a million rays of 11 entries 74 us either way.  Eight entries in flight: 7.1, 5.1, 279, 81 us.
// STATS: the idle lane of every quad also takes its ray's sample counts, which k_rays leaves per ray, and the workgroup
// adds the sums to the counter block.
template <bool STATS>
__global__ __launch_bounds__(kBlock) void k_composite(uint64_t o0, uint64_t N, const uint32_t *__restrict__ app_first,
                                                           const uint32_t *__restrict__ app_cnt, const float *__restrict__ app_w,
                                                           const float *__restrict__ rgb, const float *__restrict__ acc, int white_bg,
                                                           uint32_t row, float *__restrict__ rgb_map, RayStats stats) {
    const uint64_t o = o0 + (uint64_t)blockIdx.x * (kBlock / 4) + threadIdx.x / 4;
    const unsigned ch = threadIdx.x & 3u;
    __shared__ uint32_t s_sum[2 + LM_RAY_BINS];  // samples valid and gathered, rays by their number of valid samples
    uint32_t n_valid = 0, n_marched = 0;
    if constexpr (STATS) {
        if (threadIdx.x < 2 + LM_RAY_BINS) s_sum[threadIdx.x] = 0;
        if (o < N && ch == 3u) { n_valid = stats.valid[o]; n_marched = stats.marched[o]; }
    }
    if (o < N && ch != 3u) {
        const uint64_t r = lm_ray_order((uint32_t)o, (uint32_t)N, row);
        constexpr uint32_t kAhead = 16;
        const uint32_t n = app_cnt[r];
        const size_t first = app_first[r];
        const float a = white_bg ? acc[r] : 0.0f;
        const float *w = app_w + first, *c = rgb + 3 * first + ch;
        float sum = 0.0f;
        for (uint32_t i = 0; i < n; i += kAhead) {
            float wv[kAhead], cv[kAhead];
#pragma unroll
            for (uint32_t u = 0; u < kAhead; ++u) {
                const uint32_t at = min(i + u, n - 1u);
                wv[u] = w[at];
                cv[u] = c[3 * (size_t)at];
            }
#pragma unroll
            for (uint32_t u = 0; u < kAhead; ++u)
                if (i + u < n) sum = fmaf(wv[u], cv[u], sum);
        }
        if (white_bg) sum += 1.0f - a;
        rgb_map[3 * r + ch] = fminf(fmaxf(sum, 0.0f), 1.0f);
    }
    if constexpr (STATS) {
        __syncthreads();
        if (n_valid) {
            atomicAdd(&s_sum[0], n_valid);
            atomicAdd(&s_sum[2 + lm_ray_bin(n_valid)], 1u);
        }
        if (n_marched) atomicAdd(&s_sum[1], n_marched);
        __syncthreads();
        const unsigned t = threadIdx.x;
        if (t < 2 + LM_RAY_BINS && s_sum[t] && (t != 0u || stats.count_valid))
            atomicAdd(stats.counters + (t == 0u ? LM_STAT_N_VALID : t == 1u ? LM_STAT_N_MARCHED : LM_STAT_BINS + t - 2u), s_sum[t]);
    }
}

// Appearance list from stored weights: a contiguous slot range per ray (wave prefix + one
// atomic), filled in sample order from the weights of the ray's samples [first, p_end).
// The 64 rays a wave handles own one contiguous range of slots, a lane's slots are a short run somewhere in it: written
// directly, every access of the wave touches 64 different cache lines, each visited again a few entries later
// (partial-line writes reach the memory several times over).  A range of at most STAGE entries is therefore put together
// in LDS and written in whole lines.  A workgroup is one wave.
template <int STAGE>
__global__ __launch_bounds__(LM_WAVE) void k_app_slots(int S, uint64_t N, const uint64_t *__restrict__ bitmap,
                                                       const uint32_t *__restrict__ p_first,
                                                       const uint64_t *__restrict__ word_mask,
                                                       const float *__restrict__ w_valid, float weight_thres,
                                                       uint32_t *__restrict__ app_cnt,
                                                       const uint32_t *__restrict__ p_end,
                                                       uint32_t *__restrict__ app_first, uint32_t *__restrict__ app_idx,
                                                       float *__restrict__ app_w, uint32_t *__restrict__ app_count,
                                                       uint32_t row, uint32_t cap_app, uint32_t *__restrict__ overflow) {
    __shared__ uint32_t s_idx[STAGE];
    __shared__ float s_w[STAGE];
    const unsigned lane = lm_lane();
    const uint64_t o = (uint64_t)blockIdx.x * LM_WAVE + lane;
    const bool live = o < N;
    const uint64_t r = live ? lm_ray_order((uint32_t)o, (uint32_t)N, row) : o;
    const uint32_t cnt = live ? app_cnt[r] : 0;
    uint32_t incl = cnt;
#pragma unroll
    for (int d = 1; d < LM_WAVE; d <<= 1) {
        const uint32_t y = __shfl_up(incl, d);
        if (lane >= (unsigned)d) incl += y;
    }
    const uint32_t total = __shfl(incl, LM_WAVE - 1);
    uint32_t base = 0;
    if (total) {
        if (lane == 0) base = atomicAdd(app_count, total);
        base = __shfl(base, 0);
    }
    uint32_t slot = base + incl - cnt;
    const bool fits = lm_ray_fits(cnt, slot, cap_app, overflow);
    // through LDS when the wave's range is short enough and lies below the capacity as a whole
    const bool staged = total != 0u && total <= (uint32_t)STAGE && (uint64_t)base + total <= (uint64_t)cap_app;
    if (live) {
        app_first[r] = slot;
        if (cnt && !fits) {
            // no room for this ray's samples: it keeps the background colour (and is counted); the slots below the
            // capacity that its range covers still get a sample index of this chunk and weight zero
            app_cnt[r] = 0;
            for (uint32_t i = slot; i < cap_app && i < slot + cnt; ++i) { app_idx[i] = (uint32_t)(r * (uint64_t)S); app_w[i] = 0.0f; }
        } else if (cnt) {
            BitWalk it;
            it.start_at(bitmap, r * (uint64_t)S, (r + 1) * (uint64_t)S, p_first[r], word_mask ? word_mask[r] : ~0ull);
            const uint32_t end = p_end[r], last = slot + cnt;
            uint64_t flat;
            // eight weights per trip so that their loads overlap; the walk over the bitmap stays in order and ends
            // with the ray's last entry
            constexpr int kBatch = 8;
            for (uint32_t p = it.pos; p < end && slot < last; p += kBatch) {
                float wgt[kBatch];
#pragma unroll
                for (int u = 0; u < kBatch; ++u) wgt[u] = w_valid[p + u < end ? p + u : end - 1];
#pragma unroll
                for (int u = 0; u < kBatch; ++u) {
                    if (p + u >= end) break;
                    it.next(flat);
                    if (wgt[u] > weight_thres && slot < last) {
                        if (staged) {
                            s_idx[slot - base] = (uint32_t)flat;
                            s_w[slot - base] = wgt[u];
                        } else {
                            app_idx[slot] = (uint32_t)flat;
                            app_w[slot] = wgt[u];
                        }
                        ++slot;
                    }
                }
            }
        }
    }
    if (staged) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        for (uint32_t i = lane; i < total; i += LM_WAVE) {
            app_idx[base + i] = s_idx[i];
            app_w[base + i] = s_w[i];
        }
    }
}

__global__ void k_zero_counters(uint32_t *c) {
    if (threadIdx.x < LM_STAT_WORDS) c[threadIdx.x] = 0;
}

}  // namespace

int lm_check_geom(const lm_geom *g);

extern "C" int lm_weights(const lm_geom *geom, const float *rays, int64_t N, const uint64_t *bitmap,
                          const uint32_t *word_prefix, const float *sigma, float distance_scale, float weight_thres,
                          float term_eps, float *w_valid, float *weight_out, uint32_t *app_first, uint32_t *app_cnt,
                          uint32_t *app_idx, float *app_w, float *acc, float *depth, uint32_t *counters, void *stream) {
    if (int rc = lm_check_geom(geom)) return rc;
    LM_REQUIRE(N >= 0, "negative ray count");
    LM_REQUIRE(counters != nullptr, "counters is null");
    if (N == 0) return LM_OK;
    LM_REQUIRE(rays && bitmap && word_prefix && sigma && w_valid && app_first && app_cnt && app_idx && app_w && acc && depth,
               "null buffer");
    const unsigned grid = (unsigned)(((uint64_t)N + kBlock - 1) / kBlock);
    hipLaunchKernelGGL(k_weights, dim3(grid), dim3(kBlock), 0, (hipStream_t)stream, *geom, rays, (uint64_t)N, bitmap,
                       word_prefix, sigma, distance_scale, weight_thres, term_eps, w_valid, weight_out, app_first, app_cnt,
                       app_idx, app_w, acc, depth, counters + LM_STAT_N_APP);
    LM_CHECK_LAUNCH("k_weights");
    return LM_OK;
}

int lm_launch_composite(int64_t N, const uint32_t *app_first, const uint32_t *app_cnt, const float *app_w,
                        const float *rgb, const float *acc, int white_bg, uint32_t row, float *rgb_map,
                        const uint32_t *ray_valid, const uint32_t *ray_marched, int count_valid, uint32_t *counters,
                        hipStream_t stream) {
    if (N == 0) return LM_OK;
    const RayStats stats = {ray_valid, ray_marched, counters, count_valid};
    // four threads per ray, and fewer than 2^32 threads per launch
    constexpr uint64_t kSlice = 1ull << 29;
    for (uint64_t o0 = 0; o0 < (uint64_t)N; o0 += kSlice) {
        const dim3 grid((unsigned)((std::min((uint64_t)N - o0, kSlice) + kBlock / 4 - 1) / (kBlock / 4)));
        if (ray_valid)
            hipLaunchKernelGGL(k_composite<true>, grid, dim3(kBlock), 0, stream, o0, (uint64_t)N, app_first, app_cnt, app_w, rgb, acc,
                               white_bg, row, rgb_map, stats);
        else
            hipLaunchKernelGGL(k_composite<false>, grid, dim3(kBlock), 0, stream, o0, (uint64_t)N, app_first, app_cnt, app_w, rgb, acc,
                               white_bg, row, rgb_map, stats);
    }
    LM_CHECK_LAUNCH("k_composite");
    return LM_OK;
}

extern "C" int lm_composite_rgb(int64_t N, const uint32_t *app_first, const uint32_t *app_cnt, const float *app_w,
                                const float *rgb, const float *acc, int32_t white_bg, float *rgb_map, void *stream) {
    LM_REQUIRE(N >= 0, "negative ray count");
    if (N == 0) return LM_OK;
    LM_REQUIRE((uint64_t)N < (1ull << 32), "ray count does not fit 32 bits");
    LM_REQUIRE(app_first && app_cnt && app_w && rgb && acc && rgb_map, "null buffer");
    return lm_launch_composite(N, app_first, app_cnt, app_w, rgb, acc, white_bg, 0u, rgb_map, nullptr, nullptr, 0, nullptr,
                               (hipStream_t)stream);
}

int lm_launch_zero_counters(uint32_t *counters, hipStream_t stream) {
    hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, stream, counters);
    LM_CHECK_LAUNCH("k_zero_counters");
    return LM_OK;
}

int lm_launch_app_slots(int S, int64_t N, const uint64_t *bitmap, const uint32_t *p_first, const uint64_t *word_mask,
                        const float *w_valid,
                        float weight_thres, uint32_t *app_cnt, const uint32_t *p_end, uint32_t *app_first,
                        uint32_t *app_idx, float *app_w, uint32_t *app_count, uint32_t row, uint32_t cap_app,
                        uint32_t *overflow, hipStream_t stream) {
    const unsigned grid = (unsigned)(((uint64_t)N + LM_WAVE - 1) / LM_WAVE);
    hipLaunchKernelGGL(k_app_slots<kSlotsStage>, dim3(grid), dim3(LM_WAVE), 0, stream, S, (uint64_t)N, bitmap, p_first, word_mask,
                       w_valid, weight_thres, app_cnt, p_end, app_first, app_idx, app_w, app_count, row, cap_app, overflow);
    LM_CHECK_LAUNCH("k_app_slots");
    return LM_OK;
}
