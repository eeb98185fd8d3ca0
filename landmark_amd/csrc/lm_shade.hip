// The back half of a small chunk in one kernel: appearance gather, basis_mat, encoding and colour network, a workgroup
// of four waves for 32 appearance samples.
//
// The kernels of large chunks (k_app_feat, k_mlp) give a wave 32 samples and walk the planes and the layers' row blocks
// one after the other, with basis_mat and the layers' weights copied to LDS by every workgroup first.  A chunk of a few
// thousand rays has a few hundred such tiles: most waves idle and the launch lasts as long as one wave's chain.  Here
// four waves share a tile:
//   1. wave w gathers sample half w % 2 on planes w / 2, w / 2 + 2, ... (a plane's loads in flight while the one before
//      is used); the products meet in LDS;
//   2. one wave multiplies them by basis_mat in plane order (the accumulation order of the other kernels);
//   3. every wave encodes the 32 inputs and takes one of the four row blocks of layers 1 and 2; activations go through
//      LDS once per layer.  Each wave needs a weight fragment once per tile, so fragments come straight from the L2 into
//      registers, requested a phase ahead; nothing is copied to LDS up front;
//   4. one wave takes the last layer; in fp32 every wave its row block's share on the vector unit, and one adds them up.
// Same operations and accumulation order per sample as k_app_feat + k_mlp, hence the same bits.
// What bounds it: with nine planes the texels (20 653 entries, 0.11 GB past the L2: 22 us at the 5.2 TB/s of a large copy, 41 us
// taken, a third of the wave time waiting), with three small planes the chain list -> ray -> texels -> layers of one tile
// (0.4 TB/s, addressers 15 % busy).  The split mode on 48-channel fp16 tables spills 17 registers (72 bytes per lane).
// k_app_feat + k_mlp against this kernel:
// 12 000 entries on three 256^2 planes, fp32 network 69 -> 25 us (22 with the last layer's three rows on the vector unit);
// 20 000 entries on nine planes, split network 74 -> 41 us; 18 000 entries on three planes, a whole call 104 -> 64 us (split)
// and 99 -> 56 us (fp16).
#include <algorithm>

#include "lm_colour.h"
#include "lm_common.h"
#include "lm_gather.h"

namespace {

constexpr int kTileRays = 32;                  // samples per workgroup and trip
constexpr int kWaves = kBlock / LM_WAVE;       // one per row block of the hidden layers
constexpr int kLead = 3;                       // the wave of basis_mat and the last layer (it gathers fewest planes)
static_assert(kWaves * 32 == kHidden, "a wave per row block");

// Layer inputs travel through LDS in units of 16 bytes per lane and part: a step of the 16-bit matrix instructions, four
// steps of the fp32 one.
template <int PREC> struct Unit {
    using M = Mma<PREC>;
    static constexpr int S = M::G == 1 ? 4 : 1;            // steps
    static constexpr int U1 = kSlots1 / M::G / S;          // units of layer 1's inputs
    static constexpr int U2 = 64 / M::G / S;               // of layers 2 and 3
    static constexpr size_t kBytes = (size_t)LM_WAVE * 16 * M::NP;
    __device__ static __forceinline__ void read(const char *src, unsigned lane, typename M::frag (*x)[M::NP]) {
        if constexpr (M::G == 1) {
            const float4 v = *reinterpret_cast<const float4 *>(src + lane * 16);
            x[0][0] = v.x; x[1][0] = v.y; x[2][0] = v.z; x[3][0] = v.w;
        } else {
#pragma unroll
            for (int pt = 0; pt < M::NP; ++pt) x[0][pt] = *reinterpret_cast<const typename M::frag *>(src + (pt * LM_WAVE + lane) * 16);
        }
    }
    // four consecutive slots of a lane, the first a multiple of four
    __device__ static __forceinline__ void store4(char *base, int slot, unsigned lane, const uint32_t (*d)[4], int at) {
#pragma unroll
        for (int pt = 0; pt < M::NP; ++pt)
            *reinterpret_cast<uint2 *>(base + (size_t)(slot / 8) * kBytes + (pt * LM_WAVE + lane) * 16 + (slot / 4 % 2) * 8) =
                make_uint2(d[pt][at], d[pt][at + 1]);
    }
    __device__ static __forceinline__ void write4(char *base, int slot, unsigned lane, const float *v) {
        if constexpr (M::G == 1) {
            *reinterpret_cast<float4 *>(base + (size_t)(slot / 4) * kBytes + lane * 16) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
            uint32_t d[M::NP][4], pair[M::NP];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                M::pack_pair(v[2 * i], v[2 * i + 1], pair);
#pragma unroll
                for (int pt = 0; pt < M::NP; ++pt) d[pt][i] = pair[pt];
            }
            store4(base, slot, lane, d, 0);
        }
    }
    // the relu of accumulator registers 4 q .. 4 q + 3, in the other kernels' order of rounding and clamping
    __device__ static __forceinline__ void write4_relu(char *base, int slot, unsigned lane, const floatx16 &acc, int q) {
        if constexpr (M::G == 1) {
            *reinterpret_cast<float4 *>(base + (size_t)(slot / 4) * kBytes + lane * 16) =
                make_float4(relu_f32(acc[4 * q]), relu_f32(acc[4 * q + 1]), relu_f32(acc[4 * q + 2]), relu_f32(acc[4 * q + 3]));
        } else {
            uint32_t d[M::NP][4];
            relu_pair<PREC>(acc, 2 * q, d);
            relu_pair<PREC>(acc, 2 * q + 1, d);
            store4(base, slot, lane, d, 2 * q % 4);
        }
    }
};

// LDS: [products, then the encoded inputs, then the activations of layer 2 | features, then the activations of layer 1]
template <int PREC> struct ShadeLds {
    using N = Unit<PREC>;
    static constexpr size_t kIn1 = N::U1 * N::kBytes, kIn2 = N::U2 * N::kBytes, kRaw = (size_t)16 * LM_WAVE * sizeof(float);
    static_assert(kRaw <= kIn2 && kIn2 <= kIn1, "areas that are used again");
    __host__ __device__ static size_t first(int K) {
        const size_t p = (size_t)kTileRays * (K + 4) * sizeof(float);
        return p > kIn1 ? p : kIn1;
    }
    __host__ __device__ static size_t total(int K) { return first(K) + kIn2; }
};

// FEAT: the first half only, points to features: `rays` = xyz[M_host][3], `rgb` = feat[M_host][27]
template <int PREC, typename T, int NU, bool FEAT>  // NU = groups of 16 channels per plane
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2))) void k_shade(
    lm_geom g, PlaneSet ps, int K, const char *__restrict__ packed, PackLayout L, const float *__restrict__ rays,
    uint32_t M_host, const uint32_t *__restrict__ list, const uint32_t *__restrict__ count, uint32_t cap, float *__restrict__ rgb) {
    using Mm = Mma<PREC>;
    using frag = typename Mm::frag;
    using P = ShadeLds<PREC>;
    constexpr int V = Vec<T>::V, C = 16 * NU;
    constexpr int NG = (C + V * kQuad - 1) / (V * kQuad);
    constexpr int G = Mm::G, CW = Mm::CW, NP = Mm::NP;
    using N = Unit<PREC>;
    constexpr int T1 = kSlots1 / G, T2 = 64 / G;               // steps of layer 1, of layers 2 and 3
    constexpr int TP = C / (2 * G);                            // steps of a plane
    extern __shared__ __align__(16) char lds[];
    const int ROW = K + 4;
    float *prod = reinterpret_cast<float *>(lds);
    char *in1 = lds, *in2 = lds + P::first(K), *in3 = lds;
    float *raw_s = reinterpret_cast<float *>(in2);
    const unsigned lane = lm_lane(), j = lane & 31u, h = lane >> 5, qlane = lane & 3u, gs = lane >> 2;
    const unsigned wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / LM_WAVE));
    // fragment i of a weight matrix: uniform base, 32-bit lane offset
    auto weight = [&](size_t matrix, size_t i, uint32_t at) {
        return *reinterpret_cast<const frag *>(packed + matrix + i * (LM_WAVE * sizeof(frag)) + at);
    };
    const size_t w1 = L.w1 + (size_t)wave * T1 * NP * LM_WAVE * sizeof(frag), w2 = L.w2 + (size_t)wave * T2 * NP * LM_WAVE * sizeof(frag);
    auto bias_of = [&](size_t at, uint32_t half) { return load_bias(reinterpret_cast<const float *>(packed + at + half), 0); };
    const uint32_t M = FEAT ? M_host : min(*count, cap);  // the counter keeps counting past the list's capacity
    const uint32_t n_tiles = (uint32_t)(((uint64_t)M + kTileRays - 1) / kTileRays);
    // Workgroup b runs on XCD b % 8: granules of four neighbouring tiles stay on one XCD and share its L2
    uint32_t b = blockIdx.x;
    if (b < gridDim.x / 32u * 32u) b = (b & ~31u) + (b & 7u) * 4u + ((b & 31u) >> 3);
    // one step of a layer: the weight's parts times the input's parts, in the order of the other kernels
    auto step = [](const frag *a, const frag *x, floatx16 acc) {
        acc = Mm::mma(a[0], x[0], acc);
        if constexpr (NP == 2) {
            acc = Mm::mma(a[1], x[0], acc);
            acc = Mm::mma(a[0], x[1], acc);
        }
        return acc;
    };
    if (b >= n_tiles) return;
    auto entry = [&](uint32_t tile, uint32_t i) {
        const uint32_t at = (uint32_t)min((uint64_t)tile * kTileRays + i, (uint64_t)M - 1u);
        return FEAT ? at : list[at];
    };
    float q[4], vnext[3];  // coordinates of the lane's sample and its column's view direction
    auto position = [&](uint32_t gather, uint32_t column) {
        if constexpr (FEAT) {
#pragma unroll
            for (int i = 0; i < 3; ++i) q[i] = rays[3 * (size_t)gather + i];
            q[3] = 0.0f;
            return;
        }
        list_coords(g, rays, gather, q);
        const float *d = rays + 6 * (size_t)(column / (uint32_t)g.S) + 3;
#pragma unroll
        for (int i = 0; i < 3; ++i) vnext[i] = d[i];
    };
    position(entry(b, (wave & 1u) * 16u + gs), entry(b, j));
    for (uint32_t tile = b; tile < n_tiles; tile += gridDim.x) {
        // Weight addresses do not depend on the tile, and the compiler would load all of them ahead of the loop and spill
        // them: an offset it cannot see through keeps the loads where they are written.
        uint32_t here = lane * (uint32_t)sizeof(frag), bias = h * 64u;
        asm volatile("" : "+v"(here), "+v"(bias));
        // ---- products of the wave's 16 samples on its planes
        float vdir[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) vdir[i] = vnext[i];
        const uint32_t tn = tile + gridDim.x;
        const uint32_t gn = entry(tn, (wave & 1u) * 16u + gs), vn = entry(tn, j);  // the next tile's entries travel meanwhile
        {
            struct Loads {
                Taps2 t2;
                Taps1 t1;
                Footprint<T> f[NG];
            };
            auto load = [&](int k, Loads &x) {
                const lm_plane &pl = ps.p[k];
                x.t2 = plane_taps(pl, pick(q, pl.ax0), pick(q, pl.ax1));
                x.t1 = line_taps(pl, pick(q, pl.axl));
                block_taps(pl, ps.nblk, q, x.t2, x.t1);
#pragma unroll
                for (int gi = 0; gi < NG; ++gi) {
                    const int c = V * (int)qlane + gi * V * kQuad;
                    if (c < C) footprint_load<T>(pl, x.t2, x.t1, c, x.f[gi]);
                }
            };
            auto emit = [&](int k, const Loads &x) {
                float *row = prod + ((wave & 1u) * 16u + gs) * ROW + k * C;
#pragma unroll
                for (int gi = 0; gi < NG; ++gi) {
                    const int c = V * (int)qlane + gi * V * kQuad;
                    if (c >= C) continue;
                    float pr[V];
                    footprint_products<T>(x.f[gi], x.t2, x.t1, pr);
#pragma unroll
                    for (int i = 0; i < V; i += 2) *reinterpret_cast<float2 *>(row + c + i) = make_float2(pr[i], pr[i + 1]);
                }
            };
            for (int k = (int)(wave >> 1); k < ps.n; k += 2) {
                Loads x;
                load(k, x);
                __builtin_amdgcn_sched_barrier(0);
                emit(k, x);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // the wave's weights of layer 1 travel while basis_mat is applied
        frag wa[T1][NP];
        constexpr int kFirst = FEAT ? 0 : G == 1 || NP == 2 ? T1 / 2 : T1;  // the rest once basis_mat's fragments have left the registers
#pragma unroll
        for (int t = 0; t < kFirst; ++t)
#pragma unroll
            for (int pt = 0; pt < NP; ++pt) wa[t][pt] = weight(w1, t * NP + pt, here);
        floatx16 acc;
        __syncthreads();
        if (wave == kLead) {
            // ---- 27 features = basis_mat x products, planes in order; a plane's fragments are requested a plane ahead
            frag a0[TP][NP], a1[TP][NP];
            auto request = [&](int k, frag (*a)[NP]) {
#pragma unroll
                for (int t = 0; t < TP; ++t)
#pragma unroll
                    for (int pt = 0; pt < NP; ++pt) a[t][pt] = weight(L.basis, (size_t)((k * TP + t) * NP + pt), here);
            };
            auto multiply = [&](int k, const frag (*a)[NP]) {
#pragma unroll
                for (int it = 0; it < C / (2 * CW); ++it) {
                    float cw[CW];
                    const float4 *src = reinterpret_cast<const float4 *>(prod + j * ROW + k * C + 2 * CW * it + CW * (int)h);
#pragma unroll
                    for (int i = 0; i < CW / 4; ++i) {
                        const float4 x = src[i];
                        cw[4 * i] = x.x; cw[4 * i + 1] = x.y; cw[4 * i + 2] = x.z; cw[4 * i + 3] = x.w;
                    }
#pragma unroll
                    for (int u = 0; u < CW / G; ++u) {
                        frag bf[NP];
                        Mm::pack(cw + u * G, bf);
                        acc = step(a[it * (CW / G) + u], bf, acc);
                    }
                }
            };
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
            request(0, a0);
            for (int k = 0; k < ps.n; k += 2) {
                if (k + 1 < ps.n) request(k + 1, a1);
                multiply(k, a0);
                if (k + 2 < ps.n) request(k + 2, a0);
                if (k + 1 < ps.n) multiply(k + 1, a1);
            }
            if constexpr (FEAT) {
                const uint32_t p = tile * kTileRays + j;
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    if (p < M && row_of(v, (int)h) < kAppDim) rgb[(size_t)p * kAppDim + row_of(v, (int)h)] = acc[v];
            } else {
#pragma unroll
                for (int v = 0; v < 16; ++v) raw_s[v * LM_WAVE + lane] = acc[v];
            }
        }
        if constexpr (FEAT) {
            position(gn, vn);
            __syncthreads();  // the next tile's products overwrite this one's
            continue;
        }
        acc = bias_of(L.b1 + wave * 128u, bias);
#pragma unroll
        for (int t = kFirst; t < T1; ++t)
#pragma unroll
            for (int pt = 0; pt < NP; ++pt) wa[t][pt] = weight(w1, t * NP + pt, here);
        __syncthreads();
        // ---- encoding: wave w takes input rows 4 w .. 4 w + 3 of every lane
        {
            float x[4], s1[4], c1[4], s2[4], c2[4];
            bool big = false;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[i] = raw_s[(4 * wave + i) * LM_WAVE + lane];
                if (wave == 3u) x[i] = i < 3 ? (h ? vdir[i] : x[i]) : 0.0f;
                big |= sincos_of<PREC>(x[i], s1[i], c1[i]);
            }
            if (__builtin_expect(big, 0)) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (fabsf(x[i]) > kSincosMax) { s1[i] = sinf(x[i]); c1[i] = cosf(x[i]); }
            }
            if (wave == 3u) s1[3] = c1[3] = 0.0f;  // row 15 of a lane is zero in every group
#pragma unroll
            for (int i = 0; i < 4; i += 2) double_angle<PREC>(s1 + i, c1 + i, s2 + i, c2 + i);
            if (wave == 3u) c2[3] = 0.0f;
            const int v = 4 * (int)wave;
            N::write4(in1, v, lane, x);
            N::write4(in1, 16 + v, lane, s1);
            N::write4(in1, 32 + v, lane, c1);
            N::write4(in1, 48 + v, lane, s2);
            N::write4(in1, 64 + v, lane, c2);
        }
        __syncthreads();
        // ---- layer 1: a row block per wave; a step's weights of layer 2 are requested as registers fall free
        frag wb[T2][NP];
#pragma unroll
        for (int u = 0; u < N::U1; ++u) {
            frag x[N::S][NP];
            N::read(in1 + u * N::kBytes, lane, x);
#pragma unroll
            for (int i = 0; i < N::S; ++i) {
                const int t = u * N::S + i;
                if (!(G == 1 && t % 16 == 15)) acc = step(wa[t], x[i], acc);  // (rows 27 and 31: zero inputs, zero weights)
                if (t >= T1 - T2) {
#pragma unroll
                    for (int pt = 0; pt < NP; ++pt) wb[t - (T1 - T2)][pt] = weight(w2, (t - (T1 - T2)) * NP + pt, here);
                }
            }
        }
        auto publish = [&](char *dst) {
#pragma unroll
            for (int q = 0; q < 4; ++q) N::write4_relu(dst, (int)wave * 16 + 4 * q, lane, acc, q);
        };
        publish(in2);
        acc = bias_of(L.b2 + wave * 128u, bias);
        __syncthreads();
        // (fp32: the wave's rows of layer 3 travel meanwhile)
        float4 w3[G == 1 ? 16 : 1];
        if constexpr (G == 1) {
            const uint32_t half = (here / (uint32_t)sizeof(frag) / 32u) * 128u;
#pragma unroll
            for (int v = 0; v < 16; ++v)
                w3[v] = *reinterpret_cast<const float4 *>(packed + L.w3 + (size_t)(wave * 16 + v) * (LM_WAVE * sizeof(float)) + half);
        }
        // ---- layer 2
#pragma unroll
        for (int u = 0; u < N::U2; ++u) {
            frag x[N::S][NP];
            N::read(in2 + u * N::kBytes, lane, x);
#pragma unroll
            for (int i = 0; i < N::S; ++i) acc = step(wb[u * N::S + i], x[i], acc);
        }
        if constexpr (G == 1) {
            // ---- layer 3 in fp32: every wave its own row block's share of the three outputs, one wave adds them up
            float x[16], part[3];
#pragma unroll
            for (int v = 0; v < 16; ++v) x[v] = relu_f32(acc[v]);
            last_layer_block(x, [&](int v) { return w3[v]; }, part);
            float *sums = reinterpret_cast<float *>(in3);  // (layer 1's inputs are done with: every wave is past layer 1)
#pragma unroll
            for (int k = 0; k < 3; ++k) sums[(wave * 3 + k) * LM_WAVE + lane] = part[k];
            position(gn, vn);
            __syncthreads();
            if (wave == kLead) {
                const float *b3 = reinterpret_cast<const float *>(packed + L.b3);
                const uint32_t p = tile * kTileRays + j;
                float out[3];
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    out[k] = last_layer_sum(sums[k * LM_WAVE + lane], sums[(3 + k) * LM_WAVE + lane], sums[(6 + k) * LM_WAVE + lane],
                                            sums[(9 + k) * LM_WAVE + lane], b3[k]);
                if (p < M && h == 0) {
#pragma unroll
                    for (int i = 0; i < 3; ++i) rgb[(size_t)p * 3 + i] = colour_of<PREC>(out[i]);
                }
            }
        } else {
            frag wc[T2][NP];
            if (wave == kLead) {
#pragma unroll
                for (int t = 0; t < T2; ++t)
#pragma unroll
                    for (int pt = 0; pt < NP; ++pt) wc[t][pt] = weight(L.w3, t * NP + pt, here);
            }
            publish(in3);
            position(gn, vn);
            __syncthreads();
            // ---- layer 3
            if (wave == kLead) {
                acc = bias_of(L.b3, bias);
#pragma unroll
                for (int u = 0; u < N::U2; ++u) {
                    frag x[N::S][NP];
                    N::read(in3 + u * N::kBytes, lane, x);
#pragma unroll
                    for (int i = 0; i < N::S; ++i) acc = step(wc[u * N::S + i], x[i], acc);
                }
                const uint32_t p = tile * kTileRays + j;
                if (p < M && h == 0) {
#pragma unroll
                    for (int i = 0; i < 3; ++i) rgb[(size_t)p * 3 + i] = colour_of<PREC>(acc[i]);
                }
            }
        }
        __syncthreads();  // the next tile's products overwrite layer 3's inputs
    }
}

size_t shade_lds(int prec, int K) {
    switch (prec) {
        case LM_MLP_F32: return ShadeLds<LM_MLP_F32>::total(K);
        case LM_MLP_F16: return ShadeLds<LM_MLP_F16>::total(K);
        case LM_MLP_BF16: return ShadeLds<LM_MLP_BF16>::total(K);
        default: return ShadeLds<LM_MLP_F16X2>::total(K);
    }
}

template <int PREC, typename T, int NU, bool FEAT>
int launch_shade(const lm_geom &geom, const PlaneSet &ps, int K, const void *packed, const float *rays, uint32_t M, const uint32_t *list,
                 const uint32_t *count, uint32_t cap, float *rgb, hipStream_t st) {
    const size_t lds = ShadeLds<PREC>::total(K);
    auto kern = &k_shade<PREC, T, NU, FEAT>;
    static thread_local size_t reserved_on[LM_MAX_DEVICES] = {};  // set once per thread, device, kernel, size
    size_t &reserved = reserved_on[lm_current_device()];
    if (reserved != lds) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) LM_FAIL(LM_ERR_LAUNCH, "k_shade: LDS reservation failed: %s", hipGetErrorString(e));
        reserved = lds;
    }
    unsigned grid = (unsigned)lm_persistent_blocks(2);
    if (FEAT) grid = std::min(grid, (M + kTileRays - 1) / kTileRays);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kBlock), lds, st, geom, ps, K, (const char *)packed, pack_layout(PREC, K), rays, M, list,
                       count, cap, rgb);
    LM_CHECK_LAUNCH("k_shade");
    return LM_OK;
}

template <bool FEAT>
int shade(int prec, int dtype, int nu, const lm_geom &geom, const PlaneSet &ps, int K, const void *packed, const float *rays, uint32_t M,
          const uint32_t *list, const uint32_t *count, uint32_t cap, float *rgb, hipStream_t st) {
#define LM_SHADE_NU(PREC_, T_, NU_) launch_shade<PREC_, T_, NU_, FEAT>(geom, ps, K, packed, rays, M, list, count, cap, rgb, st)
#define LM_SHADE(PREC_)                                              \
    if (dtype == LM_F32) {                                           \
        switch (nu) {                                                \
            case 1: return LM_SHADE_NU(PREC_, float, 1);             \
            case 2: return LM_SHADE_NU(PREC_, float, 2);             \
            case 3: return LM_SHADE_NU(PREC_, float, 3);             \
            default: return LM_SHADE_NU(PREC_, float, 4);            \
        }                                                            \
    }                                                                \
    switch (nu) {                                                    \
        case 1: return LM_SHADE_NU(PREC_, Half4, 1);                 \
        case 2: return LM_SHADE_NU(PREC_, __half, 2);                \
        case 3: return LM_SHADE_NU(PREC_, Half6, 3);                 \
        default: return LM_SHADE_NU(PREC_, __half, 4);               \
    }
    switch (prec) {
        case LM_MLP_F32: LM_SHADE(LM_MLP_F32)
        case LM_MLP_F16: LM_SHADE(LM_MLP_F16)
        case LM_MLP_BF16: LM_SHADE(LM_MLP_BF16)
        default: LM_SHADE(LM_MLP_F16X2)
    }
#undef LM_SHADE
#undef LM_SHADE_NU
}

}  // namespace

int lm_check_geom(const lm_geom *g);
int lm_check_planes(const lm_plane *planes, int32_t n, int *dtype_out, int *K_out);
int lm_check_prec(int prec);
int lm_check_K(int K);
int lm_app_feat_supported(const lm_model *m);

// The models k_shade covers: equal channel counts of 16 .. 64, products that leave room for two workgroups per CU.
static bool shade_covers(const lm_model *m, int K) { return lm_app_feat_supported(m) && shade_lds(m->mlp_prec, K) <= 80 * 1024; }

// The host does not know how many entries a chunk has.  With about 100 000 of them the other kernels are as fast, which
// read the weights once per workgroup; that many are reached near 3 million candidate samples (12288 rays of 128: 227 us
// there, 217 - 225 here; 3.6 million of the production shape 337 and 337; 7.3 million 555 and 567).  The fp32 network's
// matrix steps take eight times as long, its line lies at half a million (4096 rays of 128 samples, 46 000 entries:
// 145 and 119 us; 8192 rays: 203 and 218).
// With a threshold far below the weights of a uniform fog (1 / S) nearly every valid sample is an entry, three to six times
// as many: the lines lie at a third (threshold 0, three small planes, here / there: 2048 rays of 128 samples 146 / 155 us,
// 4096 258 / 226, 12288 685 / 527; nine planes 8192 rays 344 / 348, 12288 483 / 455; fp32 network 1024 rays 139 / 155,
// 4096 443 / 363).
bool lm_shade_takes(const lm_model *m, int64_t N, int K) {
    const int64_t limit = m->mlp_prec == LM_MLP_F32 ? 1ll << 19 : 3ll << 20;
    const bool most_samples = m->weight_thres * (float)m->geom.S < 1e-2f;
    return shade_covers(m, K) && N * m->geom.S <= (most_samples ? limit / 3 : limit);
}

// compute_appfeature at given points: up to here a tile per workgroup beats k_app_feat's tile per wave.  Nine planes, split
// mode, products through memory / k_app_feat / here: 4000 points 38 / 51 / 16 us, 32000: 75 / 75 / 50, 64000: 150 / 84 / 95;
// fp16 mode (k_app_feat has two workgroups per CU there): 32000: 74 / 124 / 47, 64000: 148 / 151 / 88, 128000: 304 / 161 / 173.
bool lm_few_points_take(int prec, int K, int64_t M) {
    const int64_t limit = prec == LM_MLP_F16 || prec == LM_MLP_BF16 ? 96 * 1024 : 48 * 1024;
    return M <= limit && shade_lds(prec, K) <= 80 * 1024;
}

// `count` list entries (at most `cap`) -> rgb [count, 3]; what lm_launch_app_features + lm_launch_app_colour give.
int lm_launch_shade(const lm_model *m, const float *rays, const uint32_t *list, const uint32_t *count, uint32_t cap, float *rgb,
                    hipStream_t st) {
    int dtype, K;
    if (int rc = lm_check_planes(m->app, m->n_planes, &dtype, &K)) return rc;
    if (int rc = lm_check_prec(m->mlp_prec)) return rc;
    if (int rc = lm_check_K(K)) return rc;
    LM_REQUIRE(rays && list && count && rgb, "null buffer");
    LM_REQUIRE(m->mlp_packed && lm_aligned16(m->mlp_packed), "packed colour-network weights are null or misaligned");
    if (!shade_covers(m, K)) LM_FAIL(LM_ERR_UNSUPPORTED, "k_shade does not cover these planes");
    return shade<false>(m->mlp_prec, dtype, m->app[0].C / 16, m->geom, make_set(m->app, m->n_planes, &m->geom), K, m->mlp_packed, rays,
                        0u, list, count, cap, rgb, st);
}

// M points (M < 2^31) -> feat [M, 27]; the caller has checked the arguments and asked lm_few_points_take
int lm_launch_few_points(const lm_plane *planes, int n, int prec, int dtype, int K, const void *packed, const float *xyz, uint32_t M,
                         float *feat, hipStream_t st) {
    return shade<true>(prec, dtype, planes[0].C / 16, lm_geom{}, make_set(planes, n), K, packed, xyz, M, nullptr, nullptr, 0u, feat, st);
}
