// Device side of the colour network shared by the kernels that evaluate it: bias and activation fragments and the
// positional encoding.  See lm_mlp.hip for the register layout.
#pragma once
#include <hip/hip_fp16.h>

#include "lm_mma.h"

namespace {

using namespace lm_mma;

__device__ __forceinline__ floatx16 load_bias(const float *b, int idx) {
    floatx16 a;
    const float4 *p = reinterpret_cast<const float4 *>(b + idx * 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float4 t = p[i];
        a[4 * i] = t.x; a[4 * i + 1] = t.y; a[4 * i + 2] = t.z; a[4 * i + 3] = t.w;
    }
    return a;
}

// sin and cos of x to float rounding for |x| <= 8192 (three-constant Cody-Waite reduction by
// pi/2, then polynomials on [-pi/4, pi/4]; constants and coefficients are those published with the
// single-precision sinf / cosf of S. Moshier's Cephes library); callers redo larger arguments with the
// library routines (kSincosMax), outside their hot loop.
constexpr float kSincosMax = 8192.0f;
__device__ __forceinline__ void sincos_f32(float x, float &s, float &c) {
    const float k = rintf(x * 0.636619772367581f);
    float r = fmaf(-k, 1.5703125f, x);
    r = fmaf(-k, 4.837512969970703125e-4f, r);
    r = fmaf(-k, 7.54978995489188216e-8f, r);
    const float r2 = r * r;
    float ps = fmaf(r2, -1.9515295891e-4f, 8.3321608736e-3f);
    ps = fmaf(ps, r2, -1.6666654611e-1f);
    ps = fmaf(ps * r2, r, r);
    float pc = fmaf(r2, 2.443315711809948e-5f, -1.388731625493765e-3f);
    pc = fmaf(pc, r2, 4.166664568298827e-2f);
    pc = fmaf(pc * r2, r2, fmaf(-0.5f, r2, 1.0f));
    const int q = (int)k & 3;
    const float ss = (q & 1) ? pc : ps, cc = (q & 1) ? ps : pc;
    s = (q & 2) ? -ss : ss;
    c = ((q + 1) & 2) ? -cc : cc;
}

// sin and cos through the hardware functions (argument in revolutions) after a two-constant reduction by
// 2 pi: within 4.3e-7 of the exact values for |x| <= 8192 (measured over 2^24 arguments per range), seven
// instructions per value.  Used by the split-fp16 mode, whose products carry about 21 mantissa bits anyway.
__device__ __forceinline__ void sincos_hw(float x, float &s, float &c) {
    const float k = rintf(x * 0.15915494309189535f);
    float r = fmaf(-k, 6.28125f, x);
    r = fmaf(-k, 1.9353071795864769e-3f, r);
    const float t = r * 0.15915494309189535f;
    s = __builtin_amdgcn_sinf(t);
    c = __builtin_amdgcn_cosf(t);
}

// max(x, 0) for finite floats as one integer instruction (negative floats are negative integers)
__device__ __forceinline__ float relu_f32(float x) {
    return __builtin_bit_cast(float, max(__builtin_bit_cast(int, x), 0));
}

// relu(acc) of one row block -> G-slot B fragments of the next layer
template <int PREC>
__device__ __forceinline__ void relu_to_frags(const floatx16 &acc, typename Mma<PREC>::frag (*out)[Mma<PREC>::NP]) {
    using M = Mma<PREC>;
    constexpr int G = M::G;
    if constexpr (PREC == LM_MLP_F16) {
        // round first, then clamp two halves per instruction: rounding is monotone and keeps zero, so
        // this equals rounding relu(x)
        float hv[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) hv[v] = acc[v];
#pragma unroll
        for (int u = 0; u < 16 / G; ++u) {
            M::pack(hv + u * G, out[u]);
            const half8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
            out[u][0] = __builtin_elementwise_max(out[u][0], zero);
        }
    } else {
        float hv[16];
#pragma unroll
        for (int v = 0; v < 16; ++v) hv[v] = relu_f32(acc[v]);
#pragma unroll
        for (int u = 0; u < 16 / G; ++u) M::pack(hv + u * G, out[u]);
    }
}

// relu of two accumulator values (registers 2 q, 2 q + 1) -> register q % 4 of the next layer's B fragment q / 4
// (per part)
template <int PREC>
__device__ __forceinline__ void relu_pair(const floatx16 &acc, int q, uint32_t (*out)[4]) {
    using M = Mma<PREC>;
    uint32_t d[M::NP];
    if constexpr (PREC == LM_MLP_F16) {
        // round first, then clamp two halves with one instruction (rounding is monotone and keeps zero)
        M::pack_pair(acc[2 * q], acc[2 * q + 1], d);
        const half2v zero = {0, 0};
        d[0] = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(half2v, d[0]), zero));
    } else if constexpr (PREC == LM_MLP_BF16) {
        // round first, then clamp both halves with one packed integer maximum: a negative bf16 number is a negative
        // 16-bit integer, a non-negative one keeps its bits
        typedef short short2v __attribute__((ext_vector_type(2)));
        M::pack_pair(acc[2 * q], acc[2 * q + 1], d);
        const short2v zero = {0, 0};
        d[0] = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(short2v, d[0]), zero));
    } else {
        M::pack_pair(relu_f32(acc[2 * q]), relu_f32(acc[2 * q + 1]), d);
    }
#pragma unroll
    for (int pt = 0; pt < M::NP; ++pt) out[pt][q % 4] = d[pt];
}

// sin and cos of an input in the mode's precision; true: the argument is beyond the fast reduction's range and the caller
// takes the library routines instead, outside its hot loop
template <int PREC> __device__ __forceinline__ bool sincos_of(float x, float &s, float &c) {
    if (PREC == LM_MLP_F16X2) {
        sincos_hw(x, s, c);
    } else if (PREC == LM_MLP_F32) {
        sincos_f32(x, s, c);
    } else {
        s = __sinf(x); c = __cosf(x);
        return false;
    }
    return fabsf(x) > kSincosMax;
}

// sin and cos of twice the argument, for two arguments, as every kernel rounds them.  In the fp16 mode they are rounded
// once, from the exact product straight to fp16 (the conversion that follows is exact then): left to itself the compiler does
// so for some values in one kernel and for others in another, and rounding to fp32 first gives the wrong neighbour for one
// value in 15 000.
template <int PREC> __device__ __forceinline__ void double_angle(const float *s1, const float *c1, float *s2, float *c2) {
    if constexpr (PREC == LM_MLP_F16) {
        // In this order no instruction reads what the one before it wrote, nor a cosine that a transcendental instruction
        // may have written right before the block (2 s1 lies between the sines and here).
        half2v s, c;
        asm("v_fma_mixlo_f16 %1, -%2, %3, 1.0\n\t"
            "v_fma_mixlo_f16 %0, %2, %4, 0\n\t"
            "v_fma_mixhi_f16 %1, -%5, %6, 1.0\n\t"
            "v_fma_mixhi_f16 %0, %5, %7, 0"
            : "=&v"(s), "=&v"(c)
            : "v"(2.0f * s1[0]), "v"(s1[0]), "v"(c1[0]), "v"(2.0f * s1[1]), "v"(s1[1]), "v"(c1[1]));
#pragma unroll
        for (int i = 0; i < 2; ++i) { s2[i] = (float)s[i]; c2[i] = (float)c[i]; }
    } else {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            s2[i] = 2.0f * s1[i] * c1[i];
            c2[i] = fmaf(-2.0f * s1[i], s1[i], 1.0f);
            if (PREC == LM_MLP_F16X2) asm("" : "+v"(s2[i]), "+v"(c2[i]));  // in fp32 before the split, in every kernel
        }
    }
}

// raw[cb][16] (the lane's 16 input rows of each of its NCB samples) -> the first layer's B fragments: per lane
// five groups of 16 slots (raw, sin, cos, sin 2x, cos 2x)
template <int PREC, int NCB>
__device__ __forceinline__ void encode_inputs(const float (*raw)[16],
                                              typename Mma<PREC>::frag (*bfrag)[kSlots1 / Mma<PREC>::G][Mma<PREC>::NP]) {
    using M = Mma<PREC>;
    constexpr int G = M::G, T1 = kSlots1 / G;
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
        float slots[kSlots1];
        constexpr bool kExact = PREC == LM_MLP_F32 || PREC == LM_MLP_F16X2;
        bool big = false;
#pragma unroll
        for (int v = 0; v < 15; ++v) {
            slots[v] = raw[cb][v];
            big |= sincos_of<PREC>(slots[v], slots[16 + v], slots[32 + v]);
        }
        // row 27 / 31 (v = 15) is zero and meets zero weights
        slots[15] = 0.0f; slots[31] = 0.0f; slots[47] = 0.0f;
        if (kExact && __builtin_expect(big, 0)) {
            // arguments beyond the fast reduction's range: library routines, rarely if ever taken
#pragma unroll
            for (int v = 0; v < 15; ++v)
                if (fabsf(slots[v]) > kSincosMax) { slots[16 + v] = sinf(slots[v]); slots[32 + v] = cosf(slots[v]); }
        }
#pragma unroll
        for (int v = 0; v < 16; v += 2) double_angle<PREC>(slots + 16 + v, slots + 32 + v, slots + 48 + v, slots + 64 + v);
        slots[79] = 0.0f;
#pragma unroll
        for (int t = 0; t < T1; ++t) M::pack(slots + t * G, bfrag[cb][t]);
    }
}

// fp32 mode: a 32-row block of the last layer's input (the lane's 16 values after relu) times its three rows of weights, for the
// vector unit: `w` gives {row 0, row 1, row 2, -} of slot v.  A matrix instruction would work 32 rows for these three (64 of them
// a tile, a tenth of the network's).  2^22 rows 2616 -> 2439 us, and 2355 with the steps of the all-zero input slots left out;
// 1024 rays, where one wave did these steps alone, 49.9 -> 44.6 and 44.2 (whole call, with the rays kernel's 32-bit offsets).
// The blocks' sums are added in order, then the halves', then the bias (last_layer_sum), in every kernel.
template <typename W> __device__ __forceinline__ void last_layer_block(const float *x, const W &w, float *sum) {
    sum[0] = sum[1] = sum[2] = 0.0f;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const float4 a = w(v);
        sum[0] = fmaf(a.x, x[v], sum[0]);
        sum[1] = fmaf(a.y, x[v], sum[1]);
        sum[2] = fmaf(a.z, x[v], sum[2]);
    }
}
// blocks' sums of this lane's half -> the layer's output (on both halves); b: the bias of the row
__device__ __forceinline__ float last_layer_sum(float p0, float p1, float p2, float p3, float b) {
    const float mine = ((p0 + p1) + p2) + p3;
    return b + (mine + __shfl_xor(mine, 32));
}

// sigmoid; the hardware reciprocal is within one unit in the last place, enough for every mode
template <int PREC> __device__ __forceinline__ float colour_of(float x) {
    const float e = (PREC == LM_MLP_F32 || PREC == LM_MLP_F16X2) ? expf(-x) : __expf(-x);
    return __builtin_amdgcn_rcpf(1.0f + e);
}

}  // namespace
