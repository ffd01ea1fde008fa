// Element types of the layer-list decoders: bf16 storage with f32 arithmetic, or f32 throughout.
#pragma once
#include "epilogue.hpp"

typedef unsigned int lm_u32x4 __attribute__((ext_vector_type(4)));

template <class T> struct Piece; // 16 bytes of T
template <> struct Piece<bf16_t> {
    static constexpr int N = 8;
    static __device__ __forceinline__ void unpack(const lm_u32x4 &v, float (&f)[8]) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const unsigned pair = v[i];
            f[2 * i] = __builtin_bit_cast(float, pair << 16);
            f[2 * i + 1] = __builtin_bit_cast(float, pair & 0xffff0000u);
        }
    }
};
template <> struct Piece<float> {
    static constexpr int N = 4;
    static __device__ __forceinline__ void unpack(const lm_u32x4 &v, float (&f)[4]) {
        const float4_t w = __builtin_bit_cast(float4_t, v); // (the whole vector: a bit cast of one element reads element 0)
#pragma unroll
        for (int i = 0; i < 4; i++) f[i] = w[i];
    }
};
template <class T> __device__ __forceinline__ float dot_piece(const lm_u32x4 &w, const lm_u32x4 &x, float acc) {
    float a[Piece<T>::N], b[Piece<T>::N];
    Piece<T>::unpack(w, a);
    Piece<T>::unpack(x, b);
#pragma unroll
    for (int i = 0; i < Piece<T>::N; i++) acc = fmaf(a[i], b[i], acc);
    return acc;
}

// library exponentials: the gates and weights are wanted to f32 accuracy
__device__ __forceinline__ float lm_sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }
// z / (1 + exp(-z)).  exp(-z) = 2^r 2^f, r whole and |f| <= 1/2: the product with -1 / ln 2 in two pieces (Dekker's, with fused multiply-adds for the exact rest), so f has twice f32's
// digits, the hardware's 2^f, and a division by the hardware's 1 / d (of a quarter of d: above 2^126 its reciprocal is no normal number) with one Newton correction of the
// quotient.  These are the steps of the compiler's own expf for gfx950 without its ranges and scalings, which serve arguments that do not occur here, and its second piece of 1 / ln 2 (one unit
// below the nearest float, with which 15 results differ): the same bits as z / (1.0f + expf(-z)), for every f32 value (tested), in a quarter fewer instruction
// cycles.  A gated product's epilogue is these: 1920 x 16128 x 2048 among a model's launches 117.3 -> 112.7 us, 768 rows 50.8 -> 47.2.
__device__ __forceinline__ float lm_silu(float z) {
    constexpr float hi = -1.44269502e+00f, lo = -1.92596286e-08f; // -1 / ln 2
    const float x = __builtin_amdgcn_fmed3f(z, -200.0f, 200.0f), t = x * hi, r = __builtin_rintf(t);
    const float f = (t - r) + __builtin_fmaf(x, lo, __builtin_fmaf(x, hi, -t)), d = 1.0f + __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(f), (int)r);
    const float i = __builtin_amdgcn_rcpf(d * 0.25f) * 0.25f, q = z * i;
    return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-q, d, z), i, q), d, z); // (infinities and NaN as a division gives them)
}
__device__ __forceinline__ float lm_softcap(float z, float cap) { return cap * tanhf(z / cap); }
