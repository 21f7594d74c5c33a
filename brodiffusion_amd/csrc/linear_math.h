// Pieces shared by the kernels of the projection GEMM (linear.hip, linear_pipe.hip, linear_dma.hip): MFMA wrappers, the exact
// GELU of the GEGLU epilogue, the widening of INT8 weights and the scaling of their accumulators.
#pragma once
#include "internal.h"

namespace mi {
namespace gemm {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

template <typename T> struct Mma;
template <> struct Mma<__bf16> {
    using v8 = bf16x8;
    using v4 = bf16x4;
    static __device__ __forceinline__ f32x16 run(v8 a, v8 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ f32x4 run16(v8 a, v8 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};
template <> struct Mma<_Float16> {
    using v8 = f16x8;
    using v4 = f16x4;
    static __device__ __forceinline__ f32x16 run(v8 a, v8 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ f32x4 run16(v8 a, v8 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};

// x * Phi(x), the erf form of GELU (gelu_exact_scalar, src/fused_transformer.cu:89-92), branch free. With z = |x| / sqrt 2,
// erfc(z) = t exp(-z^2 + P(t)), t = 1 / (1 + z / 2) (the Chebyshev fit of Numerical Recipes' erfcc, fractional error below
// 1.2e-7 for all z >= 0), and Phi(x) = erfc(z) / 2 for x < 0, 1 - erfc(z) / 2 otherwise - so the left tail keeps its
// relative accuracy, which the sum 1 + erf loses to cancellation. Here in base 2 with the constants folded: the
// coefficients of P are multiplied by log2 e, its constant term also takes the factor 1/2 (-1 in the exponent), and
// z^2 log2 e = (|x| sqrt(log2 e / 2))^2. 19 FP32 instructions and 2 transcendentals; against x Phi(x) in double the
// relative error stays below 4e-6 for |x| < 6 and 1.5e-5 down to x = -12.
__device__ __forceinline__ float gelu_erf(float x) {
    const float ax = fabsf(x);
    const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(ax, 0.35355339059327373f, 1.f));
    const float zs = ax * 0.849321800288f;
    float q = 0.246517298f;
    q = __builtin_fmaf(q, t, -1.18611495f);
    q = __builtin_fmaf(q, t, 2.14747446f);
    q = __builtin_fmaf(q, t, -1.63775315f);
    q = __builtin_fmaf(q, t, 0.402321582f);
    q = __builtin_fmaf(q, t, -0.26875686f);
    q = __builtin_fmaf(q, t, 0.139630057f);
    q = __builtin_fmaf(q, t, 0.539700616f);
    q = __builtin_fmaf(q, t, 1.4427292f);
    q = __builtin_fmaf(q, t, -2.82574822f);
    const float half_erfc = t * __builtin_amdgcn_exp2f(__builtin_fmaf(-zs, zs, q));
    return x * (x < 0.f ? half_erfc : 1.f - half_erfc);
}

// acc * scale + bias of the INT8-weight forms as an FP32 value of its own. Left to itself the compiler merges the
// multiply-add with the rounding to T that follows (v_fma_mixlo_f16: one rounding of the exact result) in some places and
// not in others, and the plain and the GEGLU form of the same layer then disagree by a unit in the last place in about 3
// outputs of 100 000; as a separate FP32 operation it is the FP32 multiply-add and conversion of the reference's kernel
// everywhere.
__device__ __forceinline__ float scaled_acc(float acc, float scale, float bias) {
    float r = __builtin_fmaf(acc, scale, bias);
    asm volatile("" : "+v"(r));
    return r;
}

// 8 INT8 weights -> 8 values of T, exactly
template <typename T> __device__ __forceinline__ typename Mma<T>::v8 widen(u32x2 raw);
template <> __device__ __forceinline__ f16x8 widen<_Float16>(u32x2 raw) {
    // u = w + 128 as the low byte of 1024 + u (0x6400 | u), minus 1152
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    const f16x2 off = {static_cast<_Float16>(1152.f), static_cast<_Float16>(1152.f)};
    u32x4 r;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const unsigned u = raw[i] ^ 0x80808080u;
        const unsigned lo = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u), hi = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);
        r[2 * i] = __builtin_bit_cast(unsigned, __builtin_bit_cast(f16x2, lo) - off);
        r[2 * i + 1] = __builtin_bit_cast(unsigned, __builtin_bit_cast(f16x2, hi) - off);
    }
    return __builtin_bit_cast(f16x8, r);
}
template <> __device__ __forceinline__ bf16x8 widen<__bf16>(u32x2 raw) {
    // |w| <= 128 has at most 8 significant bits: the upper half of the FP32 value is the bf16 value
    u32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const unsigned pair = i & 1 ? raw[i >> 1] >> 16 : raw[i >> 1];
        const float a = static_cast<float>(static_cast<signed char>(pair & 0xffu)), b = static_cast<float>(static_cast<signed char>((pair >> 8) & 0xffu));
        r[i] = __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, b), __builtin_bit_cast(unsigned, a), 0x07060302u);
    }
    return __builtin_bit_cast(bf16x8, r);
}

}  // namespace gemm
}  // namespace mi
