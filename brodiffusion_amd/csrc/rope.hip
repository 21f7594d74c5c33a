// Stand-alone rotary position embedding for gfx950: out = RoPE(x) with FP32 tables.
// Bandwidth-bound elementwise pass (one read and one write of x); used where the rotated
// tensor itself must exist in HBM (the prefix cache keeps post-RoPE K). Attention calls
// apply the rotation while loading Q and K instead.
#include <type_traits>

#include "internal.h"

namespace mi {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// How the kernels with 4 heads to a thread deal rows out: a block takes rb rows, t = 0 .. rb * units of them 16-byte chunk
// positions (a unit: one chunk position of 4 heads). Row, chunk and address then come from 32-bit multiplications by inverses;
// dividing a 64-bit index by the number of units cost more than everything between the loads and the stores
// (24 heads of 128, us: head norm 300 rows 3.5 -> 2.7, 1997 5.3 -> 4.6, 4608 9.9 -> 9.4; with the rotation 3.7 -> 2.8, 5.7 -> 4.9,
// 10.7 -> 9.8; rotation alone 4608 10.1 -> 9.7; a copy of 4608 rows takes 9.1). In the head norm the sums of squares also
// left the LDS permutation network for DPP moves.
struct RowUnits {
    int units, rb, threads;      // of a row; rows and threads of a block
    unsigned inv;                // ceil(2^32 / units): t / units exactly for t * units < 2^32 (0, and no division, with one row to a block)
    long blocks;
    RowUnits(long rows, int units_) : units(units_), rb(1), inv(0xffffffffu / static_cast<unsigned>(units_) + 1u) {
        // the number of rows that leaves the fewest lanes of the block's last wavefront empty
        for (int n = 2, best = (units + 63) / 64 * 64 - units; n * units <= 256; ++n)
            if (const int empty = (n * units + 63) / 64 * 64 - n * units; empty * rb <= best * n) { rb = n; best = empty; }
        if (rb == 1) inv = 0;
        threads = rb * units < 256 ? (rb * units + 63) / 64 * 64 : 256;
        blocks = (rows + rb - 1) / rb;
    }
    unsigned grid() const { return static_cast<unsigned>(blocks < (1 << 20) ? blocks : (1 << 20)); }
};

// sum over groups of N neighbouring lanes (N = 4, 8 or 16, all of them active), in every lane of the group; the order of a butterfly
template <int N> __device__ __forceinline__ float group_sum(float v) {
    auto moved = [](float f, auto ctrl) {
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, f), decltype(ctrl)::value, 0xf, 0xf, false));
    };
    v += moved(v, std::integral_constant<int, 0xB1>{});                        // quad_perm [1, 0, 3, 2]
    v += moved(v, std::integral_constant<int, 0x4E>{});                        // quad_perm [2, 3, 0, 1]
    if constexpr (N >= 8) v += moved(v, std::integral_constant<int, 0x141>{});  // row_half_mirror: the other quad of 8
    if constexpr (N >= 16) v += moved(v, std::integral_constant<int, 0x140>{}); // row_mirror: the other half of 16
    return v;
}

// Adjacent pairs (x[2p], x[2p+1]): one thread rotates one 16-byte chunk = 4 pairs.
template <typename T>
__global__ void __launch_bounds__(256) rope_adjacent_kernel(const T* __restrict__ x, T* __restrict__ out,
                                                            const float* __restrict__ cs, const float* __restrict__ sn,
                                                            int rows, int H, int d, long x_rs, long o_rs, int per_head) {
    typedef T t8 __attribute__((ext_vector_type(8)));
    const int cpr = H * d / 8;  // chunks per row
    const long total = static_cast<long>(rows) * cpr;
    for (long idx = blockIdx.x * 256L + threadIdx.x; idx < total; idx += gridDim.x * 256L) {
        const int r = static_cast<int>(idx / cpr);
        const int c = static_cast<int>(idx - static_cast<long>(r) * cpr);
        const int col = c * 8;
        const int h = col / d;
        const int dc = col - h * d;  // multiple of 8 inside the head
        const long trow = per_head ? static_cast<long>(r) * H + h : r;
        const f32x4 cv = *reinterpret_cast<const f32x4*>(cs + trow * (d / 2) + dc / 2);
        const f32x4 sv = *reinterpret_cast<const f32x4*>(sn + trow * (d / 2) + dc / 2);
        t8 v = __builtin_bit_cast(t8, *reinterpret_cast<const u32x4*>(x + r * x_rs + col));
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const float a = static_cast<float>(v[2 * p]);
            const float b = static_cast<float>(v[2 * p + 1]);
            v[2 * p] = static_cast<T>(rope_re(a, b, cv[p], sv[p]));
            v[2 * p + 1] = static_cast<T>(rope_im(a, b, cv[p], sv[p]));
        }
        *reinterpret_cast<u32x4*>(out + r * o_rs + col) = __builtin_bit_cast(u32x4, v);
    }
}

// Adjacent pairs with one table for all heads: a thread rotates the same 16-byte chunk position of 4 heads of a row, so the
// chunk's table entries are fetched once for the four and 4 data loads are in flight per thread. The heads of a thread
// are H / 4 apart, so that for each of the four the lanes of a wavefront touch consecutive heads, i.e. one
// contiguous piece of the row. Same arithmetic per element as the kernel above.
template <typename T>
__global__ void __launch_bounds__(256) rope_adjacent_heads_kernel(const T* x, T* out, const float* __restrict__ cs, const float* __restrict__ sn, int rows,
                                                                  int d, long x_rs, long o_rs, RowUnits ru, unsigned inv_cpd) {
    typedef T t8 __attribute__((ext_vector_type(8)));
    constexpr int HB = 4;
    const int cpd = d / 8, n = ru.rb * ru.units;
    const long quarter = ru.units * 8L;
    for (long block = blockIdx.x; block < ru.blocks; block += gridDim.x)
        for (int t = threadIdx.x; t < n; t += blockDim.x) {
            const int rr = static_cast<int>(__umulhi(t, ru.inv)), u = t - rr * ru.units;
            const long r = block * ru.rb + rr;
            if (r >= rows) break;
            const int dcq = u - static_cast<int>(__umulhi(u, inv_cpd)) * cpd;
            const T* const xr = x + r * x_rs + u * 8;
            u32x4 raw[HB];
#pragma unroll
            for (int j = 0; j < HB; ++j) raw[j] = *reinterpret_cast<const u32x4*>(xr + j * quarter);
            const f32x4 cv = *reinterpret_cast<const f32x4*>(cs + r * (d / 2) + dcq * 4);
            const f32x4 sv = *reinterpret_cast<const f32x4*>(sn + r * (d / 2) + dcq * 4);
            T* const o = out + r * o_rs + u * 8;
#pragma unroll
            for (int j = 0; j < HB; ++j) {
                t8 v = __builtin_bit_cast(t8, raw[j]);
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    const float a = static_cast<float>(v[2 * p]);
                    const float b = static_cast<float>(v[2 * p + 1]);
                    v[2 * p] = static_cast<T>(rope_re(a, b, cv[p], sv[p]));
                    v[2 * p + 1] = static_cast<T>(rope_im(a, b, cv[p], sv[p]));
                }
                *reinterpret_cast<u32x4*>(o + j * quarter) = __builtin_bit_cast(u32x4, v);
            }
        }
}

// Split-half pairs (x[p], x[p + d/2]): one thread per pair (d/2 need not be a multiple of 8).
template <typename T>
__global__ void __launch_bounds__(256) rope_split_kernel(const T* __restrict__ x, T* __restrict__ out,
                                                         const float* __restrict__ cs, const float* __restrict__ sn,
                                                         int rows, int H, int d, long x_rs, long o_rs, int per_head) {
    const int half = d / 2;
    const int ppr = H * half;  // pairs per row
    const long total = static_cast<long>(rows) * ppr;
    for (long idx = blockIdx.x * 256L + threadIdx.x; idx < total; idx += gridDim.x * 256L) {
        const int r = static_cast<int>(idx / ppr);
        const int q = static_cast<int>(idx - static_cast<long>(r) * ppr);
        const int h = q / half;
        const int pp = q - h * half;
        const long trow = per_head ? static_cast<long>(r) * H + h : r;
        const float c = cs[trow * half + pp], s = sn[trow * half + pp];
        const float a = static_cast<float>(x[r * x_rs + h * d + pp]);
        const float b = static_cast<float>(x[r * x_rs + h * d + pp + half]);
        out[r * o_rs + h * d + pp] = static_cast<T>(rope_re(a, b, c, s));
        out[r * o_rs + h * d + pp + half] = static_cast<T>(rope_im(a, b, c, s));
    }
}

// Split-half pairs where half a head is whole 16-byte chunks (d % 16 == 0): one thread rotates the 8 pairs formed by
// chunk c of the lower half and chunk c of the upper half. Same arithmetic as rope_split_kernel.
template <typename T>
__global__ void __launch_bounds__(256) rope_split_vec_kernel(const T* x, T* out, const float* __restrict__ cs,
                                                             const float* __restrict__ sn, int rows, int H, int d, long x_rs,
                                                             long o_rs, int per_head) {
    typedef T t8 __attribute__((ext_vector_type(8)));
    const int half = d / 2;
    const int upr = H * half / 8;  // units (8 pairs) per row
    const long total = static_cast<long>(rows) * upr;
    for (long idx = blockIdx.x * 256L + threadIdx.x; idx < total; idx += gridDim.x * 256L) {
        const int r = static_cast<int>(idx / upr);
        const int u = static_cast<int>(idx - static_cast<long>(r) * upr);
        const int h = u / (half / 8);
        const int pp = (u - h * (half / 8)) * 8;   // first pair of the unit
        const long trow = per_head ? static_cast<long>(r) * H + h : r;
        const f32x4 c0 = *reinterpret_cast<const f32x4*>(cs + trow * half + pp), c1 = *reinterpret_cast<const f32x4*>(cs + trow * half + pp + 4);
        const f32x4 s0 = *reinterpret_cast<const f32x4*>(sn + trow * half + pp), s1 = *reinterpret_cast<const f32x4*>(sn + trow * half + pp + 4);
        t8 lo = __builtin_bit_cast(t8, *reinterpret_cast<const u32x4*>(x + r * x_rs + h * d + pp));
        t8 hi = __builtin_bit_cast(t8, *reinterpret_cast<const u32x4*>(x + r * x_rs + h * d + pp + half));
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float a = static_cast<float>(lo[e]), b = static_cast<float>(hi[e]);
            const float c = e < 4 ? c0[e & 3] : c1[e & 3], sv = e < 4 ? s0[e & 3] : s1[e & 3];
            lo[e] = static_cast<T>(rope_re(a, b, c, sv));
            hi[e] = static_cast<T>(rope_im(a, b, c, sv));
        }
        *reinterpret_cast<u32x4*>(out + r * o_rs + h * d + pp) = __builtin_bit_cast(u32x4, lo);
        *reinterpret_cast<u32x4*>(out + r * o_rs + h * d + pp + half) = __builtin_bit_cast(u32x4, hi);
    }
}

// Per-head RMS normalisation fused with the rotation (adjacent or split-half pairs) and an optional second destination for the
// leading rows: y = RoPE(x * rsqrt(mean_d(x^2) + eps) * gain), one read of x, one rounding. One thread per 16-byte
// chunk; the CPR = d/8 threads of a head row are neighbouring lanes of one wavefront (CPR is a power of two <= 16),
// so the sum of squares is CPR-lane butterfly. Everything is FP32 between the load and the single rounding.
template <typename T, int CPR>
__global__ void __launch_bounds__(256) headnorm_rope_kernel(const T* x, T* out, T* out2,
                                                            const T* __restrict__ gain, const float* __restrict__ cs,
                                                            const float* __restrict__ sn, int rows, int H, float eps,
                                                            long x_rs, long o_rs, long o2_rs, int out2_rows, int split_half) {
    typedef T t8 __attribute__((ext_vector_type(8)));
    constexpr int d = CPR * 8;
    const int cpr = H * CPR;
    const long total = static_cast<long>(rows) * cpr;
    for (long idx = blockIdx.x * 256L + threadIdx.x; idx < total; idx += gridDim.x * 256L) {
        const int r = static_cast<int>(idx / cpr);
        const int c = static_cast<int>(idx - static_cast<long>(r) * cpr);
        const int col = c * 8;
        const int dc = (c % CPR) * 8;
        const t8 v = __builtin_bit_cast(t8, *reinterpret_cast<const u32x4*>(x + r * x_rs + col));
        const t8 g = __builtin_bit_cast(t8, *reinterpret_cast<const u32x4*>(gain + dc));
        float f[8];
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) { f[e] = static_cast<float>(v[e]); ss = __builtin_fmaf(f[e], f[e], ss); }
#pragma unroll
        for (int off = 1; off < CPR; off <<= 1) ss += __shfl_xor(ss, off);
        const float inv = __builtin_amdgcn_rsqf(ss * (1.0f / d) + eps);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = f[e] * inv * static_cast<float>(g[e]);
        t8 o;
        if (cs != nullptr && split_half) {
            // the partner of chunk c is chunk c ^ (CPR / 2) of the same head row, held by the lane CPR / 2 away; the lower
            // half yields the real parts, the upper half the imaginary parts of the 8 pairs the two chunks form
            const bool upper = dc >= d / 2;
            const int pp = upper ? dc - d / 2 : dc;
            const f32x4 c0 = *reinterpret_cast<const f32x4*>(cs + static_cast<long>(r) * (d / 2) + pp);
            const f32x4 c1 = *reinterpret_cast<const f32x4*>(cs + static_cast<long>(r) * (d / 2) + pp + 4);
            const f32x4 s0 = *reinterpret_cast<const f32x4*>(sn + static_cast<long>(r) * (d / 2) + pp);
            const f32x4 s1 = *reinterpret_cast<const f32x4*>(sn + static_cast<long>(r) * (d / 2) + pp + 4);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float other = __shfl_xor(f[e], CPR / 2);
                const float a = upper ? other : f[e], b = upper ? f[e] : other;
                const float c = e < 4 ? c0[e & 3] : c1[e & 3], sv = e < 4 ? s0[e & 3] : s1[e & 3];
                o[e] = static_cast<T>(upper ? rope_im(a, b, c, sv) : rope_re(a, b, c, sv));
            }
        } else if (cs != nullptr) {
            const f32x4 cv = *reinterpret_cast<const f32x4*>(cs + static_cast<long>(r) * (d / 2) + dc / 2);
            const f32x4 sv = *reinterpret_cast<const f32x4*>(sn + static_cast<long>(r) * (d / 2) + dc / 2);
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                o[2 * p] = static_cast<T>(rope_re(f[2 * p], f[2 * p + 1], cv[p], sv[p]));
                o[2 * p + 1] = static_cast<T>(rope_im(f[2 * p], f[2 * p + 1], cv[p], sv[p]));
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = static_cast<T>(f[e]);
        }
        const u32x4 bits = __builtin_bit_cast(u32x4, o);
        *reinterpret_cast<u32x4*>(out + r * o_rs + col) = bits;
        if (r < out2_rows) *reinterpret_cast<u32x4*>(out2 + r * o2_rs + col) = bits;
    }
}

// The same for head counts that are multiples of 4: a thread takes one chunk position of 4 heads of a row (heads H / 4
// apart, so that for each of the four the lanes of a wavefront touch one contiguous piece of the row), with one fetch of
// the gain and table entries and one index computation for the four, and 4 loads in flight. Same arithmetic per element.
// kRot: 0 no rotation, 1 adjacent pairs, 2 split-half pairs.
template <typename T, int CPR, int kRot>
__global__ void __launch_bounds__(256) headnorm_rope_heads_kernel(const T* x, T* out, T* out2, const T* __restrict__ gain, const float* __restrict__ cs,
                                                                  const float* __restrict__ sn, int rows, float eps, long x_rs, long o_rs, long o2_rs,
                                                                  int out2_rows, RowUnits ru) {
    typedef T t8 __attribute__((ext_vector_type(8)));
    constexpr int d = CPR * 8, HB = 4;
    const int n = ru.rb * ru.units;
    const long quarter = ru.units * 8L;
    for (long block = blockIdx.x; block < ru.blocks; block += gridDim.x)
        for (int t = threadIdx.x; t < n; t += blockDim.x) {
            const int rr = static_cast<int>(__umulhi(t, ru.inv)), u = t - rr * ru.units;
            const long r = block * ru.rb + rr;
            if (r >= rows) break;      // (whole heads: the lanes of a sum stay together)
            const int dc = u % CPR * 8;
            const bool upper = dc >= d / 2;
            const T* const xr = x + r * x_rs + u * 8;
            u32x4 raw[HB];
#pragma unroll
            for (int j = 0; j < HB; ++j) raw[j] = *reinterpret_cast<const u32x4*>(xr + j * quarter);
            const t8 g = __builtin_bit_cast(t8, *reinterpret_cast<const u32x4*>(gain + dc));
            f32x4 c0, c1, s0, s1;
            if constexpr (kRot == 2) {
                const int pp = upper ? dc - d / 2 : dc;
                c0 = *reinterpret_cast<const f32x4*>(cs + r * (d / 2) + pp);
                c1 = *reinterpret_cast<const f32x4*>(cs + r * (d / 2) + pp + 4);
                s0 = *reinterpret_cast<const f32x4*>(sn + r * (d / 2) + pp);
                s1 = *reinterpret_cast<const f32x4*>(sn + r * (d / 2) + pp + 4);
            } else if constexpr (kRot == 1) {
                c0 = *reinterpret_cast<const f32x4*>(cs + r * (d / 2) + dc / 2);
                s0 = *reinterpret_cast<const f32x4*>(sn + r * (d / 2) + dc / 2);
            }
            T* const o_row = out + r * o_rs + u * 8;
#pragma unroll
            for (int j = 0; j < HB; ++j) {
                const t8 v = __builtin_bit_cast(t8, raw[j]);
                float f[8];
                float ss = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) { f[e] = static_cast<float>(v[e]); ss = __builtin_fmaf(f[e], f[e], ss); }
                const float inv = __builtin_amdgcn_rsqf(group_sum<CPR>(ss) * (1.0f / d) + eps);
#pragma unroll
                for (int e = 0; e < 8; ++e) f[e] = f[e] * inv * static_cast<float>(g[e]);
                t8 o;
                if constexpr (kRot == 2) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float other = __shfl_xor(f[e], CPR / 2);
                        const float a = upper ? other : f[e], b = upper ? f[e] : other;
                        const float c = e < 4 ? c0[e & 3] : c1[e & 3], sv = e < 4 ? s0[e & 3] : s1[e & 3];
                        o[e] = static_cast<T>(upper ? rope_im(a, b, c, sv) : rope_re(a, b, c, sv));
                    }
                } else if constexpr (kRot == 1) {
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        o[2 * p] = static_cast<T>(rope_re(f[2 * p], f[2 * p + 1], c0[p], s0[p]));
                        o[2 * p + 1] = static_cast<T>(rope_im(f[2 * p], f[2 * p + 1], c0[p], s0[p]));
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e) o[e] = static_cast<T>(f[e]);
                }
                const u32x4 bits = __builtin_bit_cast(u32x4, o);
                *reinterpret_cast<u32x4*>(o_row + j * quarter) = bits;
                if (r < out2_rows) *reinterpret_cast<u32x4*>(out2 + r * o2_rs + u * 8 + j * quarter) = bits;
            }
        }
}

// out[r][c] = x[r][c] * scale * (row_scale ? row_scale[r] : 1): one thread per 16-byte chunk.
template <typename T>
__global__ void __launch_bounds__(256) scale_rows_kernel(const T* x, T* out, const float* __restrict__ row_scale, float scale,
                                                         int rows, int cols, long x_rs, long o_rs) {
    typedef T t8 __attribute__((ext_vector_type(8)));
    const int cpr = cols / 8;
    const long total = static_cast<long>(rows) * cpr;
    for (long idx = blockIdx.x * 256L + threadIdx.x; idx < total; idx += gridDim.x * 256L) {
        const int r = static_cast<int>(idx / cpr);
        const int col = static_cast<int>(idx - static_cast<long>(r) * cpr) * 8;
        const float f = row_scale ? scale * row_scale[r] : scale;
        t8 v = __builtin_bit_cast(t8, *reinterpret_cast<const u32x4*>(x + r * x_rs + col));
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = static_cast<T>(static_cast<float>(v[e]) * f);
        *reinterpret_cast<u32x4*>(out + r * o_rs + col) = __builtin_bit_cast(u32x4, v);
    }
}

template <typename T>
int launch_headnorm(const mi_headnorm_rope_args* a, long x_rs, long o_rs, long o2_rs, hipStream_t st) {
    const long work = static_cast<long>(a->rows) * a->num_heads * a->head_dim / 8;
    long blocks = (work + 255) / 256;
    if (blocks > 256 * 32) blocks = 256 * 32;
    const T* x = static_cast<const T*>(a->x);
    T* o = static_cast<T*>(a->out);
    T* o2 = static_cast<T*>(a->out2);
    const T* g = static_cast<const T*>(a->gain);
    const int r2 = a->out2 ? a->out2_rows : 0;
    const bool four = a->num_heads % 4 == 0 && static_cast<long>(a->num_heads) * a->head_dim < (1L << 30);
    auto launch_four = [&](auto kernel, int cpr) {
        const RowUnits ru(a->rows, a->num_heads / 4 * cpr);
        hipLaunchKernelGGL(kernel, dim3(ru.grid()), dim3(ru.threads), 0, st, x, o, o2, g, a->cos, a->sin, a->rows, a->eps, x_rs, o_rs, o2_rs, r2, ru);
    };
#define MI_HEADNORM_CASE(CPR)                                                                                          \
    case CPR * 8:                                                                                                      \
        if (four && !a->cos) launch_four(headnorm_rope_heads_kernel<T, CPR, 0>, CPR);                                  \
        else if (four && !a->split_half) launch_four(headnorm_rope_heads_kernel<T, CPR, 1>, CPR);                      \
        else if (four) launch_four(headnorm_rope_heads_kernel<T, CPR, 2>, CPR);                                        \
        else                                                                                                           \
            hipLaunchKernelGGL((headnorm_rope_kernel<T, CPR>), dim3(blocks), dim3(256), 0, st, x, o, o2, g, a->cos,    \
                               a->sin, a->rows, a->num_heads, a->eps, x_rs, o_rs, o2_rs, r2, a->split_half);           \
        break;
    switch (a->head_dim) {
        MI_HEADNORM_CASE(4)
        MI_HEADNORM_CASE(8)
        MI_HEADNORM_CASE(16)
        default: return fail("mi_headnorm_rope: head_dim %d not supported (32, 64, 128)", a->head_dim);
    }
#undef MI_HEADNORM_CASE
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail("mi_headnorm_rope launch: %s", hipGetErrorString(e));
    return 0;
}

template <typename T>
int launch(const mi_rope_args* a, long x_rs, long o_rs, hipStream_t st) {
    const long work = a->split_half ? static_cast<long>(a->rows) * a->num_heads * (a->head_dim / 2)
                                    : static_cast<long>(a->rows) * a->num_heads * a->head_dim / 8;
    long blocks = (work + 255) / 256;
    if (blocks > 256 * 32) blocks = 256 * 32;
    if (blocks < 1) blocks = 1;
    const T* x = static_cast<const T*>(a->x);
    T* o = static_cast<T*>(a->out);
    const uintptr_t al = reinterpret_cast<uintptr_t>(a->x) | reinterpret_cast<uintptr_t>(a->out) | reinterpret_cast<uintptr_t>(a->cos) |
                         reinterpret_cast<uintptr_t>(a->sin);
    if (a->split_half && a->head_dim % 16 == 0 && x_rs % 8 == 0 && o_rs % 8 == 0 && (al & 15u) == 0) {
        long vb = (static_cast<long>(a->rows) * a->num_heads * (a->head_dim / 16) + 255) / 256;
        if (vb > 256 * 32) vb = 256 * 32;
        hipLaunchKernelGGL(rope_split_vec_kernel<T>, dim3(vb), dim3(256), 0, st, x, o, a->cos, a->sin, a->rows, a->num_heads,
                           a->head_dim, x_rs, o_rs, a->per_head);
    } else if (a->split_half) {
        hipLaunchKernelGGL(rope_split_kernel<T>, dim3(blocks), dim3(256), 0, st, x, o, a->cos, a->sin, a->rows,
                           a->num_heads, a->head_dim, x_rs, o_rs, a->per_head);
    } else if (!a->per_head && a->num_heads % 4 == 0 && a->head_dim > 8 && static_cast<long>(a->num_heads) * a->head_dim * a->head_dim < (1L << 31)) {
        // (the inverses hold: units * (d / 8) < 2^23; below two chunks to a head there is nothing to divide)
        const RowUnits ru(a->rows, a->num_heads / 4 * (a->head_dim / 8));
        hipLaunchKernelGGL(rope_adjacent_heads_kernel<T>, dim3(ru.grid()), dim3(ru.threads), 0, st, x, o, a->cos, a->sin, a->rows, a->head_dim, x_rs, o_rs,
                           ru, 0xffffffffu / static_cast<unsigned>(a->head_dim / 8) + 1u);
    } else {
        hipLaunchKernelGGL(rope_adjacent_kernel<T>, dim3(blocks), dim3(256), 0, st, x, o, a->cos, a->sin, a->rows,
                           a->num_heads, a->head_dim, x_rs, o_rs, a->per_head);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail("mi_rope_apply launch: %s", hipGetErrorString(e));
    return 0;
}

}  // namespace
}  // namespace mi

extern "C" int mi_rope_apply(const mi_rope_args* a) {
    using mi::fail;
    mi::clear_error();
    if (!a) return fail("mi_rope_apply: null args");
    if (a->struct_size != sizeof(mi_rope_args)) return fail("mi_rope_apply: struct_size mismatch");
    if (a->rows < 0 || a->num_heads <= 0 || a->head_dim <= 0) return fail("mi_rope_apply: bad shape");
    if (a->rows == 0) return 0;
    if (!a->x || !a->out || !a->cos || !a->sin) return fail("mi_rope_apply: null tensor");
    if (a->head_dim % 2 != 0) return fail("mi_rope_apply: head_dim must be even");
    const long D = static_cast<long>(a->num_heads) * a->head_dim;
    const long x_rs = a->x_row_stride ? a->x_row_stride : D;
    const long o_rs = a->out_row_stride ? a->out_row_stride : D;
    if (x_rs < D || o_rs < D) return fail("mi_rope_apply: row stride smaller than heads*head_dim");
    if (!a->split_half) {
        if (a->head_dim % 8 != 0) return fail("mi_rope_apply: adjacent-pair kernel needs head_dim %% 8 == 0");
        if (x_rs % 8 != 0 || o_rs % 8 != 0) return fail("mi_rope_apply: row strides must be multiples of 8 elements");
        const uintptr_t al = reinterpret_cast<uintptr_t>(a->x) | reinterpret_cast<uintptr_t>(a->out) |
                             reinterpret_cast<uintptr_t>(a->cos) | reinterpret_cast<uintptr_t>(a->sin);
        if (al & 15u) return fail("mi_rope_apply: pointers must be 16-byte aligned");
    }
    hipStream_t st = mi::resolve_stream(a->stream);
    if (a->dtype == MI_DTYPE_BF16) return mi::launch<__bf16>(a, x_rs, o_rs, st);
    if (a->dtype == MI_DTYPE_F16) return mi::launch<_Float16>(a, x_rs, o_rs, st);
    return fail("mi_rope_apply: dtype %d not supported", a->dtype);
}

extern "C" int mi_headnorm_rope(const mi_headnorm_rope_args* a) {
    using mi::fail;
    mi::clear_error();
    if (!a) return fail("mi_headnorm_rope: null args");
    if (a->struct_size != sizeof(mi_headnorm_rope_args)) return fail("mi_headnorm_rope: struct_size mismatch");
    if (a->rows < 0 || a->num_heads <= 0) return fail("mi_headnorm_rope: bad shape");
    if (a->head_dim != 32 && a->head_dim != 64 && a->head_dim != 128)
        return fail("mi_headnorm_rope: head_dim %d not supported (32, 64, 128)", a->head_dim);
    if (a->rows == 0) return 0;
    if (!a->x || !a->out || !a->gain) return fail("mi_headnorm_rope: x, out and gain must not be null");
    if ((a->cos == nullptr) != (a->sin == nullptr)) return fail("mi_headnorm_rope: cos and sin must be given together");
    if (!(a->eps >= 0.f)) return fail("mi_headnorm_rope: eps must be >= 0");
    if (a->out2_rows < 0 || a->out2_rows > a->rows) return fail("mi_headnorm_rope: out2_rows %d outside 0..rows", a->out2_rows);
    if (a->split_half != 0 && a->split_half != 1) return fail("mi_headnorm_rope: split_half must be 0 or 1");
    const long D = static_cast<long>(a->num_heads) * a->head_dim;
    const long x_rs = a->x_row_stride ? a->x_row_stride : D;
    const long o_rs = a->out_row_stride ? a->out_row_stride : D;
    const long o2_rs = a->out2_row_stride ? a->out2_row_stride : D;
    if (x_rs < D || o_rs < D || o2_rs < D) return fail("mi_headnorm_rope: row stride smaller than heads*head_dim");
    if (x_rs % 8 != 0 || o_rs % 8 != 0 || o2_rs % 8 != 0) return fail("mi_headnorm_rope: row strides must be multiples of 8 elements");
    const uintptr_t al = reinterpret_cast<uintptr_t>(a->x) | reinterpret_cast<uintptr_t>(a->out) | reinterpret_cast<uintptr_t>(a->out2) |
                         reinterpret_cast<uintptr_t>(a->gain) | reinterpret_cast<uintptr_t>(a->cos) | reinterpret_cast<uintptr_t>(a->sin);
    if (al & 15u) return fail("mi_headnorm_rope: pointers must be 16-byte aligned");
    hipStream_t st = mi::resolve_stream(a->stream);
    if (a->dtype == MI_DTYPE_BF16) return mi::launch_headnorm<__bf16>(a, x_rs, o_rs, o2_rs, st);
    if (a->dtype == MI_DTYPE_F16) return mi::launch_headnorm<_Float16>(a, x_rs, o_rs, o2_rs, st);
    return fail("mi_headnorm_rope: dtype %d not supported", a->dtype);
}

extern "C" int mi_scale_rows(const mi_scale_rows_args* a) {
    using mi::fail;
    mi::clear_error();
    if (!a) return fail("mi_scale_rows: null args");
    if (a->struct_size != sizeof(mi_scale_rows_args)) return fail("mi_scale_rows: struct_size mismatch");
    if (a->rows < 0 || a->cols <= 0 || a->cols % 8 != 0) return fail("mi_scale_rows: cols must be a positive multiple of 8, rows >= 0");
    if (a->rows == 0) return 0;
    if (!a->x || !a->out) return fail("mi_scale_rows: x and out must not be null");
    const long x_rs = a->x_row_stride ? a->x_row_stride : a->cols;
    const long o_rs = a->out_row_stride ? a->out_row_stride : a->cols;
    if (x_rs < a->cols || o_rs < a->cols || x_rs % 8 != 0 || o_rs % 8 != 0)
        return fail("mi_scale_rows: row strides must be multiples of 8 elements and at least cols");
    if ((reinterpret_cast<uintptr_t>(a->x) | reinterpret_cast<uintptr_t>(a->out)) & 15u) return fail("mi_scale_rows: pointers must be 16-byte aligned");
    if (reinterpret_cast<uintptr_t>(a->row_scale) & 3u) return fail("mi_scale_rows: row_scale must be 4-byte aligned");
    const long work = static_cast<long>(a->rows) * (a->cols / 8);
    long blocks = (work + 255) / 256;
    if (blocks > 256 * 32) blocks = 256 * 32;
    hipStream_t st = mi::resolve_stream(a->stream);
    if (a->dtype == MI_DTYPE_BF16)
        hipLaunchKernelGGL(mi::scale_rows_kernel<__bf16>, dim3(blocks), dim3(256), 0, st, static_cast<const __bf16*>(a->x),
                           static_cast<__bf16*>(a->out), a->row_scale, a->scale, a->rows, a->cols, x_rs, o_rs);
    else if (a->dtype == MI_DTYPE_F16)
        hipLaunchKernelGGL(mi::scale_rows_kernel<_Float16>, dim3(blocks), dim3(256), 0, st, static_cast<const _Float16*>(a->x),
                           static_cast<_Float16*>(a->out), a->row_scale, a->scale, a->rows, a->cols, x_rs, o_rs);
    else
        return fail("mi_scale_rows: dtype %d not supported", a->dtype);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail("mi_scale_rows launch: %s", hipGetErrorString(e));
    return 0;
}
