// What the two kernels for wide heads (sdpa_wide.hip, sdpa_wide_long.hip) share: work-group shape, LDS and scratch layout, and the
// output accumulators, which live in accumulation registers by name.
#pragma once
#include "sdpa_tiles.h"
#include "sdpa_wide_plan.h"

namespace mi {
namespace sdpa {

constexpr int kWideThreads = 256;

template <int D> struct WideGeo {
    using G = HeadGeo<D>;
    static constexpr int ROWB = D * 2;                  // bytes per row in LDS
    static constexpr int TILE = kWideKeys * ROWB;       // one operand stage
    static constexpr int VOFF = 2 * TILE;               // the V stages follow the K stages
    static constexpr int NDMA = TILE / 1024 / 4;        // DMA instructions per wavefront and operand tile
    static constexpr int STAGED = kWideRows * G::O_STRIDE;   // the staged Q tile, later the staged output, over the rings
    static constexpr int LDS_BYTES = 4 * TILE > STAGED ? 4 * TILE : STAGED;
    static_assert(D % 128 == 0 && TILE % 4096 == 0, "whole swizzle groups per row, whole DMA instructions per wavefront");
    static_assert(LDS_BYTES <= 160 * 1024, "one work group must fit the LDS of a compute unit");
    // A partial result, FP32: the accumulators of the four wavefronts, 16 bytes a lane (piece (w D / 8 + c) 64 + 32 u + n: head-dim
    // elements 8 c + 4 u .. + 3 of row 32 w + n), then 128 references and 128 denominators
    static constexpr long SLOT = static_cast<long>(kWideRows) * (D * 4 + 8);
};

// For every statement that touches the accumulation registers: all of them are declared clobbered, so that the compiler keeps
// nothing of its own there.
#define MI_A10(t) "a" #t "0", "a" #t "1", "a" #t "2", "a" #t "3", "a" #t "4", "a" #t "5", "a" #t "6", "a" #t "7", "a" #t "8", "a" #t "9"
#define MI_AGPRS                                                                                                              \
    "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", MI_A10(1), MI_A10(2), MI_A10(3), MI_A10(4), MI_A10(5),       \
        MI_A10(6), MI_A10(7), MI_A10(8), MI_A10(9), MI_A10(10), MI_A10(11), MI_A10(12), MI_A10(13), MI_A10(14), MI_A10(15),  \
        MI_A10(16), MI_A10(17), MI_A10(18), MI_A10(19), MI_A10(20), MI_A10(21), MI_A10(22), MI_A10(23), MI_A10(24), "a250",  \
        "a251", "a252", "a253", "a254", "a255"
template <int R> __device__ __forceinline__ float o_get() {
    float f;
    asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(f) : "n"(R) : MI_AGPRS);
    return f;
}
template <int R> __device__ __forceinline__ void o_set(float f) { asm volatile("v_accvgpr_write_b32 a[%1], %0" : : "v"(f), "n"(R) : MI_AGPRS); }
// O = 0
template <int N> __device__ __forceinline__ void o_clear() {
    [&]<int... I>(std::integer_sequence<int, I...>) { (o_set<I>(0.f), ...); }(std::make_integer_sequence<int, N>{});
}

}  // namespace sdpa
}  // namespace mi
