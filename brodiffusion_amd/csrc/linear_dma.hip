// Y = X W^T + b for large problems on gfx950 (linear_pipe.hip says which): 256 x 256 output tiles, 8 wavefronts, operand blocks moved global -> LDS
// by DMA into rings.
//
// The work group's 512 threads are 8 wavefronts in a 2 (feature halves) x 4 (token quarters) arrangement; a wavefront owns
// 128 features x 64 tokens = 8 x 4 accumulator blocks of v_mfma_f32_16x16x32 (128 registers; linear_pipe.hip says why that one). As in linear.hip the product
// is computed transposed (MFMA rows = features), so both operands are read along their contiguous contraction index.
//
// Operands arrive in blocks of 64 contraction elements: per operand a 256-row x 128-byte tile (32 KB) = 32 LDS-DMA
// instructions of 1 KB (8 rows each: whole 128-byte lines; with 64-byte row pieces the DMA path measured half the
// throughput, 33 instead of 60 bytes per clock and CU, which is no more than this kernel consumes), dealt out four per
// wavefront. An instruction deposits the 16-byte pieces of its 64 lanes back to back, so a tile row is 128 bytes in LDS
// with no padding; bank conflicts of the fragment reads (one row per lane, 16-byte pieces, 16 consecutive rows per phase)
// are avoided by an XOR swizzle applied for free on the global side: the piece that lands in position c of row r is piece
// c ^ ((r >> 1) & 7). X blocks live in a ring of two stages, W blocks in a ring of three (160 KB in all).
//
// A block is multiplied in two half-steps of 32 contraction elements (32 MFMAs per wavefront each). Half-step t of block b:
//   1. the MFMAs, and between the first 24 of them the reads of the 12 fragments of half-step t + 1 into the other register set,
//      between the last 8 this wavefront's 4 DMA instructions: first half of a block: W of block b + 2 (into the stage of W block
//      b - 1); second half: X of block b + 2 (into the stage of X block b, whose fragments are all in registers by now)
//   2. first half: wait until all but this wavefront's 4 youngest DMA instructions have landed (X and W of block b + 1);
//      barrier
// With the reads and the DMA in front of the MFMAs a block took 3078 clocks of which 2048 are products, 2700 to 2890 so. The DMA comes
// in two small bursts, each a whole half-step before what it loads is waited for (one burst of 8 per block measured 25 % slower).
// The accumulators leave through LDS (bias added in FP32, one rounding) so that global stores are full 16-byte pieces of
// consecutive threads along a row. A launch of one tile per CU spends about 11 us outside the loop (bf16, 4096 x 3456 with contractions
// of 576 to 3456: 23.8 to 81.6 us, 1.3 us per block; 25.4 to 90.9 with the half-steps as they were): hence the start after one block
// instead of two, the bias requested ahead of the operands and the write-out in batches of 8 (all three together 1 to 4 %). Rows x
// features x contraction, us, half-steps as they were / as they are, on one GPU: bf16 4096 x 3456 x 1152 37.1 / 34.3, 4608 x 3072 x 3072
// 80.4 / 72.7; fp16 38.2 / 34.5, 83.4 / 74.6.
#include <type_traits>
#include <utility>

#include "internal.h"

namespace mi {
namespace gemm_dma {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct Mma;
template <> struct Mma<__bf16> {
    using v8 = bf16x8;
    using v4 = bf16x4;
    static __device__ __forceinline__ f32x4 run(v8 a, v8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
};
template <> struct Mma<_Float16> {
    using v8 = f16x8;
    using v4 = f16x4;
    static __device__ __forceinline__ f32x4 run(v8 a, v8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
};

constexpr int kTile = 256;                       // tokens and features per work group
constexpr int kBK = 64;                          // contraction elements per block (one stage)
constexpr int kThreads = 512;
constexpr int kOpBytes = kTile * kBK * 2;        // one operand block in LDS
constexpr int kXStages = 2, kWStages = 3;
constexpr int kWRing = kXStages * kOpBytes;      // the W ring starts behind the X ring
constexpr int kOutStride = kTile * 2 + 16;       // staged output row (bytes)
constexpr int kLdsBytes = (kXStages + kWStages) * kOpBytes;
static_assert(kTile * kOutStride <= kLdsBytes, "the staged output fits the rings");
static_assert(kLdsBytes <= 160 * 1024, "LDS of a compute unit");

template <typename T>
__global__ void __launch_bounds__(kThreads, 2) linear_dma_kernel(const LinearBatch batch) {
    using M = Mma<T>;
    using V8 = typename M::v8;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];

    const LinearProblem& p = batch.p[blockIdx.y];
    const int tiles_n = (p.N + kTile - 1) / kTile;
    const int tiles_m = (p.M + kTile - 1) / kTile;
    const int n_tiles = tiles_m * tiles_n;
    // consecutive work-group ids go to the 8 XCDs in turn: give every XCD (one L2) a contiguous run of tiles, which
    // share their X rows and walk W together
    const int chunk = (n_tiles + 7) >> 3;
    // (the grid is sized for the problem of the launch with the most tiles: a smaller problem's run is shorter than the
    //  grid's, and a group past the end of its XCD's run would repeat a tile of the next XCD's)
    const int in_run = static_cast<int>(blockIdx.x) >> 3;
    const int logical = (static_cast<int>(blockIdx.x) & 7) * chunk + in_run;
    if (in_run >= chunk || logical >= n_tiles) return;
    const int m0 = (logical / tiles_n) * kTile, n0 = (logical % tiles_n) * kTile;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, lr = lane & 15, lg = lane >> 4;      // (row of a 16-row block, group of 8 contraction elements)
    const int wn = wave & 1, wm = wave >> 1;

    // ── DMA duty: instructions 4 wave .. 4 wave + 3 of either operand; instruction j fills rows 8 j .. 8 j + 7 ──
    const unsigned char* xg = static_cast<const unsigned char*>(p.x) + static_cast<long>(m0) * p.ldx * 2;
    const unsigned char* wg = static_cast<const unsigned char*>(p.w) + static_cast<long>(n0) * p.ldw * 2;
    unsigned xoff[4], woff[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int j = 4 * wave + u;
        const int r = 8 * j + (lane >> 3);
        const int piece = (lane & 7) ^ ((r >> 1) & 7);
        xoff[u] = static_cast<unsigned>(min(r, p.M - 1 - m0)) * (static_cast<unsigned>(p.ldx) * 2u) + piece * 16u;
        woff[u] = static_cast<unsigned>(min(r, p.N - 1 - n0)) * (static_cast<unsigned>(p.ldw) * 2u) + piece * 16u;
    }
    // the bias of this wavefront's 128 features, two to a lane, requested ahead of everything else (features past the end repeat the
    // last two, their outputs are not stored)
    unsigned bias2 = 0;
    if (p.bias) bias2 = *reinterpret_cast<const unsigned*>(static_cast<const T*>(p.bias) + min(n0 + wn * 128 + 2 * lane, p.N - 2));
    const unsigned lds_base = static_cast<unsigned>(reinterpret_cast<size_t>((__attribute__((address_space(3))) unsigned char*)lds));
    auto dma = [&](unsigned voff, const unsigned char* base, unsigned dst) {
        // (the LDS destination travels in m0; the s_nop is the wait state an LDS-DMA instruction needs behind a write of m0)
        asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(base), "{m0}"(dst) : "memory");
    };
    // instruction u of this wavefront's four of a block; xg / wg stand on that block
    auto dma_x = [&](int stage, int u) { dma(xoff[u], xg, lds_base + stage * kOpBytes + (4 * wave + u) * 1024); };
    auto dma_w = [&](int stage, int u) { dma(woff[u], wg, lds_base + kWRing + stage * kOpBytes + (4 * wave + u) * 1024); };
    auto dma_block = [&](int stage) {
#pragma unroll
        for (int u = 0; u < 4; ++u) dma_x(stage, u);
#pragma unroll
        for (int u = 0; u < 4; ++u) dma_w(stage, u);
        xg += kBK * 2;
        wg += kBK * 2;
    };

    // ── fragment reads: row lr of a 16-row block, 16-byte piece 4 h + lg of the row (swizzled position) ──
    unsigned frag[2];   // [half]
#pragma unroll
    for (int h = 0; h < 2; ++h) frag[h] = lr * 128 + (((4 * h + lg) ^ ((lr >> 1) & 7)) << 4);
    const unsigned x_blk = wm * 64 * 128;                         // this wavefront's first token row, in bytes
    const unsigned w_blk = kWRing + wn * 128 * 128;
    V8 wf[2][8], xf[2][4];   // [register set][block]
    // reads [R0, R1) of the 12 fragments of half-step t (block t / 2, half t % 2) into register set t % 2, in the order in which its
    // products use them: two token blocks, the feature blocks, the other token blocks
    auto read_frags = [&](auto set_tag, auto r0_tag, auto r1_tag, int t) {
        constexpr int S = decltype(set_tag)::value, R0 = decltype(r0_tag)::value, R1 = decltype(r1_tag)::value;
        const int b = t >> 1;
        const unsigned char* xs = lds + (b & 1) * kOpBytes + x_blk;
        const unsigned char* ws = lds + (b % 3) * kOpBytes + w_blk;
        [&]<int... R>(std::integer_sequence<int, R...>) {
            ([&] {
                constexpr int k = R0 + R;
                if constexpr (k >= 2 && k < 10) wf[S][k - 2] = *reinterpret_cast<const V8*>(ws + (k - 2) * 2048 + frag[S]);
                else xf[S][k < 2 ? k : k - 8] = *reinterpret_cast<const V8*>(xs + (k < 2 ? k : k - 8) * 2048 + frag[S]);
            }(), ...);
        }(std::make_integer_sequence<int, R1 - R0>{});
    };

    f32x4 acc[8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int nb = p.K / kBK;      // blocks
    const int nt = 2 * nb;         // half-steps
    // prologue: blocks 0 and 1 requested, block 0 in LDS (block 1 has landed by the first close_half; waiting for it here too
    // made every work group of the launch wait for twice the bytes before its first product)
    dma_block(0);
    if (nb > 1) {
        dma_block(1);
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    } else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    using Set0 = std::integral_constant<int, 0>;
    using Set1 = std::integral_constant<int, 1>;
    read_frags(Set0{}, std::integral_constant<int, 0>{}, std::integral_constant<int, 12>{}, 0);

    // half-step t (set S = t % 2): its 32 products, between them the fragment reads of half-step t + 1 and the DMA of half of the block
    // after next
    auto half_step = [&](auto set_tag, int t) -> bool {
        constexpr int S = decltype(set_tag)::value;
        const int nxt = (t >> 1) + 2;
        const bool more = nxt < nb;
        [&]<int... Q>(std::integer_sequence<int, Q...>) {
            ([&] {
                // (two token blocks at a time, each feature block meets both in a row)
                constexpr int i = (Q >> 1) & 7, j = 2 * (Q >> 4) + (Q & 1);
                acc[i][j] = M::run(wf[S][i], xf[S][j], acc[i][j]);
                if constexpr (Q < 24 && Q % 2 == 1)    // (behind the last half-step: a stage of no block, never used)
                    read_frags(std::integral_constant<int, 1 - S>{}, std::integral_constant<int, Q / 2>{}, std::integral_constant<int, Q / 2 + 1>{}, t + 1);
                else if (Q >= 24 && Q % 2 == 1 && more) {
                    if constexpr (S == 0) dma_w(nxt % 3, Q / 2 - 12);
                    else dma_x(nxt & 1, Q / 2 - 12);
                }
                __builtin_amdgcn_sched_barrier(0);
            }(), ...);
        }(std::make_integer_sequence<int, 32>{});
        if (more) { if constexpr (S == 0) wg += kBK * 2; else xg += kBK * 2; }
        return more;
    };
    auto close_half = [&](auto set_tag, bool more) {
        constexpr int S = decltype(set_tag)::value;
        __builtin_amdgcn_sched_barrier(0);
        // first half of a block: X and W of the next block have landed (everything but the 4 instructions just issued), and
        // this wavefront's fragment reads of the X stage that the next half-step's DMA overwrites have returned
        if constexpr (S == 0) {
            if (more) asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        }
        __builtin_amdgcn_s_barrier();
    };
    for (int t = 0; t < nt; t += 2) {
        const bool m0_ = half_step(Set0{}, t);
        close_half(Set0{}, m0_);
        const bool m1_ = half_step(Set1{}, t + 1);
        close_half(Set1{}, m1_);
    }

    // ── epilogue: acc[i][j][e] is feature wn*128 + 16 i + 4 lg + e of token wm*64 + 16 j + lr ──
    typedef T t2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int feat = wn * 128 + 16 * i + 4 * lg;
        const int src = 4 * (8 * i + 2 * lg);      // byte index of the lane that holds the bias of this and the next feature
        const t2 b01 = __builtin_bit_cast(t2, __builtin_amdgcn_ds_bpermute(src, static_cast<int>(bias2)));
        const t2 b23 = __builtin_bit_cast(t2, __builtin_amdgcn_ds_bpermute(src + 4, static_cast<int>(bias2)));
        const float bv[4] = {static_cast<float>(b01[0]), static_cast<float>(b01[1]), static_cast<float>(b23[0]), static_cast<float>(b23[1])};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            typename M::v4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = static_cast<T>(acc[i][j][e] + bv[e]);
            *reinterpret_cast<typename M::v4*>(lds + (wm * 64 + 16 * j + lr) * kOutStride + feat * 2) = o;
        }
    }
    __syncthreads();
    // (8 pieces read before the first is stored; read and stored one by one, each waited for the one before)
    const int cc = tid & 31;   // 16-byte piece of a row
    const bool in_row = n0 + cc * 8 < p.N;
    const int rows = in_row ? p.M - m0 : 0;
    unsigned char* yg = static_cast<unsigned char*>(p.y) + (static_cast<long>(m0) * p.ldy + n0 + cc * 8) * 2;
    const long step = static_cast<long>(p.ldy) * 2;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        u32x4 v[8];
        const int r0 = half * 128 + (tid >> 5);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = *reinterpret_cast<const u32x4*>(lds + (r0 + 16 * i) * kOutStride + cc * 16);
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (r0 + 16 * i < rows) *reinterpret_cast<u32x4*>(yg + (r0 + 16 * i) * step) = v[i];
    }
}

template <typename T>
int launch_t(const LinearBatch& batch, int n_problems, hipStream_t st) {
    int max_tiles = 0;
    for (int i = 0; i < n_problems; ++i) {
        const LinearProblem& p = batch.p[i];
        max_tiles = max(max_tiles, ((p.M + kTile - 1) / kTile) * ((p.N + kTile - 1) / kTile));
    }
    static thread_local bool raised = false;
    if (!raised) {
        MI_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&linear_dma_kernel<T>), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes));
        raised = true;
    }
    hipLaunchKernelGGL((linear_dma_kernel<T>), dim3(((max_tiles + 7) / 8) * 8, n_problems), dim3(kThreads), kLdsBytes, st, batch);
    MI_HIP_CHECK(hipGetLastError());
    return 0;
}

}  // namespace gemm_dma

int launch_linear_dma(const LinearBatch& batch, int n_problems, int dtype, hipStream_t st) {
    if (dtype == MI_DTYPE_BF16) return gemm_dma::launch_t<__bf16>(batch, n_problems, st);
    if (dtype == MI_DTYPE_F16) return gemm_dma::launch_t<_Float16>(batch, n_problems, st);
    return fail("linear: dtype %d is neither MI_DTYPE_F16 nor MI_DTYPE_BF16", dtype);
}

}  // namespace mi
