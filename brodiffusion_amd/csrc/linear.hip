// Y = X W^T + b for fp16 / bf16 on gfx950: the projection GEMM around the attention core.
//
// X is (M, K) and W is (N, K), both with the contraction index contiguous, which is exactly the operand layout of
// v_mfma_f32_32x32x16: a lane reads 8 consecutive contraction elements of ONE row of either operand. The product is
// computed transposed (MFMA rows = output features, MFMA columns = tokens), so a lane ends up with 4 consecutive
// output features of one token per accumulator group; bias is added in FP32 before the single rounding and the tile
// leaves through LDS as whole 16-byte pieces of rows of Y.
//
// launch_linear validates a launch and hands it to the LDS-DMA kernels of linear_pipe.hip. What those do not take (contractions
// that are no multiple of 64, operands beyond 32-bit tile offsets) runs here:
//
// linear_kernel: 256 threads = 4 wavefronts in a 2 x 2 arrangement over a BM x BN output tile (launch_t picks between two),
// contraction step 64. Operand tiles go global -> registers -> LDS with 16-byte accesses, double buffered so that the
// loads of step t+1 are in flight while step t multiplies; one barrier per step. LDS rows are 144 bytes (128 + 16): 16
// consecutive rows start on distinct 16-byte bank groups, so the ds_read_b128 fragment reads are conflict free.
// Up to three problems share one launch (blockIdx.y): the Q, K and V projections of an attention block.
#include <type_traits>
#include <utility>

#include "linear_math.h"

namespace mi {
namespace gemm {

constexpr int kBK = 64;                // contraction elements per step
constexpr int kRowBytes = kBK * 2 + 16;  // LDS row stride
constexpr int kThreads = 256;

// One 16-byte chunk column (tid % 8) and 32 rows per pass: ROWS / 32 loads per thread and tile.
// GATED (the W tile of the GEGLU form): the tile's 32-row groups alternate between the value half and the gate half
// of W — group 2j holds value features row0 + 32 j .., group 2j+1 the gate rows of the same features (n_rows further
// down) — so that one wavefront's two 32-feature blocks are the value and the gate of the same outputs.
template <int ROWS, bool GATED = false>
__device__ __forceinline__ void load_tile(u32x4 (&r)[ROWS / 32], const char* base, long ld, int row0, int n_rows,
                                          int k0, int K, int tid) {
    const int kc = k0 + (tid & 7) * 8;
    const long col = kc < K ? kc : 0;   // chunks past the end of the contraction are blanked when they are stored
#pragma unroll
    for (int i = 0; i < ROWS / 32; ++i) {
        int row;
        if constexpr (GATED) row = min(row0 + (tid >> 3) + 32 * (i >> 1), n_rows - 1) + (i & 1) * n_rows;
        else row = min(row0 + (tid >> 3) + 32 * i, n_rows - 1);  // rows past the end repeat the last one; never stored
        r[i] = *reinterpret_cast<const u32x4*>(base + (static_cast<long>(row) * ld + col) * 2);
    }
}
// INT8 weight tile: the same 8 contraction elements per thread and row are 8 bytes in memory; they are widened to T
// (exactly: |w| <= 128) on their way to LDS, the per-row scale is applied to the accumulator in the epilogue.
template <int ROWS, bool GATED = false>
__device__ __forceinline__ void load_tile_int8(u32x2 (&raw)[ROWS / 32], const char* base, long ld, int row0, int n_rows,
                                               int k0, int K, int tid) {
    const int kc = k0 + (tid & 7) * 8;
    const long col = kc < K ? kc : 0;
#pragma unroll
    for (int i = 0; i < ROWS / 32; ++i) {
        int row;
        if constexpr (GATED) row = min(row0 + (tid >> 3) + 32 * (i >> 1), n_rows - 1) + (i & 1) * n_rows;   // as in load_tile
        else row = min(row0 + (tid >> 3) + 32 * i, n_rows - 1);
        raw[i] = *reinterpret_cast<const u32x2*>(base + static_cast<long>(row) * ld + col);
    }
}

// Registers -> LDS. Nothing touches the loaded registers before this point, so the wait for the loads sits here,
// behind the MFMAs of the tile that is in LDS, and not where the loads are issued (blanking the chunks past the end
// of the contraction, or widening the weight bytes, right after the load made every step wait out the full memory
// latency before its first MFMA). k_ok: the thread's 8 contraction elements lie inside K.
template <int ROWS>
__device__ __forceinline__ void store_tile(const u32x4 (&r)[ROWS / 32], char* lds, int tid, bool k_ok) {
#pragma unroll
    for (int i = 0; i < ROWS / 32; ++i)
        *reinterpret_cast<u32x4*>(lds + ((tid >> 3) + 32 * i) * kRowBytes + (tid & 7) * 16) = k_ok ? r[i] : u32x4{0u, 0u, 0u, 0u};
}
template <typename T, int ROWS>
__device__ __forceinline__ void store_tile_int8(const u32x2 (&raw)[ROWS / 32], char* lds, int tid, bool k_ok) {
    typedef T t8 __attribute__((ext_vector_type(8)));
    typedef signed char c8 __attribute__((ext_vector_type(8)));
#pragma unroll
    for (int i = 0; i < ROWS / 32; ++i) {
        const c8 q = __builtin_bit_cast(c8, raw[i]);
        t8 w;
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = static_cast<T>(static_cast<float>(q[e]));
        *reinterpret_cast<u32x4*>(lds + ((tid >> 3) + 32 * i) * kRowBytes + (tid & 7) * 16) =
            k_ok ? __builtin_bit_cast(u32x4, w) : u32x4{0u, 0u, 0u, 0u};
    }
}

// The MFMA step and the epilogue of a BM x BN tile held by WM x WN wavefronts. GEGLU: W is (2 N, K) and bias (2 N): value half on top, gate half below; the output (M, N) is
// value * gelu_exact(gate) (diffusers' GEGLU with the erf form of GELU). A work group's 128 W-tile rows are 64 output
// features times {value, gate}; each wavefront holds both accumulators of its 32 features, so the product of the two
// halves never leaves registers and the (M, 2 N) intermediate does not exist.
// W8: W is INT8 (N, K) with one FP32 scale per row (LinearProblem::w_scale): Y = (X Wq^T) * scale + bias.
// GEGLU with W8 (2 N scales): the reference composes this one from its INT8-weight linear layer and a GEGLU pass over a
// 16-bit (M, 2 N) buffer (src/fused_transformer.cu:360-396); here the two halves are rounded to T at the same point,
// in registers, so the result is the composition's without the buffer.
template <typename T, int BM, int BN, bool GEGLU, bool W8, int WM = 2, int WN = 2>
struct TileMath {
    using M = Mma<T>;
    using V4 = typename M::v4;
    static constexpr int NT = 64 * WM * WN;                       // threads: WM x WN wavefronts over tokens x features
    static constexpr int TM = BM / (32 * WM), TN = BN / (32 * WN);  // 32 x 32 blocks per wavefront along tokens / features
    static_assert(!GEGLU || TN == 2, "the GEGLU form pairs the two feature blocks of a wavefront");
    static constexpr int BN_OUT = GEGLU ? BN / 2 : BN;   // output features per tile
    static constexpr int X_BYTES = BM * kRowBytes, W_BYTES = BN * kRowBytes;
    static constexpr int kOutRow = BN_OUT * 2 + 16;      // staged output row (bytes)
    static constexpr int kOutBytes = BM * kOutRow;

    int tid, lq, lh, wm, wn;
    __device__ __forceinline__ explicit TileMath(int tid_) : tid(tid_) {
        const int lane = tid & 63, wave = tid >> 6;
        lq = lane & 31; lh = lane >> 5; wm = wave % WM; wn = wave / WM;
    }
    static __device__ __forceinline__ void clear(f32x16 (&acc)[TN][TM]) {
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int b = 0; b < TM; ++b)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[a][b][e] = 0.f;
    }
    // The bias of this lane's features of the tile at feature n0, requested long before the epilogue (there each of these
    // loads would be a memory latency of its own). Straight-line code: lanes without a bias read the first bytes of W and
    // blank what they got, so that no wait for these loads is placed before the operand loads that follow.
    // GEGLU: [0] = value half, [1] = gate half.
    __device__ __forceinline__ void request_bias(V4 (&braw)[TN][4], const LinearProblem& p, int n0) const {
        const T* bias = static_cast<const T*>(p.bias);
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int feat = GEGLU ? n0 + wn * 32 + 8 * g + 4 * lh : n0 + (wn * TN + a) * 32 + 8 * g + 4 * lh;
                const bool there = bias != nullptr && feat < p.N;
                const T* src = there ? bias + feat + (GEGLU ? a * p.N : 0) : static_cast<const T*>(p.w);
                const V4 raw = *reinterpret_cast<const V4*>(src);
                const V4 zero = {static_cast<T>(0.f), static_cast<T>(0.f), static_cast<T>(0.f), static_cast<T>(0.f)};
                braw[a][g] = there ? raw : zero;
            }
    }
    // the four k-substeps of 16 of one step for every 32 x 32 block of this wavefront, operands from the LDS tile pair at `cur`
    __device__ __forceinline__ void multiply(f32x16 (&acc)[TN][TM], const char* cur) const {
        const char* xs = cur + (wm * TM * 32 + lq) * kRowBytes + lh * 16;
        const char* ws = cur + X_BYTES + (wn * TN * 32 + lq) * kRowBytes + lh * 16;
#pragma unroll
        for (int kk = 0; kk < kBK / 16; ++kk) {
            typename M::v8 xf[TM], wf[TN];
#pragma unroll
            for (int b = 0; b < TM; ++b) xf[b] = *reinterpret_cast<const typename M::v8*>(xs + b * 32 * kRowBytes + kk * 32);
#pragma unroll
            for (int a = 0; a < TN; ++a) wf[a] = *reinterpret_cast<const typename M::v8*>(ws + a * 32 * kRowBytes + kk * 32);
#pragma unroll
            for (int a = 0; a < TN; ++a)
#pragma unroll
                for (int b = 0; b < TM; ++b) acc[a][b] = M::run(wf[a], xf[b], acc[a][b]);
        }
    }
    // acc[a][b][4g + i]: feature n0 + (wn*TN + a)*32 + 8g + 4*lh + i of token m0 + (wm*TM + b)*32 + lq.
    // The results leave through LDS (`stage`, kOutBytes, not in use by anything else): a lane holds 4 features of one token
    // per group, and written from there a wavefront's store instruction would touch 32 rows of Y with 16 bytes each.
    // Staged, consecutive threads write consecutive 16-byte pieces of a row.
    __device__ __forceinline__ void write_tile(const f32x16 (&acc)[TN][TM], const V4 (&braw)[TN][4], const LinearProblem& p, char* stage,
                                               int m0, int n0) const {
        if constexpr (GEGLU) {
            // acc[0] = value, acc[1] = gate of features n0 + wn*32 + 8g + 4*lh + i
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int feat = wn * 32 + 8 * g + 4 * lh;
                float bv[4], bg[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) { bv[i] = static_cast<float>(braw[0][g][i]); bg[i] = static_cast<float>(braw[1][g][i]); }
                float sv[4] = {1.f, 1.f, 1.f, 1.f}, sg[4] = {1.f, 1.f, 1.f, 1.f};
                if constexpr (W8) {
                    if (n0 + feat < p.N) {   // N is a multiple of 8, so the 4 features are in or out together
#pragma unroll
                        for (int i = 0; i < 4; ++i) { sv[i] = p.w_scale[n0 + feat + i]; sg[i] = p.w_scale[p.N + n0 + feat + i]; }
                    }
                }
#pragma unroll
                for (int b = 0; b < TM; ++b) {
                    V4 o;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        float val, gate;
                        if constexpr (W8) {
                            val = static_cast<float>(static_cast<T>(scaled_acc(acc[0][b][4 * g + i], sv[i], bv[i])));
                            gate = static_cast<float>(static_cast<T>(scaled_acc(acc[1][b][4 * g + i], sg[i], bg[i])));
                        } else {
                            val = acc[0][b][4 * g + i] + bv[i];
                            gate = acc[1][b][4 * g + i] + bg[i];
                        }
                        o[i] = static_cast<T>(val * gelu_erf(gate));
                    }
                    *reinterpret_cast<V4*>(stage + ((wm * TM + b) * 32 + lq) * kOutRow + feat * 2) = o;
                }
            }
        } else {
#pragma unroll
            for (int a = 0; a < TN; ++a) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int feat = (wn * TN + a) * 32 + 8 * g + 4 * lh;
                    float bv[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) bv[i] = static_cast<float>(braw[a][g][i]);
                    float sc[4] = {1.f, 1.f, 1.f, 1.f};
                    if constexpr (W8) {
                        if (n0 + feat < p.N) {   // N is a multiple of 8, so the 4 features are in or out together
#pragma unroll
                            for (int i = 0; i < 4; ++i) sc[i] = p.w_scale[n0 + feat + i];
                        }
                    }
#pragma unroll
                    for (int b = 0; b < TM; ++b) {
                        V4 o;
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            if constexpr (W8) o[i] = static_cast<T>(scaled_acc(acc[a][b][4 * g + i], sc[i], bv[i]));
                            else o[i] = static_cast<T>(acc[a][b][4 * g + i] + bv[i]);
                        }
                        *reinterpret_cast<V4*>(stage + ((wm * TM + b) * 32 + lq) * kOutRow + feat * 2) = o;
                    }
                }
            }
        }
        __syncthreads();
        char* yg = static_cast<char*>(p.y);
        constexpr int PPR = BN_OUT / 8;   // 16-byte pieces per staged row
#pragma unroll
        for (int idx = tid; idx < BM * PPR; idx += NT) {
            const int row = idx / PPR, piece = idx % PPR;
            if (m0 + row < p.M && n0 + piece * 8 < p.N)
                *reinterpret_cast<u32x4*>(yg + (static_cast<long>(m0 + row) * p.ldy + n0 + piece * 8) * 2) =
                    *reinterpret_cast<const u32x4*>(stage + row * kOutRow + piece * 16);
        }
    }
};

// One work group per output tile, one contraction step prefetched while the previous one is multiplied.
template <typename T, int BM, int BN, bool GEGLU = false, bool W8 = false>
__global__ __launch_bounds__(kThreads) void linear_kernel(const LinearBatch batch) {
    using TM_ = TileMath<T, BM, BN, GEGLU, W8>;
    constexpr int TM = TM_::TM, TN = TM_::TN, BN_OUT = TM_::BN_OUT, X_BYTES = TM_::X_BYTES, W_BYTES = TM_::W_BYTES;
    static_assert(TM_::kOutBytes <= 2 * (X_BYTES + W_BYTES), "the staged output fits the operand buffers");
    extern __shared__ __attribute__((aligned(16))) char lds[];  // [2][X tile ; W tile]

    const LinearProblem& p = batch.p[blockIdx.y];
    const int tiles_n = (p.N + BN_OUT - 1) / BN_OUT;
    const int tiles_m = (p.M + BM - 1) / BM;
    if (static_cast<int>(blockIdx.x) >= tiles_m * tiles_n) return;  // uniform: this problem has fewer tiles than the grid
    const int m0 = (blockIdx.x / tiles_n) * BM, n0 = (blockIdx.x % tiles_n) * BN_OUT;

    const int tid = threadIdx.x;
    const TM_ tm(tid);
    const char* xg = static_cast<const char*>(p.x);
    const char* wg = static_cast<const char*>(p.w);

    f32x16 acc[TN][TM];
    TM_::clear(acc);
    typename TM_::V4 braw[TN][4];
    tm.request_bias(braw, p, n0);

    // While tile t is multiplied out of LDS, tile t + 1 is on its way into registers; it goes to the other LDS buffer at
    // the end of the step. (The loads stay under `if (more)`: issued unconditionally, the compiler sinks them behind
    // the MFMAs, next to the store, and the step waits out the memory latency again. A second register set, two tiles
    // ahead, and 256 x 256 tiles with 8 wavefronts measured no faster.)
    u32x4 xr[BM / 32];
    u32x4 wr[W8 ? 1 : BN / 32];
    u32x2 wr8[W8 ? BN / 32 : 1];
    auto load_tiles = [&](int k0) {
        load_tile<BM>(xr, xg, p.ldx, m0, p.M, k0, p.K, tid);
        if constexpr (W8) load_tile_int8<BN, GEGLU>(wr8, wg, p.ldw, n0, p.N, k0, p.K, tid);
        else load_tile<BN, GEGLU>(wr, wg, p.ldw, n0, p.N, k0, p.K, tid);
    };
    auto store_tiles = [&](char* dst, int k0) {
        const bool k_ok = k0 + (tid & 7) * 8 < p.K;
        store_tile<BM>(xr, dst, tid, k_ok);
        if constexpr (W8) store_tile_int8<T, BN>(wr8, dst + X_BYTES, tid, k_ok);
        else store_tile<BN>(wr, dst + X_BYTES, tid, k_ok);
    };
    load_tiles(0);
    store_tiles(lds, 0);
    __syncthreads();

    const int n_steps = (p.K + kBK - 1) / kBK;
    for (int t = 0; t < n_steps; ++t) {
        const char* cur = lds + (t & 1) * (X_BYTES + W_BYTES);
        char* nxt = lds + ((t + 1) & 1) * (X_BYTES + W_BYTES);
        const bool more = t + 1 < n_steps;
        if (more) load_tiles((t + 1) * kBK);
        tm.multiply(acc, cur);
        if (more) store_tiles(nxt, (t + 1) * kBK);
        __syncthreads();
    }
    tm.write_tile(acc, braw, p, lds, m0, n0);
}

template <typename T, int BM, int BN, bool GEGLU = false, bool W8 = false>
int launch_tiles(const LinearBatch& batch, int n_problems, hipStream_t st) {
    constexpr int BN_OUT = GEGLU ? BN / 2 : BN;
    int max_tiles = 0;
    for (int i = 0; i < n_problems; ++i) {
        const LinearProblem& p = batch.p[i];
        max_tiles = max(max_tiles, ((p.M + BM - 1) / BM) * ((p.N + BN_OUT - 1) / BN_OUT));
    }
    constexpr size_t lds = 2 * static_cast<size_t>(BM + BN) * kRowBytes;
    static_assert(lds <= 160 * 1024, "operand ring exceeds the LDS of a compute unit");
    // (launched by name: a launch through a pointer variable is dropped by this compiler when the host code is built with
    // -fsanitize=undefined)
    const void* const kern = reinterpret_cast<const void*>(&linear_kernel<T, BM, BN, GEGLU, W8>);
    if (lds > 64 * 1024) {
        static thread_local bool raised = false;
        if (!raised) {
            MI_HIP_CHECK(hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
            raised = true;
        }
    }
    hipLaunchKernelGGL((linear_kernel<T, BM, BN, GEGLU, W8>), dim3(max_tiles, n_problems), dim3(kThreads), lds, st, batch);
    MI_HIP_CHECK(hipGetLastError());
    return 0;
}

template <typename T>
int launch_t(const LinearBatch& batch, int n_problems, hipStream_t st, bool geglu) {
    const bool w8 = batch.p[0].w_scale != nullptr;
    // 128 tokens x 128 rows of W per tile where such tiles give every compute unit two: they read half as much per FLOP, and below
    // that the 64-token tiles fill the GPU better. The lines are the same for 16-bit and INT8 weights, plain and GEGLU, and any
    // contraction (us, 64-token / 128-token tiles, plain fp16):
    //   256 tiles: 2048 x 2048 x 328 10.1 / 10.1, x 1096 24.5 / 22.5 (INT8 24.0 / 31.1)
    //   512:       4096 x 2048 x 136 10.5 / 10.2, x 328 17.0 / 13.8, x 1096 44.7 / 29.9 (INT8 44.0 / 34.3; GEGLU 39.6 / 30.9)
    //   2048:      8192 x 4096 x 136 32.6 / 29.5, x 1096 164 / 108, x 2056 302 / 189
    long big = 0;
    for (int i = 0; i < n_problems; ++i)
        big += static_cast<long>((batch.p[i].M + 127) / 128) * ((batch.p[i].N + (geglu ? 63 : 127)) / (geglu ? 64 : 128));
    if (big >= 2L * device_cu_count()) {
        if (geglu) return w8 ? launch_tiles<T, 128, 128, true, true>(batch, 1, st) : launch_tiles<T, 128, 128, true>(batch, 1, st);
        return w8 ? launch_tiles<T, 128, 128, false, true>(batch, n_problems, st) : launch_tiles<T, 128, 128>(batch, n_problems, st);
    }
    if (geglu) return w8 ? launch_tiles<T, 64, 128, true, true>(batch, 1, st) : launch_tiles<T, 64, 128, true>(batch, 1, st);
    return w8 ? launch_tiles<T, 64, 64, false, true>(batch, n_problems, st) : launch_tiles<T, 64, 64>(batch, n_problems, st);
}

}  // namespace gemm

int launch_linear(const LinearBatch& batch, int n_problems, int dtype, hipStream_t st, bool geglu) {
    if (geglu && n_problems != 1) return fail("linear: the GEGLU form takes one problem per launch");
    if (n_problems < 1 || n_problems > kMaxLinearProblems) return fail("linear: %d problems in one launch (1..%d)", n_problems, kMaxLinearProblems);
    for (int i = 0; i < n_problems; ++i) {
        const LinearProblem& p = batch.p[i];
        if (p.M <= 0 || p.N <= 0 || p.K <= 0) return fail("linear: empty problem %d (%d x %d x %d)", i, p.M, p.N, p.K);
        if (p.N % 8 || p.K % 8) return fail("linear: in_features %d and out_features %d must be multiples of 8", p.K, p.N);
        if ((p.w_scale != nullptr) != (batch.p[0].w_scale != nullptr)) return fail("linear: INT8 and 16-bit weights cannot share a launch");
        if (reinterpret_cast<uintptr_t>(p.w_scale) & 3u) return fail("linear: weight scales must be 4-byte aligned");
        if (p.ldx % 8 || p.ldw % 8 || p.ldy % 8) return fail("linear: row strides must be multiples of 8 elements");
        if (p.ldx < p.K || p.ldw < p.K || p.ldy < p.N) return fail("linear: a row stride is smaller than the row");
        const uintptr_t al = reinterpret_cast<uintptr_t>(p.x) | reinterpret_cast<uintptr_t>(p.w) |
                             reinterpret_cast<uintptr_t>(p.y) | reinterpret_cast<uintptr_t>(p.bias);
        if (!p.x || !p.w || !p.y) return fail("linear: null operand in problem %d", i);
        if (al & 15u) return fail("linear: operands must be 16-byte aligned");
        if (static_cast<long>((p.M + 63) / 64) * ((p.N + 63) / 64) > 0x7fffffffL) return fail("linear: problem too large for one launch");
    }
    if (dtype != MI_DTYPE_BF16 && dtype != MI_DTYPE_F16) return fail("linear: dtype %d is neither MI_DTYPE_F16 nor MI_DTYPE_BF16", dtype);
    if (linear_pipe_takes(batch, n_problems, geglu)) return launch_linear_pipe(batch, n_problems, dtype, geglu, st);
    if (dtype == MI_DTYPE_BF16) return gemm::launch_t<__bf16>(batch, n_problems, st, geglu);
    if (dtype == MI_DTYPE_F16) return gemm::launch_t<_Float16>(batch, n_problems, st, geglu);
    return fail("linear: dtype %d is neither MI_DTYPE_F16 nor MI_DTYPE_BF16", dtype);
}

}  // namespace mi
