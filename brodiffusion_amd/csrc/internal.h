// Internal declarations shared by the translation units of libmi_attention.so.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>

#include "mi_attention.h"

namespace mi {

// Records the message mi_last_error() returns for this thread; always returns -1.
int fail(const char* fmt, ...) __attribute__((format(printf, 1, 2)));
void clear_error();
hipStream_t resolve_stream(void* s);
// Compute units of the current device (cached per thread; 256 if the query fails).
int device_cu_count();

#define MI_HIP_CHECK(expr)                                                          \
    do {                                                                            \
        hipError_t _e = (expr);                                                     \
        if (_e != hipSuccess) return ::mi::fail("%s: %s", #expr, hipGetErrorString(_e)); \
    } while (0)

// Split of the last, partly filled round of an attention launch without a mask other than a key mask.
//
// A launch of n_blocks equal query tiles on a GPU that runs n_cu work groups at a time takes ceil(n_blocks / n_cu)
// rounds even when the last round fills only part of the GPU (432 tiles on 256 compute units: 2 rounds for 1.69
// rounds of work). With the split, the tiles of the full rounds are processed whole and the tiles of the last round
// are cut along the KEY axis into as many equal pieces as there are work-group slots; a piece covers the end of one
// tile and the start of the next, each part leaves its output accumulators and softmax statistics, all FP32, in a
// scratch slot, and a small second kernel merges the parts of every tile. Everything is done per XCD group (work
// groups whose id is g mod 8 share an L2): group g owns the logical tiles [g*chunk, (g+1)*chunk) and cu_g work-group
// slots. All quantities are counted in key tiles of 64 keys ("steps"); T is the number of steps of one query tile.
struct SplitGeo {
    int enabled;
    int T, chunk, n_blocks, cu_g;
    int max_tail;   // most tail tiles of any group
    int max_parts;  // partial slots per tail tile
    int min_visible;  // under a key mask: a query tile with fewer visible key tiles than this is not cut, its first part takes it whole
    static constexpr int kMinPiece = 8;   // shortest piece worth a work group of its own, in steps
    __host__ __device__ int tiles_of(int g) const { const int n = n_blocks - g * chunk; return n < 0 ? 0 : (n > chunk ? chunk : n); }
    __host__ __device__ int full_of(int g) const { return tiles_of(g) / cu_g * cu_g; }
    __host__ __device__ int tail_of(int g) const { return tiles_of(g) - full_of(g); }
    // pieces the tail steps S of a group are cut into
    __host__ __device__ int pieces_for(int S) const {
        if (S <= 0) return 0;
        const int np = S / kMinPiece;
        return np < 1 ? 1 : (np > cu_g ? cu_g : np);
    }
    // piece c of np covers tail steps [piece_begin(c), piece_begin(c + 1))
    __host__ __device__ static int piece_begin(int c, int S, int np) { return static_cast<int>(static_cast<long>(c) * S / np); }
    // the piece that holds tail step x
    __host__ __device__ static int piece_of(int x, int S, int np) { return static_cast<int>((static_cast<long>(x + 1) * np + S - 1) / S) - 1; }
    // bytes of one partial slot, FP32: 256 rows of head_dim values, then 256 references and 256 denominators
    __host__ __device__ static long slot_bytes(int head_dim) { return 256L * head_dim * 4 + 256L * 8; }
};

// Device-side view of one softmax-attention launch. Strides in elements.
struct SdpaDev {
    const void* q; const void* k; const void* v; void* o;
    const void* kp; const void* vp;
    int B, H, Lq, Lk, Lp;  // Lk = Lp + fresh rows
    int kv_group;          // query heads per K/V head
    long q_rs, q_bs, k_rs, k_bs, v_rs, v_bs, o_rs, o_bs, kp_rs, kp_bs, vp_rs, vp_bs;
    float scale_log2;      // scale * log2(e)
    int mask_mode, q_offset, window;
    const int* kv_valid_len;
    const float* key_mask; long key_mask_bs;
    int n_seg;
    int seg_q_end[MI_MAX_SEGMENTS];
    int seg_k_end[MI_MAX_SEGMENTS];
    int seg_causal[MI_MAX_SEGMENTS];
    const float* cos_q; const float* sin_q;
    const float* cos_k; const float* sin_k;
    int rope_split;               // 0: adjacent pairs, 1: the two halves of a head (Q only: K then arrives rotated)
    int n_q_tiles; int n_blocks;  // logical work items = B*H*n_q_tiles
    // additive logit bias (natural-log units, added to the scaled score) for query rows >= bias_q0 and keys < bias_cols
    const float* bias; int bias_q0, bias_cols; long bias_rs;
    int bias_vec_ok;              // bias base 16-byte aligned and bias_rs a multiple of 4: rows can be read 4 floats at a time
    float inv_scale;              // 1 / scale: the bias in units of the raw dot product
    const int* cu_q; const int* cu_k;   // packed variable-length sequences: [B + 1] row offsets, or null
    float* lse;                   // [B][H][Lq] base-2 log of the softmax denominator in exponent units, or null
    int prefix_scaled;            // the rows of the cached prefix carry factors: K rows pk_scale * pk_row[j], V rows pv_scale * pv_row[j]
    float pk_scale, pv_scale;
    const float* pk_row; const float* pv_row;   // [Lp] or null
    int kbits_off;                // byte offset in dynamic LDS of the key-visibility words (256-row kernels with a key mask)
    SplitGeo split;               // enabled != 0: split the last round along the key axis
    unsigned char* split_scratch; // partial slots, [8 groups][max_tail][max_parts] of SplitGeo::slot_bytes
    size_t split_scratch_bytes;   // what the caller lent
};

// One rotation, written with explicit fused multiply-adds so that every kernel that rotates
// (stand-alone pass, Q load, K tile load) rounds identically: (a + ib)(c + is).
__device__ __forceinline__ float rope_re(float a, float b, float c, float s) { return __builtin_fmaf(a, c, -(b * s)); }
__device__ __forceinline__ float rope_im(float a, float b, float c, float s) { return __builtin_fmaf(a, s, b * c); }

// 0 = pick by problem size, 1 = 128-row kernel, 2 = 256-row ping-pong kernel (mi_sdpa_set_kernel_choice).
int sdpa_kernel_choice();

int launch_sdpa(const SdpaDev& p, int dtype, int head_dim, hipStream_t stream);
// Scratch bytes with which launch_sdpa would split the last round of this launch (0: it would not split).
size_t sdpa_split_scratch_bytes(const SdpaDev& p, int dtype, int head_dim);
bool sdpa_supported(int dtype, int head_dim);
// Head dimensions 256, 384 and 512 (sdpa_wide.hip): 128-row query tiles, the key axis in pieces when a scratch is lent.
bool sdpa_wide_head(int head_dim);
size_t sdpa_wide_split_scratch_bytes(const SdpaDev& p, int head_dim);
int launch_sdpa_wide(const SdpaDev& p, int dtype, int head_dim, hipStream_t stream);
// head_dim 512, long calls: the launch alone, planned and merged by launch_sdpa_wide
int launch_sdpa_wide_long(const SdpaDev& p, bool bf16, int n_q_tiles, int n_split, int n_blocks, hipStream_t stream);

// Calls with few query rows (sdpa_small.hip) and unmasked ones of some sizes (sdpa_flow.hip): whether the kernel takes a call at kernel
// choice 0, and the launch.
bool sdpa_small_takes(const SdpaDev& p, int head_dim);
bool sdpa_flow_runs(const SdpaDev& p);
bool sdpa_flow_takes(const SdpaDev& p, int head_dim, int n_cu);
int launch_sdpa_flow(const SdpaDev& p, int dtype, int head_dim, int n_cu, bool short_keys, hipStream_t stream);   // short_keys: the keys fit LDS
int launch_sdpa_small(const SdpaDev& p, int dtype, int head_dim, hipStream_t stream);

// Device-side view of the head-averaged attention map launch (batch 1).
struct MapDev {
    const void* q; const void* k;
    const float* lse;             // [H][Lq], as written by the attention launch
    float* map;                   // (Lq, Lk) FP32
    int H, Lq, Lk;
    long q_rs, k_rs, map_rs;
    float scale_log2;
    const float* bias; int bias_q0, bias_cols; long bias_rs;
    const float* key_mask;        // [Lk] or null
};
int launch_attention_map(const MapDev& p, int dtype, int head_dim, hipStream_t stream);

// Whether two 16-bit operands of `batch` items of `rows` rows of `len` elements (row strides of at least a row, any batch strides, in
// elements) can share an element. Column slices of one buffer share none; where strides differ, overlapping address ranges count.
inline bool operands_overlap(const void* a, long a_rs, long a_bs, const void* b, long b_rs, long b_bs, long batch, long rows, long len) {
    auto reach = [&](long rs, long bs, long& first, long& last) {
        const long items = (batch - 1) * bs;
        first = items < 0 ? items : 0;
        last = (items > 0 ? items : 0) + (rows - 1) * rs + len;
    };
    long a0, a1, b0, b1;
    reach(a_rs, a_bs, a0, a1);
    reach(b_rs, b_bs, b0, b1);
    const long apart = (static_cast<long>(reinterpret_cast<intptr_t>(a)) - static_cast<long>(reinterpret_cast<intptr_t>(b))) / 2;      // elements from b to a
    if (apart + a0 >= b1 || apart + a1 <= b0) return false;
    if (a_rs != b_rs || (batch > 1 && (a_bs % a_rs != 0 || b_bs % a_rs != 0))) return true;
    const long column = (apart % a_rs + a_rs) % a_rs;      // a's first column among b's
    return column < len || column > a_rs - len;
}

// One Y = X W^T + bias problem: X (M, K), W (N, K), Y (M, N), bias (N) or null; strides in elements.
struct LinearProblem {
    const void* x; const void* w; const void* bias; void* y;
    const float* w_scale;   // non-null: w is INT8 (N, K) with one FP32 scale per row, Y = (X Wq^T) * scale + bias
    int M, N, K;
    long ldx, ldw, ldy;
};
constexpr int kMaxLinearProblems = 3;
struct LinearBatch { LinearProblem p[kMaxLinearProblems]; };
// Validates and launches up to kMaxLinearProblems problems as one grid.
// geglu: problem 0 has W (2 N, K) and bias (2 N), value half first; Y (M, N) = value * gelu_exact(gate).
int launch_linear(const LinearBatch& batch, int n_problems, int dtype, hipStream_t stream, bool geglu = false);
// The forms with LDS-DMA operand rings: whether they take a validated launch, and the launch (linear_pipe.hip); the one with
// 256 x 256 tiles (linear_dma.hip).
bool linear_pipe_takes(const LinearBatch& batch, int n_problems, bool geglu);
int launch_linear_pipe(const LinearBatch& batch, int n_problems, int dtype, bool geglu, hipStream_t stream);
int launch_linear_dma(const LinearBatch& batch, int n_problems, int dtype, hipStream_t stream);

// Cross-attention to cached keys with its query projection in the same launch (sdpa_small.hip): p.q is not read, q projects batch * Lq
// rows to H * head_dim columns (q.y is not written).
bool sdpa_projected_takes(const SdpaDev& p, const LinearProblem& q, int head_dim);
int launch_sdpa_projected(const SdpaDev& p, const LinearProblem& q, int dtype, int head_dim, hipStream_t stream);

}  // namespace mi
