// Flash-style softmax attention forward for gfx950 (MI355X), hand-written. Four kernels share the building blocks of
// sdpa_common.h; launch_d picks one per call that sdpa_small.hip and sdpa_flow.hip do not take:
//
//   sdpa_fwd_kernel         4 wavefronts = 128 query rows per work group, K/V tiles through registers into padded LDS,
//                           double buffered. Few keys or few work groups (rows256_pay) with extras or masks, packed
//                           variable-length sequences, head_dim 160 with any of these, extras together with the prefix dial or tile-wise K rotation.
//   sdpa_fwd_pp_kernel      8 wavefronts = 256 query rows, 2 wavefronts per SIMD, one work-group barrier per key tile:
//                           between two barriers every wavefront runs the MFMA stream (O += V^T P of tile t, then
//                           S = K Q^T of tile t+1) and one softmax, in opposite order in the two groups of four, so the
//                           matrix pipe and the VALU of a SIMD are busy at the same time.
//   sdpa_fwd_pp_dma_kernel  the same schedule with K/V tiles moved global -> LDS by DMA (head_dim 72 and 128), optionally
//                           with the last, partly filled round of work groups cut along the key axis (SPLIT) and merged
//                           by sdpa_combine_kernel.
//   sdpa_shortkv_kernel     short key sequences (cross attention): K and V of a head stay in LDS, a work group walks
//                           several query tiles, no barrier in the key loop.
//
// Not in HBM: scores, probabilities, rotated Q (RoPE is applied as Q is loaded; K either the same way or by one pass into
// a caller scratch), the [prefix ; fresh] K/V concatenation (two source pointers), any mask tensor (per-row visible-key
// intervals; key tiles outside every row's interval are skipped).
#include <type_traits>

#include "sdpa_tiles.h"

namespace mi {
namespace {

using namespace sdpa;


// ───────────────────────────── 4-wavefront kernel ─────────────────────────────
constexpr int kThreads4 = 256;
template <int D> constexpr int lds_bytes_4() {
    using G = HeadGeo<D>;
    const int kv = 2 * (G::K_BYTES + G::V_BYTES + kBN * 4);
    const int o = 128 * G::O_STRIDE;
    return kv > o ? kv : o;
}

// VARLEN: the batch items are sequences of different lengths packed back to back along the row axis
// (cu_q / cu_k: device arrays of batch + 1 row offsets, the cu_seqlens convention); Lq and Lk of the launch are the
// longest sequence and only size the grid. Each work group rebuilds the launch view for its own sequence.
// PSCALE: the rows of the cached prefix carry factors (the prefix-KV dial); a separate instance so that the code for it
// costs the other instances no registers.
template <typename T, int D, bool ROPE_K, bool VARLEN = false, bool PSCALE = false>
__global__ void __launch_bounds__(kThreads4, (D > 128 ? 1 : 2)) sdpa_fwd_kernel(const SdpaDev p_in) {
    using G = HeadGeo<D>;
    using V8 = typename Mma<T>::v8;
    constexpr int BM = 128;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    __shared__ int red[8];
    constexpr int STAGE = G::K_BYTES + G::V_BYTES + kBN * 4;   // K tile, V tile, 64 key-mask floats

    int qt, bh;
    if (!block_to_tile(p_in, qt, bh)) return;
    const int h = bh % p_in.H;
    const SdpaDev& p = p_in;
    // this work group's sequence: row offsets into the packed tensors, its own lengths and causal offset
    int b = bh / p.H, Lq = p.Lq, Lk = p.Lk, q_offset = p.q_offset;
    long q_row0 = 0, k_row0 = 0;
    if constexpr (VARLEN) {
        const int qs = p.cu_q[b], ks = p.cu_k[b];
        Lq = p.cu_q[b + 1] - qs;
        Lk = p.cu_k[b + 1] - ks;
        if (qt * BM >= Lq) return;
        q_row0 = qs; k_row0 = ks;
        q_offset = Lk - Lq;   // causal: the last query meets the last key, per sequence
        b = 0;                // batch strides do not apply to packed rows
    }

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform, kept in a scalar register
    const int lane = tid & 63;
    const int lq = lane & 31;
    const int lh = lane >> 5;
    const int q0 = qt * BM;
    const int qrow = q0 + wave * 32 + lq;
    const bool qvalid = qrow < Lq;
    const int hk = h / p.kv_group;
    const T* const q_base = static_cast<const T*>(p.q) + b * p.q_bs + q_row0 * p.q_rs + h * D;
    T* const o_base = static_cast<T*>(p.o) + b * p.o_bs + q_row0 * p.o_rs + h * D;
    const float* const key_mask = p.key_mask ? p.key_mask + b * p.key_mask_bs : nullptr;
    const float* const bias_row = (p.bias && qvalid && qrow >= p.bias_q0) ? p.bias + static_cast<long>(qrow - p.bias_q0) * p.bias_rs : nullptr;

    int lo, hi;
    if constexpr (VARLEN) {
        lo = 0;
        hi = p.mask_mode == MI_MASK_CAUSAL ? min(Lk, q_offset + qrow + 1) : Lk;
        if (!qvalid || hi <= lo) { lo = 0; hi = 0; }
    } else {
        row_interval(p, b, min(qrow, p.Lq - 1), q0 + wave * 32 < p.Lq, lo, hi);
    }
    const WaveExtent we = wave_extent(lo, hi);
    if (lane == 0) { red[wave] = we.lo_min; red[4 + wave] = we.hi_max; }
    V8 qf[G::KC];
    stage_q_tile<T, D, kThreads4, BM>(smem, p, q_base, q0, tid, 1.f, Lq - 1);
    __syncthreads();
    read_q_frags<T, D>(qf, smem, wave * 32 + lq, lh);
    __syncthreads();
    zero_pads<D, kThreads4>(smem, smem + G::K_BYTES, STAGE, STAGE, 2, tid);
    __syncthreads();
    const int g_lo = __builtin_amdgcn_readfirstlane(min(min(red[0], red[1]), min(red[2], red[3])));
    const int kv_stop = __builtin_amdgcn_readfirstlane(max(max(red[4], red[5]), max(red[6], red[7])));
    const TilePlan plan(g_lo == 0x7fffffff ? 0 : g_lo, kv_stop, p.Lp);

    f32x16 oacc[G::VB];
#pragma unroll
    for (int vb = 0; vb < G::VB; ++vb)
#pragma unroll
        for (int e = 0; e < 16; ++e) oacc[vb][e] = 0.f;
    SoftmaxState st;
    const float cl2 = p.scale_log2;
    const float lazy_raw = kLazyLog2 / cl2;

    TileMover<T, D, kThreads4, ROPE_K> mv{p, plan,
                                          reinterpret_cast<const unsigned char*>(static_cast<const T*>(p.k) + b * p.k_bs + k_row0 * p.k_rs + hk * D),
                                          reinterpret_cast<const unsigned char*>(static_cast<const T*>(p.v) + b * p.v_bs + k_row0 * p.v_rs + hk * D),
                                          reinterpret_cast<const unsigned char*>(static_cast<const T*>(p.kp) + b * p.kp_bs + hk * D),
                                          reinterpret_cast<const unsigned char*>(static_cast<const T*>(p.vp) + b * p.vp_bs + hk * D),
                                          tid, {}, {}, 1.f};

    // key loop, LDS double buffered: one barrier per tile
    const int n_tiles = plan.n_tiles;
    if (n_tiles > 0) {
        mv.template issue<0>(0);
        mv.template issue<1>(0);
        if (key_mask) mv.issue_mask(0, key_mask);
        mv.store_k(0, smem);
        mv.store_v(0, smem + G::K_BYTES);
        if (key_mask) mv.store_mask(reinterpret_cast<float*>(smem + G::K_BYTES + G::V_BYTES));
        if (n_tiles > 1) {
            mv.template issue<0>(1);
            mv.template issue<1>(1);
            if (key_mask) mv.issue_mask(1, key_mask);
        }
    }
    __syncthreads();
    for (int t = 0; t < n_tiles; ++t) {
        const unsigned char* Ks = smem + (t & 1) * STAGE;
        const unsigned char* Vs = Ks + G::K_BYTES;
        const float* Ms = key_mask ? reinterpret_cast<const float*>(Vs + G::V_BYTES) : nullptr;
        const int j0 = plan.j0(t);
        const int lim = plan.limit(t);
        // wavefronts none of whose rows can see this tile only help with the loads
        if (j0 < we.hi_max && j0 + kBN > we.lo_min) {
            f32x16 sacc[2];
            V8 pf[4];
            mfma_stream<T, D, false, true>(Vs, Ks, pf, qf, oacc, sacc, lane);
            const bool biased = p.bias != nullptr && j0 < p.bias_cols;
            const bool interior = (j0 >= we.lo_max) && (j0 + kBN <= min(we.hi_min, lim)) && (key_mask == nullptr) && !biased;
            softmax_tile<T, D, PSCALE>(sacc, pf, oacc, st, cl2, lazy_raw, !interior, j0, lo, min(hi, lim), lh, Ms,
                                       biased ? bias_row : nullptr, p.bias_cols, p.inv_scale,
                                       PSCALE ? prefix_scale_of(p, plan.in_prefix(t)) : PrefixScale());
            mfma_stream<T, D, true, false>(Vs, Ks, pf, qf, oacc, sacc, lane);
        }
        if (t + 1 < n_tiles) {
            unsigned char* Kn = smem + ((t + 1) & 1) * STAGE;
            mv.store_k(t + 1, Kn);
            mv.store_v(t + 1, Kn + G::K_BYTES);
            if (key_mask) mv.store_mask(reinterpret_cast<float*>(Kn + G::K_BYTES + G::V_BYTES));
        }
        if (t + 2 < n_tiles) {
            mv.template issue<0>(t + 2);
            mv.template issue<1>(t + 2);
            if (key_mask) mv.issue_mask(t + 2, key_mask);
        }
        __syncthreads();
    }

    const float l_tot = exchange_sum(st.l);
    const float inv = row_inverse(l_tot);
    // base-2 log of the row's denominator in exponent units: p(key) = exp2(score * scale_log2 [+ bias * log2 e] - lse);
    // +inf for a row without visible keys, so that every p is 0
    if (p.lse && qvalid && lh == 0)
        p.lse[(static_cast<long>(b) * p.H + h) * Lq + qrow] = l_tot > 0.f ? st.mc + __builtin_amdgcn_logf(l_tot) : __builtin_huge_valf();
    stage_output<T, D>(smem, wave * 32 + lq, lh, oacc, inv);
    __syncthreads();
    write_output<T, D, kThreads4>(smem, o_base, p.o_rs, q0, Lq, BM, tid);
}

// ───────────────────────── short key sequences (cross attention) ─────────────────────────
// When all keys of a (batch, head) fit in LDS (cross attention to a text prompt: 77 to ~300 keys) the call moves far more
// bytes than it multiplies (Q in, O out: ~120 FLOP per byte at 77-105 keys of head_dim 72, below the ridge of ~312), so
// it is bound by HBM and by fixed costs, and the kernels above, whose work groups all stage, wait and drain at the same
// moments, are all prologue and epilogue. Here a work group of 8 wavefronts loads the K and V of its (batch, head) ONCE
// (only the tiles below the batch item's valid length, all loads in flight together), meets at one barrier, and from
// then on every wavefront is on its own: it walks 32-row query units, staging each through a private LDS slice (the
// unit's rows are fetched with full-row coalescing one unit ahead, the output leaves the same way), so no barrier stands
// in the key loop or between units and the eight wavefronts drift apart: while some wait for their rows, others
// multiply, and the memory pipe sees a steady stream instead of bursts. Unmasked calls (kv_valid_len and a 0/1 key mask
// allowed), no RoPE, no prefix. Same tile arithmetic as the 128-row kernel: bit-identical results.
constexpr int kShortMaxTiles = 5;   // 320 keys
template <int D> constexpr int shortkv_lds_bytes(int n_kt, bool with_mask) {
    using G = HeadGeo<D>;
    return 256 * G::O_STRIDE + n_kt * (G::K_BYTES + G::V_BYTES + (with_mask ? kBN * 4 : 0));
}
// most key tiles that fit in LDS next to the staging slices at head dimension D (the prologue holds that many in registers)
template <int D> constexpr int shortkv_max_tiles() {
    int n = kShortMaxTiles;
    while (n > 1 && shortkv_lds_bytes<D>(n, false) > 160 * 1024) --n;
    return n;
}

template <typename T, int D>
__global__ void __launch_bounds__(kThreads8, 2) sdpa_shortkv_kernel(const SdpaDev p, int n_kt, int units_per_group, int groups_per_head) {
    using G = HeadGeo<D>;
    using V8 = typename Mma<T>::v8;
    constexpr int UM = 32;                         // query rows of a unit (one wavefront)
    constexpr int SLICE = UM * G::O_STRIDE;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    const int logical = logical_block(p.n_blocks);
    if (logical < 0) return;
    const int bh = logical / groups_per_head;
    const int grp = logical - bh * groups_per_head;
    const int h = bh % p.H, b = bh / p.H;
    const int hk = h / p.kv_group;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, lq = lane & 31, lh = lane >> 5;
    unsigned char* const Qs = smem + wave * SLICE;            // this wavefront's staging slice
    unsigned char* const Kall = smem + 8 * SLICE;
    unsigned char* const Vall = Kall + n_kt * G::K_BYTES;
    float* const Mall = reinterpret_cast<float*>(Vall + n_kt * G::V_BYTES);
    const T* const q_base = static_cast<const T*>(p.q) + b * p.q_bs + h * D;
    T* const o_base = static_cast<T*>(p.o) + b * p.o_bs + h * D;

    // keys of this batch item (uniform): only the tiles that hold one are loaded and multiplied
    int kv_len = p.Lk;
    if (p.kv_valid_len) kv_len = min(kv_len, max(p.kv_valid_len[b], 0));
    kv_len = __builtin_amdgcn_readfirstlane(kv_len);
    const int n_kt_b = (kv_len + kBN - 1) / kBN;

    // ── a unit's Q rows: fetched with full-row coalescing into registers, stored to the slice when the unit's turn comes ──
    constexpr int CPRK = G::DK / 8;
    constexpr int NQ = UM * CPRK / 64;
    static_assert(UM * CPRK % 64 == 0, "a unit's chunks divide among the lanes");
    u32x4 qraw[NQ];
    auto q_issue = [&](int q0) {
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            const int idx = lane + 64 * i;
            const int row = idx / CPRK, cc = min(idx - row * CPRK, G::CPR - 1);
            qraw[i] = *reinterpret_cast<const u32x4*>(q_base + static_cast<long>(min(q0 + row, p.Lq - 1)) * p.q_rs + cc * 8);
        }
    };
    auto q_store = [&](int q0) {
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            const int idx = lane + 64 * i;
            const int row = idx / CPRK, cc = idx - row * CPRK;
            u32x4 v = qraw[i];
            if (q0 + row >= p.Lq || cc >= G::CPR) v = u32x4{0, 0, 0, 0};
            *reinterpret_cast<u32x4*>(Qs + row * G::O_STRIDE + cc * 16) = v;
        }
    };
    // LDS traffic of one wavefront is executed in order; the fences keep the compiler from reordering around them
    auto wave_sync = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    const int n_units = (p.Lq + UM - 1) / UM;
    const int u_end = min((grp + 1) * units_per_group, n_units);
    int u = grp * units_per_group + wave;
    if (u < u_end) q_issue(u * UM);

    // ── the K and V tiles of this (batch, head) and the key-mask values: every load is issued before the first is stored ──
    {
        constexpr int NLD = (G::NCH + kThreads8 - 1) / kThreads8;
        const unsigned char* const k_base = reinterpret_cast<const unsigned char*>(static_cast<const T*>(p.k) + b * p.k_bs + hk * D);
        const unsigned char* const v_base = reinterpret_cast<const unsigned char*>(static_cast<const T*>(p.v) + b * p.v_bs + hk * D);
        const unsigned k_rsb = static_cast<unsigned>(p.k_rs) * 2u, v_rsb = static_cast<unsigned>(p.v_rs) * 2u;
        constexpr int MAXT = shortkv_max_tiles<D>();
        u32x4 kreg[MAXT][NLD], vreg[MAXT][NLD];
        float mval = 0.f;
        if (p.key_mask && tid < n_kt_b * kBN && tid < kv_len) mval = p.key_mask[b * p.key_mask_bs + tid];
#pragma unroll
        for (int t = 0; t < MAXT; ++t) {
            if (t < n_kt_b) {
                const int last = min(kv_len - t * kBN, kBN) - 1;   // rows past the last key repeat it and are stored as zeros
#pragma unroll
                for (int i = 0; i < NLD; ++i) {
                    const int idx = min(tid + kThreads8 * i, G::NCH - 1);
                    const unsigned row = static_cast<unsigned>(t * kBN + min(idx / G::CPR, last));
                    const unsigned cc = static_cast<unsigned>(idx % G::CPR);
                    kreg[t][i] = *reinterpret_cast<const u32x4*>(k_base + (static_cast<unsigned long>(row) * k_rsb + cc * 16u));
                    vreg[t][i] = *reinterpret_cast<const u32x4*>(v_base + (static_cast<unsigned long>(row) * v_rsb + cc * 16u));
                }
            }
        }
        zero_pads<D, kThreads8>(Kall, Vall, G::K_BYTES, G::V_BYTES, n_kt_b, tid);
        if (p.key_mask && tid < n_kt * kBN) Mall[tid] = mval;
#pragma unroll
        for (int t = 0; t < MAXT; ++t) {
            if (t < n_kt_b) {
                const int nvalid = kv_len - t * kBN;
#pragma unroll
                for (int i = 0; i < NLD; ++i) {
                    const int idx = tid + kThreads8 * i;
                    const int row = idx / G::CPR, cc = idx - row * G::CPR;
                    if (idx < G::NCH) {
                        const bool live = row < nvalid;
                        *reinterpret_cast<u32x4*>(Kall + t * G::K_BYTES + row * G::K_STRIDE + cc * 16) = live ? kreg[t][i] : u32x4{0, 0, 0, 0};
                        *reinterpret_cast<u32x4*>(Vall + t * G::V_BYTES + row * G::V_STRIDE + cc * 16) = live ? vreg[t][i] : u32x4{0, 0, 0, 0};
                    }
                }
            }
        }
    }
    __syncthreads();   // K, V and the mask values are in place: the only barrier of the kernel

    const float cl2 = p.scale_log2;
    const float lazy_raw = kLazyLog2 / cl2;
    for (; u < u_end; u += 8) {
        const int q0 = u * UM;
        q_store(q0);
        wave_sync();
        V8 qf[G::KC];
        read_q_frags<T, D>(qf, Qs, lq, lh);
        wave_sync();       // the slice is free again (it takes the output next)
        // The next unit's rows, unconditionally (past its last unit a wavefront fetches the current one again, from cache):
        // vector-memory loads and stores complete in one order here, so the wait in front of the next q_store can pass over
        // this unit's output stores only if the compiler can count them, i.e. if neither the loads nor the stores sit
        // under a condition. With a conditional load the next unit waited for this unit's stores to land.
        q_issue(u + 8 < u_end ? q0 + 8 * UM : q0);

        f32x16 oacc[G::VB];
#pragma unroll
        for (int vb = 0; vb < G::VB; ++vb)
#pragma unroll
            for (int e = 0; e < 16; ++e) oacc[vb][e] = 0.f;
        SoftmaxState st;
        for (int t = 0; t < n_kt_b; ++t) {
            const int j0 = t * kBN;
            const unsigned char* Ks = Kall + t * G::K_BYTES;
            const unsigned char* Vs = Vall + t * G::V_BYTES;
            f32x16 sacc[2];
            V8 pf[4];
            mfma_stream<T, D, false, true>(Vs, Ks, pf, qf, oacc, sacc, lane);
            const bool interior = j0 + kBN <= kv_len && p.key_mask == nullptr;
            softmax_tile<T, D>(sacc, pf, oacc, st, cl2, lazy_raw, !interior, j0, 0, kv_len, lh, p.key_mask ? Mall + j0 : nullptr);
            mfma_stream<T, D, true, false>(Vs, Ks, pf, qf, oacc, sacc, lane);
        }
        const float l_tot = exchange_sum(st.l);
        const float inv = row_inverse(l_tot);
        stage_output<T, D>(Qs, lq, lh, oacc, inv);
        wave_sync();
        // (a fixed number of unconditional stores, see above: a lane without a chunk of its own, or whose row lies past the
        //  end of Q, stores a chunk that another lane stores too, same bytes to the same address)
        const int last_row = min(UM, p.Lq - q0) - 1;
#pragma unroll
        for (int i = 0; i < (UM * G::CPR + 63) / 64; ++i) {
            const int idx = min(lane + 64 * i, UM * G::CPR - 1);
            const int row = min(idx / G::CPR, last_row), cc = idx % G::CPR;
            *reinterpret_cast<u32x4*>(o_base + static_cast<long>(q0 + row) * p.o_rs + cc * 8) =
                *reinterpret_cast<const u32x4*>(Qs + row * G::O_STRIDE + cc * 16);
        }
        wave_sync();       // the staged rows are read before the next unit's Q overwrites them
    }
}

// ───────────────────────── 8-wavefront ping-pong kernel ─────────────────────────

// Eight wavefronts, 32 query rows each; wavefronts w and w + 4 share a SIMD. One work-group barrier per
// key tile. Between two barriers (step t; step -1 has no P yet and only scores tile 0) every wavefront runs
//   the MFMA stream:  O += V_t^T P_t ;  S_{t+1} = K_{t+1} Q^T   (reads LDS tiles V_t, K_{t+1}), and
//   one softmax:      P = softmax(S) of the scores it holds,
// in opposite order in the two groups: group 0 (wavefronts 0-3) streams first and then turns S_{t+1} into
// P_{t+1}; group 1 first turns S_t (scored in the previous step) into P_t and then streams. So on every SIMD
// one wavefront feeds the matrix pipe while the other is in its VALU part, and neither waits for the other
// before the end of the step: a barrier between the two halves (strict ping-pong) makes each stream run
// alone with its LDS and dependency latencies exposed and was measured ~1.6x slower.
// In the shadow of the stream the wavefront stores its share of tiles K_{t+2}, V_{t+1} into the LDS buffers
// of K_t, V_{t-1} (last read in step t-1) and issues the global loads of K_{t+3}, V_{t+2}; two buffers per
// operand suffice.
// FORM: as in the DMA form below, without prefix; kDense and kRagged are instantiated for head_dim up to 64, where kDense
// measures 2-3 % faster (at 80 the compiler's allocation of that instance goes wrong: twice as slow) and kRagged 13 %
// (head_dim 40, 8 heads, 3600 tokens: 67.0 -> 58.5 us).
// XTRA: key mask, logit bias and softmax denominators (see sdpa_fwd_pp_dma_kernel).
// F32SUM: see softmax_tile_rel.
template <typename T, int D, bool ROPE_K, int FORM = kGeneral, bool XTRA = false, bool F32SUM = false>
__global__ void __launch_bounds__(kThreads8, 2) sdpa_fwd_pp_kernel(const SdpaDev p) {
    constexpr bool DENSE = FORM != kGeneral, RAGGED = FORM == kRagged;
    static_assert(!XTRA || (!DENSE && !ROPE_K), "key mask, bias and denominators belong to the general form");
    using G = HeadGeo<D>;
    using V8 = typename Mma<T>::v8;
    constexpr int BM = 256;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    __shared__ int red[16];
    unsigned char* const Kbuf = smem;                    // 2 x K tile
    unsigned char* const Vbuf = smem + 2 * G::K_BYTES;   // 2 x V tile

    int qt, bh;
    if (!block_to_tile(p, qt, bh)) return;
    const int h = bh % p.H;
    const int b = bh / p.H;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform, kept in a scalar register
    const int grp = wave >> 2;      // phase group
    const int lane = tid & 63;
    const int lq = lane & 31;
    const int lh = lane >> 5;
    const int q0 = qt * BM;
    const int qrow = q0 + wave * 32 + lq;
    const bool qvalid = qrow < p.Lq;
    const int hk = h / p.kv_group;
    const T* const q_base = static_cast<const T*>(p.q) + b * p.q_bs + h * D;
    T* const o_base = static_cast<T*>(p.o) + b * p.o_bs + h * D;

    const int n_keys = RAGGED ? visible_keys(p, b) : p.Lk;
    int lo = 0, hi = n_keys;   // DENSE: rows past the end of Q repeat its last row and are never stored
    // (rows past the end: as in sdpa_fwd_pp_dma_kernel)
    if constexpr (!DENSE) row_interval(p, b, min(qrow, p.Lq - 1), q0 + wave * 32 < p.Lq, lo, hi);
    WaveExtent we{0, 0, n_keys, n_keys};
    if constexpr (!DENSE) {
        we = wave_extent(lo, hi);
        if (lane == 0) { red[wave] = we.lo_min; red[8 + wave] = we.hi_max; }
    }
    V8 qf[G::KC];
    stage_q_tile<T, D, kThreads8, BM>(smem, p, q_base, q0, tid);
    __syncthreads();
    read_q_frags<T, D>(qf, smem, wave * 32 + lq, lh);
    __syncthreads();
    // K pad columns must be zero; the V buffers are zeroed whole because the first pass through the
    // MFMA stream multiplies a zero P with whatever the second V buffer holds
    zero_pads<D, kThreads8>(Kbuf, Vbuf, G::K_BYTES, G::V_BYTES, 2, tid);
    for (int i = tid; i < 2 * G::V_BYTES / 16; i += kThreads8) *reinterpret_cast<u32x4*>(Vbuf + i * 16) = u32x4{0, 0, 0, 0};
    __syncthreads();
    int g_lo = 0, kv_stop = n_keys;
    if constexpr (!DENSE) {
        g_lo = red[0]; kv_stop = red[8];
#pragma unroll
        for (int w = 1; w < 8; ++w) { g_lo = min(g_lo, red[w]); kv_stop = max(kv_stop, red[8 + w]); }
        g_lo = __builtin_amdgcn_readfirstlane(g_lo);
        kv_stop = __builtin_amdgcn_readfirstlane(kv_stop);
    }
    const TilePlan plan(g_lo == 0x7fffffff ? 0 : g_lo, kv_stop, p.Lp);
    const int n_tiles = plan.n_tiles;
    // XTRA: visibility words of the plan's tiles behind the tile buffers (visible after the barrier that ends the prologue)
    const unsigned long long* const kbits = (XTRA && p.key_mask) ? reinterpret_cast<const unsigned long long*>(smem + p.kbits_off) : nullptr;
    if constexpr (XTRA) build_key_bits(p, plan, b, smem + p.kbits_off, wave, lane);
    const float* const bias_row = (XTRA && p.bias && qvalid && qrow >= p.bias_q0) ? p.bias + static_cast<long>(qrow - p.bias_q0) * p.bias_rs : nullptr;
    TileExtra xt;

    f32x16 oacc[G::VB];
#pragma unroll
    for (int vb = 0; vb < G::VB; ++vb)
#pragma unroll
        for (int e = 0; e < 16; ++e) oacc[vb][e] = 0.f;
    RelSoftmaxState st;
    const bool dead_row = hi <= lo;
    const float cl2 = p.scale_log2;

    const unsigned char* const k_head = reinterpret_cast<const unsigned char*>(static_cast<const T*>(p.k) + b * p.k_bs + hk * D);
    const unsigned char* const v_head = reinterpret_cast<const unsigned char*>(static_cast<const T*>(p.v) + b * p.v_bs + hk * D);
    // (the dense launch is whole tiles of one segment: its mover does no arithmetic per tile)
    auto make_mover = [&]() {
        if constexpr (DENSE) return DenseMover<T, D, kThreads8, RAGGED>(k_head, p.k_rs, v_head, p.v_rs, tid, wave, n_keys);
        else return TileMover<T, D, kThreads8, ROPE_K>{p, plan, k_head, v_head,
                                                       reinterpret_cast<const unsigned char*>(static_cast<const T*>(p.kp) + b * p.kp_bs + hk * D),
                                                       reinterpret_cast<const unsigned char*>(static_cast<const T*>(p.vp) + b * p.vp_bs + hk * D),
                                                       tid, {}, {}, 1.f};
    };
    auto mv = make_mover();
    auto tile_active = [&](int t) {
        if (t < 0 || t >= n_tiles) return false;
        const int j0 = plan.j0(t);
        return j0 < we.hi_max && j0 + kBN > we.lo_min;
    };
    // this thread's share of tiles K_kt, V_vt: registers -> LDS, then prefetch K_{kt+1}, V_{vt+1}
    // (the walk measured 18 % faster at head_dim 40, 9 % at 64, and no faster from 80 on, where a thread moves two chunks)
    constexpr bool WALK = !ROPE_K && D <= 64;
    static_assert(!DENSE || WALK, "the dense mover is a walk");
    auto advance_tiles = [&](int kt, int vt) {
        if constexpr (!WALK) {
            if (kt < n_tiles) mv.store_k(kt, Kbuf + (kt & 1) * G::K_BYTES);
            if (vt < n_tiles) mv.store_v(vt, Vbuf + (vt & 1) * G::V_BYTES);
            if (kt + 1 < n_tiles) mv.template issue<0>(kt + 1);
            if (vt + 1 < n_tiles) mv.template issue<1>(vt + 1);
        } else {
            // tiles are fetched strictly in order, so the mover walks them with its cursors
            if (kt < n_tiles) mv.store_held_k(Kbuf + (kt & 1) * G::K_BYTES);
            if (vt < n_tiles) mv.store_held_v(Vbuf + (vt & 1) * G::V_BYTES);
            if (kt + 1 < n_tiles) mv.template issue_next<0>();
            if (vt + 1 < n_tiles) mv.template issue_next<1>();
        }
    };
    f32x16 sacc[2];
    V8 pf[4];
#pragma unroll
    for (int c4 = 0; c4 < 4; ++c4) pf[c4] = __builtin_bit_cast(V8, u32x4{0, 0, 0, 0});

    if (n_tiles > 0) {
        // ── prologue: K_0 into LDS; registers then hold K_1, V_0 ──
        if constexpr (!WALK) {
            mv.template issue<0>(0);
            mv.store_k(0, Kbuf);
            if (n_tiles > 1) mv.template issue<0>(1);
            mv.template issue<1>(0);
        } else {
            mv.start_walk();
            mv.template issue_next<0>();
            mv.store_held_k(Kbuf);
            if (n_tiles > 1) mv.template issue_next<0>();
            mv.template issue_next<1>();
        }
        __syncthreads();
        auto softmax_of = [&](int tt) {
            if constexpr (DENSE) {
                if (tt >= 0 && tt < n_tiles) {
                    const int rows = RAGGED ? min(n_keys - tt * kBN, kBN) : kBN;
                    softmax_tile_rel<T, D, false, false, F32SUM>(sacc, pf, oacc, st, RAGGED && rows < kBN, false, 0, 0, rows, lh);
                    return;
                }
            }
            if constexpr (XTRA) {
                xt = TileExtra();
                if (kbits) {
                    const unsigned long long w = kbits[min(max(tt, 0), max(n_tiles - 1, 0))];
                    xt.kw0 = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(w));
                    xt.kw1 = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(w >> 32));
                }
                xt.bias_cols = p.bias_cols;
            }
            if (!DENSE && tile_active(tt) && (!XTRA || (xt.kw0 | xt.kw1) != 0u)) {
                const int j0 = plan.j0(tt);
                const int lim = plan.limit(tt);
                bool interior = (j0 >= we.lo_max) && (j0 + kBN <= min(we.hi_min, lim));
                if constexpr (XTRA) {
                    const bool biased = p.bias != nullptr && j0 < p.bias_cols;
                    interior = interior && (xt.kw0 & xt.kw1) == ~0u && !biased;
                    xt.bias_row = biased ? bias_row : nullptr;
                    xt.bias_vec = p.bias_vec_ok && (j0 & 3) == 0 && j0 + kBN <= p.bias_cols;
                }
                softmax_tile_rel<T, D, false, XTRA, F32SUM>(sacc, pf, oacc, st, !interior, dead_row, j0, lo, min(hi, lim), lh, PrefixScale(), xt);
            } else {
                // nothing visible to this wavefront in that tile: the next PV pass must add zero
#pragma unroll
                for (int c4 = 0; c4 < 4; ++c4) pf[c4] = __builtin_bit_cast(V8, u32x4{0, 0, 0, 0});
            }
        };
        // step -1 only scores tile 0 (there is no P yet)
        for (int t = -1; t < n_tiles; ++t) {
            if (grp == 1) {
                softmax_of(t);
                MI_SCHED_BARRIER
            }
            // Always the full stream: at t = -1 P is zero and the (zero-filled) V buffer adds nothing;
            // after the last tile the extra scores are never read. This wavefront's share of the tile
            // movement rides along in the stream (measured faster than in front of the softmax: the stores
            // and loads issue in the shadow of the matrix pipe).
            auto mover = [&]() { advance_tiles(t + 2, t + 1); };
            mfma_stream<T, D, true, true, decltype(mover), true>(Vbuf + (t & 1) * G::V_BYTES, Kbuf + ((t + 1) & 1) * G::K_BYTES, pf, qf,
                                                                 oacc, sacc, lane, mover, cl2, st.neg_ref);
            if (grp == 0) {
                MI_SCHED_BARRIER
                softmax_of(t + 1);
            }
            __syncthreads();
        }
    }

    const float l_tot = exchange_sum(st.l);
    const float inv = row_inverse(l_tot);
    if constexpr (XTRA) {
        if (p.lse && qvalid && lh == 0)
            p.lse[(static_cast<long>(b) * p.H + h) * p.Lq + qrow] = l_tot > 0.f ? __builtin_amdgcn_logf(l_tot) - st.neg_ref : __builtin_huge_valf();
    }
    stage_output<T, D>(smem, wave * 32 + lq, lh, oacc, inv);
    __syncthreads();
    write_output<T, D, kThreads8>(smem, o_base, p.o_rs, q0, p.Lq, BM, tid);
}

// ─────────────── 8-wavefront kernel with tiles by LDS DMA ───────────────
// Same schedule as sdpa_fwd_pp_kernel, but K/V tiles go from global memory straight into LDS
// (global_load_lds_dwordx4: lane i of a wavefront deposits its 16 bytes at base + 16*i), so tile
// movement costs no registers and no LDS store instructions. A DMA instruction writes 1024 contiguous
// bytes, so rows sit in LDS back to back without padding; a 64-key tile is D/8 such instructions per
// operand, dealt out to the 8 wavefronts in turn. Bank conflicts of the unpadded rows:
//   head_dim 128 (256-byte rows): avoided by an XOR swizzle, 16-byte chunk c of row r lives at chunk position
//     c ^ f(r), f(r) = 4*(r%4) + (r/4)%4, applied for free on the global side (each lane fetches the chunk that
//     belongs in its LDS slot) and undone in the LDS read addresses: K reads (one row per lane, 16 consecutive
//     rows) hit 16 distinct slots, V transpose reads (4 rows x 64 bytes per 32 lanes) 4 distinct 64-byte windows;
//   head_dim 72 (144-byte rows): 16 consecutive rows start on 16 distinct multiples of 4 banks, so the K reads are
//     conflict-free as they are; the V transpose reads overlap a little.
// Without padding, the fragment reads of the zero-padded part of the head dimension (columns D..DK-1 of K,
// D..DV-1 of V) run into the first bytes of the next row: real key rows (rows past the end of a segment are fetched
// from its last row), multiplied by the zero pad of Q, or producing output columns that are never stored. A little
// zero-filled slack behind each ring keeps the reads of the last row inside the allocation.
// Tiles are ring-buffered three deep: the loads of K_{t+3}, V_{t+2} are issued in step t, awaited at
// the end of step t+1 and read in step t+2. The key loop is unrolled by three so that every LDS offset
// is an instruction immediate; tile pointers advance incrementally in scalar registers.
constexpr int kDmaStages = 3;
template <int D> struct DmaGeo {
    using G = HeadGeo<D>;
    static constexpr int ROWB = D * 2;                       // bytes per row in LDS (no padding)
    static constexpr int TILE = kBN * ROWB;                  // = (D / 8) KB
    static constexpr int NDMA = TILE / 1024;                 // DMA instructions per operand tile
    static constexpr int SLACK = 256;                        // zero bytes behind each ring
    static constexpr int RING = kDmaStages * TILE + SLACK;
    static constexpr int VOFF = RING;
    static constexpr int MAXI = (2 * NDMA + 7) / 8;          // most DMA instructions of one wavefront per step
    static constexpr bool SWZ = D == 128;
    // The Q tile is staged behind the rings, so that the first key tiles can be in flight while it is loaded, rotated and
    // picked apart; where rings + a whole staged tile exceed the LDS of a compute unit it goes through in two halves
    // (rows 0..127 for wavefronts 0..3, then rows 128..255 for wavefronts 4..7). The output is staged over the rings,
    // which are dead by then.
    static constexpr int QOFF = 2 * RING;
    static constexpr bool Q_HALVES = QOFF + 256 * G::O_STRIDE > 160 * 1024;
    static constexpr int Q_BYTES = (Q_HALVES ? 128 : 256) * G::O_STRIDE;
    static constexpr int lds_bytes() {
        const int kvq = QOFF + Q_BYTES;
        const int o = 256 * G::O_STRIDE;
        return kvq > o ? kvq : o;
    }
    static_assert(QOFF + Q_BYTES <= 160 * 1024, "rings and Q staging exceed the LDS of a compute unit");
};
// (head_dim 40 works the same way but measured no faster than the register-staged kernel: not instantiated)
template <int D> constexpr bool dma_kernel_available() { return D == 72 || D == 128; }

// The statistics of a part's scratch slot: 256 references, then 256 denominators; in their place kWholeTile where the first part took the tile
// whole (LISTED) and wrote the result itself.
template <int D>
__device__ __forceinline__ float* part_stats(unsigned char* slot) { return reinterpret_cast<float*>(slot + 256L * D * 4); }
template <int D>
__device__ __forceinline__ const float* part_stats(const unsigned char* slot) { return reinterpret_cast<const float*>(slot + 256L * D * 4); }
constexpr float kWholeTile = -1.f;

__device__ __forceinline__ int swz(int row) { return 4 * (row & 3) + ((row >> 2) & 3); }

// SPLIT: the launch follows p.split — a work group either processes one whole query tile or one piece of the last
// round, i.e. one or more (tile, key range) parts in sequence, each leaving a partial result in its scratch slot
// (merged by sdpa_combine_kernel; plan_split has the times). Only for calls without prefix and without a mask other than a key mask: in the dense form
// where the key tiles are whole, else in the ragged form (24 heads of 128 with RoPE and K rotation, 4096 tokens: ragged 202.1, dense 194.5 us).
// The loop over parts keeps nothing of a pass for the next, the RoPE tables' registers included (QTileLoad::define_tables; carried through the key
// loop they made it spill 21 others, and each table piece was waited for as it arrived: the same call 213.5, without 203.1). Addresses that follow from
// the thread id alone it may keep: computed anew in each pass they cost every tile 0.4 to 0.8 us at its start (same call 201.0 -> 199.5; with one key
// visible under a key mask 45.0 -> 43.6), kept they fit the registers.
// FORM kDense: no mask of any kind and key counts (cached prefix, if any, and fresh) that are multiples of 64: every tile is
// whole and visible to every row, so the masked form of the softmax and the per-step bookkeeping (which tile, its limit,
// whether this wavefront sees it whole) drop out of the kernel, and with them their registers: measured 6 % faster at
// head_dim 128 and 8 % at 72 than the general form on the same dense call.
// FORM kRagged: every row sees the same keys, their number is free. All tiles but the last of a segment are as in kDense; that
// one is met by scalar branches (DMA rows clamped to the last that exists, scores past it blanked). The general form clamps and
// compares in every step: 24 heads of 128, 2500 tokens 77.5 -> 75.3 us, 16 heads of 72, 3600 tokens 84.0 -> 82.0.
// FORM kFresh: kRagged without a prefix, for calls under a key mask (the choice between prefix and fresh rows in every step is gone; launch_d has the times).
// PSCALE: the general form with the prefix-KV dial (factors on the rows of the cached prefix) in its softmax.
// XTRA: the general form with a key mask (one visibility bit per key, 64-bit words per key tile built once per work group
// in LDS behind the rings), an additive logit bias and the softmax denominators as an output (traced attention).
// XTRA with kRagged or kFresh: a key mask but no bias. The mask hides the same keys from every row (the padding of a prompt in
// the middle of a joint sequence), so the tiles without a visible key are taken out of the walk: `vis` lists the others, and a
// step looks up the tile that it loads. 48 query / 12 K/V heads of 128, 4608 tokens of which 435 are padding (6 of 72 tiles):
// 520 -> 472 us; the words used to blank the scores of a hidden tile, whose MFMAs and loads ran all the same. With SPLIT a part [s0, s1) of T
// tiles takes entries [s0 n / T, s1 n / T) of the n listed ones, so that hidden tiles shorten all parts alike; a query tile with fewer than
// split.min_visible listed ones is not cut: its first part takes it whole and writes the result, the others and the merge have nothing to do
// (cut all the same, an empty part staged Q and wrote a slot of FP32 like any other: 24 heads of 128, one key visible of 3328, unsplit 37 us, cut 59).
// F32SUM: see softmax_tile_rel.
template <typename T, int D, bool SPLIT, int FORM = kGeneral, bool PSCALE = false, bool XTRA = false, bool F32SUM = false>
__global__ void __launch_bounds__(kThreads8, 2) sdpa_fwd_pp_dma_kernel(const SdpaDev p) {
    constexpr bool DENSE = FORM != kGeneral, RAGGED = FORM == kRagged || FORM == kFresh, LISTED = XTRA && RAGGED;
    constexpr bool FRESH = SPLIT || FORM == kFresh;     // no prefix
    static_assert(!SPLIT || DENSE, "every row of a split launch sees the same keys");
    static_assert(!PSCALE || !DENSE, "the dial belongs to the general form");
    static_assert(!XTRA || (FORM != kDense && !PSCALE), "key mask, bias and denominators are not in these forms");
    static_assert(FORM != kFresh || (XTRA && !SPLIT), "only calls under a key mask gain by it");
    using G = HeadGeo<D>;
    using DG = DmaGeo<D>;
    using V8 = typename Mma<T>::v8;
    constexpr int BM = 256;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    __shared__ int red[16];

    // ── what this work group does ──
    int qt, bh;
    int kv_begin = 0, kv_end = 0x7fffffff;   // key range of the current part
    unsigned char* part = nullptr;            // scratch slot of the current part; null: the output itself
    // SPLIT bookkeeping (all wave-uniform): tail steps [seg_s, seg_end) of group xg still to do
    int xg = 0, n_full = 0, seg_s = 0, seg_end = 0, piece = 0, tail_steps = 0, n_pieces = 0;
    bool whole = true;
    if constexpr (!SPLIT) {
        if (!block_to_tile(p, qt, bh)) return;
    } else {
        xg = static_cast<int>(blockIdx.x) & 7;
        const int i = static_cast<int>(blockIdx.x) >> 3;
        n_full = p.split.full_of(xg);
        whole = i < n_full;
        if (whole) {
            const int logical = xg * p.split.chunk + i;
            qt = logical % p.n_q_tiles;
            bh = logical / p.n_q_tiles;
        } else {
            tail_steps = p.split.tail_of(xg) * p.split.T;
            n_pieces = p.split.pieces_for(tail_steps);
            piece = i - n_full;
            if (piece >= n_pieces) return;
            seg_s = SplitGeo::piece_begin(piece, tail_steps, n_pieces);
            seg_end = SplitGeo::piece_begin(piece + 1, tail_steps, n_pieces);
            qt = bh = 0;
        }
    }
    // XTRA: the visibility words of the key tiles (published by the barrier that ends the prologue). LISTED: behind them the numbers of the tiles
    // with a visible key, in order; every wavefront writes the whole list (the same values) and reads only what it wrote.
    const unsigned long long* const kbits = (XTRA && p.key_mask) ? reinterpret_cast<const unsigned long long*>(smem + p.kbits_off) : nullptr;
    unsigned short* const vis_list = LISTED ? reinterpret_cast<unsigned short*>(smem + p.kbits_off + 8 * ((p.Lk + kBN - 1) / kBN + 2)) : nullptr;
    int listed_b = -1, n_visible = 0;     // the batch item whose list it is, and its length
    auto list_tiles = [&](const TilePlan& plan, int b, int wave, int lane) -> int {
        build_key_bits(p, plan, b, smem + p.kbits_off, wave, lane);
        __syncthreads();
        int n = 0;
        for (int t0 = 0; t0 < plan.n_tiles; t0 += 64) {
            const bool on = t0 + lane < plan.n_tiles && kbits[t0 + lane] != 0ull;
            const unsigned long long m = __ballot(on);
            if (on) vis_list[n + __popcll(m & ((1ull << lane) - 1ull))] = static_cast<unsigned short>(t0 + lane);
            n += __popcll(m);
        }
        n = __builtin_amdgcn_readfirstlane(n);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        return n;
    };
    if constexpr (SPLIT && LISTED) {
        // a piece that begins inside a tile has nothing to do there if the tile is not cut; it reaches into one other tile at most, whose first part it is
        if (!whole && seg_s % p.split.T != 0) {
            listed_b = (xg * p.split.chunk + n_full + seg_s / p.split.T) / p.n_q_tiles / p.H;
            n_visible = list_tiles(TilePlan(0, p.Lk, 0), listed_b, __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6), threadIdx.x & 63);
            if (n_visible < p.split.min_visible) {
                seg_s = (seg_s / p.split.T + 1) * p.split.T;
                if (seg_s >= seg_end) return;
            }
        }
    }
  for (;;) {   // one pass per part (a single pass unless SPLIT)
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 2;
    const int lane = tid & 63;
    const int lq = lane & 31;
    const int lh = lane >> 5;
    if constexpr (SPLIT) {
        if (!whole) {
            const int tt = seg_s / p.split.T;                  // tail tile of this group
            const int s0 = seg_s - tt * p.split.T;
            const int s1 = min(seg_end - tt * p.split.T, p.split.T);
            const int logical = xg * p.split.chunk + n_full + tt;
            qt = logical % p.n_q_tiles;
            bh = logical / p.n_q_tiles;
            kv_begin = s0 * kBN;
            kv_end = s1 * kBN;
            part = nullptr;
            if (s0 != 0 || s1 != p.split.T) {
                const int k = piece - SplitGeo::piece_of(tt * p.split.T, tail_steps, n_pieces);
                part = p.split_scratch + (static_cast<long>(xg * p.split.max_tail + tt) * p.split.max_parts + k) * SplitGeo::slot_bytes(D);
            }
            seg_s = tt * p.split.T + s1;
        }
    }
    bool alone = false;                   // LISTED: the first part of a tile that is not cut
    const int Lp = FRESH ? 0 : p.Lp;      // (LISTED: a third of the key loop's scalar instructions are the choice between prefix and fresh rows)
    const int h = bh % p.H;
    const int b = bh / p.H;
    const int q0 = qt * BM;
    const int qrow = q0 + wave * 32 + lq;
    const bool qvalid = qrow < p.Lq;
    const int hk = h / p.kv_group;
    const T* const q_base = static_cast<const T*>(p.q) + b * p.q_bs + h * D;
    T* const o_base = static_cast<T*>(p.o) + b * p.o_bs + h * D;

    const int n_keys = RAGGED && !SPLIT ? visible_keys(p, b) : p.Lk;   // counts the cached prefix rows, which come first
    int lo = 0, hi = n_keys;   // DENSE: rows past the end of Q repeat its last row and are never stored
    // (rows past the end count as the last row where they share a wavefront with it: as rows without keys they put every tile
    //  of that wavefront on the masked path; 24 heads of 128, 2500 tokens, block-causal: 83.8 -> 74.5 us)
    if constexpr (!DENSE) row_interval(p, b, min(qrow, p.Lq - 1), q0 + wave * 32 < p.Lq, lo, hi);
    WaveExtent we{0, 0, n_keys, n_keys};
    if constexpr (!DENSE) {
        we = wave_extent(lo, hi);
        if (lane == 0) { red[wave] = we.lo_min; red[8 + wave] = we.hi_max; }
    }
    V8 qf[G::KC];
    // the Q rows (and their RoPE tables) are requested first; they are rotated and staged further down, behind the issue of
    // the first key tiles' DMA, so that both latencies run together
    using QL = QTileLoad<T, D, kThreads8, BM>;
    static_assert(!DG::Q_HALVES || (QL::NI % 2 == 0 && kThreads8 * (QL::NI / 2) == 128 * QL::CPRK), "half of the load rounds must be half of the rows");
    QL ql;
    if constexpr (SPLIT) ql.define_tables();
    ql.issue(p, q_base, q0, tid, p.Lq - 1);
    // the first pass through the MFMA stream multiplies a zero P with the last V buffer; the slack behind both rings is zero
    for (int i = tid; i < (DG::TILE + DG::SLACK) / 16; i += kThreads8)
        *reinterpret_cast<u32x4*>(smem + DG::VOFF + (kDmaStages - 1) * DG::TILE + i * 16) = u32x4{0, 0, 0, 0};
    for (int i = tid; i < DG::SLACK / 16; i += kThreads8)
        *reinterpret_cast<u32x4*>(smem + kDmaStages * DG::TILE + i * 16) = u32x4{0, 0, 0, 0};
    __syncthreads();
    int g_lo = 0, kv_stop = n_keys;
    if constexpr (!DENSE) {
        g_lo = red[0]; kv_stop = red[8];
#pragma unroll
        for (int w = 1; w < 8; ++w) { g_lo = min(g_lo, red[w]); kv_stop = max(kv_stop, red[8 + w]); }
        g_lo = __builtin_amdgcn_readfirstlane(g_lo);
        kv_stop = __builtin_amdgcn_readfirstlane(kv_stop);
    }
    // (a part begins at a multiple of 64 keys; its tiles are numbered from there)
    constexpr bool RANGE = SPLIT && !LISTED;
    const TilePlan plan(RANGE ? kv_begin : g_lo == 0x7fffffff ? 0 : g_lo, RANGE ? min(kv_stop, kv_end) : kv_stop, Lp);
    int n_tiles = plan.n_tiles;
    if constexpr (XTRA && !LISTED) build_key_bits(p, plan, b, smem + p.kbits_off, wave, lane);
    // LISTED: vis_t .. vis_t3 are the list's entries t .. t + 3 in step t
    const unsigned short* vis = vis_list;
    int vis_t = 0, vis_t1 = 0, vis_t2 = 0, vis_t3 = 0;
    if constexpr (LISTED) {
        if (!SPLIT || b != listed_b) n_visible = list_tiles(plan, b, wave, lane);
        listed_b = b;
        n_tiles = n_visible;
        if constexpr (SPLIT) {
            if (!whole) {
                if (n_visible < p.split.min_visible) alone = true;
                else {
                    // a part is its share of the list (keys counted in tiles: at most 3070 of them, what the LDS holds words for)
                    const int first = kv_begin / kBN * n_visible / p.split.T, stop = kv_end / kBN * n_visible / p.split.T;
                    vis += first;
                    n_tiles = stop - first;
                }
            }
        }
    }
    auto listed = [&](int i) { return __builtin_amdgcn_readfirstlane(static_cast<int>(vis[min(i, n_tiles - 1)])); };   // n_tiles > 0
    const float* const bias_row = (XTRA && p.bias && qvalid && qrow >= p.bias_q0) ? p.bias + static_cast<long>(qrow - p.bias_q0) * p.bias_rs : nullptr;

    f32x16 oacc[G::VB];
#pragma unroll
    for (int vb = 0; vb < G::VB; ++vb)
#pragma unroll
        for (int e = 0; e < 16; ++e) oacc[vb][e] = 0.f;
    RelSoftmaxState st;
    const bool dead_row = hi <= lo;
    const float cl2 = p.scale_log2;

    // ── DMA duty of this wavefront: instructions i = wave, wave + 8, ... of the list [K 0..NDMA-1, V 0..NDMA-1];
    //    instruction j of an operand fills LDS bytes [1024 j, 1024 j + 1024) of the tile = chunks 64 j + lane ──
    TileCursor kc, vc;
    kc.init(plan, reinterpret_cast<const unsigned char*>(static_cast<const T*>(p.kp) + b * p.kp_bs + hk * D), static_cast<unsigned>(p.kp_rs) * 2u,
            reinterpret_cast<const unsigned char*>(static_cast<const T*>(p.k) + b * p.k_bs + hk * D), static_cast<unsigned>(p.k_rs) * 2u, Lp);
    vc.init(plan, reinterpret_cast<const unsigned char*>(static_cast<const T*>(p.vp) + b * p.vp_bs + hk * D), static_cast<unsigned>(p.vp_rs) * 2u,
            reinterpret_cast<const unsigned char*>(static_cast<const T*>(p.v) + b * p.v_bs + hk * D), static_cast<unsigned>(p.v_rs) * 2u, Lp);
    auto seek = [&](TileCursor& c, int t, const void* pre, long pre_bs, const void* fresh, long fresh_bs) {   // (LISTED: one row stride for both)
        const int j0 = plan.j0(t);
        c.ptr = plan.in_prefix(t)
                    ? reinterpret_cast<const unsigned char*>(static_cast<const T*>(pre) + b * pre_bs + hk * D) + static_cast<unsigned long>(j0) * c.rsb
                    : reinterpret_cast<const unsigned char*>(static_cast<const T*>(fresh) + b * fresh_bs + hk * D) + static_cast<unsigned long>(j0 - Lp) * c.rsb;
        c.rows_left = plan.limit(t) - j0;
    };
    int drow[DG::MAXI];        // tile row this lane fetches in its m-th instruction
    unsigned dcol[DG::MAXI];   // byte offset inside that row
#pragma unroll
    for (int m = 0; m < DG::MAXI; ++m) {
        const int i = wave + 8 * m;
        const int j = i < DG::NDMA ? i : i - DG::NDMA;
        const int g = 64 * j + lane;
        const int row = g / G::CPR;
        int cc = g - row * G::CPR;
        if constexpr (DG::SWZ) cc ^= swz(row);     // the chunk this slot must receive
        drow[m] = row;
        dcol[m] = static_cast<unsigned>(cc) * 16u;
        if constexpr (DENSE) {
            // the lane's byte offset inside a (whole) tile never changes
            const bool is_k = DG::NDMA % 8 == 0 ? m < DG::MAXI / 2 : i < DG::NDMA;
            dcol[m] += static_cast<unsigned>(row) * (static_cast<unsigned>(is_k ? p.k_rs : p.v_rs) * 2u);
        }
    }
    // One DMA instruction. Written as inline assembly on purpose: for the compiler's builtin every later LDS read may
    // alias the DMA's LDS write, so it waits for the load to land (vmcnt(0)) before the next ds_read. The tiles
    // written here are never read before the explicit wait + barrier at the end of the following step.
    const unsigned lds_base = static_cast<unsigned>(reinterpret_cast<size_t>((__attribute__((address_space(3))) unsigned char*)smem));
    auto dma = [&](const TileCursor& c, int m, int j, int lds_off, bool last) {
        unsigned voff = dcol[m];
        if constexpr (!DENSE) voff += static_cast<unsigned>(min(drow[m], min(c.rows_left, kBN) - 1)) * c.rsb;
        // the last tile of a segment: rows past its end repeat the last one. A scalar branch that no other tile takes: the empty
        // statement keeps the compiler from computing it for every tile and selecting
        if (RAGGED && last) {
            asm volatile("" : "+v"(voff));
            voff -= static_cast<unsigned>(max(drow[m] - (c.rows_left - 1), 0)) * c.rsb;
        }
        const unsigned dst = lds_base + lds_off + j * 1024;
        // (the LDS base travels in m0 as a declared input: the compiler writes the register itself and knows it is taken;
        //  the s_nop is the wait state an LDS-DMA instruction needs behind a write of m0)
        asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(c.ptr), "{m0}"(dst) : "memory");
    };
    // this wavefront's share of the loads of one K tile (if do_k) and one V tile (if do_v); returns how many it issued.
    // head_dim 128 asks once for all loads of a step whether one of the tiles is the last (24 heads with RoPE, 4600 tokens 241.8 -> 239.6 us; under a key
    // mask 48 / 12 heads, 3000 tokens 249 -> 246), but under a key mask with a prefix for each (48 / 12 heads, 200 prefix rows: 1300 tokens 74.9 -> 73.8,
    // 2304 127.0 -> 125.6)
    constexpr bool EACH = LISTED && !FRESH;
    auto dma_tiles = [&](bool do_k, int k_off, bool do_v, int v_off) -> int {
        int n = 0;
        if constexpr (DG::NDMA % 8 == 0) {
            // every wavefront has the same duty: its first MAXI / 2 instructions are K, the others V
            auto all = [&](bool last) {
#pragma unroll
                for (int m = 0; m < DG::MAXI; ++m) {
                    const int i = wave + 8 * m;
                    if (m < DG::MAXI / 2) { if (do_k) { dma(kc, m, i, k_off, EACH ? kc.rows_left < kBN : last); ++n; } }
                    else { if (do_v) { dma(vc, m, i - DG::NDMA, v_off, EACH ? vc.rows_left < kBN : last); ++n; } }
                }
            };
            if (RAGGED && !EACH && ((do_k && kc.rows_left < kBN) || (do_v && vc.rows_left < kBN))) all(true);
            else all(false);
        } else {
#pragma unroll
            for (int m = 0; m < DG::MAXI; ++m) {
                const int i = wave + 8 * m;
                if (i < DG::NDMA) { if (do_k) { dma(kc, m, i, k_off, kc.rows_left < kBN); ++n; } }
                else if (i < 2 * DG::NDMA) { if (do_v) { dma(vc, m, i - DG::NDMA, v_off, vc.rows_left < kBN); ++n; } }
            }
        }
        return n;
    };
    auto wait_all_but = [&](int n) {     // loads complete in order: everything older than the last n has landed
        if (n >= 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        else if (n == 3) asm volatile("s_waitcnt vmcnt(3)" ::: "memory");
        else if (n == 2) asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
        else if (n == 1) asm volatile("s_waitcnt vmcnt(1)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };
    static_assert(DG::MAXI <= 4, "wait_all_but covers at most 4 loads per step");

    // ── LDS read addresses (stage and block offsets are immediates) ──
    // K fragment (kb, c): row 32kb + lq, chunk 2c + lh (at position (2c + lh) ^ f(lq) in the swizzled layout)
    const int fk = swz(lq);
    unsigned kaddr[G::KC];
#pragma unroll
    for (int c = 0; c < G::KC; ++c) kaddr[c] = lq * DG::ROWB + ((DG::SWZ ? ((2 * c + lh) ^ fk) : (2 * c + lh)) << 4);
    // V fragment (c4, vb), halves hh = 0, 1: key row 16c4 + 4lh + 8hh + trow, 8 bytes at head-dim 32vb + tcol
    const int trow = (lane & 15) >> 2;
    const int j4 = lane & 3;
    const int g1 = (lane >> 4) & 1;
    unsigned vaddr[G::VB][2];
#pragma unroll
    for (int vb = 0; vb < G::VB; ++vb)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            const int row = 4 * lh + 8 * hh + trow;
            const int chunk = 4 * vb + 2 * g1 + (j4 >> 1);
            vaddr[vb][hh] = DG::VOFF + row * DG::ROWB + ((DG::SWZ ? (chunk ^ swz(row)) : chunk) << 4) + 8 * (j4 & 1);
        }

    static_assert(G::DK == D || G::DK - D == 8, "the pad of a K row is the upper lane half of its last fragment");
    const unsigned pad_keep = lh ? 0u : ~0u;

    f32x16 sacc[2];
    V8 pf[4];
#pragma unroll
    for (int c4 = 0; c4 < 4; ++c4) pf[c4] = __builtin_bit_cast(V8, u32x4{0, 0, 0, 0});

    auto tile_active = [&](int t) {
        if (t < 0 || t >= n_tiles) return false;
        const int j0 = plan.j0(t);
        return j0 < we.hi_max && j0 + kBN > we.lo_min;
    };

    // One step t of the loop with S = (t + 1) % 3 known at compile time:
    //   reads K_{t+1} from K stage S and V_t from V stage (S + 2) % 3,
    //   loads K_{t+3} into K stage (S + 2) % 3 and V_{t+2} into V stage (S + 1) % 3.
    // head_dim 128: what a step asks is asked once, by scalar selections where that is possible. A load flag for each operand, branches around each
    // cursor and three questions for the wait are 22 scalar branches a step in the dense form, of which 9 are left (24 heads, us, with RoPE and K
    // rotation: 4608 tokens 242 -> 238, 4096 205 -> 200, 1997 62.2 -> 61.2; causal 2048 49.9 -> 49.2; with 669 prefix rows 4096 229 -> 223).
    // head_dim 72, with 9 loads per operand tile dealt to 8 wavefronts, must count its loads for the wait and is slower that way (16 heads,
    // flags for each operand / one: 4608 tokens unsplit 200.4 / 203.8, causal 4096 86.1 / 88.2, biased under a key mask 244 / 251).
    constexpr bool ONE_FLAG = DG::NDMA % 8 == 0;
    auto step = [&](auto stage_tag, int t) {
        constexpr int S = decltype(stage_tag)::value;
        constexpr int KS = S * DG::TILE, VS = ((S + 2) % 3) * DG::TILE;
        constexpr int KD = ((S + 2) % 3) * DG::TILE, VD = DG::VOFF + ((S + 1) % 3) * DG::TILE;
        // (ONE_FLAG: behind K's last tile that one is loaded once more, into the free stage)
        const bool load_v = t + 2 < n_tiles, load_k = ONE_FLAG ? load_v : t + 3 < n_tiles;
        int issued = 0;
        // XTRA: the visibility word of the tile whose softmax this wavefront runs in this step, fetched here, ahead of this
        // step's DMA instructions (an LDS read behind them would wait for them to land)
        TileExtra xt;
        if constexpr (LISTED) {
            vis_t = vis_t1; vis_t1 = vis_t2; vis_t2 = vis_t3;
            const unsigned long long w = kbits[grp == 1 ? vis_t : vis_t1];
            vis_t3 = listed(t + 3);
            xt.kw0 = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(w));
            xt.kw1 = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(w >> 32));
        } else if constexpr (XTRA) {
            if (kbits) {
                const unsigned long long w = kbits[min(max(grp == 1 ? t : t + 1, 0), max(n_tiles - 1, 0))];
                xt.kw0 = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(w));
                xt.kw1 = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(w >> 32));
            }
            xt.bias_cols = p.bias_cols;
        }
        auto softmax_of = [&](int tt) {
            if constexpr (LISTED) {
                if (tt >= 0 && tt < n_tiles) {
                    softmax_tile_rel<T, D, false, true>(sacc, pf, oacc, st, (xt.kw0 & xt.kw1) != ~0u, false, 0, 0, kBN, lh, PrefixScale(), xt);
                    return;
                }
            } else if constexpr (DENSE) {
                if (tt >= 0 && tt < n_tiles) {
                    const int rows = RAGGED ? plan.limit(tt) - plan.j0(tt) : kBN;
                    softmax_tile_rel<T, D, false, false, F32SUM>(sacc, pf, oacc, st, RAGGED && rows < kBN, false, 0, 0, rows, lh);
                    return;
                }
            }
            if (!DENSE && tile_active(tt) && (!XTRA || (xt.kw0 | xt.kw1) != 0u)) {
                const int j0 = plan.j0(tt);
                const int lim = plan.limit(tt);
                bool interior = (j0 >= we.lo_max) && (j0 + kBN <= min(we.hi_min, lim));
                if constexpr (XTRA) {
                    const bool biased = p.bias != nullptr && j0 < p.bias_cols;
                    interior = interior && (xt.kw0 & xt.kw1) == ~0u && !biased;
                    xt.bias_row = biased ? bias_row : nullptr;
                    xt.bias_vec = p.bias_vec_ok && (j0 & 3) == 0 && j0 + kBN <= p.bias_cols;
                }
                softmax_tile_rel<T, D, PSCALE, XTRA, F32SUM>(sacc, pf, oacc, st, !interior, dead_row, j0, lo, min(hi, lim), lh,
                                                     PSCALE ? prefix_scale_of(p, plan.in_prefix(tt)) : PrefixScale(), xt);
            } else {
                // nothing visible to this wavefront in that tile: the next PV pass must add zero
#pragma unroll
                for (int c4 = 0; c4 < 4; ++c4) pf[c4] = __builtin_bit_cast(V8, u32x4{0, 0, 0, 0});
            }
        };
        // An LDS read issued behind an LDS-DMA load does not return before that load has landed (measured: the
        // read takes the full memory latency), so the DMA instructions of a step go where the wavefront has no
        // LDS access ahead of it for a long time: right before its softmax.
        auto issue_dma = [&]() {
            if (ONE_FLAG && !load_v) return;
            if constexpr (LISTED) {
                seek(kc, vis_t3, p.kp, p.kp_bs, p.k, p.k_bs);
                seek(vc, vis_t2, p.vp, p.vp_bs, p.v, p.v_bs);
            }
            issued = dma_tiles(ONE_FLAG || load_k, KD, ONE_FLAG || load_v, VD);
            if constexpr (LISTED) return;
            if constexpr (ONE_FLAG) {
                kc.next(t + 4 < n_tiles);
                vc.next(t + 3 < n_tiles);
            } else if (DENSE && !RAGGED && Lp == 0) {
                if (load_k) kc.ptr += kBN * kc.rsb;
                if (load_v) vc.ptr += kBN * vc.rsb;
            } else {
                if (load_k) kc.next();
                if (load_v) vc.next();
            }
        };
        // group 1 turns the scores of its previous step into P first, so that its MFMA stream meets group 0's softmax
        if (grp == 1) {
            issue_dma();
            MI_SCHED_BARRIER
            softmax_of(t);
            MI_SCHED_BARRIER
        }
        {
            // the stream scores first (S_{t+1} = K_{t+1} Q^T), then O += V_t^T P_t; under the PV MFMAs, which do not touch
            // the scores, each raw score becomes the softmax exponent x = s * cl2 - ref (see mfma_stream)
            constexpr int NQK = 2 * G::KC, NPV = 4 * G::VB, N = NQK + NPV;
            auto fetch = [&](int i) -> V8 {
                if (i >= NQK) {
                    const int j = i - NQK;
                    const int c4 = j / G::VB, vb = j % G::VB;
                    const s16x4 v_lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (__attribute__((address_space(3))) s16x4*)(smem + VS + 16 * c4 * DG::ROWB + vaddr[vb][0]));
                    const s16x4 v_hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (__attribute__((address_space(3))) s16x4*)(smem + VS + 16 * c4 * DG::ROWB + vaddr[vb][1]));
                    const s16x8 a = __builtin_shufflevector(v_lo, v_hi, 0, 1, 2, 3, 4, 5, 6, 7);
                    return __builtin_bit_cast(V8, a);
                } else {
                    const int kb = i / G::KC, c = i % G::KC;
                    u32x4 a = *reinterpret_cast<const u32x4*>(smem + KS + 32 * kb * DG::ROWB + kaddr[c]);
                    // the upper lane half of the last fragment holds the first elements of the NEXT key row where the head
                    // dimension is padded (unpadded rows): blanked, because Q's zero pad does not silence a NaN or an
                    // infinity there, and the next row may be one that this query must not see
                    if (G::DK > D && c == G::KC - 1) a &= pad_keep;
                    return __builtin_bit_cast(V8, a);
                }
            };
            V8 ring[kAhead];
#pragma unroll
            for (int i = 0; i < kAhead; ++i) ring[i] = fetch(i);
            const float neg_ref = st.neg_ref;
            [&]<int... I>(std::integer_sequence<int, I...>) {
                ([&] {
                    constexpr int i = I;
                    const V8 a = ring[i % kAhead];
                    if constexpr (i >= NQK) {
                        constexpr int j = i - NQK;
                        constexpr int c4 = j / G::VB, vb = j % G::VB;
                        oacc[vb] = Mma<T>::run(a, pf[c4], oacc[vb]);
                    } else {
                        constexpr int kb = i / G::KC, c = i % G::KC;
                        if constexpr (c == 0) {
                            const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                            sacc[kb] = Mma<T>::run(a, qf[c], zero);
                        } else {
                            sacc[kb] = Mma<T>::run(a, qf[c], sacc[kb]);
                        }
                    }
                    if constexpr (i + kAhead < N) ring[i % kAhead] = fetch(i + kAhead);
                    if constexpr (i >= NQK) scores_to_exponents<NPV, i - NQK>(sacc, cl2, neg_ref);
                    MI_SCHED_BARRIER
                }(), ...);
            }(std::make_integer_sequence<int, N>{});
        }
        if (grp == 0) {
            MI_SCHED_BARRIER
            issue_dma();
            MI_SCHED_BARRIER
            softmax_of(t + 1);
        }
        // The tiles loaded in the PREVIOUS step are read in the next one: wait for those only (this step's
        // loads stay in flight), then meet the other wavefronts.
        if constexpr (DG::NDMA % 8 == 0) {
            // every wavefront issues NDMA / 8 loads per operand tile
            wait_all_but(load_v ? DG::NDMA / 4 : 0);
        } else {
            wait_all_but(issued);
        }
        __syncthreads();
    };

    if (n_tiles > 0) {
        // prologue: K_0, K_1, V_0 (the loop loads K_{t+3}, V_{t+2} from t = -1 on); cursors end at K_2, V_1
        if constexpr (LISTED) {
            vis_t2 = listed(0); vis_t3 = listed(1);     // (step -1 moves them up by one)
            vis_t1 = vis_t2;                            // never used as tile -1, only kept inside the words
            seek(kc, vis_t2, p.kp, p.kp_bs, p.k, p.k_bs);
            dma_tiles(true, 0, false, 0);
            if (n_tiles > 1) { seek(kc, vis_t3, p.kp, p.kp_bs, p.k, p.k_bs); dma_tiles(true, DG::TILE, false, 0); }
            seek(vc, vis_t2, p.vp, p.vp_bs, p.v, p.v_bs);
            dma_tiles(false, 0, true, DG::VOFF);
        } else {
            dma_tiles(true, 0, false, 0);
            if (n_tiles > 1) { kc.next(); dma_tiles(true, DG::TILE, false, 0); }
            if (n_tiles > 2) kc.next();
            dma_tiles(false, 0, true, DG::VOFF);
            if (n_tiles > 1) vc.next();
        }
    }
    {
        // the Q tile, rotated on its way into the staging buffer behind the rings; every lane then picks the fragments of
        // its own row
        unsigned char* const Qs = smem + DG::QOFF;
        const bool split_pairs = p.cos_q != nullptr && p.rope_split;
        if constexpr (!DG::Q_HALVES) {
            ql.store(Qs, p, q0, tid, p.Lq - 1);
            if (split_pairs) {
                __syncthreads();
                rope_split_staged<T, D, kThreads8>(Qs, p, q0, tid, p.Lq - 1, 1.f, 0, BM);
            }
            __syncthreads();
            read_q_frags<T, D>(qf, Qs, wave * 32 + lq, lh);
        } else {
            ql.template store<0, QL::NI / 2>(Qs, p, q0, tid, p.Lq - 1, 1.f, 0);
            if (split_pairs) {
                __syncthreads();
                rope_split_staged<T, D, kThreads8>(Qs, p, q0, tid, p.Lq - 1, 1.f, 0, BM / 2);
            }
            __syncthreads();
            if (grp == 0) read_q_frags<T, D>(qf, Qs, wave * 32 + lq, lh);
            __syncthreads();
            ql.template store<QL::NI / 2, QL::NI>(Qs, p, q0, tid, p.Lq - 1, 1.f, BM / 2);
            if (split_pairs) {
                __syncthreads();
                rope_split_staged<T, D, kThreads8>(Qs, p, q0, tid, p.Lq - 1, 1.f, BM / 2, BM / 2);
            }
            __syncthreads();
            if (grp == 1) read_q_frags<T, D>(qf, Qs, (wave - 4) * 32 + lq, lh);
        }
    }
    if (n_tiles > 0) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        for (int t = -1; t < n_tiles; t += 3) {
            step(std::integral_constant<int, 0>{}, t);
            if (t + 1 >= n_tiles) break;
            step(std::integral_constant<int, 1>{}, t + 1);
            if (t + 2 >= n_tiles) break;
            step(std::integral_constant<int, 2>{}, t + 2);
        }
    }

    const float l_tot = exchange_sum(st.l);
    const float inv = row_inverse(l_tot);
    if constexpr (XTRA && !SPLIT) {
        // base-2 log of the row's denominator in exponent units: p(key) = exp2(score * scale_log2 [+ bias * log2 e] - lse);
        // +inf for a row without visible keys, so that every p is 0
        if (p.lse && qvalid && lh == 0)
            p.lse[(static_cast<long>(b) * p.H + h) * p.Lq + qrow] = l_tot > 0.f ? __builtin_amdgcn_logf(l_tot) - st.neg_ref : __builtin_huge_valf();
    }
    if (SPLIT && LISTED && part != nullptr && !alone && n_tiles == 0) {
        if (tid < BM) part_stats<D>(part)[BM + tid] = 0.f;      // a part without a tile: the merge looks no further
    } else if (!SPLIT || part == nullptr || alone) {
        stage_output<T, D>(smem, wave * 32 + lq, lh, oacc, inv);
        __syncthreads();
        write_output<T, D, kThreads8>(smem, o_base, p.o_rs, q0, p.Lq, BM, tid);
        if (SPLIT && LISTED && alone && part != nullptr && tid < BM) part_stats<D>(part)[BM + tid] = kWholeTile;
    } else {
        // the accumulators of the part as the lanes hold them: 16-byte piece (wave D / 8 + c) 64 + lane is head-dim elements
        // 8 c + 4 lh .. + 3 of row 32 wave + lq; then per row the softmax reference (log2 domain) and the denominator relative
        // to it: the part's weight in the merge is 2^ref
        f32x4* const slot = reinterpret_cast<f32x4*>(part) + wave * (D / 8) * 64 + lane;
#pragma unroll
        for (int c = 0; c < D / 8; ++c) {
            const f32x16 block = oacc[c >> 2];
            const int e = 4 * (c & 3);
            slot[c * 64] = f32x4{block[e], block[e + 1], block[e + 2], block[e + 3]};
        }
        if (lh == 0) {
            float* const stat = part_stats<D>(part);
            stat[wave * 32 + lq] = -st.neg_ref;
            stat[BM + wave * 32 + lq] = l_tot;
        }
    }
    if constexpr (!SPLIT) {
        break;
    } else {
        if (whole || seg_s >= seg_end) break;
        __syncthreads();   // the staged output is read by all threads before the next part stages its Q tile
    }
  }
}

// Merge of the parts of one split query tile: out = sum_k w_k O_k / sum_k w_k l_k with w_k = 2^(ref_k - max ref), FP32, one
// rounding. blockIdx.x = (XCD group, tail tile); tiles that were written whole are skipped.
template <typename T, int D>
__global__ void __launch_bounds__(256) sdpa_combine_kernel(const SdpaDev p) {
    typedef T t8 __attribute__((ext_vector_type(8)));
    constexpr int BM = 256, CPR = D / 8;
    const SplitGeo& sg = p.split;
    const int xg = static_cast<int>(blockIdx.x) & 7, tt = static_cast<int>(blockIdx.x) >> 3;
    if (tt >= sg.tail_of(xg)) return;
    const int S = sg.tail_of(xg) * sg.T, np = sg.pieces_for(S);
    const int first = SplitGeo::piece_of(tt * sg.T, S, np);
    const int n_parts = SplitGeo::piece_of((tt + 1) * sg.T - 1, S, np) - first + 1;
    if (n_parts == 1) return;
    const int logical = xg * sg.chunk + sg.full_of(xg) + tt;
    const int qt = logical % p.n_q_tiles, bh = logical / p.n_q_tiles;
    const int h = bh % p.H, b = bh / p.H;
    const int q0 = qt * BM;
    T* const o_base = static_cast<T*>(p.o) + b * p.o_bs + h * D;
    const unsigned char* slots = p.split_scratch + static_cast<long>(xg * sg.max_tail + tt) * sg.max_parts * SplitGeo::slot_bytes(D);
    // 8 head-dim elements of one row per thread, 8 consecutive threads the same elements of 8 rows (128 bytes of a part
    // together); blockIdx.y walks the tile (many short work groups: the merge is a chain of two dependent loads per part,
    // hidden by occupancy rather than by unrolling)
    {
        const int idx = static_cast<int>(blockIdx.y) * 256 + static_cast<int>(threadIdx.x);
        if (idx >= BM * CPR) return;
        const int cc = (idx >> 3) % CPR, row = (idx >> 3) / CPR * 8 + (idx & 7);
        if (q0 + row >= p.Lq) return;
        const long piece0 = ((row >> 5) * CPR + cc) * 64 + (row & 31);
        // a part without visible keys has denominator 0 and is skipped; one whose denominator is NaN (a non-finite score)
        // must not be: it makes the row NaN, as it would in an unsplit launch. Hence the test on the bits.
        // (the bits pass through an empty asm statement: left visible, the optimiser turns the integer test back into a
        //  floating-point comparison that is false for a NaN, which -fno-honor-nans entitles it to)
        auto empty = [](float l) {
            unsigned bits = __builtin_bit_cast(unsigned, l);
            asm volatile("" : "+v"(bits));
            return (bits & 0x7fffffffu) == 0u;
        };
        if (__builtin_bit_cast(unsigned, part_stats<D>(slots)[BM + row]) == __builtin_bit_cast(unsigned, kWholeTile)) return;
        float ref = kNegInf;
        for (int k = 0; k < n_parts; ++k) {
            const float* stat = part_stats<D>(slots + k * SplitGeo::slot_bytes(D));
            if (!empty(stat[BM + row])) ref = fmaxf(ref, stat[row]);
        }
        float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        float lsum = 0.f;
        for (int k = 0; k < n_parts; ++k) {
            const unsigned char* slot = slots + k * SplitGeo::slot_bytes(D);
            const float* stat = part_stats<D>(slot);
            const float l = stat[BM + row];
            if (empty(l)) continue;           // (its values may not be written)
            const f32x4 lo = reinterpret_cast<const f32x4*>(slot)[piece0], hi = reinterpret_cast<const f32x4*>(slot)[piece0 + 32];
            const float w = __builtin_amdgcn_exp2f(stat[row] - ref);
            lsum = __builtin_fmaf(w, l, lsum);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                acc[e] = __builtin_fmaf(w, lo[e], acc[e]);
                acc[4 + e] = __builtin_fmaf(w, hi[e], acc[4 + e]);
            }
        }
        const float inv = row_inverse(lsum);
        t8 out;
#pragma unroll
        for (int e = 0; e < 8; ++e) out[e] = static_cast<T>(acc[e] * inv);
        *reinterpret_cast<t8*>(o_base + static_cast<long>(q0 + row) * p.o_rs + cc * 8) = out;
    }
}

// LDS behind the tile buffers for the visibility words of a key mask, and with the list of the tiles that have a visible key (kRagged with XTRA)
long kbits_bytes_of(const SdpaDev& p) { return p.key_mask ? 8L * ((p.Lk + kBN - 1) / kBN + 2) : 0; }
long listed_bytes_of(const SdpaDev& p) { return kbits_bytes_of(p) + kbits_bytes_of(p) / 4; }
constexpr long kMaxKbits = 24 * 1024;     // (the words share the LDS with rings and Q staging)
template <int D>
bool listed_fits(const SdpaDev& p) {
    return kbits_bytes_of(p) <= kMaxKbits && DmaGeo<D>::lds_bytes() + listed_bytes_of(p) + 256 <= 160 * 1024;
}

// Decides whether the launch splits its last round (see SplitGeo) and fills p.split. The split costs every tail work
// group a second prologue and the launch a merge pass (together about ten key steps), so it is taken only when it
// shortens the last round by more than that — and only when the last round would fill at most half of the GPU:
// under sustained MFMA load the GPU runs at its power limit, a partly idle last round runs at a higher clock, and
// measured time follows the total work rather than the number of rounds (432 tiles on 256 compute units take 1.70
// times one full round, not 2). Both sides (us, unsplit / split, with RoPE and K rotation; rounds, and the last one's share in 32):
//   dense, 128:  24 heads, 2816 tokens (1.03, 1) 140.1 / 113.9, 3328 (1.22, 7) 162.9 / 149.7, 3584 (1.31, 10) 175.1 / 166.0, 4096 (1.5, 16) 200.0 / 197.7,
//                6144 (2.25, 8) 448 / 400, 6656 (2.44, 14) 484 / 472; 32 heads, 4608 (2.25, 8) 346 / 314; 48 heads, 4352 (3.19, 6) 455 / 428, 4608
//                (3.38, 12) 480 / 470
//   ragged, 128: 24 heads, 2800 (1.03, 1) 145.7 / 117.3, 3300 (1.22, 7) 169.2 / 152.1, 4080 (1.5, 16) 205.5 / 199.3, 6600 (2.44, 14) 498 / 480; 48 heads,
//                4600 (3.38, 12) 493 / 479
//   72:          16 heads, 4608 (1.13, 4) 198.9 / 139.6, 4600 201.0 / 141.8; 40 heads, 1792 (1.09, 3) 89.5 / 79.6
// A key mask may hide tiles, which is known on the GPU only: planned as if all were visible, where that gains twice what an unmasked call has to, and
// decided there for each batch item. Visible keys: all, half, a quarter, an eighth, one:
//   48 / 12 heads of 128, 4608 (3.38, 12)  484 / 469, 268 / 272, 162 / 168, 110 / 115, 68 / 73
//   24 heads of 128, 2816 (1.03, 1)        146.7 / 119.1, 87.5 / 79.2, 58.0 / 62.0, 45.2 / 49.2, 33.1 / 37.0
//                    3328 (1.22, 7)        169.8 / 154.2, 99.6 / 102.2, 64.7 / 69.2, 49.3 / 53.7, 34.5 / 39.0
//                    4096 (1.5, 16)        206.2 / 200.0, 120.1 / 122.4, 77.2 / 81.9, 55.4 / 60.4, 38.8 / 43.6
//   16 heads of 128, 4608 (1.13, 4)        224.7 / 178.1, 127.9 / 112.3, 79.2 / 79.9, 55.0 / 59.1, 35.8 / 39.9
//   16 heads of 72, 4608 (1.13, 4)         200.5 / 145.4, 112.2 / 92.5, 67.7 / 66.6, 46.0 / 49.9, 28.1 / 32.5
// Where nothing is cut the launch still takes the merge pass (2.3 us, which then finds nothing to do) and a longer start of every tile.
template <int D>
bool plan_split(SdpaDev& p, int n_cu) {
    p.split = SplitGeo{};
    if constexpr (!dma_kernel_available<D>()) return false;
    if (sdpa_kernel_choice() == 0 && sdpa_flow_takes(p, D, n_cu)) return false;
    if (p.mask_mode != MI_MASK_NONE || p.kv_valid_len || p.Lp > 0 || p.cos_k || p.cu_q) return false;
    // (the split form neither adds a logit bias nor writes the softmax denominators)
    if (p.bias != nullptr || p.lse != nullptr) return false;
    if constexpr (dma_kernel_available<D>()) {
        if (p.key_mask && !listed_fits<D>(p)) return false;
    }
    if (n_cu < 8 || n_cu % 8 != 0 || sdpa_kernel_choice() == 1 || sdpa_kernel_choice() == 3) return false;
    const long tiles = static_cast<long>(p.B) * p.H * ((p.Lq + 255) / 256);
    const int T = (p.Lk + kBN - 1) / kBN;
    if (tiles < n_cu || tiles > (1 << 24) || T < 16 || T > (1 << 20)) return false;
    SplitGeo g{};
    g.T = T; g.n_blocks = static_cast<int>(tiles); g.chunk = static_cast<int>((tiles + 7) / 8); g.cu_g = n_cu / 8;
    const int tail0 = g.tail_of(0);
    if (tail0 == 0 || 2 * tail0 > g.cu_g) return false;
    const int np0 = g.pieces_for(tail0 * T);
    const int piece_len = (tail0 * T + np0 - 1) / np0;
    if (T - piece_len < (p.key_mask ? 24 : 12)) return false;
    // Under a key mask a tile is cut if that shortens it by 12 visible tiles, by 18 where a piece may hold two parts and so starts twice (pieces
    // that do not divide the tiles evenly). The sides meet at (visible tiles saved): 24 heads, 4096 tokens 12; 16 of 72, 4608 10, of 128 12; 24 heads, 2816 7;
    // pieces of two parts: 48 / 12 heads, 4608 19; 24 heads, 3328 18.
    const int pays = np0 % tail0 == 0 ? 12 : 18;
    g.min_visible = (pays * T + T - piece_len - 1) / (T - piece_len);
    for (int xg = 0; xg < 8; ++xg) {
        const int tail = g.tail_of(xg), S = tail * T, np = g.pieces_for(S);
        g.max_tail = max(g.max_tail, tail);
        for (int tt = 0; tt < tail; ++tt)
            g.max_parts = max(g.max_parts, SplitGeo::piece_of((tt + 1) * T - 1, S, np) - SplitGeo::piece_of(tt * T, S, np) + 1);
    }
    g.enabled = 1;
    p.split = g;
    return true;
}
template <int D>
size_t split_scratch_bytes_d(SdpaDev p, int n_cu) {
    if (!plan_split<D>(p, n_cu)) return 0;
    return static_cast<size_t>(8) * p.split.max_tail * p.split.max_parts * SplitGeo::slot_bytes(D);
}

// Every query row sees the same keys of its batch item: the kRagged form (and, with whole tiles, kDense) can take the call.
bool same_keys_for_all_rows(const SdpaDev& p) {
    return p.mask_mode == MI_MASK_NONE && !p.prefix_scaled && (p.Lp == 0 || (p.kp_rs == p.k_rs && p.vp_rs == p.v_rs));
}

// Whether a launch that comes here runs on 256-row tiles (8 wavefronts, two per SIMD, softmax of one under the MFMAs of the other) or on
// 128-row tiles. With a 256-row tile or more per CU the former always. Below that the 128-row kernel keeps more CUs busy, but
// each of them runs one wavefront per SIMD whose softmax nothing hides, and from the 257th work group on two share a CU
// anyway ("crowded"); a CU with eight wavefronts needs 2/3 of the time per row and key, and costs about 1.5 us more to start
// (rings, two-part Q staging).
// What asks below a tile per CU: calls with extras or K rotated by tile, masked ones of more rows than sdpa_small.hip takes, and plain ones
// of 40, 64 and 128 above the lines of sdpa_flow_takes (all of them on 256 rows: those of 128 are crowded and have more than three key
// tiles). The other plain lines are met only by K or V of 2 GiB and more, whose offsets sdpa_small.hip and sdpa_flow.hip do not hold. The lines are where the two sides meet (us, 128-row /
// 256-row, 8 heads of 40 and 80, 16 of 64, 72 and 96, 24 of 128; over a sweep of 156 such calls the side taken is at most 7 % slower than the
// other, 0.6 % on average):
//   128, no mask:      T = 4 11.5 / 12.5, 5 13.3 / 13.9, 8 18.0 / 17.3, 16 30.8 / 26.9, 32 (192 tiles) 74.7 / 52.7; cross, 3 key
//                      tiles, 216 query tiles 15.0 / 14.6, 96 query tiles 11.1 / 12.7
//   72, no mask:       T = 4 11.4 / 10.8, 5 12.9 / 12.0, cross with 2 9.2 / 10.1, with 5 13.4 / 13.5, 16 29.3 / 23.6, 36 (144
//                      tiles) 70.4 / 45.7
//   40 and 64:         equal or faster from one key tile on (6.4 / 5.7 and 5.7 / 5.7; 1024 tokens 24.3 / 18.5 and 24.1 / 19.2)
//   128, 72 masked:    T = 8 18.2 / 19.4 and 17.7 / 17.8, 16 31.0 / 29.7 and 29.6 / 27.1, 32 (192 tiles, block-causal) 79.1 / 54.8
//   80, 96, 112:       crowded only: 144 tiles of 96 69.1 / 56.2, 192 tiles 92.2 / 74.1, 128 of 80 100 / 111; masked never (96,
//                      160 tiles: 58.7 / 60.7)
//   K rotated by tile: crowded only: 128, 144 tiles 70.9 / 55.9, 96 tiles 40.7 / 39.0; 40, 40 tiles 35.3 / 36.9
template <int D>
bool rows256_pay(const SdpaDev& p, int n_cu, bool xtra) {
    const long heads = static_cast<long>(p.B) * p.H;
    const int T = (p.Lk + kBN - 1) / kBN;
    if (heads * ((p.Lq + 255) / 256) >= n_cu) return true;
    if (p.prefix_scaled) return false;
    const bool crowded = heads * ((p.Lq + 127) / 128) > n_cu;
    if (p.cos_k != nullptr) return crowded && T >= 16;
    const bool plain = !xtra && same_keys_for_all_rows(p);
    if constexpr (dma_kernel_available<D>()) {
        if (!plain) return T >= (crowded ? 12 : 16);
        return crowded ? T >= 3 : T >= (D == 72 ? 5 : 8);
    }
    if (D <= 64) return plain && p.Lp == 0;
    return plain && crowded && T >= 16;
}

// How many 256-row tiles of a head a work group of the short-key kernel walks, and the tiles that the busiest CU then has. The fewest
// of the latter; among equals the most tiles per group (each group loads the head's keys once). Rounding tiles per CU down instead
// gave a second, nearly empty round of groups as long as the first: with 2.5 to 7.5 tiles per CU 20 to 60 % of the launch.
struct ShortPlan { int tiles = 1; long busiest = 0; };
ShortPlan plan_short(long heads, int q_tiles, int n_cu) {
    ShortPlan best;
    auto consider = [&](int n) {
        const long groups = heads * ((q_tiles + n - 1) / n), busiest = (groups + n_cu - 1) / n_cu * n;
        if (best.busiest == 0 || busiest <= best.busiest) best = {n, busiest};
    };
    for (int n = 1; n <= min(q_tiles, 16); ++n) consider(n);
    const int per_head = max(1, static_cast<int>(n_cu / heads));      // groups of a head that one round holds
    const int one_round = (q_tiles + per_head - 1) / per_head;
    if (one_round > 16) consider(one_round);
    return best;
}

// Whether a call whose keys fit LDS is faster on the short-key kernel than on sdpa_flow.hip, which deals rows out finer and takes time
// in proportion to the rows, where the short-key kernel takes that of whole rounds of 256-row tiles per CU; it is the better one
// from a round that is nearly full on, the more so the more rounds share one load of the keys (us, short-key / flow, 16 heads of 40
// and 72, 77 keys: 1.06 tiles per CU 12.6 / 9.3 and 15.9 / 11.8, 1.5 12.8 / 9.8 and 16.6 / 12.6, 2 11.8 / 11.8 and 15.3 / 16.5, 2.5
// (as 3) 15.6 / 14.9 and 19.8 / 19.8, 3 15.6 / 17.3 and 19.8 / 22.9, 4 18.9 / 23.0 and 24.2 / 28.7; 154 keys 1.5 15.9 / 11.2). 112: 1 16.8 /
// 12.5, 8 74.7 / 67.9. 128 stays here, where it gives the same bits as the 128-row kernel (1.5 tiles per CU 20.6 / 17.2).
template <int D>
bool shortkv_pays(const ShortPlan& plan, long tiles256, int n_cu) {
    if (D == 112) return false;
    return D == 128 || plan.busiest >= 4 || 16 * tiles256 >= 15 * plan.busiest * n_cu;
}

template <typename T, int D>
int launch_d(SdpaDev p, int n_cu, hipStream_t stream) {
    const bool rope_k = p.cos_k != nullptr;
    if (p.cu_q != nullptr) {
        p.n_q_tiles = (p.Lq + 127) / 128;
        p.n_blocks = p.B * p.H * p.n_q_tiles;
        hipLaunchKernelGGL((sdpa_fwd_kernel<T, D, false, true>), dim3(grid_blocks(p)), dim3(kThreads4), lds_bytes_4<D>(), stream, p);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return fail("sdpa_fwd launch: %s", hipGetErrorString(e));
        return 0;
    }
    const int choice = sdpa_kernel_choice();
    const long tiles256 = static_cast<long>(p.B) * p.H * ((p.Lq + 255) / 256);
    // short key sequences whose K and V fit in LDS next to a query tile: one work group walks several query tiles
    const int n_kt = (p.Lk + kBN - 1) / kBN;
    const bool short_keys = D <= 128 && choice == 0 && p.mask_mode == MI_MASK_NONE && p.bias == nullptr && p.lse == nullptr && p.Lp == 0 && !rope_k &&
                            p.cos_q == nullptr && n_kt >= 1 && n_kt <= shortkv_max_tiles<(D <= 128 ? D : 128)>() && tiles256 >= n_cu &&
                            shortkv_lds_bytes<D>(n_kt, p.key_mask != nullptr) <= 160 * 1024;
    const ShortPlan short_plan = short_keys ? plan_short(static_cast<long>(p.B) * p.H, (p.Lq + 255) / 256, n_cu) : ShortPlan{};
    const bool flow = short_keys ? sdpa_flow_runs(p) && !shortkv_pays<D>(short_plan, tiles256, n_cu) : choice == 0 && sdpa_flow_takes(p, D, n_cu);
    if (flow) return launch_sdpa_flow(p, std::is_same_v<T, __bf16> ? MI_DTYPE_BF16 : MI_DTYPE_F16, D, n_cu, short_keys, stream);
    if constexpr (dma_kernel_available<D>()) {
        if (p.split_scratch != nullptr && plan_split<D>(p, n_cu) &&
            p.split_scratch_bytes >= static_cast<size_t>(8) * p.split.max_tail * p.split.max_parts * SplitGeo::slot_bytes(D)) {
            p.n_q_tiles = (p.Lq + 255) / 256;
            p.n_blocks = p.split.n_blocks;
            int per_group = 0;
            for (int xg = 0; xg < 8; ++xg)
                per_group = max(per_group, p.split.full_of(xg) + p.split.pieces_for(p.split.tail_of(xg) * p.split.T));
            const dim3 grid(8 * per_group), block(kThreads8);
            p.kbits_off = DmaGeo<D>::lds_bytes();
            if (p.key_mask) hipLaunchKernelGGL((sdpa_fwd_pp_dma_kernel<T, D, true, kRagged, false, true>), grid, block, DmaGeo<D>::lds_bytes() + listed_bytes_of(p), stream, p);
            else if (p.Lk % kBN == 0) hipLaunchKernelGGL((sdpa_fwd_pp_dma_kernel<T, D, true, kDense>), grid, block, DmaGeo<D>::lds_bytes(), stream, p);
            else hipLaunchKernelGGL((sdpa_fwd_pp_dma_kernel<T, D, true, kRagged>), grid, block, DmaGeo<D>::lds_bytes(), stream, p);
            hipLaunchKernelGGL((sdpa_combine_kernel<T, D>), dim3(8 * p.split.max_tail, (256 * (D / 8) + 255) / 256), dim3(256), 0, stream, p);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return fail("sdpa_fwd launch: %s", hipGetErrorString(e));
            return 0;
        }
        p.split = SplitGeo{};
    }
    // head_dim above 128 does not fit two wavefronts per SIMD and stays on the 128-row kernel
    // calls with a key mask, a logit bias or a request for the softmax denominators take the XTRA instances of the 256-row
    // kernels (visibility words of all key tiles in LDS behind the tile buffers), unless K is rotated tile by tile, the
    // prefix-KV dial is on as well, or the key sequence is too long for the words to fit: then the 128-row kernel
    const bool xtra = p.key_mask != nullptr || p.bias != nullptr || p.lse != nullptr;
    const long kbits_bytes = kbits_bytes_of(p);
    const bool xtra_ok = !xtra || (!rope_k && !p.prefix_scaled && kbits_bytes <= kMaxKbits);
    // calls with the prefix-KV dial stay on the 128-row kernel unless the DMA kernel (which has an instance for it) takes them
    const bool dial_ok = !p.prefix_scaled || (dma_kernel_available<D>() && !rope_k && choice != 3);
    const bool pingpong = D <= 128 && xtra_ok && dial_ok && (choice >= 2 || (choice == 0 && rows256_pay<D>(p, n_cu, xtra)));
    if (short_keys) {
        if constexpr (D <= 128) {
            p.n_q_tiles = (p.Lq + 255) / 256;
            const int n_strip = short_plan.tiles;
            const int strips_per_head = (p.n_q_tiles + n_strip - 1) / n_strip;
            p.n_blocks = p.B * p.H * strips_per_head;
            hipLaunchKernelGGL((sdpa_shortkv_kernel<T, D>), dim3(grid_blocks(p)), dim3(kThreads8), shortkv_lds_bytes<D>(n_kt, p.key_mask != nullptr), stream, p,
                               n_kt, 8 * n_strip, strips_per_head);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return fail("sdpa_fwd launch: %s", hipGetErrorString(e));
            return 0;
        }
    }
    if (pingpong) {
        p.n_q_tiles = (p.Lq + 255) / 256;
        p.n_blocks = static_cast<int>(tiles256);
        const dim3 grid(grid_blocks(p)), block(kThreads8);
        if constexpr (D <= 128) {
            if (xtra) {
                const bool dma = dma_kernel_available<D>() && sdpa_kernel_choice() != 3;
                if constexpr (dma_kernel_available<D>()) {
                    if (dma && p.key_mask && !p.bias && same_keys_for_all_rows(p) && listed_fits<D>(p)) {
                        p.kbits_off = DmaGeo<D>::lds_bytes();
                        const long lds = DmaGeo<D>::lds_bytes() + listed_bytes_of(p);
                        // (without a prefix, with RoPE and K rotation, us, looking for one / not: 48 / 12 heads of 128, 1100 tokens 43.2 / 42.4, 3000 255 / 245,
                        // 4928 548 / 532, one key visible of 3000 48.0 / 46.9; 16 of 72, 1100 34.5 / 32.9, 3000 76.6 / 72.5)
                        if (p.Lp == 0) hipLaunchKernelGGL((sdpa_fwd_pp_dma_kernel<T, D, false, kFresh, false, true>), grid, block, lds, stream, p);
                        else hipLaunchKernelGGL((sdpa_fwd_pp_dma_kernel<T, D, false, kRagged, false, true>), grid, block, lds, stream, p);
                    }
                    else if (dma) {
                        p.kbits_off = DmaGeo<D>::lds_bytes();
                        hipLaunchKernelGGL((sdpa_fwd_pp_dma_kernel<T, D, false, kGeneral, false, true>), grid, block,
                                           DmaGeo<D>::lds_bytes() + kbits_bytes, stream, p);
                    }
                }
                if (!dma) {
                    p.kbits_off = lds_bytes_8<D>();
                    hipLaunchKernelGGL((sdpa_fwd_pp_kernel<T, D, false, kGeneral, true>), grid, block, lds_bytes_8<D>() + kbits_bytes, stream, p);
                }
            }
            else {
                auto launch = [&](auto f32_sum) {
                    constexpr bool F = decltype(f32_sum)::value;
                    if (rope_k) {
                        hipLaunchKernelGGL((sdpa_fwd_pp_kernel<T, D, true, kGeneral, false, F>), grid, block, lds_bytes_8<D>(), stream, p);
                        return;
                    }
                    const bool dense = p.mask_mode == MI_MASK_NONE && p.kv_valid_len == nullptr && p.Lk % kBN == 0 && !p.prefix_scaled;
                    if constexpr (dma_kernel_available<D>()) {
                        if (sdpa_kernel_choice() != 3) {
                            constexpr int lds = DmaGeo<D>::lds_bytes();
                            // whole key tiles only; a cached prefix may come first if it is whole tiles too and laid out like K / V
                            const bool whole = dense && (p.Lp == 0 || (p.Lp % kBN == 0 && p.kp_rs == p.k_rs && p.vp_rs == p.v_rs));
                            if (whole) hipLaunchKernelGGL((sdpa_fwd_pp_dma_kernel<T, D, false, kDense, false, false, F>), grid, block, lds, stream, p);
                            else if (same_keys_for_all_rows(p)) hipLaunchKernelGGL((sdpa_fwd_pp_dma_kernel<T, D, false, kRagged, false, false, F>), grid, block, lds, stream, p);
                            else if (p.prefix_scaled) hipLaunchKernelGGL((sdpa_fwd_pp_dma_kernel<T, D, false, kGeneral, true>), grid, block, lds, stream, p);
                            else hipLaunchKernelGGL((sdpa_fwd_pp_dma_kernel<T, D, false, kGeneral, false, false, F>), grid, block, lds, stream, p);
                            return;
                        }
                    }
                    if constexpr (D <= 64) {
                        if (p.mask_mode == MI_MASK_NONE && p.Lp == 0) {
                            if (dense) hipLaunchKernelGGL((sdpa_fwd_pp_kernel<T, D, false, kDense, false, F>), grid, block, lds_bytes_8<D>(), stream, p);
                            else hipLaunchKernelGGL((sdpa_fwd_pp_kernel<T, D, false, kRagged, false, F>), grid, block, lds_bytes_8<D>(), stream, p);
                            return;
                        }
                    }
                    // (below one tile per CU only 80 and 96 come here, with K or V of 2 GiB and more: rows256_pay)
                    if constexpr (!F || D > 72) hipLaunchKernelGGL((sdpa_fwd_pp_kernel<T, D, false, kGeneral, false, F>), grid, block, lds_bytes_8<D>(), stream, p);
                };
                // the form of the denominators (from head_dim 112 on there is one)
                if constexpr (HeadGeo<D>::VB < 4) {
                    if (choice == 0 && tiles256 < n_cu) launch(std::true_type{});
                    else launch(std::false_type{});
                } else launch(std::false_type{});
            }
        }
    } else {
        p.n_q_tiles = (p.Lq + 127) / 128;
        p.n_blocks = p.B * p.H * p.n_q_tiles;
        const dim3 grid(grid_blocks(p)), block(kThreads4);
        if (p.prefix_scaled) {
            if (rope_k) return fail("mi_sdpa_forward: the prefix-KV dial with K rotated tile by tile is not supported (lend rope_k_scratch)");
            hipLaunchKernelGGL((sdpa_fwd_kernel<T, D, false, false, true>), grid, block, lds_bytes_4<D>(), stream, p);
        }
        else if (rope_k) hipLaunchKernelGGL((sdpa_fwd_kernel<T, D, true>), grid, block, lds_bytes_4<D>(), stream, p);
        else hipLaunchKernelGGL((sdpa_fwd_kernel<T, D, false>), grid, block, lds_bytes_4<D>(), stream, p);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail("sdpa_fwd launch: %s", hipGetErrorString(e));
    return 0;
}

template <typename T>
int launch_t(const SdpaDev& p, int head_dim, int n_cu, hipStream_t stream) {
    switch (head_dim) {
        case 40: return launch_d<T, 40>(p, n_cu, stream);
        case 64: return launch_d<T, 64>(p, n_cu, stream);
        case 72: return launch_d<T, 72>(p, n_cu, stream);
        case 80: return launch_d<T, 80>(p, n_cu, stream);
        case 96: return launch_d<T, 96>(p, n_cu, stream);
        case 112: return launch_d<T, 112>(p, n_cu, stream);
        case 128: return launch_d<T, 128>(p, n_cu, stream);
        case 160: return launch_d<T, 160>(p, n_cu, stream);
        default: return fail("mi_sdpa_forward: head_dim %d has no kernel (40, 64, 72, 80, 96, 112, 128, 160, 256, 384, 512)", head_dim);
    }
}

}  // namespace

bool sdpa_supported(int dtype, int head_dim) {
    if (dtype != MI_DTYPE_F16 && dtype != MI_DTYPE_BF16) return false;
    switch (head_dim) {
        case 40: case 64: case 72: case 80: case 96: case 112: case 128: case 160: return true;
        default: return sdpa_wide_head(head_dim);
    }
}

size_t sdpa_split_scratch_bytes(const SdpaDev& p, int dtype, int head_dim) {
    if (dtype != MI_DTYPE_BF16 && dtype != MI_DTYPE_F16) return 0;
    if (sdpa_wide_head(head_dim)) return sdpa_wide_split_scratch_bytes(p, head_dim);
    const int n_cu = device_cu_count();
    if (head_dim == 72) return split_scratch_bytes_d<72>(p, n_cu);
    if (head_dim == 128) return split_scratch_bytes_d<128>(p, n_cu);
    return 0;
}

int launch_sdpa(const SdpaDev& p, int dtype, int head_dim, hipStream_t stream) {
    if (sdpa_wide_head(head_dim)) return launch_sdpa_wide(p, dtype, head_dim, stream);
    if ((dtype == MI_DTYPE_BF16 || dtype == MI_DTYPE_F16) && sdpa_kernel_choice() == 0 && sdpa_small_takes(p, head_dim))
        return launch_sdpa_small(p, dtype, head_dim, stream);
    const int n_cu = device_cu_count();
    if (dtype == MI_DTYPE_BF16) return launch_t<__bf16>(p, head_dim, n_cu, stream);
    if (dtype == MI_DTYPE_F16) return launch_t<_Float16>(p, head_dim, n_cu, stream);
    return fail("mi_sdpa_forward: dtype %d not supported (fp16 = 1, bf16 = 2)", dtype);
}

}  // namespace mi
