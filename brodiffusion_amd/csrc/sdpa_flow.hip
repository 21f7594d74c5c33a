// Softmax attention, unmasked, for everything between the few-row calls of sdpa_small.hip and whole rounds of the 256-row kernels.
//
// A work group is 4 wavefronts of 32 query rows; they share 64-key tiles of K and V in LDS (panels, see PanelReads: 64-byte pieces
// of a row, no bank conflicts, two buffers) and meet at one barrier per tile. Per tile a wavefront
//   waits for its share of the tile, requested a whole tile earlier, and meets the others;
//   scores it: 2 KC products on two independent accumulators in turn (a chain on one costs a third more), the next tile's DMA
//   instructions dealt out between them without a branch (past the last tile that one is loaded again into the free buffer);
//   turns the scores into probabilities relative to the row's reference, as the 256-row kernels do (softmax_tile_rel), with FP32
//   row sums in four chains;
//   multiplies the values, fragments read four ahead.
// No LDS read waits for a DMA load: measured, a read issued right behind four of them returns in the usual 56 clocks. Two to four
// such groups share a CU (121 to 126 registers at head_dim 40, 126 to 166 at 64 to 96, 202 to 244 above) and drift apart, so that the
// softmax of one runs under the products of the other without a schedule between them, and 128-row tiles leave half as much of a last
// round idle as 256-row ones.
// At head_dim 40 and 72 the places past the end of a row are not loaded but zeroed once: the products that they feed are of zeros,
// which costs the power-limited matrix unit less (72, 8192 tokens 378 -> 365 us); at 80 to 112 that masking costs more than it saves.
// What bounds it: with all of the GPU at work the clock that the power limit leaves (72, 16 x 4096 tokens: as many cycles on zeros as on
// N(0, 1), but 2.12 against 1.65 GHz, 71 against 91 us: profiles/model_blocks_counters.txt); with fewer groups than CUs the chain above
// (about 2000 clocks per tile at head_dim 72, of which 700 are products).
// Measured (us, before -> now; 256-row kernels, 128-row kernel for 160): 16 heads of 72, 2304 tokens 45.0 -> 41.1, 4096 100 -> 97; 8
// heads of 80, batch 2, 2048 55 -> 32, 3072 93 -> 63, 4096 128 -> 98; 8 of 160, 4096 140 -> 92; 24 of 128, 1100 29.6 -> 24.2; 8 of 40, 1.25
// rounds of 256-row tiles 309 -> 234.
#include "sdpa_tiles.h"

namespace mi {
namespace {

using namespace sdpa;

constexpr int kRows = 128, kThreads = 256;

template <int D> struct FlowGeo {
    using G = HeadGeo<D>;
    static constexpr int NP = G::VB;                               // panels of 32 head-dim elements
    static constexpr int PANEL = 32 * 64;                          // bytes of 32 keys of a panel
    static constexpr int OPER = NP * PANEL, BLOCK = 2 * OPER;      // K or V of 32 keys; both
    static constexpr int TILE = 2 * BLOCK;
    static constexpr int LDS = 2 * TILE > kRows * G::O_STRIDE ? 2 * TILE : kRows * G::O_STRIDE;
    static constexpr bool ZERO_PAD = D == 40 || D == 72;
};

// How far the probabilities' rounding to 16 bits reaches a result is set by the row's reference (the probability of the key that it was
// taken from is 1, exactly) and by what the denominator sums.
struct FlowRounding {
    float sum_max;      // the reference moves to a later tile's maximum when a lane's sum reaches this
    int two_tiles;      // it is the maximum of the first two tiles, not of the first
    bool pair_sum;      // the denominators sum the rounded probabilities, in FP32 (see softmax_tile_rel), not the FP32 exponentials
};

// (40: the cap at 128 registers lets four groups share a CU; 64 spills there)
template <typename T, int D, bool PAIR_SUM>
__global__ void __launch_bounds__(kThreads, (D == 40 ? 4 : D <= 96 ? 3 : 2)) sdpa_flow_kernel(const SdpaDev p, const float sum_max, const int two_tiles) {
    using G = HeadGeo<D>;
    using FG = FlowGeo<D>;
    using V8 = typename Mma<T>::v8;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    const int logical = logical_block(p.n_blocks);
    if (logical < 0) return;
    const int qt = logical % p.n_q_tiles, bh = logical / p.n_q_tiles;
    const int h = bh % p.H, b = bh / p.H;
    const int hk = h / p.kv_group;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, lq = lane & 31, lh = lane >> 5;
    const int q0 = qt * kRows;

    QRowFrags<T, D> qr;
    qr.issue(p, b, h, min(q0 + 32 * wave + lq, p.Lq - 1), lh);
    // tiles of the cached prefix first, then of the fresh keys; none straddles the two
    const int n_keys = visible_keys(p, b);
    const int n_pre = min(p.Lp, n_keys), n_fresh = n_keys - n_pre;
    const int pre_tiles = (n_pre + kBN - 1) / kBN, n_tiles = pre_tiles + (n_fresh + kBN - 1) / kBN;

    // ── DMA duty: wavefronts 0 and 1 move K, 2 and 3 V; each the keys of one group of 16 in both blocks of a tile ──
    const unsigned lds_base = static_cast<unsigned>(reinterpret_cast<size_t>((__attribute__((address_space(3))) unsigned char*)smem));
    const int op = wave >> 1, g = wave & 1;
    const int prow = lane >> 2, pch = (lane & 3) ^ ((prow >> 2) & 3);
    constexpr int LAST = G::CPR - 4 * (FG::NP - 1);      // pieces of a row in its last panel
    const unsigned last_cut = static_cast<unsigned>(max(pch - (LAST - 1), 0)) * 16u;      // those past its end repeat its last one
    const unsigned long last_lanes = __builtin_amdgcn_ballot_w64(pch < LAST);             // ... or are not loaded (ZERO_PAD)
    const unsigned char* const fresh = reinterpret_cast<const unsigned char*>(op ? static_cast<const T*>(p.v) + b * p.v_bs + hk * D : static_cast<const T*>(p.k) + b * p.k_bs + hk * D);
    const unsigned fresh_rsb = static_cast<unsigned>(op ? p.v_rs : p.k_rs) * 2u;
    const unsigned char* src = fresh;
    unsigned rsb = fresh_rsb;
    int left = n_fresh;              // keys of the segment from the next tile to load on
    int to_load = n_tiles;           // tiles from that one on
    if (n_pre > 0) {
        src = reinterpret_cast<const unsigned char*>(op ? static_cast<const T*>(p.vp) + b * p.vp_bs + hk * D : static_cast<const T*>(p.kp) + b * p.kp_bs + hk * D);
        rsb = static_cast<unsigned>(op ? p.vp_rs : p.kp_rs) * 2u;
        left = n_pre;
    }
    unsigned va[2];
    // this lane's offsets inside the next tile; rows past the end of a segment repeat its last one
    auto set_offsets = [&]() {
        int last = min(left, kBN) - 1;
        asm volatile("" : "+s"(last));
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) va[blk] = static_cast<unsigned>(min(32 * blk + 16 * g + prow, last)) * rsb + static_cast<unsigned>(pch) * 16u;
    };
    auto dma_piece = [&](int i, unsigned buf) {       // i = blk * NP + panel
        const int blk = i / FG::NP, pn = i % FG::NP;
        const unsigned dst = lds_base + buf + blk * FG::BLOCK + op * FG::OPER + g * 1024 + pn * FG::PANEL;
        // (inline assembly: for the builtin the compiler would wait for the load in front of every later LDS read; the LDS base
        //  travels in m0, and the s_nop is the wait state an LDS-DMA instruction needs behind a write of m0)
        if (G::CPR % 4 != 0 && pn == FG::NP - 1 && FG::ZERO_PAD)      // (exec is all ones here and afterwards)
            asm volatile("s_mov_b64 exec, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1"
                         : : "v"(va[blk]), "s"(src + pn * 64), "s"(last_lanes), "{m0}"(dst) : "memory");
        else
            asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                         : : "v"(G::CPR % 4 != 0 && pn == FG::NP - 1 ? va[blk] - last_cut : va[blk]), "s"(src + pn * 64), "{m0}"(dst) : "memory");
    };
    auto dma_next = [&]() {
        if (to_load > 1) {
            --to_load;
            left -= kBN;
            src += static_cast<unsigned long>(kBN) * rsb;
            const bool crossed = left <= 0;
            if (crossed) { src = fresh; rsb = fresh_rsb; left = n_fresh; }
            if (crossed || left < kBN) set_offsets();
        }
    };
    if constexpr (FG::ZERO_PAD) {
        // the last panel of K and V, both blocks, both buffers
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (tid < FG::PANEL / 16) *reinterpret_cast<u32x4*>(smem + i * FG::OPER + (FG::NP - 1) * FG::PANEL + tid * 16) = u32x4{0, 0, 0, 0};
        __syncthreads();
    }
    if (n_tiles > 0) {
        set_offsets();
#pragma unroll
        for (int i = 0; i < 2 * FG::NP; ++i) dma_piece(i, 0);
        dma_next();
    }
    V8 qf[G::KC];
    qr.finish(p, lh, qf);

    f32x16 oacc[G::VB];
#pragma unroll
    for (int vb = 0; vb < G::VB; ++vb)
#pragma unroll
        for (int e = 0; e < 16; ++e) oacc[vb][e] = 0.f;
    RelSoftmaxState st;
    const float cl2 = p.scale_log2;
    const PanelReads at(lane);
    f32x16 sacc[2];
    V8 pf[4];

    auto tile = [&](auto parity, int t) {
        constexpr int BUF = decltype(parity)::value * FG::TILE, NEXT = FG::TILE - BUF;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        const int rows = t < pre_tiles ? n_pre - t * kBN : n_fresh - (t - pre_tiles) * kBN;
        if (rows < kBN) {
            // value rows of zeros past the end (they repeat the last row, which may hold infinities: 0 x Inf)
            for (int i = tid; i < (kBN - rows) * FG::NP * 4; i += kThreads) {
                const int row = rows + i / (FG::NP * 4), piece = i % (FG::NP * 4);
                *reinterpret_cast<u32x4*>(smem + BUF + (row >> 5) * FG::BLOCK + FG::OPER + (piece >> 2) * FG::PANEL + (row & 31) * 64 + (piece & 3) * 16) = u32x4{0, 0, 0, 0};
            }
            __syncthreads();
        }
        constexpr int NQK = 2 * G::KC, NPV = 4 * G::VB;
        auto kfetch = [&](int i) -> V8 {
            const int kb = i & 1, c = i >> 1;
            return *reinterpret_cast<const V8*>(smem + BUF + kb * FG::BLOCK + (c >> 1) * FG::PANEL + at.k[c & 1]);
        };
        V8 ring[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) ring[i] = kfetch(i);
        [&]<int... I>(std::integer_sequence<int, I...>) {
            ([&] {
                constexpr int i = I, kb = i & 1, c = i >> 1;
                const V8 a = ring[i % kAhead];
                if constexpr (c == 0) {
                    const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                    sacc[kb] = Mma<T>::run(a, qf[c], zero);
                } else sacc[kb] = Mma<T>::run(a, qf[c], sacc[kb]);
                if constexpr (i + kAhead < NQK) ring[i % kAhead] = kfetch(i + kAhead);
                constexpr int d0 = 2 * FG::NP * i / NQK, d1 = 2 * FG::NP * (i + 1) / NQK;
                if constexpr (d1 > d0) {
#pragma unroll
                    for (int j = d0; j < d1; ++j) dma_piece(j, NEXT);
                }
                MI_SCHED_BARRIER
            }(), ...);
        }(std::make_integer_sequence<int, NQK>{});
        dma_next();
        if (rows < kBN) {
            int first = 4 * lh;
            asm volatile("" : "+v"(first));     // (computed here, not kept in registers through the key loop)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const float score = sacc[kb][e];
                    sacc[kb][e] = blank_outside(score, 0, rows - 1 - first - (32 * kb + 8 * (e >> 2) + (e & 3)));
                }
        }
        auto exponentiate = [&](float mul, float add) -> float {
            float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c4 = 0; c4 < 4; ++c4)
#pragma unroll
                for (int i = 0; i < 8; i += 2) {
                    const int kb = c4 >> 1, e = 8 * (c4 & 1) + i;
                    const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[kb][e], mul, add));
                    const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[kb][e + 1], mul, add));
                    pf[c4][i] = static_cast<T>(p0);
                    pf[c4][i + 1] = static_cast<T>(p1);
                    if constexpr (PAIR_SUM) sum[i >> 1] = pair_sum<T>(pf[c4], i >> 1, sum[i >> 1]);
                    else {
                        sum[i & 2] += p0;
                        sum[(i & 2) + 1] += p1;
                    }
                }
            // (packed here: left to itself the compiler keeps the 32 FP32 values through the branch that follows)
#pragma unroll
            for (int c4 = 0; c4 < 4; ++c4) asm volatile("" : "+v"(pf[c4]));
            return (sum[0] + sum[1]) + (sum[2] + sum[3]);
        };
        float ls = exponentiate(cl2, st.neg_ref);
        const bool second = D >= 80 && D <= 112 && !PAIR_SUM && decltype(parity)::value && two_tiles && t == 1;
        if (__any(!(st.started && ls < sum_max && !second))) {
            // first tiles, or terms that grew: the reference moves to the row's maximum (see softmax_tile_rel)
            float mloc = fmaxf(sacc[0][0], sacc[1][0]);
#pragma unroll
            for (int e = 1; e < 16; ++e) mloc = fmaxf(mloc, fmaxf(sacc[0][e], sacc[1][e]));
            mloc = __builtin_fmaf(exchange_max(mloc), cl2, st.neg_ref);
            const bool visible = mloc > kNegInf;
            const float shift = !visible ? 0.f : (st.started ? fmaxf(mloc, 0.f) : mloc);
            const float alpha = st.started ? __builtin_amdgcn_exp2f(-shift) : 1.f;   // nothing accumulated before the first key
            st.started = st.started || visible;
            st.l *= alpha;
#pragma unroll
            for (int vb = 0; vb < G::VB; ++vb)
#pragma unroll
                for (int e = 0; e < 16; ++e) oacc[vb][e] *= alpha;
            st.neg_ref -= shift;
            ls = exponentiate(cl2, st.neg_ref);
        }
        st.l += ls;
        MI_SCHED_BARRIER
        auto vfetch = [&](int j) -> V8 {
            const int c4 = j / G::VB, vb = j % G::VB;
            return at.template v_frag<T>(smem + BUF + (c4 >> 1) * FG::BLOCK + FG::OPER + (c4 & 1) * 1024 + vb * FG::PANEL);
        };
#pragma unroll
        for (int i = 0; i < kAhead; ++i) ring[i] = vfetch(i);
        [&]<int... I>(std::integer_sequence<int, I...>) {
            ([&] {
                constexpr int j = I, c4 = j / G::VB, vb = j % G::VB;
                oacc[vb] = Mma<T>::run(ring[j % kAhead], pf[c4], oacc[vb]);
                if constexpr (j + kAhead < NPV) ring[j % kAhead] = vfetch(j + kAhead);
                MI_SCHED_BARRIER
            }(), ...);
        }(std::make_integer_sequence<int, NPV>{});
    };
    for (int t = 0; t < n_tiles; t += 2) {
        tile(std::integral_constant<int, 0>{}, t);
        if (t + 1 >= n_tiles) break;
        tile(std::integral_constant<int, 1>{}, t + 1);
    }
    const float inv = row_inverse(exchange_sum(st.l));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // (the repeated load of the last tile)
    __syncthreads();
    stage_output<T, D>(smem, 32 * wave + lq, lh, oacc, inv);
    __syncthreads();
    T* const o_base = static_cast<T*>(p.o) + b * p.o_bs + h * D;
    write_output<T, D, kThreads>(smem, o_base, p.o_rs, q0, p.Lq, kRows, tid);
}

template <typename T, int D>
int launch_flow(SdpaDev p, const FlowRounding& r, hipStream_t stream) {
    p.n_q_tiles = (p.Lq + kRows - 1) / kRows;
    p.n_blocks = p.B * p.H * p.n_q_tiles;
    const dim3 grid((p.n_blocks + 7) / 8 * 8), block(kThreads);
    if (D <= 96 && r.pair_sum) hipLaunchKernelGGL((sdpa_flow_kernel<T, D, D <= 96>), grid, block, FlowGeo<D>::LDS, stream, p, r.sum_max, r.two_tiles);
    else hipLaunchKernelGGL((sdpa_flow_kernel<T, D, false>), grid, block, FlowGeo<D>::LDS, stream, p, r.sum_max, r.two_tiles);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail("sdpa_fwd launch: %s", hipGetErrorString(e));
    return 0;
}

// As exact as the kernels that these calls would otherwise take:
//   a 256-row tile or more per CU, more keys than the short-key kernel holds: the 256-row kernels, which sum rounded probabilities up to
//     head_dim 96 and move the reference at 2^10;
//   below, at 40 and 64 always, at 72 from 5 and at 128 from 8 key tiles: their instances that sum exponentials;
//   otherwise the 128-row kernel or (few keys) the short-key one: exponentials, reference moved at 2^8. At 80 to 112 and four key tiles
//     or more two halves of a work group took every other tile, each with a reference of its own: hence the first two tiles here, and 2^6.
// Relative error against 64 bits, with the first tile's maximum, 2^10 and exponentials for all / so (bf16, scores N(0, 1); N(0, 3)):
//   80, 8 x 4096 rows, 231 keys 2.27e-3 / 2.22e-3; 2.18e-3 / 1.97e-3 (before there was this kernel 2.21e-3; 1.99e-3), 1000 keys 2.33e-3 /
//   2.31e-3; 2.28e-3 / 2.12e-3; 96, 16 x 4096, 300 keys 2.30e-3 / 2.28e-3; 2.22e-3 / 1.90e-3; 160, 8 x 4096, 4096 keys 2.27e-3 / 2.19e-3 (N(0, 3)).
// Time, so against that: N(0, 1) equal but for 80 to 112 with few keys (80, 231 keys 8.7 -> 9.1 us, 1000 keys 19.4 -> 19.9) and with rounded sums (40, 1.25
// rounds 99 -> 96 us; 80, 2 x 8 x 4096 bf16 90.5 -> 94); N(0, 3) up to 12 % more at 80 to 112 below a round, where the reference moves more often.
FlowRounding flow_rounding(const SdpaDev& p, int head_dim, int n_cu, bool short_keys) {
    const long heads = static_cast<long>(p.B) * p.H;
    const bool full = heads * ((p.Lq + 255) / 256) >= n_cu && !short_keys, middle = head_dim >= 80 && head_dim <= 112;
    const int tiles = (p.Lk + kBN - 1) / kBN, many = head_dim <= 64 ? 1 : head_dim == 72 ? 5 : head_dim == 128 ? 8 : 1 << 30;
    FlowRounding r;
    r.pair_sum = full && head_dim <= 96;
    r.sum_max = (full && head_dim <= 128) || (tiles >= many && p.Lp == 0 && !short_keys) ? kRelSumMax : middle ? 64.f : 256.f;
    r.two_tiles = middle && !full && tiles >= 4;
    return r;
}

template <typename T>
int launch_flow_t(const SdpaDev& p, int head_dim, const FlowRounding& r, hipStream_t stream) {
    switch (head_dim) {
        case 40: return launch_flow<T, 40>(p, r, stream);
        case 64: return launch_flow<T, 64>(p, r, stream);
        case 72: return launch_flow<T, 72>(p, r, stream);
        case 80: return launch_flow<T, 80>(p, r, stream);
        case 96: return launch_flow<T, 96>(p, r, stream);
        case 112: return launch_flow<T, 112>(p, r, stream);
        case 128: return launch_flow<T, 128>(p, r, stream);
        default: return launch_flow<T, 160>(p, r, stream);
    }
}

}  // namespace

// Calls that sdpa_small.hip (few rows) and the short-key kernel (at least a 256-row tile per CU) leave, without masks, extras,
// tile-wise K rotation, the prefix dial or packed sequences. The lines are from self-attention of 8 (batch 1 and 2), 16 and 24 heads
// and from calls of 8 heads of 300 to 4096 units (32 query rows of a head) x 2 to 128 blocks of 32 keys, against the kernels that
// took them before, with the split round where it applies (us, before / here; n = compute units; rounds of 256-row tiles):
//   80, 96, 112, 160  always: 640 units, 32 blocks 80 22 / 17, 160 34 / 24; 80, batch 2, 1536 tokens 42 / 24, 4096 128 / 98; 160, 4096
//                     units 128 blocks 352 / 313; 96 and 112, 2304 units, 64 blocks 82 / 78, 123 / 93
//   72                0.38 rounds 28.8 / 23.9, 0.56 45 / 41, 0.94 81 / 76, 1.0 95 / 89, 1.31 177 / 156; not with a last round of up to an
//                     eighth, which the split kernel cuts into its pieces
//   128               up to 4 n units (24 heads, 900 tokens 26.0 / 21.5, 1100 29.6 / 24.2; 1365 38 / 39, 1997 53.0 / 57.7, 4608 227 / 253:
//                     with the GPU full, half the operand traffic per product is worth more than finer tiles); few keys anywhere: 1536
//                     units, 10 and 16 blocks 16.4 / 15.8, 20.5 / 20.2, 4096 units 37 / 31, 48 / 42
//   40                up to 5 n units (0.28 rounds 28.8 / 28.0, 0.5 54 / 48, 0.62 75 / 71, 0.75 86 / 90) and with a last round up to half
//                     full: 1.25 309 / 234, 1.5 341 / 301, 2.5 468 / 394; 1, 2 and 3 rounds 128 / 135, 251 / 261, 555 / 571; few keys: 1536
//                     units, 10 blocks 10.8 / 10.1
//   64                up to 4 n units and 47 blocks (1024 units, 32 blocks 19.6 / 18.1), few keys, a last round up to half full (2304 units,
//                     64 blocks 72 / 55; 3072 72 / 63)
// (Calls whose keys fit LDS: launch_d asks sdpa_flow_runs and shortkv_pays instead.)
bool sdpa_flow_runs(const SdpaDev& p) {
    return !(p.mask_mode != MI_MASK_NONE || p.key_mask || p.bias || p.lse || p.cu_q || p.cos_k || p.prefix_scaled) && offsets_fit_32_bits(p);
}

bool sdpa_flow_takes(const SdpaDev& p, int head_dim, int n_cu) {
    if (!sdpa_flow_runs(p)) return false;
    const long heads = static_cast<long>(p.B) * p.H, units = heads * ((p.Lq + 31) / 32), tiles = heads * ((p.Lq + 255) / 256), last = tiles % n_cu;
    const int blocks = (p.Lp + 31) / 32 + (p.Lk - p.Lp + 31) / 32;
    const bool full = tiles >= n_cu, half_round = tiles > n_cu && last > 0 && 2 * last <= n_cu;
    switch (head_dim) {
        case 40: return units <= 5L * n_cu || half_round || (!full && blocks <= 10);
        case 64: return (units <= 4L * n_cu && blocks < 48) || half_round || (!full && blocks <= 6);
        case 72: return !full || last == 0 || 8 * last > n_cu;
        case 128: return units <= 4L * n_cu || blocks <= (full ? 30 : 10);
        default: return true;
    }
}

int launch_sdpa_flow(const SdpaDev& p, int dtype, int head_dim, int n_cu, bool short_keys, hipStream_t stream) {
    const FlowRounding r = flow_rounding(p, head_dim, n_cu, short_keys);
    if (dtype == MI_DTYPE_BF16) return launch_flow_t<__bf16>(p, head_dim, r, stream);
    return launch_flow_t<_Float16>(p, head_dim, r, stream);
}

}  // namespace mi
