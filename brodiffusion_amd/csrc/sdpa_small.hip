// Softmax attention for calls with few query rows: latency before they are anything else.
//
// Such a call is a chain: operands -> LDS -> scores -> softmax -> values -> out. The 128-row kernel makes it long (three barriers
// and a staging pass before the first key tile is even requested, then 64-key tiles one after the other on one wavefront per SIMD)
// and leaves most of the GPU out of it: 64 tokens of 8 heads of 160 took 8.5 us on 16 work groups, an empty launch takes 2.3.
// Here a work group is R x S wavefronts for 32 R query rows: wavefront (r, s) has rows 32 r .. 32 r + 31 and the 32-key blocks
// s, s + S, ..., so that S blocks are worked on at a time, and the S partial results of a row are merged through LDS in FP32.
//   * Every operand of the first block is requested before anything is waited for: query rows straight into MFMA operand
//     registers, keys and values by LDS DMA. No barrier stands in front of the first product where R = 1.
//   * A block sits in LDS as panels (PanelReads): all panels of a row share one address (the panel is a scalar offset), and the
//     fragments of K and V are read from two addresses each plus immediates.
//   * The fragments of a block are all read into registers before it is multiplied. Then its LDS is free, and the next block's
//     DMA runs under the products and the softmax of this one: one buffer, no ring. (Two and three buffers measured the same;
//     a small footprint lets more wavefronts in.)
//   * The parts meet in LDS scaled already: a wavefront first learns the maxima and sums of the others (256 B each), scales its own
//     registers and writes them, so that the last pass is loads and additions, in straight code for its number of parts.
// What bounds it: a chain of latencies. Of 9500 clocks of a work group of 64 x 160: 1300 to the first request, 2200 until its data are in
// LDS, 1600 for the one block, 1900 for scaling and writing the parts, 1600 for their sum and the write-out (4400 before it was straight).
// Measured (fp16, 8 heads; before: the 128-row kernel, for 80 in pairs of tiles, for 40 and 72 the 256-row kernels), us:
//   self, tokens x head_dim: 64 x 160 8.5 -> 5.0, 256 x 160 14.6 -> 7.0, 1024 x 160 37.4 -> 15.4; 512 x 80 14.4 -> 6.9, 2048 x 80
//   39.8 -> 22.2; 1024 x 40 18.1 -> 8.5
//   77 keys, queries x head_dim: 64 x 160 10.7 -> 5.7, 1024 x 80 8.9 -> 4.8, 4096 x 40 8.1 -> 6.3
//
// The instances with PROJ also form their query rows (project_rows): the cached cross-attention of a block, whose query projection
// is as short as the attention behind it and, as a launch of its own, mostly start, first loads and write-out.
#include "linear_math.h"
#include "sdpa_tiles.h"

namespace mi {
namespace {

using namespace sdpa;

constexpr int kKB = 32;        // keys of a block
constexpr int kMaxWaves = 8;
constexpr int kMaxLds = 160 * 1024 - 64;

template <int D> struct SmallGeo {
    using G = HeadGeo<D>;
    static constexpr int NP = G::VB;                            // panels of 32 head-dim elements
    static constexpr int PANEL = kKB * 64;                      // bytes of 32 keys of a panel
    static constexpr int OPER = NP * PANEL, BLOCK = 2 * OPER;   // K or V of a block; both
    static constexpr int P_STRIDE = D * 4 + 16;                 // bytes of one row of a partial output
    static constexpr int PART = 32 * P_STRIDE;                  // a wavefront's part of the output
};

// What the unmasked kernel needs, side by side: read one by one from the launch view, at ten places of the prologue, the arguments of a
// short call were seven scalar-load latencies in a row in front of its first key (64 x 160, with the straight sum: 6.7 -> 5.0 us).
struct SmallArgs {
    const void* q; const void* k; const void* v; const void* kp; const void* vp; void* o;
    const int* kv_valid_len; const float* cos_q; const float* sin_q;
    long q_rs, q_bs, o_bs, k_bs, v_bs, kp_bs, vp_bs;                  // elements
    unsigned k_rsb, v_rsb, kp_rsb, vp_rsb, o_rsb;                     // bytes
    int Lq, Lk, Lp, n_blocks, n_q_tiles, H, kv_group, S, rope_split;
    unsigned inv_tiles, inv_heads, inv_group;                         // 2^32 / divisor, rounded up (exact while dividend x divisor < 2^32)
    float scale_log2;
};
struct NoMask {};

// The query projection inside the kernel (project_rows): x (rows of a batch item, contraction elements), w (H D, contraction).
struct ProjArgs {
    const void* x; const void* w; const void* bias; const float* w_scale;
    long x_bsb;                          // bytes between batch items of x
    unsigned x_rsb, w_rsb; int n_steps;  // steps of 64 contraction elements
};
constexpr int kProjS = 3;                // wavefronts to a row group of 32, and steps of a round of the projection
// PROJ: 0 none, 1 16-bit weights, 2 INT8 weights. LDS: two buffers of kProjS stages each (64 rows of X, D rows of W of 64 contraction elements), the
// projected rows, the key blocks; the parts of the output will lie where the stages were.
template <int D, int PROJ> struct ProjGeo {
    using G = HeadGeo<D>;
    using SG = SmallGeo<D>;
    static constexpr int WROW = PROJ == 2 ? 64 : 128;                       // bytes of a W row in a stage
    static constexpr int MX = 8, MW = (D * WROW + 1023) / 1024;             // DMA instructions per stage
    static constexpr int X_BYTES = 8192, STAGE = X_BYTES + MW * 1024;
    static constexpr int Q_AT = 2 * kProjS * STAGE;                      // the projected rows
    static constexpr int cmax(int a, int b) { return a > b ? a : b; }
    static constexpr int BLOCKS_AT = PROJ ? (cmax(Q_AT + 64 * G::O_STRIDE, kProjS * (cmax(SG::BLOCK, 2 * SG::PART) + 512)) + 1023) / 1024 * 1024 : 0;
    static constexpr int LDS = BLOCKS_AT + kProjS * SG::BLOCK;
    static_assert(!PROJ || LDS <= 160 * 1024, "LDS of a compute unit");
    static_assert(!PROJ || kProjS * SG::BLOCK >= 4096, "fragments of W rows past the last stage's end stay inside");
};
__device__ __forceinline__ int quotient(int x, int d, unsigned inv) { return d == 1 ? x : static_cast<int>(__umulhi(static_cast<unsigned>(x), inv)); }

// Rows q0 .. q0 + 63 of x times the D rows of W of head h, into the MFMA operand registers of the score product, rounded once to T as
// the projection launch rounds them, in its order of additions: same bits. Wavefronts 0 to 2 multiply, 32 features of all 64 rows each
// (two chains of products on one fragment of W, which INT8 weights are widened into once); wavefronts 3 to 5 load: an LDS-DMA
// instruction keeps its wavefront from issuing for as long as a product takes. A round is 3 steps of 64 contraction elements, one per
// loading wavefront; round i + 2 goes into the buffer of round i once its fragments are in registers, and last come the first key
// blocks (request_keys), which land under the write-out of the rows.
template <typename T, int D, int PROJ, typename Keys>
__device__ __forceinline__ void project_rows(const ProjArgs& a, int b, int h, int q0, int Lq, int wave, int lane, unsigned char* smem, unsigned lds_base,
                                             Keys request_keys, bool has_keys, typename Mma<T>::v8 (&qf)[HeadGeo<D>::KC]) {
    using G = HeadGeo<D>;
    using SG = SmallGeo<D>;
    using PG = ProjGeo<D, PROJ>;
    using V8 = typename Mma<T>::v8;
    constexpr bool W8 = PROJ == 2;
    constexpr int KEY_LOADS = 2 * SG::NP;       // DMA instructions of request_keys
    const int lq = lane & 31, lh = lane >> 5;
    const int n = a.n_steps, rounds = (n + kProjS - 1) / kProjS;
    auto meet = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    if (wave >= kProjS) {
        const int k = wave - kProjS;
        const unsigned char* const xg = static_cast<const unsigned char*>(a.x) + b * a.x_bsb + static_cast<long>(q0) * a.x_rsb;
        const unsigned char* const wg = static_cast<const unsigned char*>(a.w) + static_cast<long>(h) * D * a.w_rsb;
        unsigned xoff[PG::MX], woff[PG::MW];
#pragma unroll
        for (int u = 0; u < PG::MX; ++u) {
            const int row = 8 * u + (lane >> 3);
            xoff[u] = static_cast<unsigned>(min(row, Lq - 1 - q0)) * a.x_rsb + ((lane & 7) ^ ((row >> 1) & 7)) * 16u;
        }
#pragma unroll
        for (int u = 0; u < PG::MW; ++u) {
            const int row = W8 ? 16 * u + (lane >> 2) : 8 * u + (lane >> 3);
            woff[u] = static_cast<unsigned>(min(row, D - 1)) * a.w_rsb + (W8 ? (lane & 3) ^ ((row >> 2) & 3) : (lane & 7) ^ ((row >> 1) & 7)) * 16u;
        }
        auto dma = [&](unsigned voff, const unsigned char* base, unsigned dst) {
            asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(base), "{m0}"(dst) : "memory");
        };
        auto request = [&](int i) {      // this wavefront's stage of round i; behind the last round its keys
            const int t = kProjS * i + k;
            if (i == rounds) request_keys();
            else if (i < rounds && t < n) {
                const unsigned dst = lds_base + ((i & 1) * kProjS + k) * PG::STAGE;
#pragma unroll
                for (int u = 0; u < PG::MX; ++u) dma(xoff[u], xg + t * 128L, dst + u * 1024);
#pragma unroll
                for (int u = 0; u < PG::MW; ++u) dma(woff[u], wg + t * static_cast<long>(PG::WROW), dst + PG::X_BYTES + u * 1024);
            }
        };
        request(0);
        request(1);
        for (int i = 0; i < rounds; ++i) {
            // the stage of round i has landed: at most what was requested after it is in flight
            if (i + 1 < rounds && kProjS * (i + 1) + k < n) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(PG::MX + PG::MW) : "memory");
            else if (i + 1 == rounds && has_keys) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(KEY_LOADS) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            meet();
            meet();
            request(i + 2);
        }
    } else {
        f32x16 acc[2];
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[r][e] = 0.f;
        const bool has_features = wave < G::VB;
        // bias and scales of this lane's features, requested here: behind the loop their latency would stand alone
        typedef T t4 __attribute__((ext_vector_type(4)));
        typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
        t4 bias[4];
        f32x4_a4 scale[W8 ? 4 : 1];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int feat = h * D + min(32 * wave + 8 * g + 4 * lh, D - 4);
            bias[g] = t4{};
            if (a.bias) bias[g] = *reinterpret_cast<const t4*>(static_cast<const T*>(a.bias) + feat);
            if constexpr (W8) scale[g] = *reinterpret_cast<const f32x4_a4*>(a.w_scale + feat);
        }
        for (int i = 0; i < rounds; ++i) {
            meet();          // the stages of round i are there
            const unsigned char* const st = smem + (i & 1) * kProjS * PG::STAGE;
            using WRaw = std::conditional_t<W8, gemm::u32x2, V8>;
            V8 xf[kProjS][4][2];
            WRaw wf[kProjS][4];
            // (stages past the last step hold something else: their fragments are read, not multiplied)
            if (has_features) {
#pragma unroll
                for (int k = 0; k < kProjS; ++k)
#pragma unroll
                    for (int kk = 0; kk < 4; ++kk) {
                        const int swz = ((2 * kk + lh) ^ ((lq >> 1) & 7)) << 4;
#pragma unroll
                        for (int r = 0; r < 2; ++r) xf[k][kk][r] = *reinterpret_cast<const V8*>(st + k * PG::STAGE + r * 4096 + lq * 128 + swz);
                        wf[k][kk] = *reinterpret_cast<const WRaw*>(st + k * PG::STAGE + PG::X_BYTES + wave * 32 * PG::WROW +
                                                                   (W8 ? lq * 64 + ((kk ^ ((lq >> 2) & 3)) << 4) + 8 * lh : lq * 128 + swz));
                    }
            }
            auto multiply = [&](int k) {
                if (!has_features || kProjS * i + k >= n) return;
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) {
                    V8 w;
                    if constexpr (W8) w = gemm::widen<T>(wf[k][kk]);
                    else w = wf[k][kk];
#pragma unroll
                    for (int r = 0; r < 2; ++r) acc[r] = Mma<T>::run(w, xf[k][kk][r], acc[r]);
                }
            };
            multiply(0);     // (while the fragments of the other two steps arrive)
            multiply(1);
            meet();          // everybody holds its fragments: the buffer is free
            if (i == rounds - 1) request_keys();
            multiply(2);
        }
        // acc[r][4 g + e] is feature 32 wave + 8 g + 4 lh + e of row 32 r + lq
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int feat = 32 * wave + 8 * g + 4 * lh;
            if (feat < D) {
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    const f32x16 v = acc[r];
                    t4 out;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if constexpr (W8) out[e] = static_cast<T>(gemm::scaled_acc(v[4 * g + e], scale[g][e], static_cast<float>(bias[g][e])));
                        else out[e] = static_cast<T>(v[4 * g + e] + static_cast<float>(bias[g][e]));
                    }
                    *reinterpret_cast<t4*>(smem + PG::Q_AT + (32 * r + lq) * G::O_STRIDE + feat * 2) = out;
                }
            }
        }
    }
    meet();
#pragma unroll
    for (int c = 0; c < G::KC; ++c) {
        u32x4 q = *reinterpret_cast<const u32x4*>(smem + PG::Q_AT + (32 * (wave & 1) + lq) * G::O_STRIDE + (2 * c + lh) * 16);
        if (G::DK > D && c == G::KC - 1 && lh) q = u32x4{0, 0, 0, 0};
        qf[c] = __builtin_bit_cast(V8, q);
    }
    meet();          // (the parts of the output will lie where the rows are)
}

template <typename T, int D, int R, bool MASKED, int PROJ>
__global__ void __launch_bounds__(64 * kMaxWaves, PROJ ? 2 : D <= 64 ? 4 : D <= 80 ? 3 : 2)
    sdpa_small_kernel(const SmallArgs p, const std::conditional_t<MASKED, SdpaDev, std::conditional_t<PROJ != 0, ProjArgs, NoMask>> ext) {
    using G = HeadGeo<D>;
    using SG = SmallGeo<D>;
    using PG = ProjGeo<D, PROJ>;
    using V8 = typename Mma<T>::v8;
    typedef T t8 __attribute__((ext_vector_type(8)));
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    __shared__ int red[2 * R];

    // (all arguments requested here, in a few wide loads)
    asm volatile("" : : "s"(p.q), "s"(p.k), "s"(p.v), "s"(p.q_rs), "s"(p.q_bs), "s"(p.k_bs), "s"(p.v_bs), "s"(p.k_rsb), "s"(p.v_rsb), "s"(p.Lq), "s"(p.Lk),
                 "s"(p.n_blocks), "s"(p.n_q_tiles), "s"(p.H), "s"(p.kv_group), "s"(p.S), "s"(p.inv_tiles), "s"(p.inv_heads), "s"(p.inv_group), "s"(p.kv_valid_len),
                 "s"(p.cos_q), "s"(p.Lp), "s"(p.o), "s"(p.o_bs), "s"(p.o_rsb), "s"(p.scale_log2));
    const int logical = logical_block(p.n_blocks);
    if (logical < 0) return;
    const int S = p.S;
    const int bh = quotient(logical, p.n_q_tiles, p.inv_tiles), qt = logical - bh * p.n_q_tiles;
    const int b = quotient(bh, p.H, p.inv_heads), h = bh - b * p.H;
    const int hk = quotient(h, p.kv_group, p.inv_group);
    const int tid = threadIdx.x, NT = 64 * R * S;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = wave % R, s = wave / R;
    const int lane = tid & 63, lq = lane & 31, lh = lane >> 5;
    const int q0 = qt * (32 * R);

    // ── requests: this lane's query row with its RoPE entries, then the first block of keys and values ──
    QRowFrags<T, D> qr;
    if constexpr (PROJ == 0) qr.issue(p, b, h, min(q0 + 32 * r + lq, p.Lq - 1), lh);
    // Visible keys [lo, hi) of this lane's row, and the blocks of the work group: those of the cached prefix, then those of the fresh
    // keys, from the first to the last that one of its rows sees; none straddles the two.
    int n_keys = p.Lk;
    if (p.kv_valid_len) n_keys = __builtin_amdgcn_readfirstlane(max(min(n_keys, p.kv_valid_len[b]), 0));
    int lo = 0, hi = n_keys, first_key = 0, stop_key = n_keys;
    WaveExtent we{0, 0, n_keys, n_keys};
    if constexpr (MASKED) {
        row_interval(ext, b, min(q0 + 32 * r + lq, p.Lq - 1), q0 + 32 * r < p.Lq, lo, hi);
        we = wave_extent(lo, hi);
        first_key = we.lo_min; stop_key = we.hi_max;
        if (R > 1) {
            if (lane == 0) { red[r] = we.lo_min; red[R + r] = we.hi_max; }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < R; ++i) { first_key = min(first_key, red[i]); stop_key = max(stop_key, red[R + i]); }
            first_key = __builtin_amdgcn_readfirstlane(first_key);
            stop_key = __builtin_amdgcn_readfirstlane(stop_key);
        }
        if (first_key >= stop_key) first_key = stop_key = 0;
    }
    const int n_pre = min(p.Lp, stop_key), n_fresh = max(stop_key - p.Lp, 0);     // keys of the two segments up to the last visible one
    const int pre0 = MASKED ? first_key / kKB : 0, fresh0 = MASKED ? max(first_key - p.Lp, 0) / kKB : 0;
    const int pre_blocks = max((n_pre + kKB - 1) / kKB - pre0, 0);
    const int n_blocks = pre_blocks + (n_fresh + kKB - 1) / kKB - fresh0;      // this wavefront takes blocks s, s + S, ...

    // ── DMA duty: a block is 2 operands x 2 groups of 16 keys x NP panels; the R wavefronts that share it take 4 / R
    //    (operand, group) pairs each ──
    constexpr int PAIRS = 4 / R;
    const unsigned lds_base = static_cast<unsigned>(reinterpret_cast<size_t>((__attribute__((address_space(3))) unsigned char*)smem));
    const int prow = lane >> 2, pch = (lane & 3) ^ ((prow >> 2) & 3);
    const unsigned last_cut = static_cast<unsigned>(max(pch - (G::CPR - 1 - 4 * (SG::NP - 1)), 0)) * 16u;   // chunks past the row's end repeat its last one
    auto load_block = [&](int blk) {
        const bool pre = blk < pre_blocks;
        const int row0 = (pre ? pre0 + blk : fresh0 + blk - pre_blocks) * kKB, last = (pre ? n_pre : n_fresh) - 1;   // rows past the end repeat the last one
#pragma unroll
        for (int i = 0; i < PAIRS; ++i) {
            const int pair = r * PAIRS + i, op = pair >> 1, g = pair & 1;
            const void* const t = op ? (pre ? p.vp : p.v) : (pre ? p.kp : p.k);
            const long bs = op ? (pre ? p.vp_bs : p.v_bs) : (pre ? p.kp_bs : p.k_bs);
            const unsigned rsb = op ? (pre ? p.vp_rsb : p.v_rsb) : (pre ? p.kp_rsb : p.k_rsb);
            const unsigned char* const base = reinterpret_cast<const unsigned char*>(static_cast<const T*>(t) + b * bs + hk * D);
            const unsigned off = static_cast<unsigned>(min(row0 + 16 * g + prow, last)) * rsb + static_cast<unsigned>(pch) * 16u;
            const unsigned dst = lds_base + PG::BLOCKS_AT + s * SG::BLOCK + op * SG::OPER + g * 1024;
            // (inline assembly: for the builtin the compiler would wait for the load in front of every later LDS read; the LDS base
            //  travels in m0, and the s_nop is the wait state an LDS-DMA instruction needs behind a write of m0)
#pragma unroll
            for (int pn = 0; pn < SG::NP; ++pn)
                asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(pn == SG::NP - 1 ? off - last_cut : off), "s"(base + pn * 64),
                             "{m0}"(dst + pn * SG::PANEL) : "memory");
        }
    };
    V8 qf[G::KC];
    if constexpr (PROJ == 0) {
        if (s < n_blocks) load_block(s);
        qr.finish(p, lh, qf);
    } else project_rows<T, D, PROJ>(ext, b, h, q0, p.Lq, wave, lane, smem, lds_base, [&] { if (s < n_blocks) load_block(s); }, s < n_blocks, qf);
    const unsigned pad_keep = lh ? 0u : ~0u;
    f32x16 oacc[G::VB];
#pragma unroll
    for (int vb = 0; vb < G::VB; ++vb)
#pragma unroll
        for (int e = 0; e < 16; ++e) oacc[vb][e] = 0.f;
    float m = kNegInf, mc = 0.f, l = 0.f, m_keep = kNegInf;      // (m_keep: the maximum up to which the reference stays)
    bool started = false;      // a block has been accumulated
    const float cl2 = p.scale_log2;
    const float lazy_raw = kLazyLog2 / cl2;
    // A wavefront's reference is the maximum of its first blocks, as many as hold the keys from which the kernels before took theirs (the
    // first 64; at head_dim 80 to 112 two halves of a work group, 64 each): the probability of the key that it comes from is 1, exactly,
    // in 16 bits too. (Error against 64 bits, bf16, scores of N(0, 3), from one block / so / before there was this kernel: causal, 256 tokens, 80
    // 2.01e-3 / 1.81e-3 / 1.81e-3, 128 2.01e-3 / 1.93e-3 / 1.93e-3; N(0, 1), 2000 tokens, 160 2.11e-3 / 2.08e-3 / 2.09e-3. Time: causal 1 % more, windows of
    // 64 in 256 tokens 6 %, others the same.)
    constexpr bool MIDDLE = D >= 80 && D <= 112;
    int exact_blocks = S == 1 ? (MIDDLE ? 4 : 2) : S == 2 && (MIDDLE || D == 160) ? 2 : 1;
    if constexpr (MASKED) { if (ext.window > 0 && S <= (MIDDLE ? 2 : 1)) exact_blocks += 2; }      // (rows whose first key lies in a later block)
    const PanelReads at(lane);

    const int n_steps = (n_blocks + S - 1) / S;
    for (int t = 0; t < n_steps; ++t) {
        const int blk = t * S + s;
        const bool pre = blk < pre_blocks;
        const int row0 = (pre ? pre0 + blk : fresh0 + blk - pre_blocks) * kKB, j0 = pre ? row0 : p.Lp + row0;
        const int rows = (pre ? n_pre : n_fresh) - row0;      // keys of the block
        const bool mine = blk < n_blocks && (!MASKED || (j0 < we.hi_max && j0 + kKB > we.lo_min));
        const unsigned char* const buf = smem + PG::BLOCKS_AT + s * SG::BLOCK;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (R > 1) __syncthreads();
        V8 kf[G::KC], vf[2][G::VB];
        if (mine) {
#pragma unroll
            for (int c = 0; c < G::KC; ++c) kf[c] = *reinterpret_cast<const V8*>(buf + at.k[c & 1] + (c >> 1) * SG::PANEL);
#pragma unroll
            for (int c4 = 0; c4 < 2; ++c4)
#pragma unroll
                for (int vb = 0; vb < G::VB; ++vb) vf[c4][vb] = at.template v_frag<T>(buf + SG::OPER + vb * SG::PANEL + c4 * 1024);
        }
        if (t + 1 < n_steps) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (R > 1) __syncthreads();
            if (blk + S < n_blocks) load_block(blk + S);
        }
        if (mine) {
            f32x16 sacc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < G::KC; ++c) {
                u32x4 a = __builtin_bit_cast(u32x4, kf[c]);
                if (G::DK > D && c == G::KC - 1) a &= pad_keep;
                sacc = Mma<T>::run(__builtin_bit_cast(V8, a), qf[c], sacc);
            }
            if (rows < kKB || (MASKED && (j0 < we.lo_max || j0 + kKB > we.hi_min))) {
                const int x0 = j0 + 4 * lh - lo, top = min(hi, j0 + rows) - 1 - lo;
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const float score = sacc[e];
                    sacc[e] = blank_outside(score, x0 + 8 * (e >> 2) + (e & 3), top);
                }
            }
            if (rows < kKB) {
                // value rows of zeros past the end (they repeat the last row, which may hold infinities)
                const int top = rows - 1 - 4 * lh;
#pragma unroll
                for (int c4 = 0; c4 < 2; ++c4) {
                    u32x4 keep;
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        const int key = 16 * c4 + 8 * (w >> 1) + 2 * (w & 1);   // and the one after it
                        keep[w] = (key <= top ? 0xffffu : 0u) | (key + 1 <= top ? 0xffff0000u : 0u);
                    }
#pragma unroll
                    for (int vb = 0; vb < G::VB; ++vb) vf[c4][vb] = __builtin_bit_cast(V8, __builtin_bit_cast(u32x4, vf[c4][vb]) & keep);
                }
            }
            float mloc = sacc[0];
#pragma unroll
            for (int e = 1; e < 16; ++e) mloc = fmaxf(mloc, sacc[e]);
            mloc = exchange_max(mloc);
            if (__any(mloc > m_keep)) {
                const float m_new = fmaxf(m, mloc);
                const float mc_new = (m_new == kNegInf) ? 0.f : m_new * cl2;
                if (started) {
                    const float alpha = __builtin_amdgcn_exp2f(m * cl2 - mc_new);
                    l *= alpha;
#pragma unroll
                    for (int vb = 0; vb < G::VB; ++vb)
#pragma unroll
                        for (int e = 0; e < 16; ++e) oacc[vb][e] *= alpha;
                }
                m = m_new;
                mc = mc_new;
                m_keep = m_new + (exact_blocks > 1 ? 0.f : lazy_raw);
            }
            started = true;
            --exact_blocks;
            V8 pf[2];
            float l0 = 0.f, l1 = 0.f;
#pragma unroll
            for (int c4 = 0; c4 < 2; ++c4)
#pragma unroll
                for (int i = 0; i < 8; i += 2) {
                    const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[8 * c4 + i], cl2, -mc));
                    const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[8 * c4 + i + 1], cl2, -mc));
                    l0 += p0;
                    l1 += p1;
                    pf[c4][i] = static_cast<T>(p0);
                    pf[c4][i + 1] = static_cast<T>(p1);
                }
            l += l0 + l1;
#pragma unroll
            for (int c4 = 0; c4 < 2; ++c4)
#pragma unroll
                for (int vb = 0; vb < G::VB; ++vb) oacc[vb] = Mma<T>::run(vf[c4][vb], pf[c4], oacc[vb]);
        }
    }
    float l_tot = exchange_sum(l);
    T* const o_base = static_cast<T*>(p.o) + b * p.o_bs + h * D;
    if (S == 1) {
        // every wavefront has all keys of its rows
        __syncthreads();     // the blocks are used up
        stage_output<T, D>(smem, 32 * r + lq, lh, oacc, row_inverse(l_tot));
        __syncthreads();
        write_output<T, D, 64 * R>(smem, o_base, static_cast<long>(p.o_rsb / 2), q0, p.Lq, 32 * R, tid);
        return;
    }
    // ── merge: maxima and denominators first, so that every wavefront scales its own part by 2^(maximum - row's maximum) / row's
    //    denominator; then the parts, FP32, whose sum is the result. (Merged piece by piece from unscaled parts, with the weights
    //    formed anew for each, this took as long as all the rest of a short call.) ──
    float* const stat = reinterpret_cast<float*>(smem + S * max(SG::BLOCK, R * SG::PART));      // [s][r][maximum, denominator][32]
    if (lh == 0) {
        stat[(s * R + r) * 64 + lq] = m;
        stat[(s * R + r) * 64 + 32 + lq] = l_tot;
    }
    __syncthreads();         // (also: the blocks are used up)
    float ms[kMaxWaves / R], ls[kMaxWaves / R];
#pragma unroll
    for (int k = 0; k < kMaxWaves / R; ++k) {
        ms[k] = k < S ? stat[(k * R + r) * 64 + lq] : kNegInf;
        ls[k] = k < S ? stat[(k * R + r) * 64 + 32 + lq] : 0.f;
    }
    float top = ms[0];
#pragma unroll
    for (int k = 1; k < kMaxWaves / R; ++k) top = fmaxf(top, ms[k]);
    const float topc = top == kNegInf ? 0.f : top * cl2;
    float lsum = 0.f;
#pragma unroll
    for (int k = 0; k < kMaxWaves / R; ++k) lsum = __builtin_fmaf(__builtin_amdgcn_exp2f(ms[k] * cl2 - topc), ls[k], lsum);     // 0 from -inf
    const float factor = __builtin_amdgcn_exp2f(m * cl2 - topc) * row_inverse(lsum);
    {
        unsigned char* const row = smem + (s * R + r) * SG::PART + lq * SG::P_STRIDE;
#pragma unroll
        for (int vb = 0; vb < G::VB; ++vb)
#pragma unroll
            for (int bb = 0; bb < 4; ++bb) {
                const int d0 = 32 * vb + 8 * bb + 4 * lh;
                if (32 * vb + 8 * bb < D) {
                    const f32x16 acc = oacc[vb];
                    *reinterpret_cast<f32x4*>(row + d0 * 4) = f32x4{acc[4 * bb] * factor, acc[4 * bb + 1] * factor, acc[4 * bb + 2] * factor, acc[4 * bb + 3] * factor};
                }
            }
    }
    __syncthreads();
    // (one straight piece of code per number of parts: with a branch per part in one loop for all, a pass took 900 clocks)
    unsigned char* const o_rows = reinterpret_cast<unsigned char*>(o_base) + static_cast<unsigned long>(q0) * p.o_rsb;
    const int n_rows = min(p.Lq - q0, 32 * R);
    auto sum_parts = [&](auto count) {
        constexpr int N = decltype(count)::value;
        for (int idx = tid; idx < n_rows * G::CPR; idx += NT) {
            const unsigned row = static_cast<unsigned>(idx) / G::CPR, cc = static_cast<unsigned>(idx) % G::CPR;
            const unsigned char* const part = smem + (row >> 5) * SG::PART + (row & 31) * SG::P_STRIDE + cc * 32;
            f32x4 lo[N], hi[N];
#pragma unroll
            for (int k = 0; k < N; ++k) {
                lo[k] = *reinterpret_cast<const f32x4*>(part + k * R * SG::PART);
                hi[k] = *reinterpret_cast<const f32x4*>(part + k * R * SG::PART + 16);
            }
#pragma unroll
            for (int k = 1; k < N; ++k) { lo[0] += lo[k]; hi[0] += hi[k]; }
            t8 out;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                out[e] = static_cast<T>(lo[0][e]);
                out[4 + e] = static_cast<T>(hi[0][e]);
            }
            *reinterpret_cast<t8*>(o_rows + static_cast<unsigned long>(row) * p.o_rsb + cc * 16) = out;
        }
    };
    [&]<int... I>(std::integer_sequence<int, I...>) {
        ([&] { if (S == I + 2) sum_parts(std::integral_constant<int, I + 2>{}); }(), ...);
    }(std::make_integer_sequence<int, kMaxWaves / R - 1>{});
}

// 32-key blocks of a call (those of the prefix and of the fresh keys apart)
int key_blocks(const SdpaDev& p) { return (p.Lp + kKB - 1) / kKB + (p.Lk - p.Lp + kKB - 1) / kKB; }

// Whether a call comes here, and with how many row groups and at most how many wavefronts to a work group.
//
// Calls without extras (key mask, logit bias, denominators), tile-wise K rotation, the prefix dial or packed sequences. The lines
// are from 8 head dimensions x 64 to 8192 units (32 query rows of a head) x 1 to 256 key blocks of 8 fp16 heads, every R and two S
// against the kernel that took the call before (us, before / here; n = compute units). Masked calls (causal, windowed, block-causal;
// 8 dimensions x 64 to 1008 units) take 0.35 to 0.98 of the time up to 4 n units (windowed ones of 96, 1008 units, 128-row kernel / here: window
// 64 11.5 / 9.3, 256 15.9 / 12.8, 1024 32.3 / 24.4, 4000 92 / 65; 1024 units of 250 tokens, window 64 11.0 / 10.0, 128 12.5 / 11.6); beyond 4 n
// they are left where their longest tiles start first.
//   units <= n       R = 1: 256 units, 5, 32 and 128 blocks: 40 8.4 / 4.8, 18.2 / 8.9, 56 / 25; 72 10.5 / 5.4, 23 / 10.2, 73 / 27; 128
//                    10.5 / 6.7, 25.7 / 12, 79 / 30; 160 13.4 / 7.9, 37 / 16.5, 134 / 43
//   units <= 2 n     R = 2: 512 units, 5, 32 and 128 blocks: 40 8.5 / 5.5, 18 / 11, 56 / 32; 80 10.5 / 6.5, 23 / 15, 73 / 40; 128 10.8 /
//                    7.9, 26 / 18, 79 / 51
//   units <= 4 n     unmasked calls go to sdpa_flow.hip, but for many keys at 64 (R = 2, two groups to a CU: 1024 units, 64 and 128
//                    blocks 33 / 30, 65 / 53; there 32, 60). Masked ones: R = 4, one wavefront per 32 rows up to 8 blocks (6 up to
//                    head_dim 64), then two: 72, 768 units, 5 blocks 7.4 and 8.2, 8 blocks 9.2 and 9.5, 16 blocks 14.1 and 13.0
struct SmallPlan { int R = 0, waves = 0; };
SmallPlan plan_small(const SdpaDev& p, int D, int n_cu) {
    if (p.key_mask || p.bias || p.lse || p.cu_q || p.cos_k || p.prefix_scaled || !offsets_fit_32_bits(p) || p.o_rs < 0 || p.o_rs >= (1L << 30)) return {};
    const long units = static_cast<long>(p.B) * p.H * ((p.Lq + 31) / 32);
    const int nb = key_blocks(p);
    const bool masked = p.mask_mode != MI_MASK_NONE;
    if (units <= n_cu) return {1, kMaxWaves};
    if (units <= 2L * n_cu) return {2, kMaxWaves};
    if (units > 4L * n_cu) return {};
    if (!masked) return D == 64 && nb >= 48 ? SmallPlan{2, kMaxWaves} : SmallPlan{};
    return {4, nb <= (D <= 64 ? 6 : 8) ? 4 : kMaxWaves};
}

SmallArgs small_args(const SdpaDev& p, int R, int S) {
    SmallArgs a{};
    a.q = p.q; a.k = p.k; a.v = p.v; a.kp = p.kp; a.vp = p.vp; a.o = p.o;
    a.kv_valid_len = p.kv_valid_len; a.cos_q = p.cos_q; a.sin_q = p.sin_q; a.rope_split = p.rope_split;
    a.q_rs = p.q_rs; a.q_bs = p.q_bs; a.o_bs = p.o_bs; a.k_bs = p.k_bs; a.v_bs = p.v_bs; a.kp_bs = p.kp_bs; a.vp_bs = p.vp_bs;
    a.k_rsb = static_cast<unsigned>(p.k_rs) * 2u; a.v_rsb = static_cast<unsigned>(p.v_rs) * 2u;
    a.o_rsb = static_cast<unsigned>(p.o_rs) * 2u;
    a.kp_rsb = static_cast<unsigned>(p.kp_rs) * 2u; a.vp_rsb = static_cast<unsigned>(p.vp_rs) * 2u;
    a.Lq = p.Lq; a.Lk = p.Lk; a.Lp = p.Lp; a.H = p.H; a.kv_group = p.kv_group; a.S = S; a.scale_log2 = p.scale_log2;
    a.n_q_tiles = (p.Lq + 32 * R - 1) / (32 * R);
    a.n_blocks = p.B * p.H * a.n_q_tiles;
    auto inverse = [](int d) { return static_cast<unsigned>(((1ull << 32) + d - 1) / static_cast<unsigned>(d)); };      // (not used for 1)
    a.inv_tiles = inverse(a.n_q_tiles); a.inv_heads = inverse(a.H); a.inv_group = inverse(a.kv_group);
    return a;
}

template <typename T, int D, int R, bool MASKED>
int launch_small(const SdpaDev& p, int most_waves, hipStream_t stream) {
    using SG = SmallGeo<D>;
    const int n_kb = key_blocks(p);
    int S = max(1, min(min(n_kb, most_waves / R), kMaxLds / (max(SG::BLOCK, R * SG::PART) + 256 * R)));
    const int steps = (n_kb + S - 1) / S;
    S = max(1, (n_kb + steps - 1) / max(steps, 1));      // as few wavefronts as take that many steps
    const int lds = S == 1 ? max(SG::BLOCK, 32 * R * HeadGeo<D>::O_STRIDE) : S * (max(SG::BLOCK, R * SG::PART) + 256 * R);
    SmallArgs a = small_args(p, R, S);
    const dim3 grid((a.n_blocks + 7) / 8 * 8), block(64 * R * S);
    if constexpr (MASKED) hipLaunchKernelGGL((sdpa_small_kernel<T, D, R, true, 0>), grid, block, lds, stream, a, p);
    else hipLaunchKernelGGL((sdpa_small_kernel<T, D, R, false, 0>), grid, block, lds, stream, a, NoMask{});
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail("sdpa_fwd launch: %s", hipGetErrorString(e));
    return 0;
}

template <typename T, int D>
int launch_small_r(const SdpaDev& p, const SmallPlan& plan, hipStream_t stream) {
    if (p.mask_mode == MI_MASK_NONE) return plan.R == 1 ? launch_small<T, D, 1, false>(p, plan.waves, stream) : launch_small<T, D, 2, false>(p, plan.waves, stream);
    switch (plan.R) {
        case 1: return launch_small<T, D, 1, true>(p, plan.waves, stream);
        case 2: return launch_small<T, D, 2, true>(p, plan.waves, stream);
        default: return launch_small<T, D, 4, true>(p, plan.waves, stream);
    }
}

template <typename T>
int launch_small_t(const SdpaDev& p, int head_dim, const SmallPlan& plan, hipStream_t stream) {
    switch (head_dim) {
        case 40: return launch_small_r<T, 40>(p, plan, stream);
        case 64: return launch_small_r<T, 64>(p, plan, stream);
        case 72: return launch_small_r<T, 72>(p, plan, stream);
        case 80: return launch_small_r<T, 80>(p, plan, stream);
        case 96: return launch_small_r<T, 96>(p, plan, stream);
        case 112: return launch_small_r<T, 112>(p, plan, stream);
        case 128: return launch_small_r<T, 128>(p, plan, stream);
        default: return launch_small_r<T, 160>(p, plan, stream);
    }
}

// ── cached cross-attention with its query projection in one launch ──
template <typename T, int D, int PROJ>
int launch_projected(const SdpaDev& p, const ProjArgs& proj, hipStream_t stream) {
    using PG = ProjGeo<D, PROJ>;
    static thread_local bool raised = false;
    if (!raised) {
        MI_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&sdpa_small_kernel<T, D, 2, false, PROJ>), hipFuncAttributeMaxDynamicSharedMemorySize, PG::LDS));
        raised = true;
    }
    const SmallArgs a = small_args(p, 2, kProjS);
    hipLaunchKernelGGL((sdpa_small_kernel<T, D, 2, false, PROJ>), dim3((a.n_blocks + 7) / 8 * 8), dim3(64 * 2 * kProjS), PG::LDS, stream, a, proj);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail("sdpa_fwd launch: %s", hipGetErrorString(e));
    return 0;
}
template <typename T>
int launch_projected_t(const SdpaDev& p, const ProjArgs& proj, int head_dim, hipStream_t stream) {
    if (head_dim == 40) return proj.w_scale ? launch_projected<T, 40, 2>(p, proj, stream) : launch_projected<T, 40, 1>(p, proj, stream);
    return proj.w_scale ? launch_projected<T, 80, 2>(p, proj, stream) : launch_projected<T, 80, 1>(p, proj, stream);
}

}  // namespace

// Where one launch less is worth the rows of x that every head projects for itself: up to a work group of 64 rows per compute unit (8
// heads, 77 keys, 16-bit weights, the whole block with its output projection in us, before / here: 40 of 320 channels, 8 groups 10.2 /
// 9.6, 256 13.8 / 11.7, 480 16.1 / 17.0; 80 of 640, 8 groups 11.7 / 12.7, 128 15.0 / 15.0, 144 15.9 / 15.0, 256 19.3 / 17.2, 480 26.2 /
// 27.0; INT8 weights: 40, 256 14.3 / 12.1, 80, 256 20.8 / 18.0; 231 keys 15.6 / 13.5 and 22.5 / 19.7). Not measured, so not taken: more
// than 640 channels or 256 keys.
bool sdpa_projected_takes(const SdpaDev& p, const LinearProblem& q, int head_dim) {
    if (head_dim != 40 && head_dim != 80) return false;
    if (sdpa_kernel_choice() != 0 || p.Lk < 1 || !sdpa_flow_runs(p) || p.kv_valid_len || p.cos_q || p.Lp != 0 || p.o_rs >= (1L << 30)) return false;
    // the projection's own conditions (launch_linear checks the rest, with its messages, when a call goes there)
    const uintptr_t al = reinterpret_cast<uintptr_t>(q.x) | reinterpret_cast<uintptr_t>(q.w) | reinterpret_cast<uintptr_t>(q.bias) | reinterpret_cast<uintptr_t>(p.k) |
                         reinterpret_cast<uintptr_t>(p.v) | reinterpret_cast<uintptr_t>(p.o);
    if ((al & 15u) || (reinterpret_cast<uintptr_t>(q.w_scale) & 3u) || q.K <= 0 || q.K % 64 != 0 || q.N % 8 != 0 || q.ldx % 8 != 0 || q.ldw % 16 != 0) return false;
    if (static_cast<long>(q.ldx) * 2 * 64 >= (1L << 31) || static_cast<long>(q.ldw) * 2 * 80 >= (1L << 31)) return false;
    const long groups = static_cast<long>(p.B) * p.H * ((p.Lq + 63) / 64);
    const int n_cu = device_cu_count();
    return groups <= n_cu && (head_dim == 40 || 2 * groups > n_cu) && q.K <= 640 && key_blocks(p) <= 8;
}

int launch_sdpa_projected(const SdpaDev& p, const LinearProblem& q, int dtype, int head_dim, hipStream_t stream) {
    ProjArgs a{};
    a.x = q.x; a.w = q.w; a.bias = q.bias; a.w_scale = q.w_scale;
    a.x_bsb = static_cast<long>(p.Lq) * q.ldx * 2;
    a.x_rsb = static_cast<unsigned>(q.ldx) * 2u; a.w_rsb = static_cast<unsigned>(q.ldw) * (q.w_scale ? 1u : 2u); a.n_steps = q.K / 64;
    if (dtype == MI_DTYPE_BF16) return launch_projected_t<__bf16>(p, a, head_dim, stream);
    return launch_projected_t<_Float16>(p, a, head_dim, stream);
}

int launch_sdpa_small(const SdpaDev& p, int dtype, int head_dim, hipStream_t stream) {
    const SmallPlan plan = plan_small(p, head_dim, device_cu_count());
    if (dtype == MI_DTYPE_BF16) return launch_small_t<__bf16>(p, head_dim, plan, stream);
    return launch_small_t<_Float16>(p, head_dim, plan, stream);
}

bool sdpa_small_takes(const SdpaDev& p, int head_dim) { return plan_small(p, head_dim, device_cu_count()).R != 0; }

}  // namespace mi
