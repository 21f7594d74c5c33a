// Y = X W^T + b for problems between the smallest and the 256 x 256-tile kernel's on gfx950 (contractions that are a
// multiple of 64; 16-bit or INT8 weights; plain or GEGLU).
//
// Operands go global -> LDS by DMA into a ring of S stages of 64 contraction elements each: no staging registers, no LDS
// store instructions, and as many steps in flight as the LDS holds (a problem of this size is a chain of memory latencies
// before it is anything else: with one step in flight, 2048 x 640 x 640 took 10 to 12 us of which 1 us is arithmetic). A
// stage holds BM rows of X and BN rows of W, 128 bytes each (INT8: 64), back to back as the DMA deposits them; bank
// conflicts of the fragment reads (16 rows, one 16-byte piece of each, per phase) are avoided by an XOR swizzle applied on
// the global side: the 16-byte piece in position c of row r is piece c ^ ((r >> 1) & 7). INT8 rows: c ^ ((r >> 2) & 3), which keeps
// reads of 8 bytes from 16 rows and two pieces apart (an operand of v_mfma_f32_16x16x32); those of 32 rows and one half of a piece
// (v_mfma_f32_32x32x16) meet in half of the banks and take two phases, and so do the operands of two blocks where the compiler
// fetches them with one ds_read2 (64 x 96 tiles: conflicts in 21 % of the busy cycles with the one, 35 % with the other).
//
// A work group is WM x WN wavefronts over tokens x features; a wavefront owns TM x TN blocks of 32 x 32 (as in linear.hip the
// product is computed transposed: MFMA rows are features). A stage is multiplied in two halves of 32 contraction elements, each
// read into a register set of its own while the other is multiplied. Step t:
//   multiply half 0 of stage t, between the products read half 1
//   wait until stage t + 1 has landed and this wavefront's reads of stage t have returned; barrier (for everybody)
//   multiply half 1 of stage t, between the products read half 0 of stage t + 1
// and the DMA of stage t + S, which goes into the ring slot of stage t, is dealt out between the MFMAs of the second half of
// step t and the first half of step t + 1: issued in one burst behind the barrier it made a step of 128 x 128 take 0.57 us
// on an otherwise empty compute unit, 0.4 dealt out. The accumulation order is the same in every form (and in linear_dma.hip):
// a problem gives the same bits whichever one takes it, alone or in a launch with others.
//
// Products are v_mfma_f32_16x16x32, two token blocks with one feature block in a row. What bounds the large forms on values of a
// real spread is the power limit, and a loop of these keeps up 2.03 PFLOP/s (bf16, N(0, 1); 1.90 fp16) at it, one of
// v_mfma_f32_32x32x16, which moves twice the accumulator registers per FLOP, 1.78 (1.64): the same bits. Reads in one burst in
// front of the products of a half kept the matrix pipe waiting for the LDS queue of all wavefronts behind each barrier: a step of
// 256 x 128 took 1427 clocks of which 1024 are products, 1260 so (halves of up to 8 products of 16-bit weights keep the burst). Both
// together (us): 4096 x 1152 x 1152 16.1 -> 14.8, 1024 x 6720 x 2240 37.6 -> 34, three of 16384 x 512 x 512 34.1 -> 32.8.
// A wavefront with one block of INT8 weights multiplies with v_mfma_f32_32x32x16 instead: its step is a chain of latencies and of
// widening, far from the power limit, and with the other product it is longer in every order of reads and widening tried (us, 32x32x16 /
// 16x16x32: fp16 32 x 1280 x 5120 15.5 / 16.7, 512 x 1280 x 5120 19.7 / 21.0; bf16 512 x 1280 x 5120 19.1 / 22.0, 1024 x 1280 x 5120
// 26.3 / 29.4, 77 x 6720 x 2240 10.5 / 11.6). Such loops of 80 to 100 instructions also take up to 3 % more or less by where they start in a cache line
// of instructions, so that this file is compiled with its loops aligned to 64 bytes (fp16, 64 x 64 tiles: 3 % faster than before).
//
// With NL > 0 the work group has NL further wavefronts that do nothing but load (a whole stage behind the barrier that frees its slot)
// and the others nothing but read and multiply: an LDS-DMA instruction keeps its wavefront from issuing for 33 clocks, the products of
// 64 contraction elements of a 32 x 32 block take 128. Steps of the small tiles become 10 to 20 % shorter, a 32 x 32 tile on one
// multiplying wavefront possible at all.
//
// Around the steps, a work group's fixed part (clocks of a 128 x 128 tile of 35 steps, 32 000 in all; before -> now): to the first DMA
// instruction 1900 -> 1250 (PipeArgs), first stage landed 2900, bias and last barrier 950 -> 390 (the bias is requested ahead of the
// loop), tile staged 1000, stored 1300 -> 570 (all pieces read before the first is stored).
//
// Measured (fp16, one launch, us, each column on a GPU of its own; first: 64 x 64 tiles through registers, one step ahead; then: this
// pipeline with the fixed part as it was; then: products of 32 x 32 x 16; now, on that GPU): 4096 x 1152 x 1152 30 / 16.9 / 15.7 / 14.3;
// 1024 x 2240 x 2240 30 / 16.3 / 15.5 / 15.2; 2048 x 640 x 640 8.4 / 6.9 / 5.3 / 5.4 (INT8 weights 11.5 / 7.8 / 6.05 / 6.04);
// 128 x 1280 x 1280 8.2 / 6.4 / 4.7 / 4.65 (INT8 - / 8.2 / 5.85 / 5.85), three of them - / 6.9 / 5.3 / 5.2 (INT8 - / 8.7 / 6.7 / 6.7);
// 256 x 1152 x 1152 - / 6.2 / 5.0 / 4.8; 3072 x 640 x 2560 - / 17.4 / 17.3 / 17.0; GEGLU 3072 x 640 -> 2 x 2560 39 / 32.0 / 29.2 / 27.2;
// three of 16384 x 512 x 512 - / 42.3 / 36.3 / 34.0.
#include <cmath>
#include <type_traits>
#include <utility>

#include "linear_forms.h"
#include "linear_math.h"

namespace mi {
namespace gemm {
namespace {

constexpr int kBK = 64;   // contraction elements per stage
// A launch as the kernel reads it. A problem is two cache lines, all of which are asked for before the first is used, and what a work
// group divides by to find its tile comes with an inverse: with the launch view and plain divisions the first DMA instruction stood
// behind four scalar-load latencies and four divisions (1900 clocks, 700 of them gone).
struct alignas(64) PipeProblem {
    const void* x; const void* w; const void* bias; void* y; const float* w_scale;
    int M, N, K, panel_tiles, width, last_width, n_panels;            // tiles of a whole panel, columns of tiles of a panel and of the last one
    unsigned ldx_b, ldw_b, inv_panel, inv_width, inv_last;            // row strides in bytes; floor(2^32 / divisor)
    long ldy_b;
};
struct PipeArgs {
    PipeProblem p[kMaxLinearProblems];
    int first[kMaxLinearProblems];       // first tile of a problem
    int n_tiles, chunk;
};
// x / d and x % d for x < 2^32; inv = floor(2^32 / d), one less for d = 1: the estimate is at most one short
struct DivMod { int q, r; };
__device__ __forceinline__ DivMod div_mod(int x, int d, unsigned inv) {
    unsigned q = __umulhi(static_cast<unsigned>(x), inv), r = static_cast<unsigned>(x) - q * d;
    if (r >= static_cast<unsigned>(d)) { ++q; r -= d; }
    return {static_cast<int>(q), static_cast<int>(r)};
}

template <typename T, bool W8, bool GEGLU, int WM, int WN, int TM, int TN, int S, int NL>
struct PipeGeo {
    static constexpr int NW = WM * WN, NT = 64 * NW;
    static constexpr int BM = WM * TM * 32, BN = WN * TN * 32;
    static constexpr int BN_OUT = GEGLU ? BN / 2 : BN;
    static constexpr int WROW = W8 ? 64 : 128;                    // bytes of a W row in a stage
    static constexpr int X_BYTES = BM * 128, W_BYTES = BN * WROW, STAGE = X_BYTES + W_BYTES;
    static constexpr int LW = NL ? NL : NW;                       // wavefronts that load
    static constexpr int MX = X_BYTES / 1024 / LW, MW = W_BYTES / 1024 / LW;   // DMA instructions of such a one per stage
    static constexpr int MI = MX + MW;
    static constexpr int OUT_ROW = BN_OUT * 2 + 16;
    static constexpr int LDS = S * STAGE > BM * OUT_ROW ? S * STAGE : BM * OUT_ROW;
    static_assert(MX * LW * 1024 == X_BYTES && MW * LW * 1024 == W_BYTES, "the same DMA duty for every loading wavefront");
    static_assert(!GEGLU || TN == 2, "the GEGLU form pairs the two feature blocks of a wavefront");
    static_assert(LDS <= 160 * 1024, "LDS of a compute unit");
    static_assert((S - 1) * MI < 64, "outstanding loads fit the counter");
};

template <typename T, bool W8, bool GEGLU, int WM, int WN, int TM, int TN, int S, int NL>
__global__ void __launch_bounds__(64 * (WM * WN + NL), 2) linear_pipe_kernel(const PipeArgs args) {
    using G = PipeGeo<T, W8, GEGLU, WM, WN, TM, TN, S, NL>;
    using M = Mma<T>;
    using V8 = typename M::v8;
    using V4 = typename M::v4;
    constexpr int BM = G::BM, BN = G::BN, BN_OUT = G::BN_OUT, MI = G::MI;
    // one block of INT8 weights per wavefront: v_mfma_f32_32x32x16 (see the top)
    constexpr bool ONE = W8 && TM == 1 && TN == 1;
    constexpr int BS = ONE ? 32 : 16, FB = TN * 32 / BS, TB = TM * 32 / BS;      // rows of a block; feature and token blocks of a wavefront
    constexpr int KS = BS / 16;                  // products of a half per pair of blocks
    constexpr int NG = ONE ? 4 : 1;              // groups of 4 features that a lane holds of a block, 8 apart
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];

    // Tiles of all problems in one row; consecutive work-group ids go to the 8 XCDs in turn, and every XCD (one L2) takes a
    // contiguous run of it. A problem's tiles are numbered panel by panel (PipeProblem::width columns of tiles, row by row), so that a
    // run is about as many rows of X as rows of W: what a run touches comes from the last-level cache, which serves a
    // compute unit 28 bytes per ns when all of them ask, once, and from then on from the L2 at 95.
#pragma unroll
    for (int i = 0; i < kMaxLinearProblems; ++i) asm volatile("" : : "s"(args.p[i].x), "s"(args.p[i].ldx_b));
    asm volatile("" : : "s"(args.first[1]), "s"(args.first[2]), "s"(args.n_tiles), "s"(args.chunk));
    int tile = (static_cast<int>(blockIdx.x) & 7) * args.chunk + (static_cast<int>(blockIdx.x) >> 3);
    if (tile >= args.n_tiles) return;
    const int pi = (tile >= args.first[1] ? 1 : 0) + (tile >= args.first[2] ? 1 : 0);
    const PipeProblem& p = args.p[pi];
    const DivMod in_problem = div_mod(tile - args.first[pi], p.panel_tiles, p.inv_panel);
    const bool last = in_problem.q == p.n_panels - 1;
    const DivMod in_panel = div_mod(in_problem.r, last ? p.last_width : p.width, last ? p.inv_last : p.inv_width);
    const int m0 = in_panel.q * BM, n0 = (in_problem.q * p.width + in_panel.r) * BN_OUT;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, lr = lane % BS, lg = lane / BS;      // (row of a block, group of 8 contraction elements)
    const int wm = wave % WM, wn = wave / WM;

    const int lw = NL ? wave - G::NW : wave;     // (NL: the loading wavefronts come last)
    // a pointer that is the same for the whole wavefront, in scalar registers
    auto uniform = [](const unsigned char* q) {
        const unsigned long u = reinterpret_cast<unsigned long>(q);
        const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(u)), hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(u >> 32));
        return reinterpret_cast<const unsigned char*>(static_cast<unsigned long>(hi) << 32 | lo);
    };
    // ── DMA duty: X instructions lw + LW m (8 rows of 128 bytes each), W instructions likewise (INT8: 16 rows of 64) ──
    const unsigned char* xg = uniform(static_cast<const unsigned char*>(p.x) + static_cast<long>(m0) * p.ldx_b);
    const unsigned char* wg = uniform(static_cast<const unsigned char*>(p.w) + (GEGLU ? 0L : static_cast<long>(n0) * p.ldw_b));
    unsigned xoff[G::MX], woff[G::MW];
#pragma unroll
    for (int u = 0; u < G::MX; ++u) {
        const int r = 8 * (lw + G::LW * u) + (lane >> 3);
        xoff[u] = static_cast<unsigned>(min(r, p.M - 1 - m0)) * p.ldx_b + ((lane & 7) ^ ((r >> 1) & 7)) * 16u;
    }
#pragma unroll
    for (int u = 0; u < G::MW; ++u) {
        const int r = W8 ? 16 * (lw + G::LW * u) + (lane >> 2) : 8 * (lw + G::LW * u) + (lane >> 3);
        const unsigned piece = W8 ? (lane & 3) ^ ((r >> 2) & 3) : (lane & 7) ^ ((r >> 1) & 7);
        // GEGLU: 32-row groups of the tile alternate between the value and the gate rows of the same features
        const int row = GEGLU ? min(n0 + 32 * (r >> 6) + (r & 31), p.N - 1) + ((r >> 5) & 1) * p.N : min(r, p.N - 1 - n0);
        woff[u] = static_cast<unsigned>(row) * p.ldw_b + piece * 16u;
    }
    const unsigned lds_base = static_cast<unsigned>(reinterpret_cast<size_t>((__attribute__((address_space(3))) unsigned char*)lds));
    // (the LDS destination travels in m0; the s_nop is the wait state an LDS-DMA instruction needs behind a write of m0)
    auto dma = [&](unsigned voff, const unsigned char* base, unsigned dst) {
        asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(base), "{m0}"(dst) : "memory");
    };
    // pieces [J0, J1) of this wavefront's share of a stage; xg / wg stand on that stage
    auto dma_piece = [&](int j, unsigned slot) {
        if (j < G::MX) dma(xoff[j < G::MX ? j : 0], xg, lds_base + slot + (lw + G::LW * j) * 1024);
        else dma(woff[j < G::MX ? 0 : j - G::MX], wg, lds_base + slot + G::X_BYTES + (lw + G::LW * (j - G::MX)) * 1024);
    };
    auto next_stage = [&]() {
        xg += kBK * 2;
        wg += W8 ? kBK : kBK * 2;
    };
    // Waits until at most `stages` of this wavefront's stages are in flight and its LDS reads have returned, then meets the others.
    auto wait_barrier = [&](int stages) {
        if (stages == S - 2) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((S - 2) * MI) : "memory");
        else {
            [&]<int... I>(std::integer_sequence<int, I...>) {
                ([&] { if (stages == I) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(I * MI) : "memory"); }(), ...);
            }(std::make_integer_sequence<int, S>{});
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
    };

    // The bias (and scale) of this lane's features, requested ahead of the first DMA: behind the loop its latency was 700 to 1800 clocks.
    // (N is a multiple of 8, so 4 features are in or out together; those past the end are not stored.)
    typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
    const T* const bias = static_cast<const T*>(p.bias);
    V4 braw[FB * NG];
    f32x4_a4 sraw[W8 ? FB * NG : 1];
    // the 4 features from feature(a) on are the lane's group a % NG of block a / NG
    // (GEGLU: blocks 0 and 1 are values, 2 and 3 the gates of the same features)
    auto feature = [&](int a) { return min(n0 + (GEGLU ? wn * 32 + 16 * (a & 1) : wn * TN * 32 + BS / NG * a) + 4 * lg, p.N - 4) + (GEGLU ? (a >> 1) * p.N : 0); };
#pragma unroll
    for (int a = 0; a < FB * NG; ++a) {
        if constexpr (W8) sraw[a] = *reinterpret_cast<const f32x4_a4*>(p.w_scale + feature(a));
        braw[a] = V4{};
    }
    if (bias != nullptr) {
#pragma unroll
        for (int a = 0; a < FB * NG; ++a) braw[a] = *reinterpret_cast<const V4*>(bias + feature(a));
    }

    // ── fragment reads: a stage is two halves of 32 contraction elements, KS MFMA operands each ──
    unsigned xaddr[2 * KS], waddr[2 * KS];
#pragma unroll
    for (int c = 0; c < 2 * KS; ++c) {
        const int piece = c * (64 / BS) + lg;       // of 8 contraction elements
        xaddr[c] = wm * TM * 4096 + lr * 128 + ((piece ^ ((lr >> 1) & 7)) << 4);
        waddr[c] = G::X_BYTES + wn * TN * 32 * G::WROW +
                   (W8 ? lr * 64 + (((piece >> 1) ^ ((lr >> 2) & 3)) << 4) + 8 * (piece & 1) : lr * 128 + ((piece ^ ((lr >> 1) & 7)) << 4));
    }
    using WRaw = std::conditional_t<W8, u32x2, V8>;
    V8 xf[2][KS * TB];
    WRaw wf[2][KS * FB];
    // reads [R0, R1) of the NR of a half, in the order in which its products use them: two token blocks, the feature blocks, the other
    // token blocks
    constexpr int NR = KS * (TB + FB);
    auto read_pieces = [&](auto half_tag, auto r0_tag, auto r1_tag, unsigned slot) {
        constexpr int H = decltype(half_tag)::value, R0 = decltype(r0_tag)::value, R1 = decltype(r1_tag)::value;
        [&]<int... R>(std::integer_sequence<int, R...>) {
            ([&] {
                constexpr int k = R0 + R;
                if constexpr (ONE) {
                    if constexpr (k % 2 == 0) xf[H][k / 2] = *reinterpret_cast<const V8*>(lds + slot + xaddr[2 * H + k / 2]);
                    else wf[H][k / 2] = *reinterpret_cast<const WRaw*>(lds + slot + waddr[2 * H + k / 2]);
                } else if constexpr (k >= 2 && k < 2 + FB) wf[H][k - 2] = *reinterpret_cast<const WRaw*>(lds + slot + waddr[H] + (k - 2) * 16 * G::WROW);
                else {
                    constexpr int b = k < 2 ? k : k - FB;
                    xf[H][b] = *reinterpret_cast<const V8*>(lds + slot + xaddr[H] + b * 2048);
                }
            }(), ...);
        }(std::make_integer_sequence<int, R1 - R0>{});
    };
    auto read_half = [&](auto half_tag, unsigned slot) { read_pieces(half_tag, std::integral_constant<int, 0>{}, std::integral_constant<int, NR>{}, slot); };
    std::conditional_t<ONE, f32x16, f32x4> acc[FB][TB];
#pragma unroll
    for (int a = 0; a < FB; ++a)
#pragma unroll
        for (int b = 0; b < TB; ++b)
#pragma unroll
            for (int e = 0; e < 4 * NG; ++e) acc[a][b][e] = 0.f;
    // the MFMAs of a half stage, and between them the reads of the next one (READ: half 1 - H from `from`) and DMA pieces [J0, J1) of
    // the stage that goes to `slot`
    auto multiply_half = [&](auto half_tag, auto read_tag, unsigned from, auto j0_tag, auto j1_tag, unsigned slot) {
        constexpr int H = decltype(half_tag)::value, J0 = decltype(j0_tag)::value, J1 = decltype(j1_tag)::value, NM = KS * TB * FB;
        constexpr bool READ = decltype(read_tag)::value;
        // (a half of few MFMAs: all reads ahead of them, as dealt out the last one returns too late; INT8 of two blocks: behind the first
        //  two, under the widening)
        constexpr bool BURST = ONE || (NM <= 8 && !W8);
        constexpr int SPAN = NM <= 8 ? 2 : NM * 3 / 4;      // MFMAs that have reads behind them
        if constexpr (READ && BURST) {
            read_pieces(std::integral_constant<int, 1 - H>{}, std::integral_constant<int, 0>{}, std::integral_constant<int, NR>{}, from);
            __builtin_amdgcn_sched_barrier(0);
        }
        // (INT8: all blocks widened ahead of the products; between them steps of two and more blocks take 1 to 4 % longer)
        V8 w[W8 ? KS * FB : 1];
        if constexpr (W8) {
#pragma unroll
            for (int a = 0; a < KS * FB; ++a) w[a] = widen<T>(wf[H][a]);
        }
        [&]<int... Q>(std::integer_sequence<int, Q...>) {
            ([&] {
                // (two token blocks at a time, each feature block meets both in a row)
                constexpr int a = ONE ? 0 : Q / 2 % FB, b = ONE ? 0 : Q / (2 * FB) * 2 + Q % 2;
                if constexpr (ONE) acc[0][0] = M::run(w[Q], xf[H][Q], acc[0][0]);
                else if constexpr (W8) acc[a][b] = M::run16(w[a], xf[H][b], acc[a][b]);
                else acc[a][b] = M::run16(wf[H][a], xf[H][b], acc[a][b]);
                if constexpr (READ && !BURST && Q < SPAN)
                    read_pieces(std::integral_constant<int, 1 - H>{}, std::integral_constant<int, NR * Q / SPAN>{}, std::integral_constant<int, NR * (Q + 1) / SPAN>{}, from);
                constexpr int j0 = J0 + (J1 - J0) * Q / NM, j1 = J0 + (J1 - J0) * (Q + 1) / NM;
                if constexpr (j1 > j0) {
#pragma unroll
                    for (int j = j0; j < j1; ++j) dma_piece(j, slot);
                }
                if constexpr (j1 > j0 || (READ && !BURST && Q < SPAN)) __builtin_amdgcn_sched_barrier(0);
            }(), ...);
        }(std::make_integer_sequence<int, NM>{});
    };

    using Half0 = std::integral_constant<int, 0>;
    using Half1 = std::integral_constant<int, 1>;
    using Mid = std::integral_constant<int, MI / 2>;
    using All = std::integral_constant<int, MI>;
    const int n = p.K / kBK;
    unsigned cur = 0, prev = (S - 1) * G::STAGE;      // ring slots of stages t and t - 1
    // Step t. D0: the second part of stage t + S - 1 is loaded, into the slot of stage t - 1; D1: the first part of stage t + S,
    // into the slot of stage t.
    auto step = [&](auto d0_tag, auto d1_tag, int t) {
        constexpr bool D0 = decltype(d0_tag)::value, D1 = decltype(d1_tag)::value;
        const unsigned nxt = cur + G::STAGE == S * G::STAGE ? 0u : cur + G::STAGE;
        if constexpr (D0) {
            multiply_half(Half0{}, std::true_type{}, cur, Mid{}, All{}, prev);
            next_stage();
        } else {
            multiply_half(Half0{}, std::true_type{}, cur, Half0{}, Half0{}, 0u);
        }
        __builtin_amdgcn_sched_barrier(0);
        wait_barrier(D1 ? S - 2 : (t + S - 1 < n - 1 ? t + S - 1 : n - 1) - (t + 1));
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (D1) multiply_half(Half1{}, std::true_type{}, nxt, Half0{}, Mid{}, cur);
        else multiply_half(Half1{}, std::true_type{}, nxt, Half0{}, Half0{}, 0u);
        __builtin_amdgcn_sched_barrier(0);
        prev = cur;
        cur = nxt;
    };
    if constexpr (NL > 0) {
        const int ahead = n < S ? n : S;
        if (wave >= G::NW) {
            unsigned slot = 0;
            auto load_stage = [&]() {
#pragma unroll
                for (int j = 0; j < MI; ++j) dma_piece(j, slot);
                next_stage();
                slot = slot + G::STAGE == S * G::STAGE ? 0u : slot + G::STAGE;
            };
            for (int s = 0; s < ahead; ++s) load_stage();
            if (ahead == S) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"((S - 1) * MI) : "memory");
            else wait_barrier(ahead - 1);
            int t = 0;
            for (; t < n - S; ++t) {       // stage t + 1 has landed, the slot of stage t is free
                wait_barrier(S - 2);
                load_stage();
            }
            for (; t < n - 1; ++t) wait_barrier(n - 2 - t);
            __syncthreads();
            __syncthreads();
            return;
        }
        asm volatile("s_barrier" ::: "memory");      // stage 0 has landed
        read_half(Half0{}, 0);
        for (int t = 0; t < n - 1; ++t) {
            const unsigned nxt = cur + G::STAGE == S * G::STAGE ? 0u : cur + G::STAGE;
            multiply_half(Half0{}, std::true_type{}, cur, Half0{}, Half0{}, 0u);
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // stage t is in registers
            __builtin_amdgcn_sched_barrier(0);
            multiply_half(Half1{}, std::true_type{}, nxt, Half0{}, Half0{}, 0u);
            __builtin_amdgcn_sched_barrier(0);
            cur = nxt;
        }
    } else if (n < S) {   // everything fits the ring
        for (int s = 0; s < n; ++s) {
#pragma unroll
            for (int j = 0; j < MI; ++j) dma_piece(j, s * G::STAGE);
            next_stage();
        }
        wait_barrier(n - 1);
        read_half(Half0{}, 0);
        for (int t = 0; t < n - 1; ++t) step(std::false_type{}, std::false_type{}, t);
    } else {
        for (int s = 0; s < S - 1; ++s) {
#pragma unroll
            for (int j = 0; j < MI; ++j) dma_piece(j, s * G::STAGE);
            next_stage();
        }
#pragma unroll
        for (int j = 0; j < MI / 2; ++j) dma_piece(j, prev);
        // stage 0 has landed: behind it are S - 2 stages and the first part of another
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"((S - 2) * MI + MI / 2) : "memory");
        read_half(Half0{}, 0);
        int t = 0;
        for (; t < n - S; ++t) step(std::true_type{}, std::true_type{}, t);
        step(std::true_type{}, std::false_type{}, t);
        for (++t; t < n - 1; ++t) step(std::false_type{}, std::false_type{}, t);
    }
    // The last step: nothing behind it to wait for or to read. It stands here once and not as a branch inside `step`: where that branch
    // met the others again, the compiler moved all accumulators, 115 to 238 registers became 131 to 256 and the GEGLU tile of 192 x 128
    // put 215 to 356 of them in scratch, each reload behind a wait for the DMA as well (GEGLU, fp16, us with the branch / without:
    // 2048 x 640 -> 2 x 2560 28.7 / 20.0, INT8 36.0 / 20.9; 4096 x 320 -> 2 x 1280 23.0 / 14.1, INT8 29.5 / 15.2; 1024 x 1280 ->
    // 2 x 5120 41.2 / 32.5, INT8 48.8 / 32.9).
    multiply_half(Half0{}, std::true_type{}, cur, Half0{}, Half0{}, 0u);
    __builtin_amdgcn_sched_barrier(0);
    multiply_half(Half1{}, std::false_type{}, 0u, Half0{}, Half0{}, 0u);

    __syncthreads();   // the ring is used up
    // ── epilogue: acc[a][b][i] is feature n0 + wn TN 32 + 16 a + 4 lg + i of token m0 + wm TM 32 + 16 b + lr; the tile
    //    leaves through LDS as 16-byte pieces of rows of Y ──
    if constexpr (GEGLU) {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < TB; ++b) {
                V4 o;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float bv = static_cast<float>(braw[a][i]), bg = static_cast<float>(braw[2 + a][i]);
                    float val, gate;
                    if constexpr (W8) {   // the two halves are rounded where the reference's 16-bit intermediate would
                        val = static_cast<float>(static_cast<T>(scaled_acc(acc[a][b][i], sraw[a][i], bv)));
                        gate = static_cast<float>(static_cast<T>(scaled_acc(acc[2 + a][b][i], sraw[2 + a][i], bg)));
                    } else {
                        val = acc[a][b][i] + bv;
                        gate = acc[2 + a][b][i] + bg;
                    }
                    o[i] = static_cast<T>(val * gelu_erf(gate));
                }
                *reinterpret_cast<V4*>(lds + (wm * TM * 32 + 16 * b + lr) * G::OUT_ROW + (wn * 32 + 16 * a + 4 * lg) * 2) = o;
            }
    } else {
#pragma unroll
        for (int a = 0; a < FB * NG; ++a)
#pragma unroll
            for (int b = 0; b < TB; ++b) {
                V4 o;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float bv = static_cast<float>(braw[a][i]), sum = acc[a / NG][b][4 * (a % NG) + i];
                    if constexpr (W8) o[i] = static_cast<T>(scaled_acc(sum, sraw[a][i], bv));
                    else o[i] = static_cast<T>(sum + bv);
                }
                *reinterpret_cast<V4*>(lds + (wm * TM * 32 + BS * b + lr) * G::OUT_ROW + (wn * TN * 32 + BS / NG * a + 4 * lg) * 2) = o;
            }
    }
    __syncthreads();
    constexpr int PPR = BN_OUT / 8;   // 16-byte pieces per staged row
    constexpr int PIECES = BM * PPR / G::NT, RSTEP = G::NT / PPR;
    static_assert(BM * PPR % G::NT == 0 && G::NT % PPR == 0, "the same pieces for every thread, one below the other");
    const int row = tid / PPR, piece = tid % PPR;
    unsigned char* const yg = static_cast<unsigned char*>(p.y) + static_cast<long>(m0 + row) * p.ldy_b + (n0 + piece * 8) * 2L;
    u32x4 out[PIECES];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) out[i] = *reinterpret_cast<const u32x4*>(lds + (row + i * RSTEP) * G::OUT_ROW + piece * 16);
    // (whole tiles without a branch: one per piece, each with its own read and wait, took 300 clocks a piece)
    if (m0 + BM <= p.M && n0 + BN_OUT <= p.N) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i) *reinterpret_cast<u32x4*>(yg + i * RSTEP * p.ldy_b) = out[i];
    } else if (n0 + piece * 8 < p.N) {
#pragma unroll
        for (int i = 0; i < PIECES; ++i)
            if (m0 + row + i * RSTEP < p.M) *reinterpret_cast<u32x4*>(yg + i * RSTEP * p.ldy_b) = out[i];
    }
}

template <typename T, bool W8, bool GEGLU, int WM, int WN, int TM, int TN, int S, int NL>
int launch_pipe(const LinearBatch& batch, int n_problems, hipStream_t st) {
    using G = PipeGeo<T, W8, GEGLU, WM, WN, TM, TN, S, NL>;
    auto tiles_m = [&](int i) { return (batch.p[i].M + G::BM - 1) / G::BM; };
    auto tiles_n = [&](int i) { return (batch.p[i].N + G::BN_OUT - 1) / G::BN_OUT; };
    long tiles = 0;
    for (int i = 0; i < n_problems; ++i) tiles += static_cast<long>(tiles_m(i)) * tiles_n(i);
    if (tiles > 0x7ffffff0L) return fail("linear: problem too large for one launch");
    if (G::LDS > 64 * 1024) {
        static thread_local bool raised = false;
        if (!raised) {
            MI_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&linear_pipe_kernel<T, W8, GEGLU, WM, WN, TM, TN, S, NL>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS));
            raised = true;
        }
    }
    auto inverse = [](int d) { return d == 1 ? 0xffffffffu : static_cast<unsigned>((1ull << 32) / static_cast<unsigned>(d)); };
    PipeArgs args{};
    args.n_tiles = static_cast<int>(tiles);
    args.chunk = (args.n_tiles + 7) / 8;
    int first = 0;
    for (int i = 0; i < kMaxLinearProblems; ++i) {
        args.first[i] = i < n_problems ? first : 0x7fffffff;
        if (i >= n_problems) continue;
        const LinearProblem& b = batch.p[i];
        PipeProblem& p = args.p[i];
        p.x = b.x; p.w = b.w; p.bias = b.bias; p.y = b.y; p.w_scale = b.w_scale;
        p.M = b.M; p.N = b.N; p.K = b.K;
        p.ldx_b = static_cast<unsigned>(b.ldx) * 2u; p.ldw_b = static_cast<unsigned>(b.ldw) * (W8 ? 1u : 2u); p.ldy_b = b.ldy * 2;
        p.width = min(tiles_n(i), max(1, static_cast<int>(std::sqrt(static_cast<double>(tiles) / 8 * G::BM / G::BN) + 0.5)));
        p.n_panels = (tiles_n(i) + p.width - 1) / p.width;
        p.last_width = tiles_n(i) - (p.n_panels - 1) * p.width;
        p.panel_tiles = tiles_m(i) * p.width;
        p.inv_panel = inverse(p.panel_tiles); p.inv_width = inverse(p.width); p.inv_last = inverse(p.last_width);
        first += tiles_m(i) * tiles_n(i);
    }
    hipLaunchKernelGGL((linear_pipe_kernel<T, W8, GEGLU, WM, WN, TM, TN, S, NL>), dim3(static_cast<unsigned>((tiles + 7) / 8 * 8)), dim3(G::NT + 64 * NL), G::LDS, st, args);
    MI_HIP_CHECK(hipGetLastError());
    return 0;
}

template <typename T>
int launch_form(const LinearBatch& b, int n, bool geglu, int dtype, hipStream_t st) {
    const bool w8 = b.p[0].w_scale != nullptr;
    const int form = pick_form(b, n, geglu, device_cu_count());
    if (geglu && w8) {
        switch (form) {
            case kG8_64x64: return launch_pipe<T, true, true, 2, 2, 1, 2, 3, 0>(b, n, st);
            case kG8_128x64_2: return launch_pipe<T, true, true, 2, 2, 2, 2, 2, 0>(b, n, st);
            case kG8_192x128: return launch_pipe<T, true, true, 2, 4, 3, 2, 3, 0>(b, n, st);
            default: return launch_pipe<T, true, true, 4, 2, 2, 2, 3, 0>(b, n, st);
        }
    }
    if (geglu) {
        switch (form) {
            case kG64x64: return launch_pipe<T, false, true, 2, 2, 1, 2, 3, 4>(b, n, st);
            case kG128x64_2: return launch_pipe<T, false, true, 2, 2, 2, 2, 2, 0>(b, n, st);
            case kG128x64: return launch_pipe<T, false, true, 2, 2, 2, 2, 3, 4>(b, n, st);
            case kG192x128: return launch_pipe<T, false, true, 2, 4, 3, 2, 2, 0>(b, n, st);
            default: return launch_pipe<T, false, true, 4, 2, 2, 2, 3, 0>(b, n, st);
        }
    }
    if (w8) {
        switch (form) {
            case k8_32x32: return launch_pipe<T, true, false, 1, 1, 1, 1, 6, 2>(b, n, st);
            case k8_64x64: return launch_pipe<T, true, false, 2, 2, 1, 1, 4, 4>(b, n, st);
            case k8_64x96: return launch_pipe<T, true, false, 2, 3, 1, 1, 5, 2>(b, n, st);
            case k8_128x64: return launch_pipe<T, true, false, 2, 2, 2, 1, 3, 4>(b, n, st);
            case k8_128x96: return launch_pipe<T, true, false, 2, 3, 2, 1, 3, 2>(b, n, st);
            case k8_128x128: return launch_pipe<T, true, false, 2, 4, 2, 1, 4, 0>(b, n, st);
            default: return launch_pipe<T, true, false, 2, 2, 2, 2, 2, 0>(b, n, st);
        }
    }
    switch (form) {
        case k32x32: return launch_pipe<T, false, false, 1, 1, 1, 1, 6, 2>(b, n, st);
        case k64x32: return launch_pipe<T, false, false, 2, 1, 1, 1, 6, 2>(b, n, st);
        case k64x64: return launch_pipe<T, false, false, 2, 2, 1, 1, 4, 4>(b, n, st);
        case k64x96: return launch_pipe<T, false, false, 2, 3, 1, 1, 5, 4>(b, n, st);
        case k128x64_load: return launch_pipe<T, false, false, 2, 2, 2, 1, 3, 4>(b, n, st);
        case k128x96: return launch_pipe<T, false, false, 2, 3, 2, 1, 4, 4>(b, n, st);
        case k128x64: return launch_pipe<T, false, false, 2, 2, 2, 1, 3, 0>(b, n, st);
        case k128x128: return launch_pipe<T, false, false, 2, 2, 2, 2, 3, 4>(b, n, st);
        case k128x128_2: return launch_pipe<T, false, false, 2, 2, 2, 2, 2, 0>(b, n, st);
        case k192x128: return launch_pipe<T, false, false, 2, 4, 3, 1, 4, 0>(b, n, st);
        case k256x128: return launch_pipe<T, false, false, 4, 2, 2, 2, 3, 0>(b, n, st);
        default: return launch_linear_dma(b, n, dtype, st);
    }
}

}  // namespace
}  // namespace gemm

// Contractions of whole stages; operands whose tiles (GEGLU: whose whole W) are addressable with 32-bit byte offsets.
bool linear_pipe_takes(const LinearBatch& batch, int n_problems, bool geglu) {
    for (int i = 0; i < n_problems; ++i) {
        const LinearProblem& p = batch.p[i];
        if (p.K % gemm::kBK != 0) return false;
        if (p.w_scale != nullptr && (p.ldw % 16 != 0)) return false;   // (rows of 16-byte pieces)
        if (static_cast<long>(p.ldx) * 2 * 256 >= (1L << 31) || static_cast<long>(p.ldw) * 2 * 256 >= (1L << 31)) return false;
        if (geglu && static_cast<long>(p.N) * 2 * p.ldw * 2 >= (1L << 32)) return false;
    }
    return true;
}

int launch_linear_pipe(const LinearBatch& batch, int n_problems, int dtype, bool geglu, hipStream_t st) {
    if (dtype == MI_DTYPE_BF16) return gemm::launch_form<__bf16>(batch, n_problems, geglu, dtype, st);
    return gemm::launch_form<_Float16>(batch, n_problems, geglu, dtype, st);
}

}  // namespace mi
