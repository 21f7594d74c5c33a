// Softmax attention of head_dim 512 on gfx950, the form for long calls that fill the GPU (sdpa_wide_plan.h says which those are; sdpa_wide.hip merges
// their parts): the same work group, LDS rings and softmax, other matrix instructions.
//
// Products are v_mfma_f32_16x16x32, each LDS fragment with both blocks of 16 query rows in turn: at the power limit they run at a
// 14 % higher clock than v_mfma_f32_32x32x16 (1.86 against 1.63 GHz, head_dim 512, N(0, 1)). But a product covers 16 clocks instead
// of 32, and what stands between two of them in one piece (two V reads; a DMA instruction behind a read) no longer fits: cycles
// per CU 794 k before, 963 k so, 16384 tokens of one head 485 -> 518 us on one GPU. Hence the order of a slot: first product, one LDS
// read, second product, then one other thing (the second half of a V fragment; a DMA instruction or an exponential in turn), and the
// scale and reference of the scores go under the PV product. The times differ from GPU to GPU: 16384 tokens, fp16, us, the kernel of
// sdpa_wide.hip / this one, three of them: 498 / 455 (without the turns 459), 490 / 454, 508 / 468. Mid-block around it on another (540 before): DMA
// ahead of the second product 521, exponentials there 537, fragments 5 or 7 ahead instead of 6 523 and 526 (518 in that build).
// Mid-block of 16384 tokens: 560 -> 553 and 559 -> 549 on two GPUs.
//   Register layouts (lq = lane % 16, g = lane / 16): A row lq, B column lq, 8 contraction elements from 8 g on; C column lq, element
//   i is row 4 g + i. A lane holds scores of two query rows (16 r + lq of the wavefront's 32), each shared with the lanes 16, 32 and
//   48 away; P goes into the PV product as it lies (slot 8 g + t of the contraction is key 4 g + t, for t >= 4 key 16 + 4 g + t - 4).
//   LDS: rows back to back as the DMA deposits them, 16-byte chunk c of row r at position c ^ f(r) within its group of 16
//   chunks, f(r) = 2 (r % 8 ^ (r & 8) / 2) + r / 8 % 2: the K fragment reads (16 rows, one chunk column) and the V transpose reads
//   (8 rows, two chunks) are both free of bank conflicts.
#include "sdpa_wide.h"

namespace mi {
namespace {

using namespace sdpa;

// (inline assembly with O in a[0 : 8 VB) by name, block vb of query rows r in a[8 vb + 4 r : + 4), for the reasons given in
// sdpa_wide.hip. The wait that VALU code needs before it touches the result of an MFMA of 4 passes, 8 wait states, is kept by
// construction: the last MFMAs of a score tile and the four that follow them are one statement, four slots pass before the
// scores are scaled, and wide_settle stands in front of the code that works on O.)
template <typename T> struct WideMma;
#define MI_WIDE_MMA(TYPE, NAME)                                                                                               \
    template <> struct WideMma<TYPE> {                                                                                        \
        using V8 = typename Mma<TYPE>::v8;                                                                                    \
        static __device__ __forceinline__ void first(f32x4& s, V8 a, V8 b) {                                                  \
            asm volatile(NAME " %0, %1, %2, 0" : "=&v"(s) : "v"(a), "v"(b));                                                  \
        }                                                                                                                     \
        static __device__ __forceinline__ void score(f32x4& s, V8 a, V8 b) {                                                  \
            asm volatile(NAME " %0, %1, %2, %0" : "+v"(s) : "v"(a), "v"(b));                                                  \
        }                                                                                                                     \
        /* O block B += a b */                                                                                                \
        template <int B> static __device__ __forceinline__ void out(V8 a, V8 b) {                                             \
            asm volatile(NAME " a[%2:%3], %0, %1, a[%2:%3]" : : "v"(a), "v"(b), "n"(4 * B), "n"(4 * B + 3) : MI_AGPRS);       \
        }                                                                                                                     \
        /* the last two MFMAs of a score tile together with the first four of the PV product (O blocks 0 to 3) */             \
        static __device__ __forceinline__ void tail(f32x4& s0, f32x4& s1, V8 ak, V8 q0, V8 q1, V8 a0, V8 a1, V8 p0, V8 p1) {  \
            asm volatile(NAME " %0, %2, %3, %0\n\t" NAME " %1, %2, %4, %1\n\t"                                                \
                         NAME " a[0:3], %5, %7, a[0:3]\n\t" NAME " a[4:7], %5, %8, a[4:7]\n\t"                                \
                         NAME " a[8:11], %6, %7, a[8:11]\n\t" NAME " a[12:15], %6, %8, a[12:15]"                             \
                         : "+v"(s0), "+v"(s1) : "v"(ak), "v"(q0), "v"(q1), "v"(a0), "v"(a1), "v"(p0), "v"(p1) : MI_AGPRS);    \
        }                                                                                                                     \
    };
MI_WIDE_MMA(__bf16, "v_mfma_f32_16x16x32_bf16")
MI_WIDE_MMA(_Float16, "v_mfma_f32_16x16x32_f16")
#undef MI_WIDE_MMA
// every MFMA in flight has written its result when this returns
__device__ __forceinline__ void wide_settle(f32x4 (&s)[2][2]) {
    asm volatile("s_nop 15\n\ts_nop 15" : "+v"(s[0][0]), "+v"(s[0][1]), "+v"(s[1][0]), "+v"(s[1][1]) : : MI_AGPRS);
}
// O *= f, per row of the lane (the reads of a block go out before its writes: a value just read is not touched in the next instruction)
template <int B> __device__ __forceinline__ void o_scale_block(const float (&f)[2]) {
    [&]<int... I>(std::integer_sequence<int, I...>) {
        const float v[16] = {o_get<16 * B + I>()...};
        (o_set<16 * B + I>(v[I] * f[(I >> 2) & 1]), ...);
    }(std::make_integer_sequence<int, 16>{});
}
template <int N> __device__ __forceinline__ void o_scale(const float (&f)[2]) {
    [&]<int... B>(std::integer_sequence<int, B...>) { (o_scale_block<B>(f), ...); }(std::make_integer_sequence<int, N / 16>{});
    asm volatile("s_nop 7" : : : MI_AGPRS);   // accumulation registers written by the VALU and read by the next MFMA
}

// max / sum over the four lanes of a row (lane % 16): permlane16_swap exchanges the odd rows of 16 lanes of one operand with the
// even ones of the other, as permlane32_swap does with halves (exchange_max)
__device__ __forceinline__ float quad_max(float v) {
    const int i = __builtin_bit_cast(int, v);
    const auto r = __builtin_amdgcn_permlane16_swap(i, i, false, false);
    const int r0 = r[0], r1 = r[1];
    return exchange_max(fmaxf(__builtin_bit_cast(float, r0), __builtin_bit_cast(float, r1)));
}
__device__ __forceinline__ float quad_sum(float v) {
    const int i = __builtin_bit_cast(int, v);
    const auto r = __builtin_amdgcn_permlane16_swap(i, i, false, false);
    const int r0 = r[0], r1 = r[1];
    return exchange_sum(__builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1));
}

// position of 16-byte chunk `c` of row `row` (XOR within groups of 16 chunks)
__device__ __forceinline__ int wide_swz(int row) { return 2 * ((row ^ ((row >> 1) & 4)) & 7) + ((row >> 3) & 1); }

constexpr int D = 512;     // a row of K or V is one DMA instruction

template <typename T>
__global__ void __launch_bounds__(kWideThreads, 1) sdpa_wide_long_kernel(const SdpaDev p, int n_q_tiles, int n_split, int n_blocks) {
    using G = HeadGeo<D>;
    using W = WideGeo<D>;
    using V8 = typename Mma<T>::v8;
    constexpr int KC = D / 32, VB = D / 16;     // 32-element chunks of K Q^T, 16-row blocks of O^T
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    // pieces of the key axis outermost: the work groups of one XCD walk the same keys
    const int logical = logical_block(n_blocks);
    if (logical < 0) return;
    const int tiles = n_blocks / n_split;
    const int piece = logical / tiles, tile = logical - piece * tiles;
    const int bh = tile / n_q_tiles, qt = tile - bh * n_q_tiles;
    const int h = bh % p.H, b = bh / p.H;
    const int hk = h / p.kv_group;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, lq = lane & 15, g = lane >> 4;
    const int q0 = qt * kWideRows;
    const int wrow = wave * 32;     // the lane's own rows: wrow + 16 r + lq
    const T* const q_base = static_cast<const T*>(p.q) + b * p.q_bs + h * D;
    T* const o_base = static_cast<T*>(p.o) + b * p.o_bs + h * D;
    const float* const key_mask = p.key_mask ? p.key_mask + b * p.key_mask_bs : nullptr;

    int lo, hi;    // visible interval of row wrow + lane % 32
    // (rows past the end count as the last row where they share a wavefront with it: as rows without keys they would put every
    //  step of that wavefront on the masked path)
    row_interval(p, b, min(q0 + wrow + (lane & 31), p.Lq - 1), q0 + wrow < p.Lq, lo, hi);
    if (n_split > 1) {   // this work group's piece of the key axis, in whole steps
        const int steps = (p.Lk + kWideKeys - 1) / kWideKeys;
        lo = max(lo, static_cast<int>(static_cast<long>(piece) * steps / n_split) * kWideKeys);
        hi = min(hi, static_cast<int>(static_cast<long>(piece + 1) * steps / n_split) * kWideKeys);
        if (hi <= lo) { lo = 0; hi = 0; }
    }
    const WaveExtent we = wave_extent(lo, hi);
    const int row_lo[2] = {__shfl(lo, lq), __shfl(lo, 16 + lq)}, row_hi[2] = {__shfl(hi, lq), __shfl(hi, 16 + lq)};
    const bool dead_row[2] = {row_hi[0] <= row_lo[0], row_hi[1] <= row_lo[1]};

    // ── Q rows through LDS (RoPE, if any, applied on the way), 32 rows at a time; every lane picks its row's fragments ──
    V8 qf[KC][2];
#pragma unroll 1
    for (int r = 0; r < 4; ++r) stage_q_tile<T, D, kWideThreads, 32>(smem + r * 32 * G::O_STRIDE, p, q_base, q0 + 32 * r, tid);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < KC; ++c)
#pragma unroll
        for (int r = 0; r < 2; ++r)
            qf[c][r] = __builtin_bit_cast(V8, *reinterpret_cast<const u32x4*>(smem + (wrow + 16 * r + lq) * G::O_STRIDE + (32 * c + 8 * g) * 2));
    __syncthreads();
    // the extents of the four wavefronts
    if (lane == 0) { reinterpret_cast<int*>(smem)[wave] = we.lo_min; reinterpret_cast<int*>(smem)[4 + wave] = we.hi_max; }
    __syncthreads();
    int g_lo = 0x7fffffff, g_hi = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) { g_lo = min(g_lo, reinterpret_cast<int*>(smem)[w]); g_hi = max(g_hi, reinterpret_cast<int*>(smem)[4 + w]); }
    g_lo = __builtin_amdgcn_readfirstlane(g_lo);
    g_hi = __builtin_amdgcn_readfirstlane(g_hi);
    __syncthreads();
    const int k_first = g_lo == 0x7fffffff ? 0 : g_lo / kWideKeys * kWideKeys;
    const int n_steps = g_lo == 0x7fffffff ? 0 : (g_hi - k_first + kWideKeys - 1) / kWideKeys;

    o_clear<8 * VB>();
    float l_sum[2] = {0.f, 0.f}, neg_ref[2] = {0.f, 0.f};     // as RelSoftmaxState
    bool started[2] = {false, false};
    const float cl2 = p.scale_log2;

    // ── DMA duty: instructions wave, wave + 4, ... of a tile; instruction j fills LDS bytes [1024 j, 1024 j + 1024) ──
    const unsigned k_rsb = static_cast<unsigned>(p.k_rs) * 2u, v_rsb = static_cast<unsigned>(p.v_rs) * 2u;
    const unsigned char* kptr = reinterpret_cast<const unsigned char*>(static_cast<const T*>(p.k) + b * p.k_bs + hk * D) + static_cast<unsigned long>(k_first) * k_rsb;
    const unsigned char* vptr = reinterpret_cast<const unsigned char*>(static_cast<const T*>(p.v) + b * p.v_bs + hk * D) + static_cast<unsigned long>(k_first) * v_rsb;
    int k_left = g_hi - k_first, v_left = k_left;     // rows from the tile under the cursor on
    // the tile row of the wavefront's m-th instruction, and the byte offset of this lane's chunk in that row, which depends on m % 4 only
    auto drow = [&](int m) -> int { return wave + 4 * m; };
    unsigned dcol[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) dcol[m] = static_cast<unsigned>(lane ^ wide_swz(drow(m))) * 16u;
    const unsigned lds_base = static_cast<unsigned>(reinterpret_cast<size_t>((__attribute__((address_space(3))) unsigned char*)smem));
    // (inline assembly: for the compiler's builtin every later LDS read may alias the DMA's LDS write, so it would wait for the
    //  load to land before the next LDS read. The s_nop is the wait state an LDS-DMA instruction needs behind a write of m0.
    //  Rows past the last visible key repeat it: their scores are blanked.)
    auto dma = [&](const unsigned char* base, unsigned rsb, int left, int m, unsigned dst) {
        const unsigned voff = dcol[m % 4] + static_cast<unsigned>(min(drow(m), left - 1)) * rsb;
        asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(base), "{m0}"(lds_base + dst + (wave + 4 * m) * 1024) : "memory");
    };
    auto dma_tile = [&](bool is_k, unsigned dst) {
#pragma unroll
        for (int m = 0; m < W::NDMA; ++m) dma(is_k ? kptr : vptr, is_k ? k_rsb : v_rsb, is_k ? k_left : v_left, m, dst);
    };

    // ── LDS read addresses (stage, 32-row and 256-byte group offsets are immediates) ──
    // K fragment (kb, c): row 16 kb + lq, chunk 4 c + g; V fragment vb: rows 4 g + trow and 16 further on, 8 bytes at 16 vb + 4 j4
    unsigned kaddr[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) kaddr[c] = lq * W::ROWB + (((4 * c + g) ^ wide_swz(lq)) << 4);
    const int trow = lq >> 2, j4 = lq & 3;
    unsigned vaddr[8];
#pragma unroll
    for (int v = 0; v < 8; ++v) {
        const int row = 4 * g + trow;
        vaddr[v] = W::VOFF + row * W::ROWB + (((2 * v + (j4 >> 1)) ^ wide_swz(row)) << 4) + 8 * (j4 & 1);
    }

    f32x4 x[2][2];      // scores of the tile whose softmax is due: blocks of 16 keys x 16 rows
    V8 pf[2];
    constexpr int NQK = 2 * KC;
    constexpr int kFetch = 7;    // LDS reads run one less than this many fragments ahead of their two MFMAs
    // fragment i of the score product: key block i % 2, chunk i / 2
    auto fetch_k = [&](int stage, int i) -> V8 {
        const int kb = i & 1, c = i >> 1;
        return __builtin_bit_cast(V8, *reinterpret_cast<const u32x4*>(smem + stage * W::TILE + kb * 16 * W::ROWB + (c >> 2) * 256 + kaddr[c & 3]));
    };
    auto fetch_v = [&](int stage, int vb, int half) -> s16x4 {
        const unsigned off = stage * W::TILE + (vb >> 3) * 256 + half * 16 * W::ROWB;
        return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(smem + off + vaddr[vb & 7]));
    };
    auto step_end = [&]() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };

    if (n_steps > 0) {
        // prologue: K_0, K_1 and V_0 in LDS, x = raw scores of tile 0
        dma_tile(true, 0);
        dma_tile(false, W::VOFF);
        if (n_steps > 1) {
            kptr += kWideKeys * k_rsb; k_left -= kWideKeys;
            dma_tile(true, W::TILE);
        }
        step_end();
#pragma unroll
        for (int i = 0; i < NQK; ++i) {
            const V8 a = fetch_k(0, i);
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                if (i < 2) WideMma<T>::first(x[i & 1][r], a, qf[i >> 1][r]);
                else WideMma<T>::score(x[i & 1][r], a, qf[i >> 1][r]);
            }
        }
        wide_settle(x);
#pragma unroll
        for (int e = 0; e < 16; ++e) x[(e >> 2) & 1][e >> 3][e & 3] *= cl2;
    }
    // K_0 has been read by everybody before its stage is overwritten
    __syncthreads();

    // Step t (PAR = t % 2): reads K_{t+1} (stage 1 - PAR) and V_t (stage PAR), loads K_{t+2} into stage PAR and V_{t+1} into
    // stage 1 - PAR (their former tiles were used up in step t - 1).
    auto step = [&](auto par_tag, int t) {
        constexpr int PAR = decltype(par_tag)::value;
        if (t + 2 < n_steps) { kptr += kWideKeys * k_rsb; k_left -= kWideKeys; }
        if (t + 1 < n_steps) { vptr += kWideKeys * v_rsb; v_left -= kWideKeys; }
        const int j0 = k_first + t * kWideKeys;
        if (j0 < we.lo_max || j0 + kWideKeys > we.hi_min || key_mask != nullptr) {   // wave-uniform
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int key = j0 + 16 * kb + 4 * g + i;
                    int hidden = 0;
                    // a key-mask value of +-0 hides the key: (bits of |m|) - 1 is negative exactly then
                    if (key_mask) hidden = static_cast<int>(__builtin_bit_cast(unsigned, key_mask[min(key, p.Lk - 1)]) & 0x7fffffffu) - 1;
#pragma unroll
                    for (int r = 0; r < 2; ++r) {
                        const float score = x[kb][r][i];
                        x[kb][r][i] = blank_outside(score, key - row_lo[r], row_hi[r] - 1 - row_lo[r], hidden);
                    }
                }
        }
        f32x4 s[2][2];
        float sum[2] = {0.f, 0.f};
        V8 ring[kFetch];
        s16x4 vlo[kFetch], vhi[kFetch];
        constexpr int NPV = VB, N = NQK + NPV;
        auto fetch = [&](auto i_tag) {
            constexpr int i = decltype(i_tag)::value;
            if constexpr (i < NQK) ring[i % kFetch] = fetch_k(1 - PAR, i);
            else if constexpr (i < N) vlo[i % kFetch] = fetch_v(PAR, i - NQK, 0);
        };
        auto fetch2 = [&](auto i_tag) {     // second half of a V fragment
            constexpr int i = decltype(i_tag)::value;
            if constexpr (i >= NQK && i < N) vhi[i % kFetch] = fetch_v(PAR, i - NQK, 1);
        };
        auto frag = [&](auto i_tag) -> V8 {
            constexpr int i = decltype(i_tag)::value;
            return __builtin_bit_cast(V8, s16x8(__builtin_shufflevector(vlo[i % kFetch], vhi[i % kFetch], 0, 1, 2, 3, 4, 5, 6, 7)));
        };
        // element e of the tile: row e / 8, its keys in the order of the PV contraction (key block e / 4 % 2)
        auto exponentials = [&](int e0, int e1) {
#pragma unroll
            for (int e = e0; e < e1; ++e) {
                const float pr = __builtin_amdgcn_exp2f(x[(e >> 2) & 1][e >> 3][e & 3]);
                pf[e >> 3][e & 7] = static_cast<T>(pr);
                sum[e >> 3] += pr;
            }
        };
        [&]<int... I>(std::integer_sequence<int, I...>) { (fetch(std::integral_constant<int, I>{}), ...); }(std::make_integer_sequence<int, kFetch - 1>{});
        // ── S_{t+1} = K_{t+1} Q^T (after the last tile: of a stage that holds none, never read) over the exponentials of tile t;
        //    the last of these MFMAs goes out with the first of the PV product ──
        [&]<int... I>(std::integer_sequence<int, I...>) {
            ([&] {
                constexpr int i = I;
                constexpr int e0 = (16 * i + (NQK - 1) / 2) / (NQK - 1), e1 = (16 * (i + 1) + (NQK - 1) / 2) / (NQK - 1);
                if constexpr (i < 2) WideMma<T>::first(s[i & 1][0], ring[i % kFetch], qf[i >> 1][0]);
                else WideMma<T>::score(s[i & 1][0], ring[i % kFetch], qf[i >> 1][0]);
                MI_SCHED_BARRIER
                fetch(std::integral_constant<int, i - 1 + kFetch>{});
                fetch2(std::integral_constant<int, i - 1 + kFetch>{});
                MI_SCHED_BARRIER
                if constexpr (i < 2) WideMma<T>::first(s[i & 1][1], ring[i % kFetch], qf[i >> 1][1]);
                else WideMma<T>::score(s[i & 1][1], ring[i % kFetch], qf[i >> 1][1]);
                MI_SCHED_BARRIER
                // (past the last tile the cursors stand still and that tile is loaded again, into a stage nobody reads)
                constexpr int m0 = 2 * W::NDMA * i / (NQK - 1), m1 = 2 * W::NDMA * (i + 1) / (NQK - 1);
#pragma unroll
                for (int n = m0; n < m1; ++n) {
                    const int m = n >> 1;
                    if (n & 1) dma(vptr, v_rsb, v_left, m, W::VOFF + (1 - PAR) * W::TILE);
                    else dma(kptr, k_rsb, k_left, m, PAR * W::TILE);
                }
                MI_SCHED_BARRIER
                exponentials(e0, e1);
                MI_SCHED_BARRIER
            }(), ...);
        }(std::make_integer_sequence<int, NQK - 1>{});
        const bool fine = (started[0] || dead_row[0]) && sum[0] < kRelSumMax && (started[1] || dead_row[1]) && sum[1] < kRelSumMax;   // false also for inf / nan sums
        if (__any(!fine)) {   // first visible tile of a row, or its terms grew: move the reference (see softmax_tile_rel)
            wide_settle(s);
            float alpha[2];
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                float mloc = x[0][r][0];
#pragma unroll
                for (int e = 1; e < 8; ++e) mloc = fmaxf(mloc, x[e >> 2][r][e & 3]);
                mloc = quad_max(mloc);
                const bool visible = mloc > kNegInf;
                const float shift = !visible ? 0.f : (started[r] ? fmaxf(mloc, 0.f) : mloc);
                alpha[r] = started[r] ? __builtin_amdgcn_exp2f(-shift) : 1.f;
                started[r] = started[r] || visible;
                l_sum[r] *= alpha[r];
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e >> 2][r][e & 3] -= shift;
                neg_ref[r] -= shift;
                sum[r] = 0.f;
            }
            o_scale<8 * VB>(alpha);
            exponentials(0, 16);
        }
        l_sum[0] += sum[0];
        l_sum[1] += sum[1];
        MI_SCHED_BARRIER
        // ── O^T += V_t^T P_t ──
        fetch(std::integral_constant<int, NQK - 2 + kFetch>{});
        fetch2(std::integral_constant<int, NQK - 2 + kFetch>{});
        WideMma<T>::tail(s[1][0], s[1][1], ring[(NQK - 1) % kFetch], qf[KC - 1][0], qf[KC - 1][1], frag(std::integral_constant<int, NQK>{}), frag(std::integral_constant<int, NQK + 1>{}), pf[0], pf[1]);
        fetch(std::integral_constant<int, NQK - 1 + kFetch>{});
        fetch2(std::integral_constant<int, NQK - 1 + kFetch>{});
        fetch(std::integral_constant<int, NQK + kFetch>{});
        fetch2(std::integral_constant<int, NQK + kFetch>{});
        MI_SCHED_BARRIER
        [&]<int... I>(std::integer_sequence<int, I...>) {
            ([&] {
                constexpr int i = NQK + 2 + I, vb = I + 2;
                const V8 a = frag(std::integral_constant<int, i>{});
                WideMma<T>::template out<2 * vb>(a, pf[0]);
                MI_SCHED_BARRIER
                fetch(std::integral_constant<int, i - 1 + kFetch>{});
                MI_SCHED_BARRIER
                WideMma<T>::template out<2 * vb + 1>(a, pf[1]);
                MI_SCHED_BARRIER
                fetch2(std::integral_constant<int, i - 1 + kFetch>{});
                // the next tile's scores (complete since the first slots) into exponents, in front of their mask
                if constexpr (I >= 4) {
                    constexpr int e0 = 16 * (I - 4) / (NPV - 6), e1 = 16 * (I - 3) / (NPV - 6);
#pragma unroll
                    for (int e = e0; e < e1; ++e) s[(e >> 2) & 1][e >> 3][e & 3] = __builtin_fmaf(s[(e >> 2) & 1][e >> 3][e & 3], cl2, neg_ref[e >> 3]);
                }
                MI_SCHED_BARRIER
            }(), ...);
        }(std::make_integer_sequence<int, NPV - 2>{});
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e >> 1][e & 1] = s[e >> 1][e & 1];
        step_end();
    };
    for (int t = 0; t < n_steps; t += 2) {
        step(std::integral_constant<int, 0>{}, t);
        if (t + 1 >= n_steps) break;
        step(std::integral_constant<int, 1>{}, t + 1);
    }

    wide_settle(x);
    const float l_tot[2] = {quad_sum(l_sum[0]), quad_sum(l_sum[1])};
    // accumulation registers 8 vb + 4 r .. + 3: head-dim elements 16 vb + 4 g .. + 3 of row wrow + 16 r + lq
    if (n_split == 1) {
        const float inv[2] = {row_inverse(l_tot[0]), row_inverse(l_tot[1])};
        [&]<int... B>(std::integer_sequence<int, B...>) {
            ([&] {
                typedef T t4 __attribute__((ext_vector_type(4)));
                constexpr int r = B & 1;
                const float o0 = o_get<4 * B>(), o1 = o_get<4 * B + 1>(), o2 = o_get<4 * B + 2>(), o3 = o_get<4 * B + 3>();
                const t4 ov = {static_cast<T>(o0 * inv[r]), static_cast<T>(o1 * inv[r]), static_cast<T>(o2 * inv[r]), static_cast<T>(o3 * inv[r])};
                *reinterpret_cast<t4*>(smem + (wrow + 16 * r + lq) * G::O_STRIDE + (16 * (B >> 1) + 4 * g) * 2) = ov;
            }(), ...);
        }(std::make_integer_sequence<int, 2 * VB>{});
        __syncthreads();
        write_output<T, D, kWideThreads>(smem, o_base, p.o_rs, q0, p.Lq, kWideRows, tid);
    } else {
        unsigned char* const slot = p.split_scratch + (static_cast<long>(tile) * n_split + piece) * W::SLOT;
        f32x4* const part = reinterpret_cast<f32x4*>(slot) + wave * (D / 8) * 64 + (g >> 1) * 64 + (g & 1) * 32 + lq;
        [&]<int... B>(std::integer_sequence<int, B...>) {
            ([&] {
                const float o0 = o_get<4 * B>(), o1 = o_get<4 * B + 1>(), o2 = o_get<4 * B + 2>(), o3 = o_get<4 * B + 3>();
                part[(B >> 1) * 128 + (B & 1) * 16] = f32x4{o0, o1, o2, o3};
            }(), ...);
        }(std::make_integer_sequence<int, 2 * VB>{});
        if (g == 0) {   // the weight of the part in the merge is 2^ref
            float* const stat = reinterpret_cast<float*>(slot + static_cast<long>(kWideRows) * D * 4);
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                stat[wrow + 16 * r + lq] = -neg_ref[r];
                stat[kWideRows + wrow + 16 * r + lq] = l_tot[r];
            }
        }
    }
}

template <typename T>
int launch(const SdpaDev& p, int n_q_tiles, int n_split, int n_blocks, hipStream_t stream) {
    using W = WideGeo<D>;
    static thread_local bool raised = false;
    if (!raised) {
        MI_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&sdpa_wide_long_kernel<T>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                         W::LDS_BYTES));
        raised = true;
    }
    hipLaunchKernelGGL((sdpa_wide_long_kernel<T>), dim3(static_cast<unsigned>((n_blocks + 7) / 8 * 8)), dim3(kWideThreads), W::LDS_BYTES,
                       stream, p, n_q_tiles, n_split, n_blocks);
    return 0;
}

}  // namespace

int launch_sdpa_wide_long(const SdpaDev& p, bool bf16, int n_q_tiles, int n_split, int n_blocks, hipStream_t stream) {
    return bf16 ? launch<__bf16>(p, n_q_tiles, n_split, n_blocks, stream) : launch<_Float16>(p, n_q_tiles, n_split, n_blocks, stream);
}

}  // namespace mi
