// Softmax attention for head dimensions 256, 384 and 512 on gfx950: the single wide head of a VAE mid-block
// (src/vae.cpp:259-277: one head over all 512 channels of a 64 x 64 latent; src/vae_qwenimage.cpp:322-340: 384 channels),
// through the same entry point as every other head dimension.
//
// Bound: MFMA (4 L^2 d FLOPs against 8 L d bytes). A work group is 4 wavefronts, one per SIMD, each with 32 query rows of its
// own and all of the head dimension: at 512 the output accumulator of 32 rows is 256 registers per lane, the Q fragments
// are 128, and one wavefront per SIMD may use 512 (that instance is still nine registers short: 40 bytes per lane of scratch, of
// which a step reloads 4). So no partial score ever leaves a wavefront (the earlier form dealt the
// head dimension out to the wavefronts and summed four FP32 score tiles through LDS at every step: 240 TFLOP/s at 16384
// tokens, 2.37 ms). The key axis goes in steps of 32: with rows of up to 1 KB two stages of K and two of V are 128 KB of LDS.
//
// With one wavefront per SIMD nothing but the wavefront itself can cover its softmax, so the step is one instruction
// stream in which the two overlap: the MFMAs of S_{t+1} = K_{t+1} Q^T carry the exponentials of tile t between them
// (elementwise: the softmax is taken relative to a reference that is raised only when a tile grows past it, see
// softmax_tile_rel), then O^T += V_t^T P_t. The DMA of tiles K_{t+2} and V_{t+1} is dealt out under the first half, so it
// has the rest of the step to land; one barrier per step.
//   LDS: rows back to back as the DMA deposits them, 16-byte chunk c of row r at position c ^ f(r) within its group of 16
//   chunks, f(r) = 4 (r % 4) + (r / 4) % 4: the K fragment reads (16 rows, one chunk column) and the V transpose reads
//   (4 rows, one 64-byte window) are both free of bank conflicts.
//
// Long calls of head_dim 512 that fill the GPU take the form of sdpa_wide_long.hip; planning (sdpa_wide_plan.h), scratch and merge are
// the same.
//
// A query tile is 128 rows, so a VAE mid-block has 32 (64 x 64 latent) to 128 tiles for 256 compute units: the key axis is
// cut into as many pieces as shorten the launch (wide_split), each leaving its output accumulators and softmax statistics in
// the caller's scratch, all FP32, merged in a fixed order by wide_combine_kernel: the result is rounded once.
//
// Masks work as everywhere (per-row visible key interval, kv_valid_len, key mask); cached prefixes, logit bias, lse output,
// packed sequences and K rotated tile by tile are not offered at these widths (K rotated into a scratch and Q rotated on
// load are).
#include "sdpa_wide.h"

namespace mi {
namespace {

using namespace sdpa;

// The MFMAs of this kernel are inline assembly. At head_dim 512 the output accumulator of a wavefront is exactly the 256
// accumulation registers; left to the compiler, which also puts every other MFMA result there, the scores spill (640 to
// 1840 bytes of scratch per lane). Here O lives in a[0 : 16 VB) by name (block vb in a[16 vb : 16 vb + 16)), every statement
// that touches it declares all of a0..a255 clobbered, so that the compiler keeps nothing of its own there, and the scores are
// in ordinary registers. The compiler does not see the wait that VALU code needs before it touches the result of an
// MFMA of 8 passes (12 wait states); it is kept by construction: the last MFMA of a score tile and the two that follow it
// are one statement (wide_tail), so the scores are complete before anything can read them, and wide_settle stands in front
// of the code that works on O.
template <typename T> struct WideMma;
#define MI_WIDE_MMA(TYPE, NAME)                                                                                               \
    template <> struct WideMma<TYPE> {                                                                                        \
        using V8 = typename Mma<TYPE>::v8;                                                                                    \
        static __device__ __forceinline__ void first(f32x16& s, V8 a, V8 b) {                                                 \
            asm volatile(NAME " %0, %1, %2, 0" : "=&v"(s) : "v"(a), "v"(b));                                                  \
        }                                                                                                                     \
        static __device__ __forceinline__ void score(f32x16& s, V8 a, V8 b) {                                                 \
            asm volatile(NAME " %0, %1, %2, %0" : "+v"(s) : "v"(a), "v"(b));                                                  \
        }                                                                                                                     \
        /* O block VB += a b */                                                                                               \
        template <int VB> static __device__ __forceinline__ void out(V8 a, V8 b) {                                            \
            asm volatile(NAME " a[%2:%3], %0, %1, a[%2:%3]" : : "v"(a), "v"(b), "n"(16 * VB), "n"(16 * VB + 15) : MI_AGPRS);  \
        }                                                                                                                     \
        /* the last MFMA of a score tile together with the first two of the PV product (O blocks 0 and 1) */                  \
        static __device__ __forceinline__ void tail(f32x16& s, V8 ak, V8 q, V8 a0, V8 a1, V8 p) {                             \
            asm volatile(NAME " %0, %1, %2, %0\n\t" NAME " a[0:15], %3, %5, a[0:15]\n\t" NAME " a[16:31], %4, %5, a[16:31]"   \
                         : "+v"(s) : "v"(ak), "v"(q), "v"(a0), "v"(a1), "v"(p) : MI_AGPRS);                                   \
        }                                                                                                                     \
    };
MI_WIDE_MMA(__bf16, "v_mfma_f32_32x32x16_bf16")
MI_WIDE_MMA(_Float16, "v_mfma_f32_32x32x16_f16")
#undef MI_WIDE_MMA
// every MFMA in flight has written its result when this returns
__device__ __forceinline__ void wide_settle(f32x16& s) { asm volatile("s_nop 15\n\ts_nop 15" : "+v"(s) : : MI_AGPRS); }
// O *= f (the reads of a block go out before its writes: a value just read is not touched in the next instruction)
template <int B> __device__ __forceinline__ void o_scale_block(float f) {
    [&]<int... I>(std::integer_sequence<int, I...>) {
        const float v[16] = {o_get<16 * B + I>()...};
        (o_set<16 * B + I>(v[I] * f), ...);
    }(std::make_integer_sequence<int, 16>{});
}
template <int N> __device__ __forceinline__ void o_scale(float f) {
    [&]<int... B>(std::integer_sequence<int, B...>) { (o_scale_block<B>(f), ...); }(std::make_integer_sequence<int, N / 16>{});
    asm volatile("s_nop 7" : : : MI_AGPRS);   // accumulation registers written by the VALU and read by the next MFMA
}

// position of 16-byte chunk `c` of row `row` (XOR within groups of 16 chunks)
__device__ __forceinline__ int wide_swz(int row) { return 4 * (row & 3) + ((row >> 2) & 3); }

template <typename T, int D>
__global__ void __launch_bounds__(kWideThreads, 1) sdpa_wide_kernel(const SdpaDev p, int n_q_tiles, int n_split, int n_blocks) {
    using G = HeadGeo<D>;
    using W = WideGeo<D>;
    using V8 = typename Mma<T>::v8;
    constexpr int KC = D / 16, VB = D / 32;     // 16-element chunks of K Q^T, 32-row blocks of O^T
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
    const int lane = tid & 63, lq = lane & 31, lh = lane >> 5;
    const int q0 = qt * kWideRows;
    const int qrow = q0 + wave * 32 + lq;
    const T* const q_base = static_cast<const T*>(p.q) + b * p.q_bs + h * D;
    T* const o_base = static_cast<T*>(p.o) + b * p.o_bs + h * D;
    const float* const key_mask = p.key_mask ? p.key_mask + b * p.key_mask_bs : nullptr;

    int lo, hi;
    // (rows past the end count as the last row where they share a wavefront with it: as rows without keys they would put every
    //  step of that wavefront on the masked path)
    row_interval(p, b, min(qrow, p.Lq - 1), q0 + wave * 32 < p.Lq, lo, hi);
    if (n_split > 1) {   // this work group's piece of the key axis, in whole steps
        const int steps = (p.Lk + kWideKeys - 1) / kWideKeys;
        lo = max(lo, static_cast<int>(static_cast<long>(piece) * steps / n_split) * kWideKeys);
        hi = min(hi, static_cast<int>(static_cast<long>(piece + 1) * steps / n_split) * kWideKeys);
        if (hi <= lo) { lo = 0; hi = 0; }
    }
    const bool dead_row = hi <= lo;
    const WaveExtent we = wave_extent(lo, hi);

    // ── Q rows through LDS (RoPE, if any, applied on the way), 32 rows at a time; every lane picks its row's fragments ──
    V8 qf[KC];
#pragma unroll 1
    for (int r = 0; r < 4; ++r) stage_q_tile<T, D, kWideThreads, 32>(smem + r * 32 * G::O_STRIDE, p, q_base, q0 + 32 * r, tid);
    __syncthreads();
    read_q_frags<T, D>(qf, smem, wave * 32 + lq, lh);
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

    o_clear<16 * VB>();
    float l_sum = 0.f, neg_ref = 0.f;     // as RelSoftmaxState
    bool started = false;
    const float cl2 = p.scale_log2;

    // ── DMA duty: instructions wave, wave + 4, ... of a tile; instruction j fills LDS bytes [1024 j, 1024 j + 1024) ──
    const unsigned k_rsb = static_cast<unsigned>(p.k_rs) * 2u, v_rsb = static_cast<unsigned>(p.v_rs) * 2u;
    const unsigned char* kptr = reinterpret_cast<const unsigned char*>(static_cast<const T*>(p.k) + b * p.k_bs + hk * D) + static_cast<unsigned long>(k_first) * k_rsb;
    const unsigned char* vptr = reinterpret_cast<const unsigned char*>(static_cast<const T*>(p.v) + b * p.v_bs + hk * D) + static_cast<unsigned long>(k_first) * v_rsb;
    int k_left = g_hi - k_first, v_left = k_left;     // rows from the tile under the cursor on
    // this lane's tile row in its m-th instruction, and the byte offset of its chunk in that row (at 512 a row is one instruction,
    // and the chunk depends on m % 4 only: a scalar row and four registers)
    auto drow = [&](int m) -> int { return D == 512 ? wave + 4 * m : (64 * (wave + 4 * m) + lane) / G::CPR; };
    constexpr int NCOL = D == 512 ? 4 : W::NDMA;
    unsigned dcol[NCOL];
#pragma unroll
    for (int m = 0; m < NCOL; ++m) dcol[m] = static_cast<unsigned>((64 * (wave + 4 * m) + lane - drow(m) * G::CPR) ^ wide_swz(drow(m))) * 16u;
    const unsigned lds_base = static_cast<unsigned>(reinterpret_cast<size_t>((__attribute__((address_space(3))) unsigned char*)smem));
    // (inline assembly: for the compiler's builtin every later LDS read may alias the DMA's LDS write, so it would wait for the
    //  load to land before the next LDS read. The s_nop is the wait state an LDS-DMA instruction needs behind a write of m0.
    //  Rows past the last visible key repeat it: their scores are blanked.)
    auto dma = [&](const unsigned char* base, unsigned rsb, int left, int m, unsigned dst) {
        const unsigned voff = dcol[m % NCOL] + static_cast<unsigned>(min(drow(m), left - 1)) * rsb;
        asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(base), "{m0}"(lds_base + dst + (wave + 4 * m) * 1024) : "memory");
    };
    auto dma_tile = [&](bool is_k, unsigned dst) {
#pragma unroll
        for (int m = 0; m < W::NDMA; ++m) dma(is_k ? kptr : vptr, is_k ? k_rsb : v_rsb, is_k ? k_left : v_left, m, dst);
    };

    // ── LDS read addresses (stage, 32-row and 256-byte group offsets are immediates) ──
    const int fk = wide_swz(lq);
    unsigned kaddr[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) kaddr[c] = lq * W::ROWB + (((2 * c + lh) ^ fk) << 4);
    const int trow = (lane & 15) >> 2, j4 = lane & 3, g1 = (lane >> 4) & 1;
    unsigned vaddr[4][2];
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            const int row = 4 * lh + 8 * hh + trow;
            vaddr[v][hh] = W::VOFF + row * W::ROWB + (((4 * v + 2 * g1 + (j4 >> 1)) ^ wide_swz(row)) << 4) + 8 * (j4 & 1);
        }

    f32x16 x;           // scores of the tile whose softmax is due
    V8 pf[2];
    constexpr int kFetch = 6;    // LDS reads run this many operands ahead of their MFMA
    auto fetch_k = [&](int stage, int c) -> V8 {
        return __builtin_bit_cast(V8, *reinterpret_cast<const u32x4*>(smem + stage * W::TILE + (c >> 3) * 256 + kaddr[c & 7]));
    };
    auto fetch_v = [&](int stage, int j) -> V8 {
        const int c2 = j / VB, vb = j % VB;
        const unsigned off = stage * W::TILE + c2 * 16 * W::ROWB + (vb >> 2) * 256;
        const s16x4 v_lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(smem + off + vaddr[vb & 3][0]));
        const s16x4 v_hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(smem + off + vaddr[vb & 3][1]));
        return __builtin_bit_cast(V8, __builtin_shufflevector(v_lo, v_hi, 0, 1, 2, 3, 4, 5, 6, 7));
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
        WideMma<T>::first(x, fetch_k(0, 0), qf[0]);
#pragma unroll
        for (int c = 1; c < KC; ++c) WideMma<T>::score(x, fetch_k(0, c), qf[c]);
        wide_settle(x);
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
            const int d0 = j0 + 4 * lh - lo, top = hi - 1 - lo;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int c = 8 * (e >> 2) + (e & 3);
                int hidden = 0;
                // a key-mask value of +-0 hides the key: (bits of |m|) - 1 is negative exactly then
                if (key_mask) hidden = static_cast<int>(__builtin_bit_cast(unsigned, key_mask[min(j0 + 4 * lh + c, p.Lk - 1)]) & 0x7fffffffu) - 1;
                const float score = x[e];
                x[e] = blank_outside(score, d0 + c, top, hidden);
            }
        }
        f32x16 s;
        float s0 = 0.f, s1 = 0.f;
        const float nr = neg_ref;
        V8 ring[kFetch];
        constexpr int NPV = 2 * VB, N = KC + NPV;
        auto fetch = [&](auto i_tag) {
            constexpr int i = decltype(i_tag)::value;
            if constexpr (i < KC) ring[i % kFetch] = fetch_k(1 - PAR, i);
            else if constexpr (i < N) ring[i % kFetch] = fetch_v(PAR, i - KC);
        };
        auto exponentials = [&](int e0, int e1) {
#pragma unroll
            for (int e = e0; e < e1; ++e) {
                const float pr = __builtin_amdgcn_exp2f(x[e]);
                pf[e >> 3][e & 7] = static_cast<T>(pr);
                if (e & 1) s1 += pr; else s0 += pr;
            }
        };
        [&]<int... I>(std::integer_sequence<int, I...>) { (fetch(std::integral_constant<int, I>{}), ...); }(std::make_integer_sequence<int, kFetch>{});
        // ── S_{t+1} = K_{t+1} Q^T (after the last tile: of a stage that holds none, never read) over the exponentials of tile t;
        //    the last of these MFMAs goes out with the first of the PV product ──
        [&]<int... I>(std::integer_sequence<int, I...>) {
            ([&] {
                constexpr int i = I;
                if constexpr (i == 0) WideMma<T>::first(s, ring[0], qf[0]);
                else WideMma<T>::score(s, ring[i % kFetch], qf[i]);
                fetch(std::integral_constant<int, i + kFetch>{});
                constexpr int e0 = 16 * i / (KC - 1), e1 = 16 * (i + 1) / (KC - 1);
#pragma unroll
                for (int e = e0; e < e1; ++e) x[e] = __builtin_fmaf(x[e], cl2, nr);
                exponentials(e0, e1);
                // (past the last tile the cursors stand still and that tile is loaded again, into a stage nobody reads)
                constexpr int m0 = W::NDMA * i / (KC - 1), m1 = W::NDMA * (i + 1) / (KC - 1);
#pragma unroll
                for (int m = m0; m < m1; ++m) {
                    dma(kptr, k_rsb, k_left, m, PAR * W::TILE);
                    dma(vptr, v_rsb, v_left, m, W::VOFF + (1 - PAR) * W::TILE);
                }
                MI_SCHED_BARRIER
            }(), ...);
        }(std::make_integer_sequence<int, KC - 1>{});
        const bool fine = (started || dead_row) && s0 + s1 < kRelSumMax;   // false also for inf / nan sums
        if (__any(!fine)) {   // first visible tile of a row, or its terms grew: move the reference (see softmax_tile_rel)
            wide_settle(s);
            float mloc = x[0];
#pragma unroll
            for (int e = 1; e < 16; ++e) mloc = fmaxf(mloc, x[e]);
            mloc = exchange_max(mloc);
            const bool visible = mloc > kNegInf;
            const float shift = !visible ? 0.f : (started ? fmaxf(mloc, 0.f) : mloc);
            const float alpha = started ? __builtin_amdgcn_exp2f(-shift) : 1.f;
            started = started || visible;
            l_sum *= alpha;
            o_scale<16 * VB>(alpha);
#pragma unroll
            for (int e = 0; e < 16; ++e) x[e] -= shift;
            neg_ref -= shift;
            s0 = s1 = 0.f;
            exponentials(0, 16);
        }
        l_sum += s0 + s1;
        MI_SCHED_BARRIER
        // ── O^T += V_t^T P_t ──
        WideMma<T>::tail(s, ring[(KC - 1) % kFetch], qf[KC - 1], ring[KC % kFetch], ring[(KC + 1) % kFetch], pf[0]);
        fetch(std::integral_constant<int, KC - 1 + kFetch>{});
        fetch(std::integral_constant<int, KC + kFetch>{});
        fetch(std::integral_constant<int, KC + 1 + kFetch>{});
        MI_SCHED_BARRIER
        [&]<int... I>(std::integer_sequence<int, I...>) {
            ([&] {
                constexpr int i = KC + 2 + I, c2 = (I + 2) / VB, vb = (I + 2) % VB;
                WideMma<T>::template out<vb>(ring[i % kFetch], pf[c2]);
                fetch(std::integral_constant<int, i + kFetch>{});
                MI_SCHED_BARRIER
            }(), ...);
        }(std::make_integer_sequence<int, NPV - 2>{});
        x = s;
        step_end();
    };
    for (int t = 0; t < n_steps; t += 2) {
        step(std::integral_constant<int, 0>{}, t);
        if (t + 1 >= n_steps) break;
        step(std::integral_constant<int, 1>{}, t + 1);
    }

    wide_settle(x);
    const float l_tot = exchange_sum(l_sum);
    // accumulation registers 4 B .. 4 B + 3: head-dim elements 8 B + 4 lh ..
    if (n_split == 1) {
        const float inv = row_inverse(l_tot);
        [&]<int... B>(std::integer_sequence<int, B...>) {
            ([&] {
                typedef T t4 __attribute__((ext_vector_type(4)));
                const float o0 = o_get<4 * B>(), o1 = o_get<4 * B + 1>(), o2 = o_get<4 * B + 2>(), o3 = o_get<4 * B + 3>();
                const t4 ov = {static_cast<T>(o0 * inv), static_cast<T>(o1 * inv), static_cast<T>(o2 * inv), static_cast<T>(o3 * inv)};
                *reinterpret_cast<t4*>(smem + (wave * 32 + lq) * G::O_STRIDE + (8 * B + 4 * lh) * 2) = ov;
            }(), ...);
        }(std::make_integer_sequence<int, 4 * VB>{});
        __syncthreads();
        write_output<T, D, kWideThreads>(smem, o_base, p.o_rs, q0, p.Lq, kWideRows, tid);
    } else {
        unsigned char* const slot = p.split_scratch + (static_cast<long>(tile) * n_split + piece) * W::SLOT;
        f32x4* const part = reinterpret_cast<f32x4*>(slot) + wave * (D / 8) * 64 + lane;
        [&]<int... B>(std::integer_sequence<int, B...>) {
            ([&] {
                const float o0 = o_get<4 * B>(), o1 = o_get<4 * B + 1>(), o2 = o_get<4 * B + 2>(), o3 = o_get<4 * B + 3>();
                part[B * 64] = f32x4{o0, o1, o2, o3};
            }(), ...);
        }(std::make_integer_sequence<int, 4 * VB>{});
        if (lh == 0) {   // the weight of the part in the merge is 2^ref
            float* const stat = reinterpret_cast<float*>(slot + static_cast<long>(kWideRows) * D * 4);
            stat[wave * 32 + lq] = -neg_ref;
            stat[kWideRows + wave * 32 + lq] = l_tot;
        }
    }
}

// out = sum_k w_k O_k / sum_k w_k l_k with w_k = 2^(ref_k - max ref) over the pieces of a query tile, in a fixed order.
// blockIdx.x = query tile; a thread takes 8 head-dim elements of a row, 8 consecutive threads the same elements of 8 rows, so that
// 128 bytes of a part are together on the way in and (in a wavefront) 128 bytes of a row on the way out.
template <typename T, int D>
__global__ void __launch_bounds__(256) wide_combine_kernel(const SdpaDev p, int n_q_tiles, int n_split) {
    using W = WideGeo<D>;
    typedef T t8 __attribute__((ext_vector_type(8)));
    constexpr int CPR = D / 8;
    const int tile = blockIdx.x;
    const int bh = tile / n_q_tiles, q0 = (tile - bh * n_q_tiles) * kWideRows;
    const int h = bh % p.H, b = bh / p.H;
    const int idx = static_cast<int>(blockIdx.y) * 256 + static_cast<int>(threadIdx.x);
    const int cc = (idx >> 3) % CPR, row = (idx >> 3) / CPR * 8 + (idx & 7);
    if (row >= kWideRows || q0 + row >= p.Lq) return;
    const unsigned char* const slots = p.split_scratch + static_cast<long>(tile) * n_split * W::SLOT;
    const long piece0 = ((row >> 5) * CPR + cc) * 64 + (row & 31);
    // (a part without visible keys has denominator 0 and is skipped; one whose denominator is NaN is not. The bits pass
    //  through an empty asm statement because -fno-honor-nans entitles the optimiser to a comparison that is false for NaN.)
    auto empty = [](float l) {
        unsigned bits = __builtin_bit_cast(unsigned, l);
        asm volatile("" : "+v"(bits));
        return (bits & 0x7fffffffu) == 0u;
    };
    float ref = kNegInf;
    for (int k = 0; k < n_split; ++k) {
        const float* stat = reinterpret_cast<const float*>(slots + k * W::SLOT + static_cast<long>(kWideRows) * D * 4);
        if (!empty(stat[kWideRows + row])) ref = fmaxf(ref, stat[row]);
    }
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    float lsum = 0.f;
    for (int k = 0; k < n_split; ++k) {
        const unsigned char* slot = slots + k * W::SLOT;
        const float* stat = reinterpret_cast<const float*>(slot + static_cast<long>(kWideRows) * D * 4);
        const f32x4 lo = reinterpret_cast<const f32x4*>(slot)[piece0], hi = reinterpret_cast<const f32x4*>(slot)[piece0 + 32];
        const float l = stat[kWideRows + row];
        if (empty(l)) continue;
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
    *reinterpret_cast<t8*>(static_cast<T*>(p.o) + b * p.o_bs + static_cast<long>(q0 + row) * p.o_rs + h * D + cc * 8) = out;
}

template <typename T, int D>
int launch_wide_d(const SdpaDev& p, hipStream_t stream) {
    using W = WideGeo<D>;
    const int n_q_tiles = (p.Lq + kWideRows - 1) / kWideRows;
    const long tiles = wide_tiles(p);
    int n_split = wide_split(p, D, device_cu_count());
    if (p.split_scratch == nullptr || p.split_scratch_bytes < static_cast<size_t>(tiles) * n_split * W::SLOT) n_split = 1;
    const long blocks = tiles * n_split;
    if (blocks > 0x7fffff00L) return fail("mi_sdpa_forward: problem too large for one launch");
    if (D == 512 && wide_long_pays(p, n_split, device_cu_count())) {
        if (launch_sdpa_wide_long(p, std::is_same_v<T, __bf16>, n_q_tiles, n_split, static_cast<int>(blocks), stream) != 0) return -1;
    } else {
        static thread_local bool raised = false;
        if (!raised) {
            MI_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&sdpa_wide_kernel<T, D>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                             W::LDS_BYTES));
            raised = true;
        }
        hipLaunchKernelGGL((sdpa_wide_kernel<T, D>), dim3(static_cast<unsigned>((blocks + 7) / 8 * 8)), dim3(kWideThreads), W::LDS_BYTES, stream, p,
                           n_q_tiles, n_split, static_cast<int>(blocks));
    }
    if (n_split > 1)
        hipLaunchKernelGGL((wide_combine_kernel<T, D>), dim3(static_cast<unsigned>(tiles), kWideRows * (D / 8) / 256), dim3(256), 0, stream, p,
                           n_q_tiles, n_split);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail("sdpa_wide launch: %s", hipGetErrorString(e));
    return 0;
}

}  // namespace

bool sdpa_wide_head(int head_dim) { return head_dim == 256 || head_dim == 384 || head_dim == 512; }

size_t sdpa_wide_split_scratch_bytes(const SdpaDev& p, int head_dim) {
    const int n_split = wide_split(p, head_dim, device_cu_count());
    if (n_split == 1) return 0;
    const size_t slot = static_cast<size_t>(kWideRows) * (static_cast<size_t>(head_dim) * 4 + 8);
    return static_cast<size_t>(wide_tiles(p)) * n_split * slot;
}

int launch_sdpa_wide(const SdpaDev& p, int dtype, int head_dim, hipStream_t stream) {
    const char* what = nullptr;
    if (p.Lp > 0) what = "a cached prefix";
    else if (p.cos_k) what = "K rotated tile by tile (lend rope_k_scratch)";
    else if (p.bias) what = "a logit bias";
    else if (p.lse) what = "lse_out";
    else if (p.cu_q) what = "packed variable-length sequences";
    if (what) return fail("mi_sdpa_forward: head_dim %d does not offer %s", head_dim, what);
    if (dtype != MI_DTYPE_BF16 && dtype != MI_DTYPE_F16) return fail("mi_sdpa_forward: dtype %d not supported (fp16 = 1, bf16 = 2)", dtype);
    const bool bf = dtype == MI_DTYPE_BF16;
    switch (head_dim) {
        case 256: return bf ? launch_wide_d<__bf16, 256>(p, stream) : launch_wide_d<_Float16, 256>(p, stream);
        case 384: return bf ? launch_wide_d<__bf16, 384>(p, stream) : launch_wide_d<_Float16, 384>(p, stream);
        case 512: return bf ? launch_wide_d<__bf16, 512>(p, stream) : launch_wide_d<_Float16, 512>(p, stream);
        default: return fail("mi_sdpa_forward: head_dim %d has no kernel", head_dim);
    }
}

}  // namespace mi
