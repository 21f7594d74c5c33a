// Which tile a projection takes: the forms of linear_pipe.hip (and the 256 x 256 tiles of linear_dma.hip) with what a launch on each is
// expected to cost. Host code without HIP in it, so that a test can ask which form a problem gets.
#pragma once
#include <algorithm>

#include "internal.h"

namespace mi {
namespace gemm {

// ── which form a launch takes ──
// A launch of n tiles on a GPU of C compute units costs about
//     phi + steps lam + (m - 1) (steps tau + eps),   m = ceil(n / C) tiles on the busiest compute unit,
// with steps = K / 64: phi what a launch of one tile per compute unit costs beyond its steps (start, first loads, write-out), lam
// a step when the compute unit has one tile, tau and eps a step and the rest of every further tile. The constants (us) are fitted
// on MI355X to 350 problems (32 to 16384 rows, eleven layers of the supported models, one or three of a launch; 16-bit: jointly with a
// term for the bytes of the operands, the same for every form), with all products v_mfma_f32_32x32x16. As built now steps of the large
// tiles are 6 to 12 % shorter and the others much as they were, and the constants still rank the forms: every form timed on 452 such
// problems (profiles/linear_form_times.txt), the form taken is 0.7 (INT8 0.5 to 0.8, GEGLU 1.2 to 1.7, GEGLU of INT8 0.6 to 0.7) % slower
// than the fastest one on average, where the same form timed twice differs by 0.8 %; at worst 16 % (GEGLU 6144 x 640 -> 2 x 2560 56.5 us on
// 192 x 128 tiles, 48.5 on 128 x 64). Large tiles
// need fewer bytes per FLOP: a compute unit takes 1 KB from its L2 in 16 to 24 clocks, so a step of 128 x 128 (32 KB) took 600 to 700 where its products take 512, one of 128 x 64 (24 KB) 450 to 650 where they take
// 256 (with products of 32 x 32 x 16). Small ones fill the GPU: 128 x 1280 x 1280 takes 4.8 us with 160 tiles of 32 x 32, 5.1 with 80 of 64 x 32, 7.0 with 20 of
// 128 x 64; 1024 x 2240 x 2240 takes 15.6 us with 192 tiles of 128 x 96, 23 with 280 of 128 x 64, 46 with 36 of 256 x 256.
// The tiles 96 features wide and the GEGLU tile of 192 x 128 (constants set by hand from 17 problems of their own) are for
// the counts between (us, best other form / theirs, profiles/linear_form_times.txt): 1024 x 2240 x 2240 16.8 / 15.6 on
// 192 tiles of 128 x 96, 2048 x 1152 x 1152 10.5 / 9.9, 2048 x 640 x 2560 15.0 / 13.2 on 224 of 64 x 96; GEGLU 2048 x 640 ->
// 2 x 2560 21.6 / 21.1 and 1024 x 1280 -> 2 x 5120 35.5 / 33.8 (INT8 22.9 / 21.3, 38.2 / 33.1) on 220 and 240 of 192 x 128; INT8
// 1024 x 1280 x 1280 8.7 (128 x 64) / 8.8, 4096 x 640 x 640 8.4 / 7.8. Wavefronts that own 128 x 64
// or 96 x 64 instead of 64 x 64 (a quarter fewer LDS reads) gave nothing with products of 32 x 32 x 16: 1024 x 6720 x 2240 32.8 -> 32.9.
// Loading wavefronts (see the top) pay where the products of a step are short. They are no help where a compute unit holds two work
// groups of large register use (products of 32 x 32 x 16): GEGLU 3072 x 640 -> 2 x 2560 29 -> 37 us, three of 16384 x 512 x 512 37 -> 42.
struct Form {
    int bm, bn_out;
    float phi, lam, tau, eps;
};
enum { k32x32, k64x32, k64x64, k64x96, k128x64_load, k128x64, k128x96, k128x128, k128x128_2, k192x128, k256x128, k256x256, kPlainForms };
constexpr Form kPlain[kPlainForms] = {{32, 32, 2.46f, 0.091f, 0.058f, 0.22f},   {64, 32, 2.60f, 0.111f, 0.126f, 0.34f},   {64, 64, 2.52f, 0.154f, 0.190f, 0.42f},
                                      {64, 96, 3.10f, 0.225f, 0.240f, 1.50f},   {128, 64, 2.53f, 0.250f, 0.322f, 0.76f},  {128, 64, 2.57f, 0.274f, 0.322f, 0.59f},
                                      {128, 96, 3.50f, 0.318f, 0.360f, 2.30f},  {128, 128, 3.95f, 0.356f, 0.529f, 3.18f}, {128, 128, 3.19f, 0.515f, 0.465f, 1.20f},
                                      {192, 128, 4.67f, 0.511f, 0.727f, 4.11f}, {256, 128, 5.03f, 0.656f, 0.839f, 6.17f}, {256, 256, 8.05f, 1.379f, 1.789f, 6.40f}};
// INT8 weights: the widening makes small steps dearer and the large tiles no better (those above 128 x 128 are not built)
enum { k8_32x32, k8_64x64, k8_64x96, k8_128x64, k8_128x96, k8_128x128, k8_128x128_2, kPlainW8Forms };
constexpr Form kPlainW8[kPlainW8Forms] = {{32, 32, 2.47f, 0.155f, 0.049f, 0.33f},
                                          {64, 64, 2.75f, 0.209f, 0.187f, 0.80f},
                                          {64, 96, 3.30f, 0.245f, 0.235f, 0.90f},
                                          {128, 64, 3.03f, 0.325f, 0.286f, 1.43f},
                                          {128, 96, 4.00f, 0.350f, 0.360f, 1.50f},
                                          {128, 128, 4.03f, 0.420f, 0.562f, 3.98f},
                                          {128, 128, 2.89f, 0.658f, 0.382f, 3.13f}};
enum { kG64x64, kG128x64_2, kG128x64, kG256x64, kG192x128, kGegluForms };   // output features; the W tile holds twice as many rows
constexpr Form kGeglu[kGegluForms] = {{64, 64, 2.65f, 0.377f, 0.330f, 1.20f}, {128, 64, 3.66f, 0.648f, 0.496f, 2.09f}, {128, 64, 4.41f, 0.442f, 0.588f, 4.08f},
                                      {256, 64, 5.99f, 0.800f, 0.834f, 8.98f}, {192, 128, 7.00f, 1.200f, 1.250f, 7.00f}};
enum { kG8_64x64, kG8_128x64_2, kG8_256x64, kG8_192x128, kGegluW8Forms };
constexpr Form kGegluW8[kGegluW8Forms] = {{64, 64, 3.92f, 0.315f, 0.302f, 1.17f}, {128, 64, 3.92f, 0.653f, 0.429f, 2.93f}, {256, 64, 7.90f, 0.816f, 1.031f, 6.53f},
                                          {192, 128, 9.30f, 1.290f, 1.500f, 5.50f}};

// 256 x 256 tiles take contractions from 512 on (below, their prologue is most of the launch).
inline int pick_form(const Form* forms, int n_forms, const LinearBatch& batch, int n_problems, int n_cu) {
    int best = 0;
    double best_cost = 1e30;
    for (int f = 0; f < n_forms; ++f) {
        long tiles = 0;
        int k = 0;
        for (int i = 0; i < n_problems; ++i) {
            const LinearProblem& p = batch.p[i];
            tiles += static_cast<long>((p.M + forms[f].bm - 1) / forms[f].bm) * ((p.N + forms[f].bn_out - 1) / forms[f].bn_out);
            k = std::max(k, p.K);
        }
        if (forms[f].bn_out == 256 && k < 512) continue;
        const double steps = k / 64, m = static_cast<double>((tiles + n_cu - 1) / n_cu);
        const double cost = forms[f].phi + steps * forms[f].lam + (m - 1) * (steps * forms[f].tau + forms[f].eps);
        if (cost < best_cost) { best_cost = cost; best = f; }
    }
    return best;
}

// The form of a launch: an index into the table of its kind.
inline int pick_form(const LinearBatch& batch, int n_problems, bool geglu, int n_cu) {
    if (batch.p[0].w_scale != nullptr)
        return geglu ? pick_form(kGegluW8, kGegluW8Forms, batch, n_problems, n_cu) : pick_form(kPlainW8, kPlainW8Forms, batch, n_problems, n_cu);
    return geglu ? pick_form(kGeglu, kGegluForms, batch, n_problems, n_cu) : pick_form(kPlain, kPlainForms, batch, n_problems, n_cu);
}

}  // namespace gemm
}  // namespace mi
