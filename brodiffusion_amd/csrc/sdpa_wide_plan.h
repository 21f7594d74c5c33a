// How attention of the wide heads is laid out on the GPU: the pieces of the key axis and, at head_dim 512, which of the two kernels
// (sdpa_wide.hip, sdpa_wide_long.hip) takes a launch. Host code, so that a test can ask.
#pragma once
#include "internal.h"

namespace mi {
namespace sdpa {

constexpr int kWideRows = 128;    // query rows per work group, 32 per wavefront
constexpr int kWideKeys = 32;     // key rows per step

inline long wide_tiles(const SdpaDev& p) { return static_cast<long>(p.B) * p.H * ((p.Lq + kWideRows - 1) / kWideRows); }

// Pieces of the key axis: as many as minimise the launch, counted in steps: rounds x (steps of a piece + kOverhead: Q staging,
// first tiles, write-out), and for the merge kMerge plus kParts per part on every compute unit (128 x D FP32 values written and
// read again), the same once more for what the parts of the launch exceed kNear by (the L2s no longer hold them). Fitted on
// MI355X to up to 16 pieces of 45 problems (1 to 24 batch items, 300 to 16384 rows, 320 to 16384 keys) at each head dimension:
// the number taken is 1.2 % slower than the best one on average, 10 % at worst (counting no parts: 3.1 and 21 %). The kernel of
// sdpa_wide_long.hip, 22 problems of 3 to 192 tiles: 0.6 % on average, 6 % at worst. At 512 with the kernel of sdpa_wide.hip, us:
//   1024 tokens (8 tiles)      1 piece 54.6   3 34.6   5 32.4           6 33.2 (taken)   8 35.4
//   4096 (32)                  1 168          4 67.0   6 63.6 (taken)   8 67.1   9 (a second round) 91.8
//   9216 (72)                  1 358          2 208    3 185 (taken)    7 210
//   16384 (128)                1 638          2 493 (taken)             4 515
//   8 x 600 (40)               1 45.7         3 38.0   4 37.2           5 40.1       3 taken
// Only unmasked calls (a valid length or key mask may be on): with causal masks the tiles are unequal and fill the GPU in their
// own way.
inline int wide_split(const SdpaDev& p, int head_dim, int n_cu) {
    if (p.mask_mode != MI_MASK_NONE) return 1;
    const long tiles = wide_tiles(p);
    const int steps = (p.Lk + kWideKeys - 1) / kWideKeys;
    constexpr int kMaxSplit = 16, kMinSteps = 5;
    constexpr double kOverhead = 6, kMerge = 1, kParts = 16, kNear = 47e6;
    int best = 1;
    double best_cost = 0;
    for (int s = 1; s <= kMaxSplit && (s == 1 || steps / s >= kMinSteps); ++s) {
        const double parts = static_cast<double>(tiles) * s, far = parts * kWideRows * head_dim * 4 - kNear;
        const double rounds = static_cast<double>((tiles * s + n_cu - 1) / n_cu);
        double cost = rounds * ((steps + s - 1) / s + kOverhead);
        if (s > 1) cost += kMerge + kParts * (parts / n_cu + (far > 0 ? far / (n_cu * kWideRows * 512.0 * 4) : 0));
        if (s == 1 || cost < best_cost) { best = s; best_cost = cost; }
    }
    return best;
}

// Whether a launch of head_dim 512 goes to sdpa_wide_long.hip. Its products pay by a higher clock at the power limit, so only
// while the GPU is full; on a GPU that is not, the clock is the same and their cycles are more. Work groups of one round, this
// kernel's time as a share of the other's (fp16 and bf16, 19 to 512 key steps a work group): 32 to 160 of 256 compute units 1.04 to
// 1.09, 192 0.95 to 1.04 by GPU, 204 to 224 0.94 to 0.98 (one 1.03), 240 and 256 0.92 to 0.97. So a round counts as full from
// 3 of 4 compute units on, and there must be more full rounds than rounds that are not (1 full round and 32 to 128 groups:
// 0.99 to 1.01). us, that kernel / this one: 16384 tokens 490 / 454, without a scratch for parts 662 / 706; 16 x 1024 58 / 62;
// 9216 186 / 180. From 16 key steps per compute unit on (8 x 1024, 8 of them, 48.2 / 47.9 fp16, 47.7 / 48.1 bf16) and 4 per work group (1 and 2: 1.00
// to 1.01, 3: 0.99, 4: 0.97 to 0.98: a fixed part of 2000 clocks more). With a causal mask the tiles are unequal and the launch ends with a few
// long ones on an otherwise empty GPU: below 2 tiles per compute unit 1.00 to 1.08 (one head of 4096 to 9216 tokens 1.07 to 1.08),
// from there on 0.97 to 0.99. Valid lengths are not known here. At head_dim 256 and 384 there are fewer products per exponential,
// and that form is the slower one at nearly every length (256: 4096 tokens 41.3 / 42.4, 9216 105 / 110; 384 bf16: 9216 141 / 146).
inline bool wide_long_pays(const SdpaDev& p, int n_split, int n_cu) {
    const long tiles = wide_tiles(p), groups = tiles * n_split;
    const int steps = (p.Lk + kWideKeys - 1) / kWideKeys;
    if (tiles * steps < 16L * n_cu || steps < 4L * n_split) return false;
    if (p.mask_mode != MI_MASK_NONE) return tiles >= 2L * n_cu;
    const long rest = groups % n_cu;
    const bool rest_full = 4 * rest >= 3L * n_cu;
    return groups / n_cu + (rest_full ? 1 : 0) > (rest != 0 && !rest_full ? 1 : 0);
}

}  // namespace sdpa
}  // namespace mi
