// launch_rules.hpp — which launch a shape takes: plain host arithmetic on sizes, no HIP (the tests compile it with the
// host compiler).
//
// Prefill launches.  A launch's blocks run in rounds of one per compute unit, so its time is close to
//     fixed + rounds (round + step K / 128) + partial (f32 partials written and summed, in millions),
// also past one resident block per unit: they share its matrix cores.  The constants are least-squares fits to launches
// on MI355X (256 compute units) over copies of the weights in turn (none in an L2), captured in graphs: m = 17 .. 4096,
// n = 256 .. 151936, K = 128 .. 18944, 4485 unsplit calls and 2190 with room for partials, each in every shape: half of
// them lie within 5 %, nine in ten within 17 %.  Counting rounds is what decides: a tile half full of padding costs what
// a full one does.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace kr {

// The launch shapes of plain projections.  Narrow: q4_prefill.hip's 64 x 64 tiles (token rows x weight rows), or 128 x
// 128 with K split; the others: q4_prefill_wide.hip's 128 x 256, 64 x 256 and 64 x 128 tiles.
enum PrefillShape : int { kPrefillAuto = 0, kPrefillNarrow = 1, kPrefillWide42 = 42, kPrefillWide22 = 22, kPrefillWide21 = 21 };

struct PrefillChoice {
    int shape;
    uint32_t ksplit;
};

struct PrefillCost {
    int shape;
    uint32_t rows, cols;
    float fixed, round, step, partial;
};
constexpr PrefillCost kCostNarrow = {kPrefillNarrow, 64, 64, 3.6f, 2.2f, 0.41f, 0.0f};
constexpr PrefillCost kCostNarrowSplit = {kPrefillNarrow, 128, 128, 12.3f, 0.0f, 1.09f, 1.26f};
constexpr PrefillCost kCostWide[3] = {{kPrefillWide42, 128, 256, 4.3f, 4.0f, 1.62f, 0.0f},
                                      {kPrefillWide22, 64, 256, 4.3f, 1.5f, 1.1f, 0.0f},
                                      {kPrefillWide21, 64, 128, 4.1f, 0.7f, 0.64f, 0.0f}};
constexpr PrefillCost kCostWideSplit = {kPrefillWide42, 128, 256, 9.9f, 0.0f, 1.66f, 1.41f};
// A wide shape has to be this much faster by estimate: at 0.93 one of those calls comes out more than 3 % slower
// than on the narrow kernel (by 5 %).
constexpr float kWideMargin = 0.93f;

// 64-column groups per K split, even (two per step).
constexpr uint32_t groups_per_split(uint32_t k, uint32_t split) {
    return split > 1 ? ((k / 64 + split - 1) / split + 1) & ~1u : k / 64;
}

// Output tiles of rows x cols over np problems of ns[i] weight rows.
inline uint64_t prefill_tiles(uint32_t m, const uint32_t *ns, int np, uint32_t rows, uint32_t cols) {
    uint64_t t = 0;
    for (int i = 0; i < np; ++i) t += (uint64_t)((m + rows - 1) / rows) * ((ns[i] + cols - 1) / cols);
    return t;
}

// Estimated microseconds.
inline float prefill_us(const PrefillCost &c, uint32_t m, const uint32_t *ns, int np, uint32_t k, uint32_t split, uint32_t cus) {
    const uint64_t rounds = (prefill_tiles(m, ns, np, c.rows, c.cols) * split + cus - 1) / cus;
    float us = c.fixed + (float)rounds * (c.round + c.step * (float)groups_per_split(k, split) * 0.5f);
    if (split > 1) us += c.partial * (float)m * (float)ns[0] * (float)split * 1e-6f;
    return us;
}

// K splits of the narrow kernel: about one 128 x 128 block per compute unit, at least eight groups each.
inline uint32_t narrow_split(uint32_t m, uint32_t n, uint32_t k, uint32_t max_split, uint32_t cus) {
    const uint64_t tiles = prefill_tiles(m, &n, 1, kCostNarrowSplit.rows, kCostNarrowSplit.cols);
    uint32_t split = 1;
    while (split < max_split && tiles * split < cus && k / 64 / (split * 2) >= 8) split *= 2;
    return split;
}

// Plain projections (k % 128 == 0) of one x.  max_split > 1 (one problem): there is room for that many K splits'
// partials.  converted: x may come as the fp16 operand, which of the wide shapes only 128 x 256 reads.
inline PrefillChoice prefill_choice(uint32_t m, const uint32_t *ns, int np, uint32_t k, uint32_t max_split, bool converted,
                                    uint32_t cus) {
    const uint32_t ns_split = max_split > 1 ? narrow_split(m, ns[0], k, max_split, cus) : 1;
    PrefillChoice best = {kPrefillNarrow, ns_split};
    float us = kWideMargin * prefill_us(ns_split > 1 ? kCostNarrowSplit : kCostNarrow, m, ns, np, k, ns_split, cus);
    auto consider = [&](const PrefillCost &c, uint32_t split, float scale) {
        const float t = scale * prefill_us(c, m, ns, np, k, split, cus);
        if (t < us) {
            us = t;
            best = {c.shape, split};
        }
    };
    for (const PrefillCost &c : kCostWide) {
        float scale = 1.0f;
        if (converted && c.shape != kPrefillWide42) continue;
        // One round of 64 x 128 tiles has fewer loads in flight than two of 64 x 64, which shows on long rows, rows a
        // power of two apart and single token tiles: this / that, 15.7 / 17.4 us at K = 1536, 30.5 / 31.1 at 3584, but
        // 15.0 / 14.3 at K = 1024 (the norm and [2048 + 512 + 512], m = 377), 18.9 / 18.0 at 2048, 35.5 / 33.3 at 4096, 90
        // / 78 at 11008 and, m <= 64, 27.4 / 25.6 at 3072 (m = 2048, n = 1024, K = 4096: 36.5 / 41.4).  With room for
        // partials a split is as good: 23.9 / 20.7 at K = 2816.
        const bool one_round = prefill_tiles(m, ns, np, c.rows, c.cols) <= cus;
        if (c.shape == kPrefillWide21 && one_round &&
            ((k > 1536 && (max_split > 1 || m <= 64)) || (m < 2048 && (k % 1024 == 0 || k > 3584))))
            scale = 1.5f;
        consider(c, 1, scale);
    }
    for (uint32_t split = 2; split <= max_split && k / 64 / split >= 8; split *= 2) consider(kCostWideSplit, split, 1.0f);
    return best;
}

// ---- the few-token kernel's slab loop (q4_skinny.hip): K of several slabs, no room for partials
constexpr uint32_t kSlabColumns = 2048;      // K columns per slab
constexpr uint32_t kSlabLoopBlocks = 256;    // KR_OPT_SKINNY_MAX_BLOCKS' default

// Estimated microseconds over `tiles` weight tiles (16 rows; gate/up 8 pairs) in groups of 16 mg token rows, at most
// `blocks` blocks: per slab, the staging of X and the block's tiles.  Fitted to 2160 calls as above, m = 17 .. 63, n =
// 256 .. 49152, K = 2112 .. 18944 (nine in ten within 12 %).  One or two rows in the last group take up to 25 % longer
// over a long run of tiles (n = 65536, K = 3072: 61.9 us at m = 17, 51.5 at m = 20).
inline float slab_loop_us(uint32_t m, uint32_t tiles, uint32_t k, uint32_t mg, uint32_t blocks) {
    const uint32_t groups = (m + 16 * mg - 1) / (16 * mg), cap = std::max<uint32_t>(1, blocks / groups);
    const float per = (float)((tiles + cap - 1) / cap), slabs = (float)((k + kSlabColumns - 1) / kSlabColumns);
    const float us = mg == 1 ? 2.4f + slabs * (1.6f + 1.43f * per) : 2.2f + slabs * (3.75f + 1.42f * per);
    return (m % 16 == 1 || m % 16 == 2) && m > 16 && per > 4.0f ? 1.15f * us : us;
}

// Groups of 16 token rows per block: one, on more blocks, while there are few tiles, else two per unpacked word.
// options: KR_OPT_SKINNY_GROUPS and KR_OPT_SKINNY_MAX_BLOCKS (the same bits under any).
inline uint32_t slab_loop_groups(uint32_t m, uint32_t tiles, uint32_t k, uint32_t groups_option, uint32_t blocks) {
    return m > 16 && groups_option != 1 && slab_loop_us(m, tiles, k, 2, blocks) < slab_loop_us(m, tiles, k, 1, blocks) ? 2 : 1;
}

// Whether the slab loop takes m token rows over `rows` weight rows in all (ns[i] of np problems; gate/up: one).  Before /
// with it, us: gate/up [2 x 9536, 3072], m = 2 .. 16 67-70 / 17, m = 32 41 / 22, m = 40 41 / 39; q/k/v [4608, 3584], m = 2
// 45 / 10; linear [3584, 18944], m = 8 255 / 28, m = 32 77 / 39; [2048, 11008], m = 27 46 / 20, m = 63 46 / 27.  So: gate/up
// up to 32 tokens; other launches up to 16, and above where it is estimated faster than the prefill launch these sizes
// would take: [65536, 3072], m = 32 51.7 us against 38.3 there, [32768, 8192], m = 32 59.8 / 73.0; [6144, 4096], m = 33
// 21.5 / 19.9; [2048, 2112] (an odd group count: 64-column steps), m = 33 11.5 / 18.5.  With one token tile no other
// block reads a block's weights: about 0.05 us per MB over prefill_us.  13 of the 2160 calls come out 3 to 7 % slower than
// on the prefill kernel, none more.  (Defaults on purpose, not the options: results must not depend on those.)
inline bool slab_loop_pays(uint32_t m, const uint32_t *ns, int np, uint32_t k, bool gate_up, uint32_t cus) {
    if (m <= (gate_up ? 32u : 16u)) return true;
    if (gate_up) return false;
    uint32_t tiles = 0, rows = 0;
    for (int i = 0; i < np; ++i) {
        tiles += (ns[i] + 15) / 16;
        rows += ns[i];
    }
    float prefill;
    if (k % 128 == 0) {
        const int shape = prefill_choice(m, ns, np, k, 1, false, cus).shape;
        prefill = prefill_us(kCostNarrow, m, ns, np, k, 1, cus);
        for (const PrefillCost &w : kCostWide)
            if (w.shape == shape) prefill = prefill_us(w, m, ns, np, k, 1, cus);
    } else {
        const uint64_t rounds = (prefill_tiles(m, ns, np, 64, 64) + cus - 1) / cus;
        prefill = 5.0f + 0.36f * (float)(rounds + 1) * (float)k / 128.0f;
    }
    prefill += 0.05e-6f * (float)rows * (float)k * 0.5f;
    const float loop = std::min(slab_loop_us(m, tiles, k, 1, kSlabLoopBlocks), slab_loop_us(m, tiles, k, 2, kSlabLoopBlocks));
    return loop < 0.99f * prefill;
}

// ---- routed experts (q4_grouped.hip, q4_skinny.hip, moe.hip); tokens per expert as if they were even

// Grouped matrix products instead of the few-token kernel, which takes 16 tokens of an expert at a time and moves fewer
// zero rows: from 8 to 10 tokens per expert where there are many experts (one of them has 17 by then; the later the larger
// their matrices), later still where few experts leave compute units idle.  Measured crossings (random routing, tokens
// per expert): 60 experts [1408, 2048] 10, 32 11, 16 13, 8 15, 4 25, 2 40; 16 [2048, 2048] 12, 8 15, 4 28; 64 [768, 2048] 9,
// 32 9, 16 10, 8 14, 4 26; 32 [512, 1024] below 8, 16 8, 8 13, 4 24, 2 28.  The rule: 10.9, 11.8, 13.5, 17, 24, 38; 13.5, 17, 24;
// 8.9, 9.8, 11.5, 15, 22; 9.8, 11.5, 15, 22, 36.
inline bool moe_grouped_pays(uint32_t assign, uint32_t experts, uint32_t hidden, uint32_t inter) {
    return assign >= ((uint64_t)hidden * inter >= 2500000 ? 10u : 8u) * (uint64_t)experts + 56;
}

// 96-token tiles instead of 32-token ones, ntiles of them side by side per expert: once they hold a second fragment on
// average (the third is skipped where there are no tokens), if they still give two blocks per three compute units (down:
// or one per two, well filled).  This / 32-token tiles: gate/up of [1408, 2048], 60 experts 1.00 at 22 tokens per expert,
// 0.96 at 28, 0.79 at 40; 8 (176 blocks) 1.03 at 28, 0.89 at 40; 4 (88) 1.15 at 64, 0.97 at 128 (176); [2048, 2048], 8 (256)
// 1.00 at 24, 0.90 at 28; down: 60 experts 1.00 at 20, 0.93 at 32; 16 (256) 0.91 at 28; 8 (128) 1.04 at 40, 0.97 at 64.
inline bool moe_wide_tiles(uint32_t assign, uint32_t experts, uint32_t ntiles, bool gate_up, uint32_t cus) {
    const uint32_t e = std::max(1u, std::min(experts, assign)), per = assign / e;
    const uint64_t blocks = (uint64_t)e * ((per + 95) / 96) * ntiles;
    if (!gate_up && per > 56 && blocks * 2 >= cus) return true;
    return per > (gate_up ? 23u : 20u) && blocks * 3 >= 2 * (uint64_t)cus;
}

// Slots of the sorted list in parts, one per wave (3.6 us plus 0.6 per 1000 assignments), instead of a pass over all
// assignments for every sixteen experts (3.0 us plus 1.2 per 1000 and sixteen): 8 experts, 256 assignments 3.65 / 3.35 us,
// 512 3.79 / 3.87, 2048 5.2 / 7.2; 32 experts, 192 3.60 / 3.68; 60 experts, 128 3.60 / 3.88, 4096 6.8 / 35.6.
inline bool moe_route_parts(uint32_t assign, uint32_t experts) { return (uint64_t)((experts + 15) / 16) * assign > 480; }

}  // namespace kr
