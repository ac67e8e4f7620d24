// launch_rules.hpp — which prefill launch a shape takes: plain host arithmetic on sizes, no HIP (the tests compile it
// with the host compiler).
//
// A launch's blocks run in rounds of one per compute unit, so its time is close to
//     fixed + rounds (round + step K / 128) + partial (f32 partials written and summed, in millions),
// also past one resident block per unit: they share its matrix cores.  The constants are least-squares fits to launches
// on MI355X (256 compute units) over copies of the weights in turn (none in an L2), captured in graphs: m = 17 .. 4096,
// n = 256 .. 151936, K = 1024 .. 18944, 2913 unsplit calls and 2190 with room for partials, each in every shape; the
// median error is 5 %.  Counting rounds is what decides: a tile half full of padding costs what a full one does.
#pragma once

#include <stdint.h>

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
constexpr PrefillCost kCostNarrow = {kPrefillNarrow, 64, 64, 5.3f, 0.3f, 0.45f, 0.0f};
constexpr PrefillCost kCostNarrowSplit = {kPrefillNarrow, 128, 128, 16.2f, -5.4f, 1.17f, 2.03f};
constexpr PrefillCost kCostWide[3] = {{kPrefillWide42, 128, 256, 3.2f, 4.5f, 1.64f, 0.0f},
                                      {kPrefillWide22, 64, 256, 5.4f, 0.1f, 1.13f, 0.0f},
                                      {kPrefillWide21, 64, 128, 8.7f, -3.3f, 0.83f, 0.0f}};
constexpr PrefillCost kCostWideSplit = {kPrefillWide42, 128, 256, 12.9f, -3.7f, 1.67f, 1.74f};
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
        // One round of 64 x 128 tiles has fewer loads in flight than two of 64 x 64: 16.0 / 17.3 us at K = 1536, but
        // 18.9 / 18.0 at K = 2048, 35.5 / 33.3 at K = 4096 and 90 / 78 at 11008 (m = 2048, n = 1024, K = 4096: 36.5 /
        // 41.4, but 33 with K split).
        if (c.shape == kPrefillWide21 && prefill_tiles(m, ns, np, c.rows, c.cols) <= cus && k > 1536 &&
            (m < 2048 || max_split > 1))
            scale = 1.25f;
        consider(c, 1, scale);
    }
    for (uint32_t split = 2; split <= max_split && k / 64 / split >= 8; split *= 2) consider(kCostWideSplit, split, 1.0f);
    return best;
}

}  // namespace kr
