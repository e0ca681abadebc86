// How the prompt's matrix products (prefill.hip) are cut up: plain host code, which a test compiles by itself.
// Needs ceil_div of common.hpp.
#pragma once

namespace l2 {

constexpr int kTile = 32; // rows of a token tile, columns of a weight tile (v_mfma_f32_32x32x16_f16)

// How a product is cut up: MT token tiles and WN pairs of weight tiles per workgroup, WK groups per step, and
// pieces of K per launch.
struct GemmShape {
    int mt, wn, splits;
    int mt2, first; // mt2 other than mt: the first `first` blocks of weights of every XCD with mt token tiles, the rest with mt2
};

constexpr int kMaxSplits = 8;

// The cheapest of the shapes that fit into LDS, by an estimate in ns that was fitted to the times of 700 launches of 7B and
// 13B (all shapes, 32 to 1003 rows): a launch takes 4.3 us, every round of workgroups (one per compute unit) 3.1 us to fill
// and drain and its steps; the last round's steps go faster the fewer compute units it has, because the clock follows the
// power that the matrix cores take.  Blocks of weights go to the 8 XCDs in turn, so the rounds are those of the XCD with the
// most blocks.  A piece of K is written and read once more at about 4.5 TB/s.  Over those launches the shapes
// picked take 0.8 % more than the best ones of each size together; with the XCDs and the clock left out 3.4 % (13B, 1003
// rows, o-proj: 20 blocks of 11, 33 workgroups on 32 compute units, 131 us instead of 89).
inline GemmShape gemm_shape(int tiles, int pairs, int groups, bool may_split, int cus)
{
    static constexpr int kStepNs[5] = {0, 900, 1330, 1710, 2070}; // by token tiles, one group of K
    static constexpr int kLaunchNs = 4300, kRoundNs = 3100, kXcds = 8;
    const int per_xcd = cus >= kXcds ? cus / kXcds : 1;
    GemmShape best{};
    long long least = -1;
    for (int wn = 4; wn >= 1; wn /= 2)
        for (int mt = wn; mt >= 1; --mt)
            for (int splits = 1; splits <= (may_split ? kMaxSplits : 1) && (splits == 1 || splits * 4 <= groups); ++splits) {
                const int wk = 4 / wn;
                const int units = ceil_div(ceil_div(pairs, wn) * splits, kXcds) * ceil_div(tiles, mt); // of one XCD
                const int rounds = ceil_div(units, per_xcd), last = units - (rounds - 1) * per_xcd;
                const long long steps = ceil_div(ceil_div(groups, splits), wk);
                const long long step = kStepNs[mt] * (wk > 1 ? 107 : 100) / 100;
                const long long cost = kLaunchNs + kRoundNs * rounds +
                                       steps * step * ((rounds - 1) * 10 * per_xcd + 6 * per_xcd + 4 * last) / (10 * per_xcd) +
                                       (may_split ? static_cast<long long>(splits) * tiles * kTile * pairs * 64 * 4 / 4500 : 0);
                if (least < 0 || cost < least)
                    least = cost, best = GemmShape{mt, wn, splits, mt, 0};
            }
    if (may_split)
        return best;
    // Two heights of workgroup, the higher ones in full rounds.  7B, 511 rows, SwiGLU: 44 workgroups for the 32 compute units of an
    // XCD; 32 of them and 24 of half the height instead.  The whole prompt, one height -> two: 7B 350 / 512 / 740 / 1004 tokens
    // 9.33 / 10.92 / 14.98 / 18.31 ms -> 9.15 / 10.60 / 14.78 / 17.97, 13B 310 / 940 / 1004 14.86 / 35.7 / 36.9 -> 14.47 / 34.8 / 36.2.
    // Only for 2 % of the product at least, which is more than the estimate's error: 7B and 13B have 3 % or more
    // wherever they have any, but for SwiGLU of 385 .. 448 rows of 7B (0.3 %), whose prompts took 1.0 .. 1.4 % longer with two
    // heights (400 tokens 9.74 -> 9.85 ms).  One height stays for 7B up to 320 rows, at 385 .. 480, 513 .. 672 and 769 .. 896.
    least = least * 98 / 100;
    static constexpr int kMixed[][2] = {{4, 3}, {4, 2}, {3, 2}};
    const int rows = ceil_div(ceil_div(pairs, 4), kXcds);
    for (const auto& m : kMixed)
        for (int first = 1; first < rows; ++first) {
            const int units = first * ceil_div(tiles, m[0]), units2 = (rows - first) * ceil_div(tiles, m[1]);
            if (units % per_xcd)
                continue;
            const int rounds = units / per_xcd, rounds2 = ceil_div(units2, per_xcd), last = units2 - (rounds2 - 1) * per_xcd;
            const long long cost = kLaunchNs + kRoundNs * (rounds + rounds2) + static_cast<long long>(groups) * rounds * kStepNs[m[0]] +
                                   static_cast<long long>(groups) * kStepNs[m[1]] *
                                       ((rounds2 - 1) * 10 * per_xcd + 6 * per_xcd + 4 * last) / (10 * per_xcd);
            if (cost < least)
                least = cost, best = GemmShape{m[0], 4, 1, m[1], first};
        }
    return best;
}

} // namespace l2
