// Tile plans of the K kernels: the width of the BF16x3 half-transform's column
// tiles, the tiles of the FP64 contraction and their P splits.  No device code.
#pragma once
#include <algorithm>
#include <cstdint>

namespace f2jk {

// The tile width, in units of 32 columns, for `need` occupied units and tiles of
// at most `cap` units.
//
// 256-row kernel (every width but 9, which spills): a column tile loads and
// splits all of B again, which takes as long as the products of 2 units (nbf
// 384, 2224 P) to 4 (nbf 960, 2000 P), and the widest is slower than its columns
// say (nbf 960: 2.24, 2.54, 2.67 and 3.22 ms with 6, 7, 8 and 10 units).  A tile
// costs its units and 2.5 more, 13 for the widest.  Counting the columns alone
// takes a divisor of `need`, for most prime numbers one tile per unit: at nbf
// 960 9 units took 4.18 ms as 3 x 3 and take 3.14 as 1 x 10, 11 units 6.39 as
// 11 x 1 and 4.02 as 2 x 6, 19 units 10.3 as 19 x 1 and 6.00 as 2 x 10.
//
// 128-row kernel (widths 10, 8, 6, 5, 4, 2): the fewest columns, then the wider
// tile.  Up to 5 units two workgroups share a CU, and narrow tiles cost less
// (nbf 384, 11 units: 1.20 ms as 3 x 4, 1.42 as 2 x 6).
inline int bf16_tile_units(int need, int cap, int rows) {
    constexpr int flat[] = {10, 8, 6, 5, 4, 2}, tall[] = {10, 8, 7, 6, 5, 4, 3, 2, 1};
    int best = 0, cost = 0;
    auto take = [&](int w, int tile) {
        const int c = (need + w - 1) / w * tile;
        if (w <= cap && (best == 0 || c < cost)) best = w, cost = c;
    };
    if (rows == 256)
        for (int w : tall) take(w, w == 10 ? 26 : 2 * w + 5);
    else
        for (int w : flat) take(w, w);
    return best;
}

constexpr int kDTileEdge = 128;
// The lower triangle of K in tiles of 8 x 8 blocks of 16; the last tile row has
// rl <= 8 blocks.  Four kinds of tiles, by the blocks of their busiest wave:
// 0 full (16), 1 diagonal (9), 2 last row, 3 last diagonal.
struct DTiles {
    int nt;        // tile rows
    int rl;        // 16-row blocks of the last tile row
    int cnt[4];    // tiles of each kind
    int ns[4];     // P splits of each kind
    int G;         // max ns of the kinds present
    int total;     // workgroups: sum cnt * ns
};

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Tiles of the FP64 contraction of an N x N matrix and the P splits of each
// kind, in proportion to the cost of a tile: the blocks of its busiest wave,
// 1.6 times that for a diagonal tile (its waves read two fragments per block
// and lose the matrix pipe to full tiles on the same CU: workgroups of a
// diagonal tile took 2.1 times their share of blocks).  A step takes no less
// than its loads, which are in flight for one step: as long as the products of
// 9 blocks, so the last row's tiles, of 4 blocks when nbf is a little above a
// multiple of 128, cost 9.  At 4 their workgroups had four times a full tile's
// steps and ended last (K at nbf 520, 100 columns, 1500 P: 3.39 ms with 4, 2.35
// with 9; 400 1.47 and 1.07, 288 0.73 and 0.57, 130 92 and 68 us; 8 and 10 are
// within 2% but at 130 and 150).
//
// All workgroups at once (512) is best when the shares round well; a tile count
// that does not fit runs in more, shorter workgroups that even out over several
// rounds, at ~5 us a round, the traffic of their partials and the reduction's
// chain of loads (~0.03 us per split).  The estimate below orders the measured
// times of nbf 318 (64.7 us per density at 512 workgroups, 71 at 1024, 85 at
// 2048), 384 (491, 562, 529), 960 (6.2-7.1 ms, 5.6, 5.3, 4.9 at 4096) and 1152
// (8.1-9.0 ms, 9.1, 8.6, 8.3).
inline DTiles dtile_plan(int N, int64_t Pc, int width, int slots) {
    DTiles m{};
    m.nt = (int)ceil_div(N, kDTileEdge);
    m.rl = (int)ceil_div(N - (m.nt - 1) * kDTileEdge, 16);
    m.cnt[0] = (m.nt - 1) * (m.nt - 2) / 2;
    m.cnt[1] = m.nt - 1;
    m.cnt[2] = m.nt - 1;
    m.cnt[3] = 1;
    const double cost[4] = {16, 1.6 * 9, std::max(9.0, 4.0 * ((m.rl + 1) / 2)),
                            std::max(9.0, 1.6 * ((m.rl * (m.rl + 1) / 2 + 3) / 4))};
    const double unit_us = 0.225 * (double)width / 16;  // one block for one P, two workgroups on the CU
    double sum = 0;
    for (int k = 0; k < 4; ++k) sum += m.cnt[k] * cost[k];
    double best = -1;
    for (double r : {0.25, 0.5, 1.0, 2.0, 4.0, 8.0})
        for (int i = 0; i < 4; ++i) {
            const double target = (double)slots * r * (1.0 - 0.04 * i);
            int ns[4], total = 0, G = 1;
            double work = 0, longest = 0;
            for (int k = 0; k < 4; ++k) {
                ns[k] = (int)std::max<int64_t>(1, std::min<int64_t>(Pc, (int64_t)(target * cost[k] / sum)));
                total += m.cnt[k] * ns[k];
                if (!m.cnt[k]) continue;
                G = std::max(G, ns[k]);
                longest = std::max(longest, cost[k] * (double)ceil_div(Pc, ns[k]));
            }
            // the partials stay within the workspace the serving layer reserves for a job
            if (G > 80 + (8 << 20) / ((int64_t)N * N) && best >= 0) continue;
            work = sum * (double)Pc / slots;
            const int rounds = (int)ceil_div(total, slots);
            // one round ends with its longest workgroup; several fill in behind each other
            const double span = rounds == 1 ? longest : std::max(work, longest) + 0.6 * longest;
            // up to one workgroup per CU has the matrix pipes to itself
            const double us = span * unit_us * (total <= slots / 2 ? 0.55 : 1.0) + 5.0 * rounds +
                              (double)G * N * N * 8 / 4e6 + 0.03 * G;
            if (best < 0 || us < best) {
                best = us;
                for (int k = 0; k < 4; ++k) m.ns[k] = ns[k];
                m.G = G;
                m.total = total;
            }
            if (slots < 256) break;  // a small cap: no variants
        }
    return m;
}

}  // namespace f2jk
