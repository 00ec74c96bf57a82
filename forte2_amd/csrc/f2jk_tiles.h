// Width of the BF16x3 half-transform's column tiles.  Host code only.
#pragma once

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

}  // namespace f2jk
