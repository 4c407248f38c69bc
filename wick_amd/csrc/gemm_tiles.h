// gemm_tiles.h -- the tile of gemm_kernel (model.hip) that a product of several
// tokens runs on.  Plain C++, so that a host program can ask for it too.
#pragma once

namespace wick {

// rb x tb blocks of 16 rows x 16 tokens; waves per workgroup; 16-column k-steps
// a wave takes per batch of loads
struct GemmTile {
    int rb, tb, waves, ku;
};

// 8 waves, or 6 where those take no more batches of 32 columns each (576 columns
// are 18: 3 either way; 16 tokens of gate/up 6.2 against 6.5 us, 251 tokens of o
// 6.3 against 6.5; where they take more, up to a quarter slower).
inline int gemm_waves(int cols) {
    const int nbat = (int)((cols + 31LL) / 32);
    return (nbat + 5) / 6 == (nbat + 7) / 8 ? 6 : 8;
}

// What a tile of rb x tb blocks costs: the products of the busiest of the 256
// CUs, each dearer the less the tile reuses what it loads.  The model's order
// is the measured one where the tiles differ by more than a few percent: 64
// tokens at 2048 x 2048: 1x2 10 us, 2x2 12.6; 251 tokens at 2560 x 2048: 5x2
// 27.5, 1x2 30.2, 2x2 30.7; at 2048 x 5632: 2x4 47.3, 2x2 50.4; at 576 x 576:
// 2x2 6.3, 1x2 6.6, 2x4 8.
inline double gemm_cost(int rows, int t, int rb, int tb) {
    const long long wgs = ((rows + 16LL * rb - 1) / (16 * rb)) * ((t + 16LL * tb - 1) / (16 * tb));
    return (double)((wgs + 255) / 256) * (rb * tb + 0.5 * (rb + tb));
}

inline GemmTile gemm_tile(bool gate_up, int rows, int cols, int t) {
    if (t <= 16) {
        // bound by the weights' arrival: more of them in flight per wave where a
        // wave takes several batches (4 tokens, 2048 x 5632: 13.7 against 17.4
        // us; at 576 columns a batch of 4 leaves waves idle, 4.1 against 3.5)
        if (!gate_up && cols >= 2048) return {1, 1, 8, 4};
        return {1, 1, gemm_waves(cols), 2};
    }
    // Larger tiles of both matrices fill a CU's LDS with one workgroup: 251
    // tokens at 5632 x 2048 114 us on 2x2 against 110.  8 waves leave room for
    // two; with 4 more workgroups fit where a wave takes few batches.  251 tokens
    // on 4 / 8 waves: 1536 x 576 13.6 / 20.7 us, 4864 x 896 47 / 59, 5632 x 2048
    // 111 / 109.  Between, a few tokens want 8 and many want 4: 17 and 251 tokens at
    // 3072 x 1024 11.3 / 10.8 and 36 / 38, at 3456 x 1280 14.1 / 12.6 and 46 / 53.
    if (gate_up) return {1, 2, cols < 1024 ? 4 : 8, 2};
    const int tiles[][2] = {{1, 2}, {2, 2}, {2, 4}, {5, 2}};
    int best = 0;
    for (int i = 1; i < 4; i++)
        if (gemm_cost(rows, t, tiles[i][0], tiles[i][1]) < gemm_cost(rows, t, tiles[best][0], tiles[best][1])) best = i;
    return {tiles[best][0], tiles[best][1], best < 2 ? gemm_waves(cols) : 8, 2};
}

}  // namespace wick
