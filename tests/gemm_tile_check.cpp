// Prints the tile of wick_amd/csrc/gemm_tiles.h, "rb tb waves ku", for every line
// "gate_up rows cols t" of its input.
#include "gemm_tiles.h"

#include <cstdio>

int main() {
    int gate_up, rows, cols, t;
    while (scanf("%d %d %d %d", &gate_up, &rows, &cols, &t) == 4) {
        const wick::GemmTile x = wick::gemm_tile(gate_up != 0, rows, cols, t);
        printf("%d %d %d %d\n", x.rb, x.tb, x.waves, x.ku);
    }
    return 0;
}
