// Walks the row blocks of the products on 96-row tiles: every one lies inside the operands' layout, and a block with rows of the output is
// the block itself.  The room of the other formats' operands takes every height of tile.  Prints the number of blocks looked at.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "gemm_rows.h"

int main() {
    long long looked = 0;
    for (int m = 1; m <= 4100; m++) {
        const int rows = skn_blocks_padded_rows(m), tiles = (m + 95) / 96;
        bool ok = rows >= m && rows % 32 == 0 && (m <= 32 || rows % 64 == 0) && rows - m < 64;
        for (int block = 0; block < 3 * tiles; block++, looked++) {
            const int from = skn_blocks_of_96(block, m);
            ok = ok && from >= 0 && 32 * from + 32 <= rows && (32 * block >= m || from == block);
        }
        for (int height : {32, 64, 128, 256})
            if (m > 128 || height < 128) ok = ok && skn_tall_rows(m) >= (m + height - 1) / height * height;
        if (!ok) {
            std::printf("%d rows\n", m);
            return 1;
        }
    }
    std::printf("%lld blocks\n", looked);
    return 0;
}
