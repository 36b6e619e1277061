// Answers what a dense product would take, a line for each line read:
//   tile bytes m rows k units                                                          -> the tile
//   pitch bytes elements                                                               -> whether the GEMM's offsets reach all of a tile
//   once mode bytes rows k_pad ld k0 groups dim splits second_input units segments row0 .. -> wavefronts, pieces each, rows of a workgroup (0: staged)
#include <cstdio>
#include <cstring>

#include "dense_plan.h"

int main() {
    char what[16];
    int v[12];
    auto read = [](int* to, int n) {
        for (int i = 0; i < n; i++)
            if (std::scanf("%d", to + i) != 1) return false;
        return true;
    };
    while (std::scanf("%15s", what) == 1) {
        if (std::strcmp(what, "tile") == 0 && read(v, 5)) {
            std::printf("%d\n", skn_dense_tile(v[0], v[1], v[2], v[3], v[4]));
        } else if (std::strcmp(what, "pitch") == 0 && read(v, 2)) {
            std::printf("%d\n", (int)skn_dense_pitch_ok(v[0], v[1]));
        } else if (std::strcmp(what, "once") == 0 && read(v, 12) && v[11] >= 0 && v[11] <= 8) {
            skn_dense_call c = {v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8], v[9] != 0, v[11], {}};
            if (!read(c.row0, c.nseg)) return 1;
            const skn_dense_once p = skn_dense_once_plan(c, v[10]);
            std::printf("%d %d %d\n", p.parts, p.pieces, p.rows);
        } else {
            return 1;
        }
    }
    return 0;
}
