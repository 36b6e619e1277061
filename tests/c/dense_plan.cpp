// Answers what a dense product would take, a line for each line read: "tile bytes m rows k units".
#include <cstdio>
#include <cstring>

#include "dense_plan.h"

int main() {
    char what[16];
    int v[5];
    while (std::scanf("%15s", what) == 1) {
        if (std::strcmp(what, "tile") != 0 || std::scanf("%d %d %d %d %d", v, v + 1, v + 2, v + 3, v + 4) != 5) return 1;
        std::printf("%d\n", skn_dense_tile(v[0], v[1], v[2], v[3], v[4]));
    }
    return 0;
}
