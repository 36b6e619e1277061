// Walks the loads of the products of few rows over every lane: each ends inside its buffer or has a vector offset past its end, and what a
// row's lanes read is the row.  Prints the number of loads looked at.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "gemm_few_loads.h"

static long long looked = 0;

static void check(bool ok, const char* what, int n, int k, int lane, int x) {
    looked++;
    if (ok) return;
    std::printf("%s: %d rows of %d elements, lane %d, load %d\n", what, n, k, lane, x);
    std::exit(1);
}

// a load of sixteen bytes: past the end by its vector offset, or `row`'s bytes from `from` on
static void load(uint32_t vector, uint64_t scalar, uint64_t bytes, int row, int rows, uint64_t row_bytes, uint64_t from, const char* what, int k, int lane, int x) {
    if (row >= rows) check(vector >= bytes, what, rows, k, lane, x);
    else check(vector + scalar == row * row_bytes + from && vector + scalar + 16 <= bytes, what, rows, k, lane, x);
}

template <int PIECES, int BYTES>
void weights(int n, int k) {
    using L = FewWeightLoads<PIECES, BYTES>;
    const int nb = k / 256;
    const uint32_t row = nb * BYTES, bytes = n * row;
    for (int n0 = (n - 1) / 16 * 16; n0 >= 0; n0 -= std::max(16, n0 / 32 * 16))  // (the last tile, some others, the first)
        for (int sb = 0; sb < nb; sb += std::max(1, nb - 1))
            for (int lane = 0; lane < 64; lane++) {
                for (int x = 0; x < L::COUNT; x++) {
                    const uint32_t at = L::wide(lane, n0, row, bytes) + x * L::step(row);
                    if (!L::wide_lane(lane)) check(at >= bytes, "weights, no piece", n, k, lane, x);
                    else load(at, (uint64_t)sb * BYTES, bytes, n0 + x * (64 / L::WIDE) + lane / L::WIDE, n, row, (uint64_t)sb * BYTES + std::min(lane % L::WIDE * 16, BYTES - 16), "weights", k, lane, x);
                }
                if (!L::REST) continue;
                const uint32_t at = L::rest(lane, n0, row, bytes);
                if (!L::rest_lane(lane)) check(at >= bytes, "weights, no rest", n, k, lane, -1);
                else load(at, (uint64_t)sb * BYTES, bytes, n0 + L::rest_row(lane), n, row, (uint64_t)sb * BYTES + L::rest_piece(lane) * 16, "weights, rest", k, lane, -1);
            }
}

template <int CH, int MT>
void activations(int m, int k) {
    using L = FewActivationLoads<CH>;
    const uint32_t row = 2 * k, bytes = m * row;
    for (int m0 = (m - 1) / (16 * MT) * 16 * MT; m0 >= 0; m0 -= 16 * MT)
        for (int chunk = 0; chunk < k / (32 * CH); chunk += std::max(1, k / (32 * CH) - 1))
            for (int lane = 0; lane < 64; lane++)
                for (int x = 0; x < CH * MT; x++)
                    load(L::first(lane, m0, row) + x * L::step(row), (uint64_t)chunk * 64 * CH, bytes, m0 + x * L::ROWS + lane / L::LANES, m, row,
                         (uint64_t)chunk * 64 * CH + lane % L::LANES * 16, "activations", k, lane, x);
}

int main() {
    for (int k : {256, 512, 2304, 11008, 16384})
        for (int n : {1, 2, 3, 4, 5, 7, 8, 9, 11, 12, 13, 15, 16, 17, 31, 33, 100, 4095, 32003}) {
            weights<9, 144>(n, k), weights<11, 176>(n, k), weights<17, 272>(n, k);
            weights<14, 210>(n, k);
        }
    weights<17, 272>(((1u << 31) - 1) / (64 * 272), 16384);  // (as many rows as the path takes: no offset wraps)
    weights<14, 210>(((1u << 31) - 1) / 210, 256);
    for (int k : {256, 2304, 16384})
        for (int m = 1; m <= 130; m++) activations<4, 1>(m, k), activations<2, 2>(m, k), activations<2, 3>(m, k), activations<2, 4>(m, k);
    activations<2, 4>(393216, 256);
    std::printf("%lld loads\n", looked);
    return 0;
}
