// Which kernel and tile a dense product takes (plain C++, so that a host program can ask for any shape and any number of compute units).
#pragma once
#include <cmath>

// ---- tiles of the batched GEMM (dense_gemm.hip), tokens x weight rows; "dense.tile" is one more than these -----------------
enum {
    SKN_TILE_64x64 = 0,
    SKN_TILE_128x64 = 1,
    SKN_TILE_128x128 = 2,
    SKN_TILE_256x256 = 3,
    SKN_TILE_32x64_K4 = 4,   // k divided in four
    SKN_TILE_256x192 = 5,
    SKN_TILE_128x192 = 6,
    SKN_TILE_128x128_K2 = 7  // k divided in two
};

// A shape's time: of a launch, of the loop over k = 4096 with one, two or three tiles on a compute unit, and of the store of a tile to each.
struct skn_dense_tile_cost {
    int rows_a, rows_w, resident;  // resident 0: not chosen by its cost
    float launch, loop[3], store;
};

// m tokens, weights of [rows, k_pad] elements of elem_bytes (2: bf16, 4: fp32)
static inline int skn_dense_tile(int elem_bytes, int m, int rows, int k_pad, int units) {
    // bf16 rows of 512 elements and more, us, fitted to 476 shapes (40 to 2048 tokens, 256 to 18496 rows, k from 512 to 8192, weights not in any cache;
    // profiles/dense_gemm_tiles.md).  On those shapes the choice takes 1.015 times the best one's time in the mean, 1 / 1.047 of what it takes by the loops
    // alone (2048 x 2048 x 8192 94 -> 88 us, 1000 x 18496 x 2048 in a model 151 -> 142) and at worst 1.035 times as long as that; at worst 1.54 times
    // the best one's (see the end).
    static const skn_dense_tile_cost fitted[8] = {
        {64, 64, 3, 8.2f, {28.6f, 38.8f, 35.4f}, 0.8f}, {128, 64, 2, 10.3f, {33.f, 51.8f}, 3.6f}, {128, 128, 2, 8.6f, {65.9f, 62.f}, 5.5f},
        {256, 256, 1, 12.2f, {88.3f}, 22.7f},           {0, 0, 0, 0.f, {0.f}, 0.f},               {256, 192, 1, 13.f, {60.1f}, 21.5f},
        {128, 192, 2, 20.6f, {47.f, 55.8f}, 8.9f},      {128, 128, 1, 7.7f, {49.8f}, 5.f}};
    // fp32, and shorter rows: of the loop alone, in relative units.  An fp32 loop takes sixteen times as long, so that launches and stores are
    // nothing beside it, and in rows of less than 512 elements it is not what the fit above saw.  us at fp32, by the fitted costs | by these: 1000 x 8512 x 2048
    // 515 | 339, 954 x 8512 x 2048 485 | 282, 512 x 18496 x 2048 489 | 391, 1700 x 10752 x 2048 976 | 692, 2048 x 10752 x 2048 977 | 727, 1000 x 18496 x 512
    // 295 | 206; at bf16: 1000 x 8512 x 256 30.7 | 23.5, 954 x 8512 x 448 33.6 | 27.1, 1700 x 10752 x 256 54.2 | 44.6, 2048 x 10752 x 448 69.3 | 59.5.
    static const skn_dense_tile_cost loops[8] = {
        {64, 64, 3, 0.f, {25.f, 40.f, 40.f}, 0.f}, {128, 64, 2, 0.f, {31.f, 48.f}, 0.f}, {128, 128, 2, 0.f, {59.f, 87.f}, 0.f},  {256, 256, 1, 0.f, {145.f}, 0.f},
        {0, 0, 0, 0.f, {0.f}, 0.f},                {256, 192, 1, 0.f, {116.f}, 0.f},     {128, 192, 2, 0.f, {80.f, 118.f}, 0.f}, {128, 128, 0, 0.f, {0.f}, 0.f}};
    const bool known = elem_bytes == 2 && k_pad >= 512;
    const skn_dense_tile_cost* costs = known ? fitted : loops;
    const float length = known ? (float)k_pad / 4096.f : 1.f;
    int best = 0;
    float best_time = INFINITY;
    for (int i = 0; i < 8; i++) {
        const skn_dense_tile_cost& c = costs[i];
        if (c.resident == 0) continue;
        const int tiles = ((m + c.rows_a - 1) / c.rows_a) * ((rows + c.rows_w - 1) / c.rows_w), round = c.resident * units;
        const int rest = tiles % round;
        // (by loops alone, 192 rows are for the rounds of widths that 128 and 256 leave a third of idle: only with four fifths of the last round)
        if (!known && c.rows_w == 192 && rest != 0 && 5 * rest < 4 * (rest <= units ? units : round)) continue;
        const float turns = tiles / round * c.loop[c.resident - 1] + (rest == 0 ? 0.f : c.loop[(rest - 1) / units]);
        const float time = c.launch + length * turns + (float)tiles / units * c.store;
        if (time < best_time) best = i, best_time = time;
    }
    // Few outputs: k divided in four.  Rows of eight slices and more (512 elements of bf16, 256 of fp32) where half of the compute units have a
    // tile: bf16 40 x 512 x 512 7.3 -> 5.0 us, fp32 64 x 2048 x 256 10.8 -> 7.1, 40 x 4096 x 256 10.4 -> 7.0; of sixteen slices where all have one.  (Between,
    // at k = 512, it would be faster too: eleven of the measured shapes, 333 x 1024 x 512 8.7 us on 64 x 64 tiles and 5.7 on these.)
    const int few = ((m + 31) / 32) * ((rows + 63) / 64), slices = k_pad * elem_bytes / 128;
    if ((few <= units && slices >= 16) || (2 * few <= units && slices >= 8)) best = SKN_TILE_32x64_K4;
    return best;
}
