// Which kernel and tile a dense product takes (plain C++, so that a host program can ask for any shape and any number of compute units).
#pragma once
#include <cmath>
#include <cstdint>

constexpr int kDenseRowPad = 32, kDenseColPad = 64;  // what the projections of a stacked matrix and its rows are padded to

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

// Whether 32-bit offsets reach every element of a tile's rows (256 at most) whose pitch is `pitch` elements.
static inline bool skn_dense_pitch_ok(int elem_bytes, int64_t pitch) { return pitch * elem_bytes * 256 <= INT32_MAX; }

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
    // Rows of 8192 and more, fitted to 160 shapes (40 to 8192 tokens, 256 to 18496 rows, k to 18432): a long loop takes up to 1.5 times as long a piece of k in the
    // larger tiles as the costs above have it.  us, by those | by these: 2048 x 4096 x 18432 408 | 333, x 10240 239 | 199, 4096 x 2048 x 10240 232 | 198, 8192 x 4096 x
    // 8192 555 | 479; 1.003 times the best one's time in the mean of 100 shapes that the fit above never saw.
    static const skn_dense_tile_cost longer[8] = {
        {64, 64, 3, 2.4f, {22.2f, 31.3f, 41.7f}, 0.f}, {128, 64, 2, 0.f, {27.5f, 44.3f}, 3.9f}, {128, 128, 2, 0.f, {53.9f, 68.6f}, 1.4f},
        {256, 256, 1, 0.f, {84.4f}, 69.4f},            {0, 0, 0, 0.f, {0.f}, 0.f},              {256, 192, 1, 0.f, {73.6f}, 44.9f},
        {128, 192, 2, 0.f, {62.3f, 81.8f}, 7.4f},      {128, 128, 1, 0.f, {43.1f}, 7.1f}};
    // fp32, and shorter rows: of the loop alone, in relative units.  An fp32 loop takes sixteen times as long, so that launches and stores are
    // nothing beside it, and in rows of less than 512 elements it is not what the fit above saw.  us at fp32, by the fitted costs | by these: 1000 x 8512 x 2048
    // 515 | 339, 954 x 8512 x 2048 485 | 282, 512 x 18496 x 2048 489 | 391, 1700 x 10752 x 2048 976 | 692, 2048 x 10752 x 2048 977 | 727, 1000 x 18496 x 512
    // 295 | 206; at bf16: 1000 x 8512 x 256 30.7 | 23.5, 954 x 8512 x 448 33.6 | 27.1, 1700 x 10752 x 256 54.2 | 44.6, 2048 x 10752 x 448 69.3 | 59.5.
    static const skn_dense_tile_cost loops[8] = {
        {64, 64, 3, 0.f, {25.f, 40.f, 40.f}, 0.f}, {128, 64, 2, 0.f, {31.f, 48.f}, 0.f}, {128, 128, 2, 0.f, {59.f, 87.f}, 0.f},  {256, 256, 1, 0.f, {145.f}, 0.f},
        {0, 0, 0, 0.f, {0.f}, 0.f},                {256, 192, 1, 0.f, {116.f}, 0.f},     {128, 192, 2, 0.f, {80.f, 118.f}, 0.f}, {128, 128, 0, 0.f, {0.f}, 0.f}};
    const bool known = elem_bytes == 2 && k_pad >= 512;
    const skn_dense_tile_cost* costs = !known ? loops : k_pad < 8192 ? fitted : longer;
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

// ---- the batch-1 product (dense_matvec.hip) ----------------------------------------------------------------------------------
enum { SKN_XSRC_PLAIN = 0, SKN_XSRC_GROUP_NORM = 1, SKN_XSRC_MERGE = 2, SKN_XSRC_ADD_NORM = 3 };  // what its input is made of (dense.h)

struct skn_dense_call {
    int mode, elem_bytes, rows, k_pad;
    int64_t ld;               // elements from row to row
    int k0, groups, dim, splits;  // columns of the input, norm groups, elements of a merged head, its splits
    bool second_input;
    int nseg;                 // segments and where they begin; 0: residual form
    int row0[8];
};

constexpr int kOnceGroups = 8;  // norm groups
constexpr int kOnceParts = 16;  // wavefronts of a workgroup on a plain input, half of them where the input is worked on

// dense_matvec_once_kernel: wavefronts of a workgroup, 1 KiB pieces of a row that each has, rows; rows 0: the staged kernel.
struct skn_dense_once {
    int parts, pieces, rows;
};

// Rows of a workgroup whose `parts` wavefronts share `rows` rows; 0: the input takes so much that many rows are better
// behind one staging of it.  (Figures of one comparison are of one sweep; two sweeps differ by boxes and by what a cache holds.)
// Four rows where the input is taken as it is (two where that leaves compute units without work): 2048 x 2048 3.52 | 3.49 | 3.59 us
// with 2 | 4 | 8, 2048 x 8192 8.0 | 7.3 | 7.7, 256 x 2048 and 2048 x 256 4.96 | 4.80 | 5.20.  A norm's launch takes rounds of compute
// units, a round of 2, 4, 8, 16 rows as 0.38, 0.6, 1, 1.9 (960 x 3072 behind a sum and a norm 5.2 | 4.2 | 4.6 | 5.5, 2624 x 3072
// 9.5 | 7.4 | 7.2 | 6.1, 5120 x 3072 15.0 | 10.8 | 9.6 | 10.2); more than two rounds of sixteen fp32 rows are better as eights
// (12000 x 1536 15.4 | 13.7, 16384 x 1536 19.4 | 18.4).
// The staged kernel, us of it | of the other: behind a sum and a norm 13312 x 2048 11.8 | 12.7, x 3072 16.6 | 18.6, and from two rounds of sixteen bf16 rows on, each
// of three pieces or more, 13312 x 1536 9.9 | 11.3, 9600 x 2048 10.5 | 11.2, but 8192 x 2048 10.2 | 8.9, 16384 x 1024 9.7 | 9.3; behind a merge of eight splits
// 4096 x 3072 9.5 | 9.7, 2624 x 4096 9.6 | 10.4, but 5120 x 2048 9.1 | 8.5, 2048 x 4096 7.7 | 7.0; of sixteen, whose partials are twice as many, 2624 x 3072 9.6 | 11.1,
// 5120 x 2048 9.8 | 10.7, but 8192 x 1024 8.8 | 8.2.  All shapes of profiles/dense_matvec_once.md, and those between, are within 3.5 % of the
// staged kernel or faster (but 16384 x 3072 behind a norm, 18.9 | 19.6).
static inline int skn_dense_once_rows(int mode, int elem_bytes, int rows, int parts, int splits, int units) {
    const int64_t pieces = (int64_t)rows * parts;
    if (mode == SKN_XSRC_PLAIN) return parts == 1 ? 8 : rows <= 2 * units ? 2 : 4;
    if (mode == SKN_XSRC_MERGE) return pieces > (splits > 8 && parts > 2 ? 60 : 80) * units ? 0 : rows <= 4 * units ? 4 : 8;
    if (mode == SKN_XSRC_ADD_NORM && (pieces > 176 * units || (elem_bytes == 2 && parts > 2 && rows > 32 * units))) return 0;
    const float round_cost[4] = {0.38f, 0.6f, 1.0f, 1.9f};
    int best = 0;
    float least = INFINITY;
    const int most = mode == SKN_XSRC_GROUP_NORM && elem_bytes == 4 && rows > 32 * units ? 8 : 16;
    for (int i = 0; i < 4; i++) {
        const int r = 2 << i;
        const float rounds = (float)rows / (float)(r * units), cost = round_cost[i] * (0.7f * std::ceil(rounds) + 0.3f * rounds);
        if (r <= 8 * parts && r <= most && cost < least) best = r, least = cost;
    }
    return best;
}

static inline skn_dense_once skn_dense_once_plan(const skn_dense_call& c, int units) {
    const int v = 16 / c.elem_bytes, pieces = (c.k_pad + 64 * v - 1) / (64 * v);  // elements of a request, 1 KiB pieces of a row
    const int each = c.mode != SKN_XSRC_PLAIN || pieces <= kOnceParts ? 1 : pieces <= 2 * kOnceParts ? 2 : 4, parts = (pieces + each - 1) / each;
    const skn_dense_once staged = {0, 0, 0};
    if (c.second_input || parts > (c.mode == SKN_XSRC_PLAIN ? kOnceParts : kOnceParts / 2) || c.ld * c.elem_bytes >= (int64_t)1 << 30) return staged;
    // The kernel has whole workgroups of rows, each of one segment: stacked as the projections of a matrix are, the first from its first
    // row on.  (The staged kernel goes row by row, and leaves out what lies ahead of the first segment.)
    if (c.rows % kDenseRowPad != 0) return staged;
    for (int i = 0; i < c.nseg; i++)
        if (c.row0[i] % kDenseRowPad != 0 || (i == 0 ? c.row0[0] != 0 : c.row0[i] <= c.row0[i - 1])) return staged;
    // a head, a norm group takes whole requests of a lane
    if (c.mode == SKN_XSRC_MERGE && c.dim % v != 0) return staged;
    if (c.mode == SKN_XSRC_GROUP_NORM && (c.groups > kOnceGroups || (c.groups > 1 && c.k0 / c.groups % v != 0))) return staged;
    if (c.mode == SKN_XSRC_ADD_NORM && c.groups != 1) return staged;
    const int r = each > 1 ? 4 : skn_dense_once_rows(c.mode, c.elem_bytes, c.rows, parts, c.splits, units);
    return r == 0 ? staged : skn_dense_once{parts, each, r};
}
