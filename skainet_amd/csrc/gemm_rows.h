// The rows that the products' activation operands take room for (plain C++, so that a host program can walk them).  That follows the number
// of rows alone: a caller that captures calls runs one of the same type and activations before, with whatever matrix, and must find the
// workspace grown to what the captured ones need.
#pragma once

// Q4_K and Q6_K: the tiles' height follows the matrix too, 64 rows (Q6_K also 32) or, above 128 rows, up to 256.
constexpr int skn_tall_rows(int m) { return m <= 128 ? (m + 63) / 64 * 64 : (m + 255) / 256 * 256; }

// Formats in blocks of 32: the layout, and which of its blocks of 32 rows a tile of 96 rows reads.

// 32 for up to 32 rows, else whole tiles of 64: what 64-row tiles read, and 96-row tiles too.
constexpr int skn_blocks_padded_rows(int m) { return m <= 32 ? 32 : (m + 63) / 64 * 64; }

// The layout's block of 32 rows for block `block` of the tiles of 96 rows.  Their last tile may reach past the layout: it repeats the last
// block there, whose products no row of the output takes.
constexpr int skn_blocks_of_96(int block, int m) { return block < skn_blocks_padded_rows(m) / 32 ? block : skn_blocks_padded_rows(m) / 32 - 1; }
