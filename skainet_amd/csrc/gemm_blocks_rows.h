// The rows that the activation operands of gemm_blocks.hip are laid out for, and which of their blocks of 32 a tile of 96 rows reads
// (plain C++, so that a host program can walk them).  The layout follows the number of rows alone: a caller that captures calls runs one
// of the same type and activations before, with whatever matrix, and must find the workspace grown to what the captured ones need.
#pragma once

// 32 for up to 32 rows, else whole tiles of 64: what 64-row tiles read, and 96-row tiles too.
constexpr int skn_blocks_padded_rows(int m) { return m <= 32 ? 32 : (m + 63) / 64 * 64; }

// The layout's block of 32 rows for block `block` of the tiles of 96 rows.  Their last tile may reach past the layout: it repeats the last
// block there, whose products no row of the output takes.
constexpr int skn_blocks_of_96(int block, int m) { return block < skn_blocks_padded_rows(m) / 32 ? block : skn_blocks_padded_rows(m) / 32 - 1; }
