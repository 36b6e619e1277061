// Byte offsets of the loads of gemm_few.hip (plain C++, so that a host program can walk them all).  The range check of a raw buffer load
// is defined for its vector offset; the scalar offset is no part of it.  So the vector offset of every load holds the row, which may lie
// past the last one (it then is the buffer's size at least, and the load reads as zero), and the scalar offset moves within a row only.
#pragma once
#include <cstdint>

// Sixteen rows of weights from row n0 on, a superblock of BYTES bytes each in PIECES pieces of sixteen bytes (the last one is the
// superblock's last sixteen): a row's first pieces go to WIDE neighbouring lanes, 64 / WIDE rows at a time, those past them to REST
// lanes.  From one load to the next a lane's offset grows by step(); the scalar offset is the superblock's place in its row.
template <int PIECES, int BYTES>
struct FewWeightLoads {
    static constexpr int WIDE = PIECES > 12 ? 16 : 8, REST = PIECES <= WIDE ? 0 : PIECES - WIDE == 1 ? 1 : 4;
    static constexpr int COUNT = WIDE / 4;  // (and one more with REST)
    static constexpr bool wide_lane(int lane) { return lane % WIDE < PIECES; }
    static constexpr uint32_t wide(int lane, int n0, uint32_t row_bytes, uint32_t bytes) {
        const int piece = lane % WIDE * 16;
        return wide_lane(lane) ? (uint32_t)(n0 + lane / WIDE) * row_bytes + (uint32_t)(piece < BYTES - 16 ? piece : BYTES - 16) : bytes;
    }
    static constexpr uint32_t step(uint32_t row_bytes) { return 64 / WIDE * row_bytes; }
    static constexpr int rest_row(int lane) { return REST ? lane / (REST ? REST : 1) : 16; }
    static constexpr int rest_piece(int lane) { return WIDE + lane % (REST ? REST : 1); }
    static constexpr bool rest_lane(int lane) { return rest_row(lane) < 16 && rest_piece(lane) < PIECES; }
    static constexpr uint32_t rest(int lane, int n0, uint32_t row_bytes, uint32_t bytes) {
        return rest_lane(lane) ? (uint32_t)(n0 + rest_row(lane)) * row_bytes + (uint32_t)rest_piece(lane) * 16 : bytes;
    }
};

// Rows of bf16 activations from row m0 on, CH blocks of 32 elements each: 4 CH lanes to a row, 16 / CH rows of a load.  The scalar offset is
// the chunk's place in its row.
template <int CH>
struct FewActivationLoads {
    static constexpr int LANES = 4 * CH, ROWS = 64 / LANES;
    static constexpr uint32_t first(int lane, int m0, uint32_t row_bytes) { return (uint32_t)(m0 + lane / LANES) * row_bytes + lane % LANES * 16; }
    static constexpr uint32_t step(uint32_t row_bytes) { return ROWS * row_bytes; }
};
