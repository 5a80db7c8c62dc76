// Where the lanes of the tiled GEMM's async loads find their 16 bytes (no HIP types: the CPU tests compile
// this header too).
#pragma once

#include <stdint.h>

namespace mk {

// A stage of the LDS ring holds rows of BKB bytes of K.  16-byte chunk c of row r sits at slot c ^ swz(r), so
// the 16 lanes of a ds_read_b128 phase (16 consecutive rows, same chunk) hit 16 distinct 4-bank groups.
template <int BKB>
constexpr int swz(int row) {
  return BKB == 64 ? (row >> 2) & 3 : (row >> 1) & 7;
}

// the chunk of its row that lane `lane` of a load loads (BKB / 16 consecutive lanes share a row)
template <int BKB>
constexpr int stage_chunk(int lane, int row) {
  return (lane % (BKB / 16)) ^ swz<BKB>(row);
}

// Lane offset of a load of the last stage when K ends halfway through it: `voff` is the lane's offset at K
// byte 0, kb the stage's first K byte.  Lanes whose chunk lies past K get an offset that the buffer's range
// check refuses (operands span less than 4 GiB), so they read nothing and leave zeros: past K there is the
// next row, or, after the last row of an operand that is a column range of a wider matrix, memory that need
// not belong to the caller.
template <int BKB>
constexpr uint32_t half_stage_offset(uint32_t voff, int lane, int row, uint32_t kb) {
  return stage_chunk<BKB>(lane, row) < BKB / 32 ? voff + kb : 0xfffffff0u;
}

}  // namespace mk
