// Where gemm_short.hip reads activation rows of any length at any address: in whole aligned 16-byte chunks, and a row's bytes out of
// those.  Plain integer arithmetic, so that the addresses can be checked on the host (tests/test_row_chunks.py).
#pragma once

#include <stdint.h>

#include "weight_loads.h"

namespace mi {

// The rows of a tile of at most 32, k bytes each and end to end: `address` is that of its first, `left` the rows from there to the tensor's
// last.  Offsets count from the 16-byte boundary at or in front of the address.
struct RowChunks {
  int skew, rows, k, end;
  // end: the last chunk with a byte of the tensor in it, which the blocks of its last row reach past
  MI_HOST_DEVICE RowChunks(uintptr_t address, int left, int k_) : skew((int)(address & 15)), rows(left < 32 ? left : 32), k(k_) {
    const int64_t last = (int64_t)skew + (int64_t)left * k - 1;
    end = (int)(last < 0x7fffffff ? last : 0x7fffffff) & ~15;
  }
  MI_HOST_DEVICE int row_at(int r) const { return skew + (r < rows ? r : rows - 1) * k; }  // (past the last row: that row again)
  // Chunk `id` of a block of 128 bytes of every row, nine to a row; `first` of block 0, what the others add to that, and not past the end.
  MI_HOST_DEVICE int first(int id) const {
    id = id < 32 * 9 ? id : 32 * 9 - 1;
    const int row = id * 57 >> 9;  // id / 9
    return (row_at(row) & ~15) + (id - 9 * row) * 16;
  }
  MI_HOST_DEVICE int of_block(int first, int block) const { return first + 128 * block < end ? first + 128 * block : end; }
  // Where row r's first byte of a block stands behind the first of its nine chunks.
  MI_HOST_DEVICE uint32_t odd(int r) const { return (uint32_t)row_at(r) & 15; }
};

}  // namespace mi
