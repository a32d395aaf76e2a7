// Rows of row-strided arrays as consecutively numbered 16-byte chunks (8 bf16
// each): the numbering of swiglu_vec.  constexpr and free of HIP, so that the
// kernels and the host-side unit test (g++) run this one definition.
#pragma once

#include <stdint.h>

#include "kp_div32.hpp"

namespace kp {

// Chunks of one launch over several rows: chunk numbers are 32-bit and a
// div32 numerator is below 2^31.
constexpr int64_t kMaxRowChunks = 0x7fff0000LL;

// Chunk k of rows of cpr.d chunks: its row, and its first column -- 64-bit, a
// row of 2^29 chunks has 2^32 columns.
struct RowChunk {
  uint32_t row;
  int64_t col;
};
constexpr RowChunk row_chunk(uint32_t k, const Div32& cpr) {
  const uint32_t row = div32(k, cpr);
  return RowChunk{row, (int64_t)(k - row * cpr.d) * 8};
}

}  // namespace kp
