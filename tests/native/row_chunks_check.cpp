// Host check of kernelproblems_amd/csrc/kp_row_chunks.hpp: rows of 1 to
// kMaxRowChunks chunks, around the 2^29 chunks where a row's columns pass 32
// bits among them, at both ends of the rows and of the launch.
#include <cstdio>
#include <initializer_list>

#include "kp_row_chunks.hpp"

using namespace kp;

int main() {
  long checked = 0, bad = 0;
  for (int64_t cpr : {(int64_t)1, (int64_t)2, (int64_t)683, (int64_t)1 << 20, ((int64_t)1 << 28) + 1, ((int64_t)1 << 29) - 1,
                      (int64_t)1 << 29, ((int64_t)1 << 29) + 1, ((int64_t)1 << 30) - 1, kMaxRowChunks / 3,
                      kMaxRowChunks / 2, kMaxRowChunks}) {
    const Div32 by = make_div32((uint32_t)cpr);
    const int64_t rows = kMaxRowChunks / cpr, total = rows * cpr;
    for (int64_t row : {(int64_t)0, (int64_t)1, rows / 2, rows - 1})
      for (int64_t c : {(int64_t)0, (int64_t)1, cpr / 2, ((int64_t)1 << 29) - 1, (int64_t)1 << 29, cpr - 2, cpr - 1}) {
        const int64_t k = row * cpr + c;
        if (row < 0 || row >= rows || c < 0 || c >= cpr || k >= total) continue;
        const RowChunk p = row_chunk((uint32_t)k, by);
        ++checked;
        if (p.row != row || p.col != c * 8) {
          ++bad;
          std::printf("chunk %lld of rows of %lld: row %u column %lld\n", (long long)k, (long long)cpr, p.row,
                      (long long)p.col);
        }
      }
  }
  std::printf("%ld checked, %ld bad\n", checked, bad);
  return bad != 0 || checked < 100;
}
