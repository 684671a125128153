// host_staging.cpp -- cable_amd/csrc/staging.h by itself, for
// tests/test_staging.py: prints, one line each, the offsets of a batch's arrays
// modulo the alignment they need, and how often the pieces of a buffer of some
// sizes were handed out.
#include <stdio.h>

#include "../cable_amd/csrc/staging.h"

using namespace staging;

int main() {
  // the first arrays of a batch of single-value FP64 fields of 77 tiles
  size_t off = TABLE_BYTES;
  printf("offsets");
  for (int k = 0; k < 4; k++, off += align_up(77 * 8)) printf(" %zu", off % ALIGN);
  printf("\n");
  // each byte once, whatever the threads
  for (size_t bytes : {(size_t)1, (size_t)65536, (size_t)UNIT - 1, (size_t)UNIT + 1, 9 * (size_t)UNIT + 12345}) {
    const size_t piece = 512 << 10, n = (bytes + piece - 1) / piece;
    std::vector<std::atomic<int>> seen(n);
    for (auto &x : seen) x = 0;
    on_threads(bytes, piece, [] { return true; }, [&](size_t q) { seen[q]++; });
    size_t once = 0;
    for (auto &x : seen) once += x == 1;
    printf("pieces %zu %zu\n", n, once);
    // threads that cannot start leave the work to the first
    for (auto &x : seen) x = 0;
    on_threads(bytes, piece, [] { return false; }, [&](size_t q) { seen[q]++; });
    once = 0;
    for (auto &x : seen) once += x == 1;
    printf("pieces %zu %zu\n", n, once);
  }
  return 0;
}
