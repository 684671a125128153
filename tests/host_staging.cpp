// host_staging.cpp -- cable_amd/csrc/staging.h by itself, for
// tests/test_staging.py: prints, one line each, the offsets of a batch's arrays
// modulo the alignment they need, and how the bytes of a buffer of some sizes were
// handed out.
#include <stdio.h>

#include "../cable_amd/csrc/staging.h"

using namespace staging;

int main() {
  // the first arrays of a batch of single-value FP64 fields of 77 tiles
  size_t off = TABLE_BYTES;
  printf("offsets");
  for (int k = 0; k < 4; k++, off += align_up(77 * 8)) printf(" %zu", off % ALIGN);
  printf("\n");
  // each byte once, whether threads start or leave the work to the first; the
  // most threads that have a part of one aligned 2 MiB; pieces beyond their unit
  const size_t unit = UNIT, large = 2 << 20;
  for (size_t bytes : {(size_t)1, (size_t)65536, unit - 1, unit + 1, 4 * unit - 1, 4 * unit, 9 * unit + 12345}) {
    for (bool starts : {true, false}) {
      std::vector<std::atomic<int>> seen(bytes), parts(bytes / large + 1);
      for (auto &x : seen) x = 0;
      for (auto &x : parts) x = 0;
      std::atomic<size_t> beyond(0);
      on_threads(bytes, [&] { return starts; }, [&](size_t b0, size_t b1) {
        for (size_t b = b0; b < b1; b++) seen[b]++;
        beyond += b0 / unit != (b1 - 1) / unit;
        for (size_t p = b0 / large; p <= (b1 - 1) / large; p++) parts[p]++;
      });
      size_t once = 0;
      int most = 0;
      for (auto &x : seen) once += x == 1;
      for (size_t p = 0; p + 1 < parts.size() && (p + 1) * large + unit + large <= bytes; p++)
        most = std::max(most, parts[p].load());
      printf("pieces %zu %zu %zu %d\n", bytes, once, (size_t)beyond, bytes < 4 * unit ? 1 : most);
    }
  }
  // what a context of some tiles asks for in turn: its forcing's inputs, the surface
  // fluxes and the soil (29 values), and the times it pins for them
  for (size_t mp : {77, 1000, 4093, 20011}) {
    size_t have = 0, pins = 0;
    for (size_t need : {16 * mp, TABLE_BYTES + 14 * ALIGN + 29 * 8 * mp}) {
      if (need <= have) continue;
      have = capacity(need);
      pins += have >= need;
    }
    printf("pins %zu %zu\n", mp, pins);
  }
  return 0;
}
