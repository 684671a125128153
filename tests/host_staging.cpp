// host_staging.cpp -- cable_amd/csrc/staging.h by itself, for
// tests/test_staging.py: prints, one line each, the offsets of a batch's arrays
// modulo the alignment they need, and how the bytes of a buffer of some sizes were
// handed out.
#include <stdio.h>

#include <mutex>

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
      std::mutex m;
      std::vector<Range> got;
      on_threads(bytes, [&] { return starts; }, [&](size_t b0, size_t b1) {
        std::lock_guard<std::mutex> l(m);
        got.push_back({b0, b1});
      });
      std::sort(got.begin(), got.end(), [](const Range &x, const Range &y) { return x.from < y.from; });
      size_t upto = 0, beyond = 0;
      std::vector<int> parts(bytes / large + 1);
      for (const Range &r : got) {
        upto = r.from == upto && r.end > r.from ? r.end : bytes + 1;
        beyond += r.from / unit != (r.end - 1) / unit;
        for (size_t p = r.from / large; p <= (r.end - 1) / large; p++) parts[p]++;
      }
      int most = 0;
      for (size_t p = 0; (p + 1) * large + unit + large <= bytes; p++) most = std::max(most, parts[p]);
      printf("pieces %zu %zu %zu %d\n", bytes, upto, beyond, bytes < 4 * unit ? 1 : most);
    }
  }
  // more than the buffer holds, through its two halves, behind what stays there:
  // chunk q's bytes packed, sent and taken over by whoever closes it
  for (size_t half : {(size_t)300000, (size_t)2 * SMALL, unit + 70000}) {
    const size_t stay = 1000, all = 11 * half - 12345;
    std::vector<unsigned char> src(all), dst(all), host(stay + 2 * half), dev(host.size());
    for (size_t b = 0; b < all; b++) src[b] = (unsigned char)(b * 2654435761u >> 13);
    std::vector<Range> chunks;
    for (size_t q = 0; q * half < all; q++) {
      const size_t at = stay + (q & 1) * half;
      chunks.push_back({q ? at : 0, at + std::min(half, all - q * half)});
    }
    std::atomic<size_t> closed[2] = {{0}, {0}}, begun(0), early(0);
    chunks_on_threads(
        chunks, [] { return true; },
        [&](size_t q) {
          if (q > 1)
            while (closed[q & 1] < q / 2) std::this_thread::yield();
          begun++;
        },
        [&](size_t q, size_t b0, size_t b1) {
          const size_t at = stay + (q & 1) * half, b = std::max(b0, at);
          if (b < b1) std::copy(src.begin() + q * half + (b - at), src.begin() + q * half + (b1 - at), host.begin() + b);
        },
        [&](size_t b0, size_t b1) { std::copy(host.begin() + b0, host.begin() + b1, dev.begin() + b0); },
        [&](size_t q) {
          early += closed[q & 1] != q / 2;
          const size_t at = stay + (q & 1) * half;
          std::copy(dev.begin() + at, dev.begin() + chunks[q].end, dst.begin() + q * half);
          closed[q & 1]++;
        });
    printf("chunks %zu %zu %zu %d\n", chunks.size(), closed[0] + closed[1], (size_t)early, (int)(src == dst));
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
