// staging.h -- the host side of the batched transfers' staging buffer: its
// layout, its size, and how the host's threads share its packing.  Host code
// without HIP, so that the test suite can run it by itself.
#pragma once
#include <stddef.h>

#include <algorithm>
#include <atomic>
#include <thread>
#include <vector>

#include "../../include/cable_fields.h"

namespace staging {

// One entry per field of a batched transfer: the field's device array, its
// offset in the staging buffer, its rows of mp values and a value's bytes.
struct Entry {
  void *dev;
  unsigned long long off;
  int rows, bytes;
};
// Every array in the buffer starts at a multiple of ALIGN, the first behind the
// table of entries: the transfer kernel moves 16 bytes at a time.
constexpr size_t ALIGN = 256;
constexpr size_t align_up(size_t n) { return (n + ALIGN - 1) / ALIGN * ALIGN; }
constexpr size_t TABLE_BYTES = align_up(sizeof(Entry) * CABLE_NFIELDS);
static_assert(TABLE_BYTES % ALIGN == 0 && ALIGN % 16 == 0, "the kernel's 16-byte accesses");

// The buffer is packed (unpacked) in pieces on up to eight threads, one per
// PER_THREAD bytes (starting one costs as much as it saves below: 11 fields of
// 8,000 tiles down, 0.7 MB, 67 us with one thread, 76 with three), and copied
// in units, each when its pieces are packed or before they are unpacked, so
// that the copies and the host's work overlap: every field of 49,149 tiles up
// in 3.9 ms (152 MB; 4.9 packed first), down in 2.9 ms (3.6).  Units of 1 and
// 2 MiB were slower (4.7 and 4.1 ms up), of 8 MiB faster for this and slower
// for small batches.
constexpr size_t PER_THREAD = 1 << 20, UNIT = 4 << 20;
constexpr unsigned THREADS = 8;

// f(piece) for every piece of `bytes`; init() on each thread that is started,
// which takes no piece if it is false
template <class Init, class F>
void on_threads(size_t bytes, size_t piece, Init &&init, F &&f) {
  const size_t pieces = (bytes + piece - 1) / piece;
  std::atomic<size_t> next(0);
  auto run = [&]() {
    for (size_t q; (q = next.fetch_add(1)) < pieces;) f(q);
  };
  const unsigned nt = (unsigned)std::min<size_t>(
      {THREADS, pieces, bytes / PER_THREAD + 1, std::max(1u, std::thread::hardware_concurrency())});
  std::vector<std::thread> th;
  for (unsigned t = 1; t < nt; t++) {
    try {
      th.emplace_back([&]() {
        if (init()) run();
      });
    } catch (...) {  // no more threads: those there do the work
      break;
    }
  }
  run();
  for (auto &t : th) t.join();
}

}  // namespace staging
