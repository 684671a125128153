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

// The size of a buffer that `need` bytes ask for: at least 256 KiB, so that a
// small context pins once for what it sends and reads (its forcing's inputs, then
// the first read-back with the soil: 77 tiles 0.2 ms against 0.25 to 0.55, 1,000
// in FP64 0.36 against 0.43).  Not more: pinning 1 MiB takes 0.05 to 0.1 ms longer,
// which a context that needs less pays, and a buffer given back for a larger
// one as much again.
constexpr size_t capacity(size_t need) { return std::max(need, (size_t)256 << 10); }

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

// Pieces of 512 KiB share a few MiB out to all threads.  From the size on that
// gives each thread 2 MiB, pieces of 2 MiB, but for the end, where small ones
// let the threads finish together: there the caller's arrays are large enough
// for huge pages of 2 MiB, and where they or the buffer have not been touched
// before, threads with pieces of one page between them waited for each
// other's page faults.  Every field of 49,149 tiles (113 MB) down to new arrays
// 70 ms in pieces of 512 KiB, 40 in these (56 with a field to a thread), and
// up from new arrays 13 and 8 ms; of 8,000 tiles down 7.0 and 4.4 ms.  On touched
// pages the same (2.9 and 0.75 ms down).
constexpr size_t SMALL = 512 << 10, LARGE = 2 << 20;
static_assert(UNIT % LARGE == 0 && LARGE % SMALL == 0, "a piece lies within a unit");
struct Pieces {
  size_t bytes, large;  // the first `large` pieces are LARGE
  explicit constexpr Pieces(size_t n) : bytes(n), large(n < THREADS * LARGE ? 0 : (n - UNIT) / LARGE) {}
  constexpr size_t begin(size_t q) const {
    return q < large ? q * LARGE : std::min(bytes, large * LARGE + (q - large) * SMALL);
  }
  constexpr size_t count() const { return large + (bytes - large * LARGE + SMALL - 1) / SMALL; }
};

// f(q) for every q below `count`, claimed in order by the threads that `bytes` of
// work ask for; init() on each thread that is started, which claims none if it
// is false
template <class Init, class F>
void share_out(size_t bytes, size_t count, Init &&init, F &&f) {
  std::atomic<size_t> next(0);
  auto run = [&]() {
    for (size_t q; (q = next.fetch_add(1)) < count;) f(q);
  };
  const unsigned nt = (unsigned)std::min<size_t>(
      {THREADS, count, bytes / PER_THREAD + 1, std::max(1u, std::thread::hardware_concurrency())});
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

// f(b0, b1) for every piece [b0, b1) of `bytes`
template <class Init, class F>
void on_threads(size_t bytes, Init &&init, F &&f) {
  const Pieces p(bytes);
  share_out(bytes, p.count(), init, [&](size_t q) { f(p.begin(q), p.begin(q + 1)); });
}

// Chunks of a buffer that is smaller than what goes through it: chunk q is packed
// when release(q) has returned, sent unit by unit when its parts are packed and
// closed by the thread that sent its last unit.  Chunks are begun in order, so
// that release(q) may wait for the closing of an earlier one.
struct Range {
  size_t from, end;
};
template <class Init, class Release, class Fill, class Send, class Close>
void chunks_on_threads(const std::vector<Range> &chunks, Init &&init, Release &&release, Fill &&fill, Send &&send,
                       Close &&close) {
  struct Part {
    size_t chunk, b0, b1, unit, of;  // bytes [b0, b1) of unit `unit`, of which there are `of`
  };
  std::vector<Part> parts;
  size_t units = 0, total = 0;
  for (size_t q = 0; q < chunks.size(); q++) {
    const size_t bytes = chunks[q].end - chunks[q].from;
    const Pieces p(bytes);
    for (size_t k = 0; k < p.count(); k++) {
      const size_t b0 = p.begin(k), u0 = b0 / UNIT * UNIT;
      parts.push_back({q, b0, p.begin(k + 1), units + b0 / UNIT, std::min(bytes, u0 + UNIT) - u0});
    }
    units += (bytes + UNIT - 1) / UNIT;
    total += bytes;
  }
  std::vector<std::atomic<size_t>> packed(units), sent(chunks.size());
  for (auto &x : packed) x = 0;
  for (auto &x : sent) x = 0;
  share_out(total, parts.size(), init, [&](size_t k) {
    const Part &t = parts[k];
    const Range &r = chunks[t.chunk];
    release(t.chunk);
    fill(t.chunk, r.from + t.b0, r.from + t.b1);
    if (packed[t.unit].fetch_add(t.b1 - t.b0) + (t.b1 - t.b0) != t.of) return;
    const size_t u0 = r.from + t.b0 / UNIT * UNIT;
    send(u0, u0 + t.of);
    if (sent[t.chunk].fetch_add(t.of) + t.of == r.end - r.from) close(t.chunk);
  });
}

}  // namespace staging
