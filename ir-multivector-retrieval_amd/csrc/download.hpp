// download.hpp — the staged device-to-host copy of large outputs, over a port
// that stands for the device: the library's is HipDownload (tac_gpu.hip), the
// CPU check's a buffer in memory.  Plain C++.
//
// The port offers, with 0 or an error as every int result:
//   bool known(dst)                 dst is no pageable memory: the direct copy is DMA
//   bool ring()                     the ring of pinned buffers can be had
//   const char *buffer(b)           buffer b of the ring, kDownChunk bytes
//   int fetch(b, off, len)          enqueues bytes [off, off + len) into buffer b
//   int wait(b)                     until buffer b's last fetch is done
//   int attach()                    once in every thread, before its first wait
//   bool skip()                     after a wait: the output is to be left alone
//   int drain()                     until every fetch is done
//   int direct(dst, bytes)          the whole copy without ring or threads
//   std::thread spawn(f)            may throw, as std::thread does
#pragma once

#include <stddef.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <exception>
#include <thread>

namespace tacgpu {

constexpr int kDownThreads = 8;
constexpr int kDownBufs = 4;
constexpr size_t kDownChunk = 4u << 20;  // most bytes per staged copy
// Smaller outputs take the direct copy.  Decode, us a call, direct | staged: 2 MB
// 169 | 243, 3 MB 227 | 262, 4 MB 288 | 291, 5 MB 350 | 303-329, 6 MB 410 | 330,
// 8 MB 540 | 397.
constexpr size_t kDownMin = 5u << 20;

// Copies `bytes` to dst; returns when dst is written.  Large copies to pageable
// memory pass in chunks through the ring: kDownThreads host threads each write
// their share of every chunk to dst (and take its page faults, when dst is
// fresh memory) while the DMA fetches the next ones.  A chunk costs some 15 us
// beside its bytes, so there are at least four of at most 4 MB.  Decode of
// 65,537 rows to 16.8 MB: 620 us a call, 715 with chunks of 1 MB, 1,040 with
// the direct copy, which one thread empties.  Where no ring or not every
// thread is to be had, the direct copy serves, and to pinned memory it is the
// faster one (16 MB 415 us a call, 600 through the ring; 64 MB 1,410, 1,830).
template <class Port>
int download(Port &port, void *dst, size_t bytes) {
  if (bytes < kDownMin || port.known(dst) || !port.ring()) return port.direct(dst, bytes);
  constexpr int T = kDownThreads;
  constexpr size_t B = kDownBufs;
  const size_t chunk = std::min(kDownChunk, (bytes / B + 65535) / 65536 * 65536);
  const size_t nch = (bytes + chunk - 1) / chunk;
  auto fetch = [&](size_t c) {  // chunk c into buffer c % B
    return port.fetch(c % B, c * chunk, std::min(bytes - c * chunk, chunk));
  };
  int first = 0;
  size_t ahead = 0;
  for (; ahead < std::min(nch, B) && !first; ++ahead) first = fetch(ahead);
  if (first) {
    port.drain();
    return first;
  }
  std::atomic<size_t> issued{ahead};  // chunks that are fetched or under way
  std::atomic<int> left[kDownBufs];   // threads yet to empty a buffer
  for (auto &l : left) l = T;
  std::atomic<int> failed{0};
  std::atomic<bool> stop{false};
  auto work = [&](int tid) {
    int e = port.attach();
    for (size_t c = 0; c < nch && !e; ++c) {
      while (issued.load(std::memory_order_acquire) <= c) {
        if (failed.load(std::memory_order_acquire) || stop.load(std::memory_order_acquire)) return;
        std::this_thread::yield();
      }
      if ((e = port.wait(c % B))) break;
      if (port.skip()) return;
      const size_t off = c * chunk, len = std::min(bytes - off, chunk);
      // shares of whole pages
      const size_t share = (len / T + 4095) / 4096 * 4096;
      const size_t lo = std::min(len, share * tid);
      const size_t hi = tid + 1 == T ? len : std::min(len, lo + share);
      memcpy(static_cast<char *>(dst) + off + lo, port.buffer(c % B) + lo, hi - lo);
      if (left[c % B].fetch_sub(1, std::memory_order_acq_rel) == 1 && c + B < nch) {
        // the last to leave the buffer refills it; buffers empty in order
        left[c % B].store(T, std::memory_order_release);
        if (!(e = fetch(c + B))) issued.fetch_add(1, std::memory_order_acq_rel);
      }
    }
    if (e) failed.store(e, std::memory_order_release);
  };
  std::thread helpers[T - 1];
  int made = 0;
  try {
    for (; made < T - 1; ++made) helpers[made] = port.spawn([&work, made] { work(made + 1); });
  } catch (const std::exception &) {
    // Without all of them no buffer is ever emptied: the others end at the
    // latest where they wait for a fifth chunk.
    stop.store(true, std::memory_order_release);
  }
  if (made == T - 1) work(0);
  for (int t = 0; t < made; ++t) helpers[t].join();
  const int drained = port.drain();  // no fetch outlives the call
  if (failed.load()) return failed.load();
  if (drained) return drained;
  return made == T - 1 ? 0 : port.direct(dst, bytes);
}

}  // namespace tacgpu
