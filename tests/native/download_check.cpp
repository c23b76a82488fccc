// CPU check of the staged device-to-host copy (csrc/download.hpp): every size at
// the edges of its chunks, with a thread that cannot be made (each of the
// seven), no ring, a pinned output, a fetch that fails and a raised skip word.  The device is a
// buffer in memory whose fetches run at once.
#include <cstdio>
#include <new>
#include <system_error>
#include <vector>

#include "../../ir-multivector-retrieval_amd/csrc/download.hpp"

using namespace tacgpu;

struct Port {
  const std::vector<char> &src;
  std::vector<char> mem = std::vector<char>(kDownBufs * kDownChunk);
  int spawn_limit = kDownThreads;  // threads that can be made
  bool no_memory = false;          // the one past them: bad_alloc, else system_error
  bool have_ring = true, pinned = false, raised = false;
  size_t fail_at = ~(size_t)0;  // offset whose fetch fails
  int directs = 0, made = 0;
  std::atomic<size_t> fetched{0};

  bool known(const void *) const { return pinned; }
  bool ring() { return have_ring; }
  const char *buffer(size_t b) const { return mem.data() + b * kDownChunk; }
  int fetch(size_t b, size_t off, size_t len) {
    if (off == fail_at) return 7;
    fetched += len;
    memcpy(mem.data() + b * kDownChunk, src.data() + off, len);
    return 0;
  }
  int wait(size_t) { return 0; }
  int attach() { return 0; }
  bool skip() const { return raised; }
  int drain() { return 0; }
  int direct(void *dst, size_t bytes) {
    ++directs;
    if (!raised) memcpy(dst, src.data(), bytes);
    return 0;
  }
  template <class F>
  std::thread spawn(F f) {
    if (made == spawn_limit) {
      if (no_memory) throw std::bad_alloc();
      throw std::system_error(std::make_error_code(std::errc::resource_unavailable_try_again));
    }
    ++made;
    return std::thread(f);
  }
};

static int bad = 0;
static void expect(bool ok, const char *what, size_t bytes, int arg) {
  if (!ok) {
    std::printf("WRONG %s: %zu bytes, %d\n", what, bytes, arg);
    ++bad;
  }
}

int main() {
  const size_t sizes[] = {1, kDownMin - 1, kDownMin, kDownMin + 1, kDownMin + 70000,
                          3 * kDownMin + 4097,
                          4 * kDownChunk, 4 * kDownChunk + 1, 9 * kDownChunk + 65537};
  for (size_t bytes : sizes) {
    std::vector<char> src(bytes);
    uint32_t x = (uint32_t)bytes;
    for (auto &c : src) c = (char)((x = x * 1664525u + 1013904223u) >> 24);
    const bool staged = bytes >= kDownMin;
    for (int limit = 0; limit <= kDownThreads - 1; ++limit)
      for (bool no_memory : {false, true}) {
        std::vector<char> dst(bytes, 1);
        Port p{src};
        p.spawn_limit = limit;
        p.no_memory = no_memory;
        expect(download(p, dst.data(), bytes) == 0 && dst == src, "threads", bytes, limit);
        const bool whole = staged && limit == kDownThreads - 1;
        expect(p.directs == (whole ? 0 : 1), "copies", bytes, limit);
        if (whole) expect(p.fetched == bytes, "fetched", bytes, limit);
      }
    std::vector<char> dst(bytes, 1);
    Port none{src};
    none.have_ring = false;
    expect(download(none, dst.data(), bytes) == 0 && dst == src && none.made == 0, "no ring", bytes, 0);
    Port pinned{src};
    pinned.pinned = true;
    std::fill(dst.begin(), dst.end(), 1);
    expect(download(pinned, dst.data(), bytes) == 0 && dst == src, "pinned", bytes, 0);
    expect(pinned.directs == 1 && pinned.made == 0, "pinned copies", bytes, 0);
    for (size_t c = 0; staged && c < 9; ++c) {
      const size_t chunk = std::min(kDownChunk, (bytes / kDownBufs + 65535) / 65536 * 65536);
      if (c * chunk >= bytes) break;
      Port f{src};
      f.fail_at = c * chunk;
      expect(download(f, dst.data(), bytes) == 7, "failing fetch", bytes, (int)c);
    }
    for (int limit : {0, 3, kDownThreads - 1}) {
      std::vector<char> keep(bytes, 9);
      Port s{src};
      s.raised = true;
      s.spawn_limit = limit;
      expect(download(s, keep.data(), bytes) == 0 && keep == std::vector<char>(bytes, 9), "skip", bytes,
             limit);
    }
  }
  std::printf("%d wrong\n%s\n", bad, bad ? "download check FAILED" : "download check passed");
  return bad ? 1 : 0;
}
