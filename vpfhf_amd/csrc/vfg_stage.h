// vfg_stage.h -- small host-to-device uploads gathered into one launch (internal).
//
// A work-list update is a dozen arrays of a few hundred bytes; a copy of each
// costs about 10 us of the stream.  Here their contents go to pinned memory at
// once (the sources may change or go away) and one kernel writes them to their
// places, in stream order.  The pinned bytes of a flush are in use until its
// kernel has run: idle() reuses them, after the owner has synchronised the
// stream.
#pragma once
#include <hip/hip_runtime.h>
#include <string.h>
#include <vector>

namespace vfg {

struct StageSeg {
  void *dst;
  const void *src;  // pinned
  size_t bytes;     // a multiple of 4
};
void launch_stage(const StageSeg *seg, int n, size_t max_bytes, hipStream_t s);

struct Stage {
  char *h = nullptr;
  size_t cap = 0, used = 0, max_bytes = 0;
  std::vector<StageSeg> segs;
  Stage() = default;
  Stage(const Stage &) = delete;
  Stage &operator=(const Stage &) = delete;
  ~Stage() {
    if (h) hipHostFree(h);
  }
  void idle() {
    if (segs.empty()) used = 0;
  }
  bool room(size_t bytes, hipStream_t s) {
    if (used + bytes <= cap) return true;
    if (!flush(s) || hipStreamSynchronize(s) != hipSuccess) return false;
    used = 0;
    if (bytes <= cap) return true;
    if (h) hipHostFree(h);
    cap = 0;
    h = nullptr;
    size_t c = (size_t)1 << 18;
    while (c < bytes) c *= 2;
    if (hipHostMalloc((void **)&h, c, hipHostMallocDefault) != hipSuccess) {
      h = nullptr;
      return false;
    }
    cap = c;
    return true;
  }
  static size_t up(size_t b) { return (b + 15) / 16 * 16; }
  bool put(void *dst, const void *src, size_t bytes, hipStream_t s) {
    if (!bytes) return true;
    // room for the table entry too, so that a flush always has it
    if (!room(up(bytes) + (segs.size() + 1) * sizeof(StageSeg) + 16, s)) return false;
    memcpy(h + used, src, bytes);
    segs.push_back({dst, h + used, bytes});
    used += up(bytes);
    if (bytes > max_bytes) max_bytes = bytes;
    return true;
  }
  bool flush(hipStream_t s) {
    if (segs.empty()) return true;
    const size_t tb = segs.size() * sizeof(StageSeg);
    memcpy(h + used, segs.data(), tb);
    launch_stage((const StageSeg *)(h + used), (int)segs.size(), max_bytes, s);
    used += up(tb);
    if (used > cap) used = cap;
    segs.clear();
    max_bytes = 0;
    return hipGetLastError() == hipSuccess;
  }
};

}  // namespace vfg
