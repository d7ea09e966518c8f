// A buffer that only grows (host code; builds without HIP).
#pragma once

#include <stddef.h>

namespace llmhip {

// Bytes to allocate for a request: the next power of two up to 8 MiB, the
// request itself above. A caller whose request grows a little from call to
// call (a generation's history) then reallocates once per doubling; exactly
// sized, one row of 32000 with a history of 1 to 512 ids took 65 us a call,
// half of it in hipHostFree and hipHostMalloc.
constexpr size_t kRoundedBytes = (size_t)8 << 20;
inline size_t grown_capacity(size_t bytes) {
  if (bytes > kRoundedBytes) return bytes;
  size_t cap = 256;
  while (cap < bytes) cap *= 2;
  return cap;
}

// Mem: static int alloc(void** p, size_t bytes) and static int free(void* p),
// 0 on success. A failed ensure leaves the buffer empty.
template <class Mem>
struct GrowBuf {
  void* ptr = nullptr;
  size_t cap = 0;
  int ensure(size_t bytes) {
    if (bytes <= cap) return 0;
    int st = release();
    if (st) return st;
    const size_t want = grown_capacity(bytes);
    if ((st = Mem::alloc(&ptr, want))) {
      ptr = nullptr;
      return st;
    }
    cap = want;
    return 0;
  }
  int release() {
    void* p = ptr;
    ptr = nullptr;
    cap = 0;
    return p ? Mem::free(p) : 0;
  }
};

}  // namespace llmhip
