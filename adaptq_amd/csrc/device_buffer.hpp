// device_buffer.hpp -- device memory that grows with the calls that use it.
#pragma once

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <new>
#include <vector>

namespace aq {

// Memory that only one call at a time uses and whose address no graph holds.
struct DevBuf {
  void *p = nullptr;
  size_t bytes = 0;
  hipError_t ensure(size_t need) {
    if (need <= bytes) return hipSuccess;
    if (p) (void)hipFree(p);  // hipFree waits for the device: no kernel still uses it
    p = nullptr;
    bytes = 0;
    size_t want = std::max(need, (size_t)4096);
    hipError_t e = hipMalloc(&p, want);
    if (e == hipSuccess) bytes = want;
    return e;
  }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
  }
};

// Memory whose address a captured graph may hold: workspaces, copies of a
// call's rows and descriptor lists of the calls on a caller's stream.  Any later
// call may need more of it (more queries, other rings: split counts are not
// monotone in the ring's length, 64 queries of 8 heads d128 K4/V4 take 15.7 MB
// at 8,300 tokens and 17.3 MB at 8,192), and the graph's replays still use the
// old address.  So a buffer that is grown out of stays until release; each is at
// least twice the one before, so that the kept ones together are smaller than
// the one in use.  Where twice as much is not there, as much as is needed is
// taken; where that is not there either, ensure fails and nothing is lost.
struct KeptBuf {
  void *p = nullptr;
  size_t bytes = 0;
  hipError_t ensure(size_t need) {
    if (need <= bytes) return hipSuccess;
    if (p) {  // a place for the old address before the new one is taken
      try {
        kept.reserve(kept.size() + 1);
      } catch (const std::bad_alloc &) {
        return hipErrorOutOfMemory;
      }
    }
    size_t want = std::max({need, 2 * bytes, (size_t)4096});
    void *bigger = nullptr;
    hipError_t e = hipMalloc(&bigger, want);
    if (e == hipErrorOutOfMemory && need < want) {
      (void)hipGetLastError();  // (the failure is not the caller's next error)
      want = need;
      e = hipMalloc(&bigger, want);
    }
    if (e != hipSuccess) return e;
    if (p) kept.push_back(p);
    p = bigger;
    bytes = want;
    return hipSuccess;
  }
  void release() {
    if (p) (void)hipFree(p);
    for (void *q : kept) (void)hipFree(q);
    kept.clear();
    p = nullptr;
    bytes = 0;
  }

 private:
  std::vector<void *> kept;
};

}  // namespace aq
