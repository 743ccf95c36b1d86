// device_buffer_check.cpp -- KeptBuf (adaptq_amd/csrc/device_buffer.hpp) over a
// hipMalloc and a hipFree that only keep books: prints "ok", or the first line
// that does not hold.
#include "../../adaptq_amd/csrc/device_buffer.hpp"

#include <cstdint>
#include <cstdio>
#include <map>

namespace {
std::map<uintptr_t, size_t> live;
size_t limit = SIZE_MAX, held = 0;
uintptr_t next_at = 4096;
int mallocs = 0, other = 0;
}  // namespace

extern "C" hipError_t hipMalloc(void **p, size_t n) {
  ++mallocs;
  if (other) return hipErrorStreamCaptureUnsupported;
  if (n > limit - held) return hipErrorOutOfMemory;
  *p = reinterpret_cast<void *>(next_at);
  live[next_at] = n;
  held += n;
  next_at += n;
  return hipSuccess;
}
extern "C" hipError_t hipFree(void *p) {
  const auto it = live.find(reinterpret_cast<uintptr_t>(p));
  if (it == live.end()) return hipErrorInvalidValue;
  held -= it->second;
  live.erase(it);
  return hipSuccess;
}
extern "C" hipError_t hipGetLastError() { return hipSuccess; }

#define CHECK(x)                                      \
  do {                                                \
    if (!(x)) {                                       \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x); \
      return 1;                                       \
    }                                                 \
  } while (0)

int main() {
  auto alive = [](void *p) { return live.count(reinterpret_cast<uintptr_t>(p)) == 1; };
  // sizes below, across and above 8 MiB, up and down: the split partials of 64
  // queries of 8 heads d128 at 8,300 and 8,192 tokens among them
  const size_t sizes[] = {1, 5000, 3 << 20, 7 << 20, 9 << 20, 15679488, 17301504,
                          4096, 17301505, 100 << 20, 60 << 20, 101 << 20};
  aq::KeptBuf b;
  std::map<void *, size_t> handed;  // address -> bytes a caller may still use there
  size_t most = 0;
  for (const size_t n : sizes) {
    CHECK(b.ensure(n) == hipSuccess);
    most = n > most ? n : most;
    CHECK(b.p && b.bytes >= n);
    handed[b.p] = b.bytes;
    for (const auto &h : handed) CHECK(alive(h.first));
    CHECK(held < 4 * most + 8192);  // the kept ones less than the one in use, that at most twice
  }
  const int before = mallocs;
  for (const size_t n : sizes) CHECK(b.ensure(n) == hipSuccess);  // all there already
  CHECK(mallocs == before);

  // twice as much is not there, as much as needed is
  void *old = b.p;
  const size_t had = b.bytes, need = had + 1000;
  limit = held + need;
  CHECK(b.ensure(need) == hipSuccess && b.bytes == need && alive(old) && b.p != old);
  // not even that: the buffer in hand stays as it is
  old = b.p;
  CHECK(b.ensure(2 * need) == hipErrorOutOfMemory);
  CHECK(b.p == old && b.bytes == need && alive(old));
  // another failure is not tried again
  limit = SIZE_MAX;
  other = 1;
  const int tries = mallocs;
  CHECK(b.ensure(2 * need) == hipErrorStreamCaptureUnsupported && mallocs == tries + 1);
  CHECK(b.p == old && b.bytes == need);
  other = 0;
  b.release();
  CHECK(live.empty() && held == 0 && !b.p && b.bytes == 0);
  CHECK(b.ensure(10) == hipSuccess && live.size() == 1);
  b.release();
  CHECK(live.empty());
  std::printf("ok\n");
  return 0;
}
