// Out of device memory, on a made-up device: this program's hipMalloc and
// hipFree (they take the place of the runtime's for the library too) hand out
// host memory within a budget.  A plan's arrays (fmmdev::DevArray) get the
// room that the builders' cached scratch holds, of their own and of other
// streams, and an exact fit where the spare quarter does not fit.
#include <cstdio>
#include <cstdlib>
#include <map>

#include "fmm_device.hpp"

namespace {
size_t budget = 0, used = 0;
std::map<void *, size_t> live;
}  // namespace

extern "C" hipError_t hipMalloc(void **p, size_t n) {
  if (used + n > budget) return hipErrorOutOfMemory;
  *p = std::malloc(n);
  live[*p] = n;
  used += n;
  return hipSuccess;
}
extern "C" hipError_t hipFree(void *p) {
  if (p) {
    used -= live.at(p);
    live.erase(p);
    std::free(p);
  }
  return hipSuccess;
}
extern "C" hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
extern "C" hipError_t hipGetLastError() { return hipSuccess; }
extern "C" hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
extern "C" hipError_t hipSetDevice(int) { return hipSuccess; }

int bad = 0;
#define EXPECT(x) (x) ? 0 : (bad++, std::printf("line %d: %s\n", __LINE__, #x))

int main() {
  constexpr size_t kMB = (size_t)1 << 20;
  hipStream_t st = reinterpret_cast<hipStream_t>(1), other = reinterpret_cast<hipStream_t>(2);
  budget = 100 * kMB;
  for (hipStream_t s : {st, other}) {
    void *p;
    size_t cap;
    EXPECT(fmmdev::plan_scratch_get(&p, &cap, 40 * kMB, s) == hipSuccess);
    fmmdev::plan_scratch_put(p, cap, s);  // idle
  }
  EXPECT(used == 80 * kMB);
  fmmdev::DevArray a;
  EXPECT(a.alloc(70 * kMB, 0) == hipSuccess && a.p && a.bytes == 70 * kMB);
  EXPECT(a.alloc(90 * kMB, 0) == hipSuccess && a.p && a.cap == 90 * kMB);  // 112 do not fit
  void *q = a.p;
  EXPECT(a.alloc(10 * kMB, 0) == hipSuccess && a.p == q && a.bytes == 10 * kMB);
  EXPECT(a.alloc(101 * kMB, 0) == hipErrorOutOfMemory && !a.p && a.bytes == 0 && a.cap == 0 && used == 0);
  EXPECT(a.alloc(100 * kMB, 0) == hipSuccess);
  void *p;
  size_t cap;
  EXPECT(fmmdev::plan_scratch_get(&p, &cap, kMB, st) == hipErrorOutOfMemory && !p && cap == 0);
  a.reset();
  EXPECT(used == 0);
  std::puts(bad ? "bad" : "ok");
  return bad != 0;
}
