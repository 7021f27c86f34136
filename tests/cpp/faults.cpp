// Failures forced from the host: this program's hipMalloc (it takes the place
// of the runtime's for the library too) passes on to the runtime's, or refuses
// as told.  Every kernel that is launched has its memory and ends.
#include <dlfcn.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <functional>
#include <string>
#include <vector>

#include <hip/hip_runtime.h>

#include "exafmm_amd.h"

namespace {
std::function<bool(size_t)> refuse;  // a request of this size
int refused = 0;
hipError_t refusal = hipErrorOutOfMemory;  // with this
}  // namespace

extern "C" hipError_t hipMalloc(void **p, size_t n) {
  static const auto real = reinterpret_cast<hipError_t (*)(void **, size_t)>(dlsym(RTLD_NEXT, "hipMalloc"));
  if (refuse && refuse(n)) {
    refused++;
    return refusal;
  }
  return real(p, n);
}

namespace {
int bad = 0;
#define EXPECT(x) (x) ? 0 : (bad++, std::printf("line %d: %s\n", __LINE__, #x))

struct System {
  std::vector<double> x, q;
  System(int n, const char *dist, int seed) : x(3 * (size_t)n), q(n) {
    fmm_make_bodies(n, dist, seed, x.data(), q.data());
  }
  int n() const { return (int)q.size(); }
};
fmm_ctx *context(int P, int images = 0) {
  fmm_params p;
  fmm_default_params(&p);
  p.P = P;
  p.images = images;
  fmm_ctx *c = nullptr;
  if (fmm_create(&c, &p) != FMM_OK) bad++;
  return c;
}
std::vector<double> solve(fmm_ctx *c, int n) {
  std::vector<double> t(4 * (size_t)n);
  EXPECT(fmm_evaluate(c) == FMM_OK);
  EXPECT(fmm_get_targets(c, t.data(), 1) == FMM_OK);
  return t;
}
double rel(const std::vector<double> &a, const std::vector<double> &b) {
  double d = 0, s = 0;
  for (size_t i = 0; i < a.size(); i++) {
    d += (a[i] - b[i]) * (a[i] - b[i]);
    s += b[i] * b[i];
  }
  return std::sqrt(d / s);
}

// the offset groups' table (2^20 keys) does not fit on the device: the host groups the pairs
void groups() {
  const System s(20000, "cube", 1);
  for (int images : {0, 2}) {
    fmm_ctx *c = context(8, images), *d = context(8, images);
    EXPECT(fmm_set_bodies(c, s.n(), s.x.data(), s.q.data()) == FMM_OK);
    refused = 0;
    refuse = [](size_t n) { return n == (size_t)8 << 20; };
    EXPECT(fmm_set_bodies(d, s.n(), s.x.data(), s.q.data()) == FMM_OK);
    refuse = nullptr;
    EXPECT(refused > 0);
    fmm_stats a, b;
    fmm_get_stats(c, &a);
    fmm_get_stats(d, &b);
    EXPECT(a.m2l_groups == b.m2l_groups && b.m2l_ungrouped == 0);
    const double e = rel(solve(d, s.n()), solve(c, s.n()));
    std::printf("images %d: %.1e\n", images, e);
    EXPECT(e < 1e-12);  // the same translations in another order
    fmm_destroy(c);
    fmm_destroy(d);
  }
}

// an allocation fails while the next system's tree, lists or groups are made:
// the context still has the system before, and takes the next one afterwards
void kept() {
  const System a(20000, "cube", 1), b(30000, "plummer", 2);
  for (bool device : {false, true}) {
    const auto set = [&](fmm_ctx *c, const System &s) {
      return (device ? fmm_set_bodies_device : fmm_set_bodies)(c, s.n(), s.x.data(), s.q.data());
    };
    int total = 0, at = 0;  // allocations of b's plan
    {
      fmm_ctx *c = context(8);
      EXPECT(set(c, a) == FMM_OK);
      refuse = [&](size_t) { return total++, false; };
      fmm_plan *p = nullptr;
      EXPECT(fmm_plan_build_device(c, &p, b.n(), b.x.data(), 64, 0.4, 5000) == FMM_OK);
      refuse = nullptr;
      fmm_plan_destroy(p);
      fmm_destroy(c);
    }
    EXPECT(total > 8);
    // fmm_set_bodies makes the lists alone there: its first allocations
    for (int k : device ? std::vector<int>{0, total / 4, total / 2, 3 * total / 4} : std::vector<int>{0, 1, 2}) {
      fmm_ctx *c = context(8), *d = context(8);
      EXPECT(set(c, a) == FMM_OK);
      const std::vector<double> ta = solve(c, a.n());
      refused = at = 0;
      refusal = hipErrorUnknown;  // no second try, nothing falls back
      refuse = [&](size_t) { return at++ == k; };
      const int rc = set(c, b);
      refuse = nullptr;
      refusal = hipErrorOutOfMemory;
      std::printf("%s, allocation %d of %d: %d, refused %d\n", device ? "device" : "host", k, total, rc, refused);
      EXPECT(refused == 1 && rc == FMM_ERR_DEVICE);
      EXPECT(rel(solve(c, a.n()), ta) < 1e-12);  // the order of the atomic additions
      EXPECT(set(c, b) == FMM_OK);
      EXPECT(set(d, b) == FMM_OK);
      EXPECT(rel(solve(c, b.n()), solve(d, b.n())) < 1e-12);
      fmm_destroy(c);
      fmm_destroy(d);
    }
  }
}
}  // namespace

int main(int argc, char **argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "groups") groups();
  else if (what == "kept") kept();
  else bad++;
  std::puts(bad ? "bad" : "ok");
  return bad != 0;
}
