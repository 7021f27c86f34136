// The bounds of the device walk's 32-bit counts (csrc/fmm_host.hpp): whatever a
// round of n pairs splits into (up to 64 each), a count that an int cannot hold
// is added up in 64 bits and refused; rounds in all keep to 2^30 pairs.
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <initializer_list>

#include "fmm_host.hpp"

int main() {
  int bad = 0;
  for (int64_t n : {(int64_t)1, (int64_t)27, (int64_t)33554431, (int64_t)33554432, (int64_t)67108864, (int64_t)67108865,
                    (int64_t)70000001, (int64_t)536870912, fmm::kVisitMaxPairs})
    for (int64_t children : {(int64_t)0, n, 8 * n, 63 * n, 64 * n, ((int64_t)1 << 31) - 1, (int64_t)1 << 31,
                             ((int64_t)1 << 32) + 1, ((int64_t)1 << 33) + 4096}) {
      if (children > 64 * n) continue;
      const int32_t sum = (int32_t)(uint32_t)children;  // as the scan gives it
      const int64_t seen = fmm::visit_sum_wraps(n) ? children : sum;
      bad += seen != children;
      const bool takes = fmm::visit_fits(n, seen);
      bad += takes != (n + children <= ((int64_t)1 << 30));
    }
  std::puts(bad ? "bad" : "ok");
  return bad != 0;
}
