// The lanes of p2m_kernel (csrc/fmm_p2m_lanes.hpp), walked on the host: every
// entry that a lane reads when a leaf's groups are added lies in the step's
// row of the buffer (64 (P + 1) entries) and was written by a lane of the same
// leaf and column, each group once; every leaf of a wavefront is added by one
// lane a column; lanes that hold no leaf read nothing.
#include <cstdio>
#include <set>
#include <utility>

#include "fmm_p2m_lanes.hpp"

template <int P, int S> int check() {
  using Ln = fmmdev::P2MLanes<P, S>;
  int bad = 0;
  std::set<std::pair<int, int>> sums;  // (leaf, column)
  for (int lane = 0; lane < 64; lane++) {
    if (!Ln::adds(lane)) continue;
    bad += !Ln::holds(lane);
    bad += !sums.insert({Ln::leaf(lane), Ln::column(lane)}).second;
    for (int t = 0; t <= P; t++)
      for (int k = 0; k < S; k++) {
        const int e = Ln::entry(t, lane, k), from = e - 64 * t;
        bad += e >= 64 * (P + 1) || from < 0 || from >= 64 || Ln::leaf(from) != Ln::leaf(lane) ||
               Ln::column(from) != Ln::column(lane) || Ln::slot(from) != k;
      }
  }
  bad += Ln::LW < 1 || (int)sums.size() != Ln::LW * Ln::H;
  if (bad) std::printf("P = %d, S = %d: %d\n", P, S, bad);
  return bad;
}
template <int P> int orders() {
  int bad = check<P, 64 / ((P + 1) / 2)>() + check<P, 2>();  // the two forms that run
  if constexpr (P < 20) bad += orders<P + 1>();
  return bad;
}
int main() {
  const int bad = orders<2>();
  if (!bad) std::puts("ok");
  return bad != 0;
}
