// fmm_p2m_lanes.hpp -- how p2m_kernel<P, S> deals the 64 lanes of a wavefront:
// H lanes a group (each two columns of the harmonics), S groups a leaf (its
// bodies dealt to them), LW leaves a wavefront.  Where H S LW < 64 (every
// order but 2, 3, 4, 7, 8, 15 and 16) the lanes behind the last leaf hold
// none; `slot` wraps to 0 for them too, so what a lane does is decided by
// holds() and adds(), not by the slot alone.
#pragma once

namespace fmmdev {

template <int P, int S> struct P2MLanes {
  static constexpr int H = (P + 1) / 2, LW = 64 / (H * S);
  static constexpr int column(int lane) { return lane % H; }
  static constexpr int slot(int lane) { return lane / H % S; }
  static constexpr int leaf(int lane) { return lane / (H * S); }
  static constexpr bool holds(int lane) { return leaf(lane) < LW; }
  // adds up its leaf's groups: entry(t, lane, k), k = 0 .. S - 1, of rows of 64
  static constexpr bool adds(int lane) { return holds(lane) && slot(lane) == 0; }
  static constexpr int entry(int t, int lane, int k) { return t * 64 + lane + H * k; }
  // every such entry is its row's, and one of the lane's own leaf and column
  static constexpr bool sound() {
    if (LW < 1) return false;
    for (int lane = 0; lane < 64; lane++)
      for (int k = 0; adds(lane) && k < S; k++) {
        const int from = entry(0, lane, k);
        if (from >= 64 || leaf(from) != leaf(lane) || column(from) != column(lane) || slot(from) != k) return false;
      }
    return true;
  }
};

}  // namespace fmmdev
