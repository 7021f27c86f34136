// Work items of a forest's M2L tiles (csrc/fmm_host.cpp, merge_plans): as long
// as all the slices together allow, whatever the parts' own items; every slice
// is in one item, and a tile of one item is stored, not added.
#include <cstdio>
#include <map>

#include "fmm_host.hpp"

int main() {
  fmm::set_host_threads(1);
  const int k = 32, n = 3000;
  std::vector<fmm::Tree> t(k);
  std::vector<fmm::Lists> l(k);
  std::vector<fmm::M2LGroups> g(k);
  std::vector<fmm::M2LTiles> tl(k);
  std::vector<fmm::PlanPart> parts;
  size_t slices = 0;
  for (int i = 0; i < k; i++) {
    std::vector<double> x(3 * n), q(n);
    fmm::make_bodies(n, "cube", i, x.data(), q.data());
    double a[3], b[3];
    const double zero[3] = {0, 0, 0};
    fmm::get_bounds(n, x.data(), a, b);
    t[i] = fmm::build_tree(n, x.data(), 32, a, b);
    l[i] = fmm::build_lists(t[i], 0.4, 5000, zero, 0, zero);
    g[i] = fmm::build_m2l_groups(t[i], l[i], 512, false, nullptr);
    tl[i] = fmm::build_m2l_tiles(t[i], g[i], 16, 4, 0);
    slices += tl[i].slice.size() / 4;
    parts.push_back({&t[i], &l[i], &g[i], &tl[i]});
  }
  fmm::Tree T;
  fmm::Lists L;
  fmm::M2LGroups G;
  fmm::M2LTiles X;
  fmm::merge_plans(parts, T, L, &G, 512, &X);
  int bad = X.slice.size() / 4 != slices || slices < 64 * 1700;  // enough for the longest items
  std::vector<int> seen(slices, 0);
  std::map<int, int> items;
  for (size_t i = 0; i < X.item.size(); i += 4) {
    if (X.item[i + 2] > X.item[i + 1]) items[X.item[i]]++;
    for (int s = X.item[i + 1]; s < X.item[i + 2]; s++) {
      seen[s]++;
      bad += s < X.ptr[X.item[i]] || s >= X.ptr[X.item[i] + 1];
    }
  }
  for (int v : seen) bad += v != 1;
  for (size_t i = 0; i < X.item.size(); i += 4)
    if (X.item[i + 2] > X.item[i + 1]) bad += X.item[i + 3] != (items[X.item[i]] > 1);
  for (int b = 0; b < X.ntile; b++) bad += items[b] > (X.ptr[b + 1] - X.ptr[b] + 63) / 64;
  std::printf("%zu slices, %d tiles, %zu items: %s\n", slices, X.ntile, X.item.size() / 4, bad ? "bad" : "ok");
  return bad != 0;
}
