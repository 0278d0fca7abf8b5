// Rows of a tree's tiles (tree.hpp): the uniform tree's fullest tile, and the mean over the
// walked sources on an irregular tree of a lat-lon grid's points, which follows the leaves'
// points and not the proxies alone.
#include <cmath>
#include <cstdio>

#include "irreg_tree.hpp"

using namespace sbslpm;

int main() {
  Tree u;
  if (!build_tree(TreeConfig{4, 8, 5, 0.7, 1}, u).empty()) return 1;
  if (fullest_tile(u.tiles) != 41) return 2;  // 81 proxies in tiles of 41 and 40, 36 points
  if (fullest_tile({}) != 0 || mean_tile({}, {}) != 0) return 3;
  std::vector<double> x, y, z;
  const int rows = 60;
  for (int i = 0; i < rows; ++i)
    for (int j = 0; j < 2 * rows; ++j) {
      const double la = M_PI * ((i + 0.5) / rows - 0.5), lo = M_PI * (j + 0.5) / rows;
      x.push_back(std::cos(la) * std::cos(lo));
      y.push_back(std::cos(la) * std::sin(lo));
      z.push_back(std::sin(la));
    }
  const int degree[2] = {4, 8}, leaf[2] = {64, 324};
  for (int k = 0; k < 2; ++k) {
    IrregTree t;
    if (!build_irreg_tree(x.data(), y.data(), z.data(), (int64_t)x.size(), leaf[k], degree[k], 0.7, t).empty()) return 4;
    double w = 0, r = 0;
    for (const TargetTile& tl : t.tiles) {
      double s = 0;
      for (int e = tl.src_begin; e < tl.src_end; ++e) s += t.sets[e].count;
      w += s;
      r += s * tl.count;
    }
    const int m = mean_tile(t.tiles, t.sets);
    std::printf("degree %d, %d points a leaf: %d rows of at most %d\n", degree[k], leaf[k], m, fullest_tile(t.tiles));
    if (std::fabs(m - r / w) > 1 || (k == 0) != (m <= 42)) return 5;
  }
  return 0;
}
