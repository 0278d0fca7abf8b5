// Tile lists of the uniform tree: every order holds the same tiles; lists shorter
// than kBalancedTiles run from the most pairs per lane to the fewest, longer ones
// stay in breadth-first panel order.
#include <algorithm>
#include <cstdio>
#include <cmath>
#include <cstdlib>

#include "tree.hpp"

using namespace sbslpm;

static long cost(const TargetTile& t, const std::vector<SourceSet>& sets) {
  long w = 0;
  for (int e = t.src_begin; e < t.src_end; ++e) w += sets[e].count + 16;
  return w;
}

static int check(const std::vector<TargetTile>& tiles, std::vector<TargetTile> bfs, const std::vector<SourceSet>& sets) {
  auto same = [](const TargetTile& a, const TargetTile& b) {
    return a.panel == b.panel && a.first == b.first && a.count == b.count && a.src_begin == b.src_begin &&
           a.src_end == b.src_end;
  };
  if (tiles.size() != bfs.size()) return 1;
  const bool sorted = (int)tiles.size() < kBalancedTiles;
  for (size_t k = 1; k < tiles.size(); ++k) {
    if (bfs[k].panel < bfs[k - 1].panel) return 2;
    if (sorted && cost(tiles[k], sets) > cost(tiles[k - 1], sets)) return 3;
  }
  if (!sorted) return std::equal(tiles.begin(), tiles.end(), bfs.begin(), same) ? 0 : 4;
  auto t2 = tiles;
  auto by_first = [](const TargetTile& a, const TargetTile& b) { return a.first < b.first; };
  std::sort(t2.begin(), t2.end(), by_first);
  std::sort(bfs.begin(), bfs.end(), by_first);
  return std::equal(t2.begin(), t2.end(), bfs.begin(), same) ? 0 : 5;
}

int main(int argc, char** argv) {
  if (argc < 5) return 100;
  Tree t;
  const TreeConfig cfg{std::atoi(argv[1]), std::atoi(argv[2]), std::atoi(argv[3]), std::atof(argv[4]), 1};
  if (!build_tree(cfg, t).empty()) return 101;
  if (int rc = check(t.tiles, t.bfs_tiles, t.srcsets)) return rc;
  std::vector<TargetTile> nonleaf;
  for (const TargetTile& tl : t.bfs_tiles)
    if (!t.pn[tl.panel].is_leaf) nonleaf.push_back(tl);
  if (int rc = check(t.nonleaf_tiles, nonleaf, t.srcsets)) return 10 + rc;
  SourceMajor sm;
  build_source_major(t, sm);
  if (int rc = check(sm.tiles, sm.bfs_tiles, sm.targets)) return 20 + rc;
  // the XCD ranges cover their list and hold equal work to within a tile's
  if (t.xcd_start.size() != 36) return 30;
  for (int range = 0; range < 4; ++range) {
    const std::vector<TargetTile>& list = range < 2 ? t.tiles : t.bfs_tiles;
    const int* xs = t.xcd_start.data() + 9 * range;
    if (xs[0] != 0 || xs[8] != (int)list.size()) return 31;
    double all = 0, most = 0, part[8] = {};
    for (int x = 0; x < 8; ++x)
      for (int k = xs[x]; k < xs[x + 1]; ++k) {
        const TargetTile& tl = list[k];
        double w = 0;
        for (int e = tl.src_begin; e < tl.src_end; ++e)
          w += range & 1 ? t.srcsets[e].count + 16.0
                         : ((tl.count + 15) / 16) * ((t.srcsets[e].count + 15) / 16) + 1.0;
        part[x] += w;
        all += w;
        most = std::max(most, w);
      }
    for (int x = 0; x < 8; ++x)
      if (std::abs(part[x] - all / 8) > most) return 32 + range;
  }
  std::printf("%zu tiles, %zu non-leaf, %zu source-major\n", t.tiles.size(), nonleaf.size(), sm.tiles.size());
  return 0;
}
