// tile_choice_check.cpp - the choice of the pair form's tiles: tile_ids, whose
// passes are split over threads, against the tiles numbered one point after
// the other, and crowded() against the whole count that it shortens, on ice
// masks from none to contiguous and limits on both sides of the count.
#include <cstdint>
#include <cstdio>
#include <map>
#include <random>
#include <tuple>
#include <vector>

#include "evp1d_tiles.hpp"

extern "C" int evp1d__set_error(int code, const char *) { return code; }

namespace {
int failures = 0;
void check(bool ok, const char *what, int a, int b, double c) {
  if (!ok) {
    ++failures;
    std::printf("FAILED %s (%d, %d, %g)\n", what, a, b, c);
  }
}
}  // namespace

int main() {
  static const int dx[6] = {-1, -1, 0, 1, 1, 0}, dy[6] = {0, -1, -1, 0, 1, 1};
  std::mt19937 rng(3);
  std::uniform_real_distribution<double> u(0.0, 1.0);
  for (auto [nx, ny, land] : {std::tuple<int, int, double>{1, 1, 0.0}, {400, 330, 0.0}, {401, 333, 0.2}}) {
    std::vector<int32_t> pos((size_t)nx * ny, -1), cx, cy;
    for (int i = 0; i < nx * ny; ++i)
      if (u(rng) >= land) {
        pos[(size_t)i] = (int32_t)cx.size();
        cx.push_back(i % nx);
        cy.push_back(i / nx);
      }
    const int na = (int)cx.size(), navel = na + 1;
    std::vector<int32_t> nb[6];
    const int32_t *idx[6];
    for (int k = 0; k < 6; ++k) {
      for (int q = 0; q < na; ++q) {
        const int x = cx[(size_t)q] + dx[k], y = cy[(size_t)q] + dy[k];
        const int32_t r = x < 0 || x >= nx || y < 0 || y >= ny ? -1 : pos[(size_t)y * nx + x];
        nb[k].push_back(r < 0 ? na : r);
      }
      idx[k] = nb[k].data();
    }
    evp1d::GridCoords c;
    c.ok = true;
    c.width = nx;
    c.height = ny;
    c.gx = cx;
    c.gy = cy;
    for (auto [w, h] : {std::pair<int, int>{31, 17}, {31, 19}, {22, 16}, {1, 1}}) {
      const evp1d::TileIds t = evp1d::tile_ids(c, w, h, 0);
      std::map<std::pair<int, int>, int32_t> seen;   // (row, column) of the tiles that hold a point
      for (int q = 0; q < na; ++q) seen[{cy[(size_t)q] / h, cx[(size_t)q] / w}] = 0;
      int32_t n = 0;
      for (auto &s : seen) s.second = n++;
      bool same = t.ntiles == n;
      for (int q = 0; q < na; ++q) same = same && t.tid[(size_t)q] == seen[{cy[(size_t)q] / h, cx[(size_t)q] / w}];
      check(same, "tile ids", nx, w, h);
      for (double ice : {0.0, 0.5, 0.7, 0.8, 0.9, 0.97, 1.0}) {
        std::vector<uint8_t> skip((size_t)na);
        for (uint8_t &s : skip) s = (uint8_t)((u(rng) >= ice ? 1 : 0) | (u(rng) >= ice ? 2 : 0));
        const int most = evp1d::max_level2(na, idx, skip.data(), t);
        check(most <= (w + 1) * (h + 1), "level-2 points", nx, w, ice);
        for (int limit : {0, most - 60, most - 1, most, most + 1, most + 60, 512})
          check(evp1d::crowded(na, idx, skip.data(), t, limit) == (most > limit), "crowded", nx, limit, ice);
      }
    }
  }
  std::printf(failures ? "%d failures\n" : "ok\n", failures);
  return failures ? 1 : 0;
}
