// Host-side check of the maps of the stencils by planes (kernels.hpp):
// plane_group must give every group of 64 sites to exactly one (XCD, walk
// index), and pair_count / pair_site must list every link of constraint
// classes 1 and 10 exactly once and no other. Also tile_map over a grid
// rounded up to a multiple of 8 blocks: every tile exactly once, the surplus
// blocks past the lattice. One line per shape and mag;
// exits non-zero on the first violation.
#include <cstdio>
#include <vector>

#include "../../mag_amd/csrc/kernels.hpp"

using namespace mag;

int main() {
  const int shapes[][4] = {{4, 4, 4, 4},  {5, 7, 4, 9},    {9, 7, 11, 13},  {8, 8, 8, 8},    {6, 6, 6, 12},
                           {12, 8, 4, 24}, {16, 16, 16, 16}, {8, 4, 6, 32}, {24, 24, 24, 24}, {32, 32, 4, 32}};
  for (const auto& L : shapes) {
    const Geom g = make_geom(L);
    const int n = (g.V + PLANE_SITES - 1) / PLANE_SITES, per = (n + 7) / 8;
    std::vector<int> hit((size_t)n, 0);
    for (int x = 0; x < 8; ++x)
      for (int i = 0; i < per; ++i) {
        const int q = plane_group(g, x, i);
        if (q >= n) return std::printf("FAIL group %d of %d\n", q, n), 1;
        if (q >= 0) ++hit[(size_t)q];
      }
    for (int q = 0; q < n; ++q)
      if (hit[(size_t)q] != 1) return std::printf("FAIL group %d hit %d times\n", q, hit[(size_t)q]), 1;
    const int nbs = (g.V + BLOCK - 1) / BLOCK, nb = (4 * nbs + 7) / 8 * 8;
    std::vector<int> tiles((size_t)(4 * nbs), 0);
    for (int b = 0; b < nb; ++b) {
      int mu = -1, sblk = -1;
      tile_map<false>(g, nb, b, mu, sblk);
      if (mu < 0 || mu > 3 || sblk < 0) return std::printf("FAIL tile (%d, %d)\n", mu, sblk), 1;
      if (sblk < nbs) ++tiles[(size_t)(4 * sblk + mu)];
    }
    for (int t = 0; t < 4 * nbs; ++t)
      if (tiles[(size_t)t] != 1) return std::printf("FAIL tile %d hit %d times\n", t, tiles[(size_t)t]), 1;
    for (int mag = 1; mag <= 4; ++mag)
      for (int mu = 0; mu < 4; ++mu) {
        std::vector<int> seen((size_t)g.V, 0);
        const int np = pair_count(g, mu, mag);
        for (int t = 0; t < np; ++t) {
          const Site p = pair_site(g, mu, mag, t);
          if (p.s < 0 || p.s >= g.V) return std::printf("FAIL pair site %d\n", p.s), 1;
          ++seen[(size_t)p.s];
        }
        for (int s = 0; s < g.V; ++s) {
          const Site p = site_of(g, s);
          const int cls = link_class_rt(p, mu, mag);
          if (seen[(size_t)s] != ((cls == 1 || cls == 10) ? 1 : 0))
            return std::printf("FAIL mag %d mu %d site %d class %d listed %d times\n", mag, mu, s, cls,
                               seen[(size_t)s]), 1;
        }
      }
    std::printf("ok %dx%dx%dx%d\n", L[0], L[1], L[2], L[3]);
  }
  return 0;
}
