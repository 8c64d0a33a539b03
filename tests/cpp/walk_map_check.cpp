// Host-side check of the walks that deal site blocks to the XCDs (kernels.hpp):
// run_block (plaquette and rectangle sums) must be a permutation of the blocks,
// and the identity up to one block per CU; wloop_block (Wilson loops) must be a
// permutation on any lattice, x3 in one piece or by eights with a remainder; and
// tile_map, in both its orders over the grid that stencils are launched on (whole
// rounds over the XCDs), must give every tile once and nothing but site blocks
// past the lattice to the surplus blocks. One line per check; exits non-zero on
// the first violation.
#include <cstdio>
#include <vector>

#include "../../mag_amd/csrc/kernels.hpp"
#include "../../mag_amd/csrc/runtime.hpp"

using namespace mag;

template <class Map>
static int permutation(const char* what, int nb, Map map) {
  std::vector<int> hit((size_t)nb, 0);
  for (int b = 0; b < nb; ++b) {
    const int t = map(b);
    if (t < 0 || t >= nb) return std::printf("FAIL %s: block %d of %d -> %d\n", what, b, nb, t), 1;
    ++hit[(size_t)t];
  }
  for (int t = 0; t < nb; ++t)
    if (hit[(size_t)t] != 1) return std::printf("FAIL %s: block %d of %d hit %d times\n", what, t, nb, hit[(size_t)t]), 1;
  return 0;
}

template <bool X2>
static int tiles(const Geom& g) {
  const int nbs = (g.V + BLOCK - 1) / BLOCK, nb = (int)grid_stencil(g).x;
  std::vector<int> hit((size_t)(4 * nbs), 0);
  int surplus = 0;
  for (int b = 0; b < nb; ++b) {
    int mu = -1, sblk = -1;
    tile_map<X2>(g, nb, b, mu, sblk);
    if (mu < 0 || mu > 3 || sblk < 0) return std::printf("FAIL tile_map: block %d -> (%d, %d)\n", b, mu, sblk), 1;
    if (sblk < nbs) ++hit[(size_t)(4 * sblk + mu)];
    else ++surplus;
  }
  if (surplus != nb - 4 * nbs) return std::printf("FAIL tile_map: %d surplus blocks of %d\n", surplus, nb - 4 * nbs), 1;
  for (int t = 0; t < 4 * nbs; ++t)
    if (hit[(size_t)t] != 1) return std::printf("FAIL tile_map: tile %d hit %d times\n", t, hit[(size_t)t]), 1;
  return 0;
}

int main() {
  for (int nb = 1; nb < 1300; ++nb) {
    if (permutation("run_block", nb, [&](int b) { return run_block(b, nb); })) return 1;
    for (int b = 0; nb <= 256 && b < nb; ++b)
      if (run_block(b, nb) != b) return std::printf("FAIL run_block: %d of %d moved\n", b, nb), 1;
  }
  std::printf("ok run_block\n");
  const int shapes[][4] = {{4, 4, 4, 4},    {5, 7, 4, 9},    {16, 16, 16, 8}, {8, 4, 4, 32},  {8, 4, 4, 33},
                           {8, 16, 4, 37},  {16, 8, 4, 40},  {4, 4, 8, 71},   {24, 16, 8, 48}, {32, 32, 4, 64},
                           {12, 12, 12, 48}, {8, 8, 6, 100}};
  for (const auto& L : shapes) {
    const Geom g = make_geom(L);
    const int nb = (g.V + WLOOP_SITES - 1) / WLOOP_SITES;
    if (permutation("wloop_block", nb, [&](int b) { return wloop_block(g, b, nb); })) return 1;
  }
  std::printf("ok wloop_block\n");
  const int grids[][4] = {{4, 4, 4, 4},    {6, 6, 6, 6},     {5, 7, 4, 9},     {16, 16, 5, 5},  {12, 12, 12, 12}, {14, 14, 14, 14},
                          {20, 20, 20, 20}, {16, 16, 16, 16}, {24, 24, 24, 24}, {32, 32, 4, 32}, {8, 8, 4, 16},    {64, 64, 4, 8}};
  for (const auto& L : grids)
    if (tiles<false>(make_geom(L)) || tiles<true>(make_geom(L))) return 1;
  std::printf("ok tile_map\n");
  return 0;
}
