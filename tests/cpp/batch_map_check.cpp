// Host-side check of the block maps of batched stencils (kernels.hpp), split by
// planes and with one thread per link: over the grid of a batch of n chains,
// every site block and direction of every chain must come from exactly one
// block, no chain, site block or direction may be out of range, and each XCD
// (block id mod 8) must hold as many blocks with work as any other, up to one
// chain's share. One line per shape; exits non-zero on the first violation.
#include <algorithm>
#include <cstdio>
#include <vector>

#include "../../mag_amd/csrc/kernels.hpp"
#include "../../mag_amd/csrc/runtime.hpp"

using namespace mag;

// sites per block, blocks per chain of the grid, and the map of one form
template <class Map>
static int check(const Geom& g, const char* form, int sites, int gx, Map map) {
  const int nb = (g.V + sites - 1) / sites;
  if (gx % 8) return std::printf("FAIL %s: grid of %d blocks\n", form, gx), 1;
  for (int n : {1, 2, 3, 7, 8, 9, 15, 16, 17, 64}) {
    std::vector<int> hit((size_t)n * nb * 4, 0);
    long xcd[8] = {};
    for (int z = 0; z < n; ++z)
      for (int x = 0; x < gx; ++x) {
        const ChainBlock q = chain_block(gx, n, x, z, 4 * nb);
        if (q.chain == -1) continue;
        if (q.chain < 0 || q.chain >= n || q.block < 0 || q.block >= gx)
          return std::printf("FAIL %s: chain %d block %d\n", form, q.chain, q.block), 1;
        int mu = -1, blk = -1;
        map(q.block, q.whole, mu, blk);
        if (mu < 0 || mu > 3) return std::printf("FAIL %s: direction %d\n", form, mu), 1;
        if (blk < 0 || blk >= nb) continue;
        ++hit[((size_t)q.chain * nb + blk) * 4 + mu];
        ++xcd[((long)x + (long)gx * z) % 8];
      }
    for (size_t i = 0; i < hit.size(); ++i)
      if (hit[i] != 1) return std::printf("FAIL %s, %d chains: tile %zu hit %d times\n", form, n, i, hit[i]), 1;
    const auto mm = std::minmax_element(xcd, xcd + 8);
    if (*mm.second - *mm.first > 4 * ((nb + 7) / 8))
      return std::printf("FAIL %s, %d chains of %d blocks: %ld to %ld per XCD\n", form, n, nb, *mm.first, *mm.second), 1;
  }
  return 0;
}

int main() {
  const int shapes[][4] = {{4, 4, 4, 4}, {6, 6, 6, 6}, {5, 7, 4, 9}, {8, 8, 8, 8}, {9, 7, 11, 13}, {12, 12, 12, 12}, {8, 4, 6, 32}};
  for (const auto& L : shapes) {
    const Geom g = make_geom(L);
    const int gu = (int)grid_stencil(g).x;
    if (check(g, "split", PLANE_SITES, (int)grid_split(g).x,
              [&](int b, bool whole, int& mu, int& blk) { split_tile(g, b, whole, mu, blk); }) ||
        check(g, "one thread per link", BLOCK, gu,
              [&](int b, bool whole, int& mu, int& blk) { unsplit_tile(g, gu, b, whole, mu, blk); }))
      return 1;
    std::printf("ok %dx%dx%dx%d\n", L[0], L[1], L[2], L[3]);
  }
  return 0;
}
