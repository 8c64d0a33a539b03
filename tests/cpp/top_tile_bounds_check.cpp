// Host-side run of the LDS-tiled FP32 Iwasaki top kernel (kernels.hpp,
// k_stout_top_tile_body) over the grid it is launched on, which is rounded up
// to whole rounds over the 8 XCDs: the blocks past the lattice must load and
// store nothing. The device functions are compiled for the host; a block is
// 256 host threads with a barrier, and the blocks are run in order, the
// surplus blocks again at the end. Every field lies in an allocation with
// guard reals behind it: links there hold NaN, outputs there must stay as
// they were, and outputs of the lattice must be the same after the surplus
// blocks as before them. One line per shape; exits non-zero on a violation.
#include <hip/hip_runtime.h>

#include <barrier>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>
#include <thread>
#include <vector>

namespace sim {
struct Dim {
  unsigned x = 0, y = 0, z = 0;
};
thread_local Dim tid;
Dim bid, grid;
std::barrier<>* gate = nullptr;
inline void sync() { gate->arrive_and_wait(); }
}  // namespace sim
#undef __device__
#define __device__ __attribute__((host)) __attribute__((device))
#undef __shared__
#define __shared__ static
#define threadIdx sim::tid
#define blockIdx sim::bid
#define gridDim sim::grid
#define __syncthreads sim::sync

#include "../../mag_amd/csrc/kernels.hpp"
#include "../../mag_amd/csrc/runtime.hpp"

using namespace mag;

static constexpr int GUARD = 4096;  // reals behind a field

struct Buf {
  std::vector<float> v;
  size_t n;
  Buf(const Geom& g, int nc, float guard) : v((size_t)g.V * 4 * nc + GUARD, guard), n((size_t)g.V * 4 * nc) {}
};

// A block: its threads run the body; one that leaves early leaves the barrier.
template <int NCL>
static void run_block(const StoutTopArgs<float, 12, 12>& a, int b) {
  sim::bid.x = (unsigned)b;
  std::barrier<> gate(BLOCK);
  sim::gate = &gate;
  std::vector<std::thread> pool;
  for (unsigned t = 0; t < (unsigned)BLOCK; ++t)
    pool.emplace_back([&, t] {
      sim::tid.x = t;
      k_stout_top_tile_body<NCL>(a);
      gate.arrive_and_drop();
    });
  for (auto& t : pool) t.join();
}

template <int NCL>
static int check(const int L[4]) {
  const Geom g = make_geom(L);
  const float nan = std::numeric_limits<float>::quiet_NaN();
  if (!top_tile_ok(g)) return std::printf("FAIL the tile does not take %dx%dx%dx%d\n", L[0], L[1], L[2], L[3]), 1;
  Buf un(g, 12, nan), ulo(g, 12, nan), q(g, 8, nan), c(g, 18, nan), lam(g, 8, 7.f), w(g, 18, 7.f);
  std::mt19937 r(5);
  std::uniform_real_distribution<float> u(-0.5f, 0.5f);
  for (Buf* f : {&un, &ulo, &q, &c})
    for (size_t i = 0; i < f->n; ++i) f->v[i] = u(r);
  const StoutTopArgs<float, 12, 12> a{g,
                                      {un.v.data(), g.V},
                                      {ulo.v.data(), g.V},
                                      {q.v.data(), g.V},
                                      {c.v.data(), g.V},
                                      {lam.v.data(), g.V},
                                      {w.v.data(), g.V},
                                      2.6,
                                      -0.331,
                                      0.1};
  const int nb = (int)grid_stencil(g).x, tiles = 4 * ((g.V + BLOCK - 1) / BLOCK);
  sim::grid.x = (unsigned)nb;
  std::vector<int> surplus;
  for (int b = 0; b < nb; ++b) {
    int mu, sblk;
    tile_map<false>(g, nb, b, mu, sblk);
    if (sblk * BLOCK >= g.V) surplus.push_back(b);
    else run_block<NCL>(a, b);
  }
  if ((int)surplus.size() != nb - tiles) return std::printf("FAIL %zu surplus blocks\n", surplus.size()), 1;
  for (size_t i = 0; i < lam.n; ++i)
    if (!std::isfinite(lam.v[i])) return std::printf("FAIL Lambda[%zu] is not finite\n", i), 1;
  const std::vector<float> lam0 = lam.v, w0 = w.v;
  for (int b : surplus) run_block<NCL>(a, b);
  if (std::memcmp(lam0.data(), lam.v.data(), lam0.size() * sizeof(float)) ||
      std::memcmp(w0.data(), w.v.data(), w0.size() * sizeof(float)))
    return std::printf("FAIL %dx%dx%dx%d, %d reals staged: a block past the lattice stored\n", L[0], L[1], L[2], L[3],
                       NCL), 1;
  for (int i = 0; i < GUARD; ++i)
    if (lam.v[lam.n + i] != 7.f || w.v[w.n + i] != 7.f) return std::printf("FAIL guard %d overwritten\n", i), 1;
  std::printf("ok %dx%dx%dx%d %d reals staged, %zu surplus blocks\n", L[0], L[1], L[2], L[3], NCL, surplus.size());
  return 0;
}

int main() {
  // whole grids (no surplus), an odd number of site blocks (4 surplus)
  const int shapes[][4] = {{16, 16, 4, 4}, {16, 16, 5, 5}};
  for (const auto& L : shapes)
    if (check<12>(L) || check<20>(L)) return 1;
  return 0;
}
