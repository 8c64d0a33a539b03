// Kernel launch layer. Every launch on the trajectory path goes through
// launch(): with no recorder attached it launches the single-chain kernel
// on the context stream; with a recorder attached (serving, see server.hip)
// it records the call instead. A batch of chains of one shape class records
// the same call sequence once per chain; the recorder then emits one launch
// per call of the batched kernel variant (of two, the one for the number of
// chains), whose argument table holds one entry per chain. The emitted sequence
// has fixed arguments, so it can be captured in a HIP graph and replayed.
#pragma once
#include <cstring>
#include <string>
#include <vector>

#include "kernels.hpp"
#include "runtime.hpp"

namespace mag {

// A batched kernel, void(*)(const A*), and its launch for one chain.
struct BatchKernel {
  const void* k = nullptr;
  dim3 grid, block;
};

struct RecCall {
  BatchKernel few, many;  // for fewer than many_from chains, for that many and more
  int many_from = 0;      // 0: `few` for any number
  size_t argsz = 0;
  std::vector<char> blob;  // argsz bytes per recorded chain
  void* table = nullptr;   // device copy of blob (set when the plan is built)
  const BatchKernel& kernel(size_t chains) const { return many_from && (int)chains >= many_from ? many : few; }
};

struct Recorder {
  std::vector<RecCall> calls;
  size_t pos = 0;
  int chain = 0;
  bool mismatch = false;
  void begin_chain(int i) {
    chain = i;
    pos = 0;
  }
  void add(const BatchKernel& few, const BatchKernel& many, int many_from, const void* args, size_t argsz) {
    if (chain == 0) {
      RecCall c;
      c.few = few;
      c.many = many;
      c.many_from = many_from;
      c.argsz = argsz;
      calls.push_back(std::move(c));
    } else if (pos >= calls.size() || calls[pos].few.k != few.k || calls[pos].argsz != argsz ||
               calls[pos].few.grid.x != few.grid.x || calls[pos].few.grid.y != few.grid.y) {
      mismatch = true;
      return;
    }
    RecCall& c = calls[pos++];
    const size_t o = c.blob.size();
    c.blob.resize(o + argsz);
    std::memcpy(c.blob.data() + o, args, argsz);
  }
};

template <class A>
int launch(mag_ctx c, const char* timer, void (*ks)(A), void (*kb)(const A*), dim3 grid, const A& a,
           int block = BLOCK, const BatchKernel& many = {}, int many_from = 0) {
  if (c->rec) {
    c->rec->add({(const void*)kb, grid, dim3(block)}, many, many_from, &a, sizeof(A));
    return MAG_OK;
  }
  KTimer t(c, timer);
  A copy = a;
  void* args[] = {&copy};
  HIPCHK(c, hipLaunchKernel((const void*)ks, grid, dim3(block), args, 0, c->stream));
  return MAG_OK;
}

// A stencil kernel in its split form: one wavefront per plane, 64 sites per
// block; `many` from many_from chains in a batch.
template <class K>
struct Stencil {};
template <class A, class K>
int launch_split(mag_ctx c, const char* timer, Stencil<K>, const Geom& g, const A& a, const BatchKernel& many = {},
                 int many_from = 0) {
  return launch(c, timer, k_split<K>, k_split_b<K>, grid_split(g), a, PLANE_THREADS, many, many_from);
}

// The split form up to a number of sites, else one thread per link (ks, kb).
// Below the line one thread per link leaves most SIMDs with one wavefront or
// none; above it all are busy either way, and two of three wavefronts idle
// while the first goes on costs 5-30 %. Iwasaki + 3-stout force, back to back,
// one thread per link -> split:
//   FP32   8^4 93 -> 57 us, 10^4 100 -> 71, 12^4 117 -> 113, 27,648 sites 122 -> 136, 32,768 134 -> 151
//   FP64   8^4 119 -> 93,   10^4 134 -> 130, 12^4 212 -> 212, 27,648 sites 238 -> 256, 32,768 276 -> 293
// Time of the split form over that of one thread per link, by sites:
//                               8,192  12,288  16,384  18,432  20,736  24,576  28,672  32,768
//   FP32 Wilson + 3-stout force   0.65    0.77    0.81    0.87    0.97    1.05    1.13    1.14
//   FP32 smearing                 0.65    0.76    0.82    0.83    1.02    1.04    1.14    1.15
//   FP64 Wilson + 3-stout force   0.74    1.01    1.19    0.92    0.99    1.08    1.12    1.10
//   FP64 smearing                 0.76    1.04    1.28    0.96    1.01    1.16    1.22    1.06
//   FP64 thin Wilson force        0.70    0.85    0.96    0.77    0.83    0.93    0.97    0.80
//   FP64 thin, 12-real links      0.74    0.88    0.95    0.84    0.93    0.98    1.02    1.06
// FP64 one thread per link takes as long for any lattice up to 16,384 sites (one
// wavefront per SIMD) and nearly twice that from there; the split form, two blocks
// per CU, needs a second round from 8,192, which costs it the gain by 12,288, and a
// smearing by itself, without the backward kernels, already 4-9 % (smear() gives
// split_max). Six wavefronts (plane and side) took 50 us at FP32 8^4 but 149 at
// 12^4; three groups of sites per block, every wavefront going on with one, gave
// the split's gain back.
constexpr int SPLIT_MAX_SITES = 20736;  // 12^4
template <class K>
constexpr bool split_wins(int V) {
  if constexpr (sizeof(typename K::Real) == sizeof(float)) return V <= SPLIT_MAX_SITES;
  else if constexpr (!K::smears) return V <= (K::reals == 12 ? 24576 : 32768);
  else return V <= 12288 || (V > 16384 && V <= SPLIT_MAX_SITES);
}
// A served batch fills the chip with lattices that do not alone: from this many
// sites in all its launches go one thread per link, with the same bits (from two
// chains on, so that a chain alone keeps the form of Chain.run). FP64 rectangles
// stay split. Trajectories, split and one thread per link, against the kernels
// of larger lattices: FP32 Iwasaki + 3-stout, 16 chains of 6^4 (20,736 sites) 0.76
// and 0.78, 7 of 8^4 (28,672) 1.11 split, 64 of 8^4 1.09 and 1.00; FP64 Wilson
// + 2-stout 8^4, 2 chains 0.79 and 1.05, 4 chains 1.13 and 1.04, 64 chains 1.07 and
// 0.99.
template <class K>
constexpr int unsplit_from(int V) {
  const int sites = sizeof(typename K::Real) == sizeof(float) || !K::smears ? 24576 : 16384;
  return (sites + V - 1) / V < 2 ? 2 : (sites + V - 1) / V;
}
template <class A, class K>
int launch_stencil(mag_ctx c, const char* timer, void (*ks)(A), void (*kb)(const A*), Stencil<K> k, const Geom& g,
                   const A& a, int split_max = SPLIT_MAX_SITES) {
  if (split_wins<K>(g.V) && (!K::smears || g.V <= split_max))
    return launch_split(c, timer, k, g, a, {(const void*)k_unsplit_b<K>, grid_stencil(g), dim3(BLOCK)},
                        unsplit_from<K>(g.V));
  return launch(c, timer, ks, kb, grid_stencil(g), a);
}

// Device-to-device copy of `bytes` (a multiple of 16) through a kernel.
inline int copy_async(mag_ctx c, void* dst, const void* src, size_t bytes) {
  CopyArgs a{(double2*)dst, (const double2*)src, bytes / 16};
  const unsigned nb = (unsigned)std::min<size_t>((a.n + BLOCK - 1) / BLOCK, (size_t)1 << 30);
  return launch(c, "copy", k_copy<0>, k_copy_b<0>, dim3(nb ? nb : 1), a);
}

inline int fill_async(mag_ctx c, double* p, double v, int n) {
  FillArgs a{p, v, n};
  return launch(c, "fill", k_fill<0>, k_fill_b<0>, dim3((n + BLOCK - 1) / BLOCK), a);
}

}  // namespace mag
