// Kernel launch layer. Every launch on the trajectory path goes through
// launch(): with no recorder attached it launches the single-chain kernel
// on the context stream; with a recorder attached (serving, see server.hip)
// it records the call instead. A batch of chains of one shape class records
// the same call sequence once per chain; the recorder then emits one launch
// per call of the batched kernel variant, whose argument table holds one
// entry per chain (blockIdx.z = chain). The emitted sequence has fixed
// arguments, so it can be captured in a HIP graph and replayed.
#pragma once
#include <cstring>
#include <string>
#include <vector>

#include "kernels.hpp"
#include "runtime.hpp"

namespace mag {

struct RecCall {
  const void* kb = nullptr;  // batched kernel entry, void(*)(const A*)
  dim3 grid, block;
  size_t argsz = 0;
  std::vector<char> blob;  // argsz bytes per recorded chain
  void* table = nullptr;   // device copy of blob (set when the plan is built)
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
  void add(const void* kb, dim3 grid, dim3 block, const void* args, size_t argsz) {
    if (chain == 0) {
      RecCall c;
      c.kb = kb;
      c.grid = grid;
      c.block = block;
      c.argsz = argsz;
      calls.push_back(std::move(c));
    } else if (pos >= calls.size() || calls[pos].kb != kb || calls[pos].argsz != argsz ||
               calls[pos].grid.x != grid.x || calls[pos].grid.y != grid.y) {
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
           int block = BLOCK) {
  if (c->rec) {
    c->rec->add((const void*)kb, grid, dim3(block), &a, sizeof(A));
    return MAG_OK;
  }
  KTimer t(c, timer);
  A copy = a;
  void* args[] = {&copy};
  HIPCHK(c, hipLaunchKernel((const void*)ks, grid, dim3(block), args, 0, c->stream));
  return MAG_OK;
}

// A stencil kernel in its split form: one wavefront per plane, 64 sites per block.
template <class K>
struct Stencil {};
template <class A, class K>
int launch_split(mag_ctx c, const char* timer, Stencil<K>, const Geom& g, const A& a) {
  return launch(c, timer, k_split<K>, k_split_b<K>, grid_split(g), a, PLANE_THREADS);
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
// per CU, needs a second round from 8,192. Six wavefronts (plane and side) took 50
// us at FP32 8^4 but 149 at 12^4; three groups of sites per block, every wavefront
// going on with one, gave the split's gain back.
constexpr int SPLIT_MAX_SITES = 20736;  // 12^4
template <class K>
constexpr bool split_wins(int V) {
  if (sizeof(typename K::Real) == sizeof(float)) return V <= SPLIT_MAX_SITES;
  if (!K::smears) return V <= 24576;
  return V <= 8192 || (V > 16384 && V <= SPLIT_MAX_SITES);
}
template <class A, class K>
int launch_stencil(mag_ctx c, const char* timer, void (*ks)(A), void (*kb)(const A*), Stencil<K> k, const Geom& g,
                   const A& a) {
  if (split_wins<K>(g.V)) return launch_split(c, timer, k, g, a);
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
