// Host <-> device movement of fields (mag_field_upload_aos /
// mag_field_download_aos): the qlat layout on the host ([site][mu][3x3
// complex], or [site][mu] for one real per link) against the grouped
// structure-of-arrays in HBM (lattice.hpp).
//
// What bounds it: the PCIe link (57 GB/s for a pinned buffer) and the host
// memory of a fresh user buffer (page faults: 15 GB/s on one thread with
// huge pages, 50 GB/s on four or more). The conversion itself is done by a
// kernel that stores the host layout straight into pinned memory (or loads
// it from there): a block turns 64 sites x 4 directions through LDS, so that
// its accesses over the link are whole contiguous lines (51-54 GB/s, within
// 5 % of the DMA engine, without a second copy in HBM). The field goes in
// chunks through a ring of pinned slots; host threads, two slots each, launch
// their chunks on the context's stream and copy finished slots to (or fill
// them from) the caller's buffer, so conversion, link and host copies
// overlap: 12 ms up and 13-14 ms down (46 GB/s) for any field of 32^4, whose
// host layout is 604 MB. Converting on one host thread beside a pageable copy
// of the raw field took 309 / 269 ms for its FP64 links, 106 / 133 ms for the
// FP32 links and 91 / 101 ms for the momenta.
//
// Momenta and forces of few sites cross as they are stored and are converted by
// the calling thread (convert_here).
//
// Conversions are the host's own arithmetic (no fused multiply-adds), so the
// values are bitwise the same either way.
#pragma clang fp contract(off)
#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <thread>
#include <vector>

#include "lattice.hpp"
#include "runtime.hpp"

using namespace mag;

namespace {

constexpr int TB = 256;           // threads: 64 sites x 4 directions
constexpr int ROW = 4 * 18;       // doubles per site in the host layout
constexpr int LROW = ROW + 1;     // LDS row, odd so that the 64 sites of a wave hit different banks
constexpr size_t CHUNK_MAX = (size_t)4 << 20, CHUNK_MIN = (size_t)512 << 10;
constexpr int WORKERS_MAX = 4;    // host threads (8 or 12: no faster); 32 MiB of pinned slots at most

typedef double V2 __attribute__((ext_vector_type(2)));

// ALG: eight generator components per link, expanded to (projected from) the 3x3 matrix
template <class TS, int NC, bool ALG>
__global__ __launch_bounds__(TB) void k_to_host(TS* p, int V, int s0, int ns, double* out) {
  __shared__ double buf[64 * LROW];
  const int lane = threadIdx.x & 63, mu = threadIdx.x >> 6, b0 = blockIdx.x * 64;
  if (b0 + lane < ns) {
    TS r[NC];
    Packed<TS, NC>::template get<NC, true>(p, V, mu, s0 + b0 + lane, r);
    M3<double> m;
    if constexpr (ALG) {
      double h[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) h[k] = double(r[k]);
      m = alg_to_mat(h);
    } else {
#pragma unroll
      for (int k = 0; k < NC / 2; ++k) m.e[k] = {double(r[2 * k]), double(r[2 * k + 1])};
      if constexpr (NC == 12) reconstruct_row2(m);
    }
    double* b = buf + lane * LROW + mu * 18;
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      b[2 * k] = m.e[k].r;
      b[2 * k + 1] = m.e[k].i;
    }
  }
  __syncthreads();
  const int n2 = min(64, ns - b0) * (ROW / 2);
  V2* o = (V2*)(out + (size_t)b0 * ROW);
  for (int i = threadIdx.x; i < n2; i += TB) {
    const int site = i / (ROW / 2), c = 2 * (i - site * (ROW / 2));
    o[i] = V2{buf[site * LROW + c], buf[site * LROW + c + 1]};
  }
}

// AHEAD of a thread's nine loads over the link are on their way at a time.
template <class TS, int NC, bool ALG, int AHEAD>
__global__ __launch_bounds__(TB) void k_from_host(TS* p, int V, int s0, int ns, const double* in) {
  __shared__ double buf[64 * LROW];
  const int lane = threadIdx.x & 63, mu = threadIdx.x >> 6, b0 = blockIdx.x * 64;
  const int n2 = min(64, ns - b0) * (ROW / 2);
  const V2* src = (const V2*)(in + (size_t)b0 * ROW);
  constexpr int PER = 64 * (ROW / 2) / TB;
#pragma unroll 1
  for (int k0 = 0; k0 < PER; k0 += AHEAD) {
    V2 v[AHEAD];
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) {
      const int i = threadIdx.x + (k0 + k) * TB;
      if (i < n2) v[k] = src[i];
    }
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) {
      const int i = threadIdx.x + (k0 + k) * TB, site = i / (ROW / 2), c = 2 * (i - site * (ROW / 2));
      if (i < n2) {
        buf[site * LROW + c] = v[k][0];
        buf[site * LROW + c + 1] = v[k][1];
      }
    }
  }
  __syncthreads();
  if (b0 + lane >= ns) return;
  const double* b = buf + lane * LROW + mu * 18;
  TS r[NC];
  if constexpr (ALG) {
    M3<double> m;
#pragma unroll
    for (int k = 0; k < 9; ++k) m.e[k] = {b[2 * k], b[2 * k + 1]};
    double h[8];
    mat_to_alg(m, h);
#pragma unroll
    for (int k = 0; k < 8; ++k) r[k] = TS(h[k]);
  } else {
#pragma unroll
    for (int k = 0; k < NC; ++k) r[k] = TS(b[k]);
  }
  Packed<TS, NC>::template put<false>(p, V, mu, s0 + b0 + lane, r);
}

// One real per link: [site][mu] on the host, [mu][site] in the field.
__global__ __launch_bounds__(TB) void k_real_to_host(const double* p, int V, int s0, int ns, double* out) {
  const int i = blockIdx.x * TB + threadIdx.x;
  if (i < 4 * ns) out[i] = p[(size_t)(i & 3) * V + s0 + (i >> 2)];
}
__global__ __launch_bounds__(TB) void k_real_from_host(double* p, int V, int s0, int ns, const double* in) {
  const int i = blockIdx.x * TB + threadIdx.x;
  if (i < 4 * ns) p[(size_t)(i & 3) * V + s0 + (i >> 2)] = in[i];
}

// Up, a chunk of at most 16 blocks waits for the link's latency, so its threads ask
// for all they need at once (4^4 links 27 -> 20.5 us, 8^4 115 -> 102); with more
// blocks the link is busy anyway, and nine lines per thread out of order take it
// longer (16^4 853 -> 1069 us, 24^3 x 32 5.2 -> 6.7 ms).
template <class TS, int NC, bool ALG>
const void* matrix_kernel(bool down, int ns) {
  if (down) return (const void*)k_to_host<TS, NC, ALG>;
  return ns <= 16 * 64 ? (const void*)k_from_host<TS, NC, ALG, 9> : (const void*)k_from_host<TS, NC, ALG, 1>;
}

// Sites [s0, s0 + ns) of f to (from) a pinned slot. Answers with the launch's
// own status: the thread's last error may have been left by an earlier call.
hipError_t launch_chunk(mag_field f, bool down, int s0, int ns, double* slot) {
  const bool f64 = f->prec == MAG_F64;
  const void* k = nullptr;
  int nb = (ns + 63) / 64;
  switch (f->kind) {
    case MAG_REAL1:
      k = down ? (const void*)k_real_to_host : (const void*)k_real_from_host;
      nb = (4 * ns + TB - 1) / TB;
      break;
    case MAG_ALG8: k = f64 ? matrix_kernel<double, 8, true>(down, ns) : matrix_kernel<float, 8, true>(down, ns); break;
    case MAG_LINK12: k = f64 ? matrix_kernel<double, 12, false>(down, ns) : matrix_kernel<float, 12, false>(down, ns); break;
    default: k = matrix_kernel<double, 18, false>(down, ns);  // MAG_LINK18 fields are FP64
  }
  int V = f->g.V;
  void* args[] = {&f->p, &V, &s0, &ns, &slot};
  return hipLaunchKernel(k, dim3(nb), dim3(TB), args, 0, f->ctx->stream);
}

// The calling thread on the context's device for the length of a call: pinned
// slots and events are made on the current device, and an event of another
// device is refused on the context's stream. The caller's device is put back.
struct OnDevice {
  int before = -1;
  hipError_t status;
  explicit OnDevice(int device) {
    int d = device;
    status = hipGetDevice(&d);
    if (status != hipSuccess || d == device) return;
    status = hipSetDevice(device);
    if (status == hipSuccess) before = d;
  }
  ~OnDevice() {
    if (before >= 0) (void)hipSetDevice(before);
  }
};

// The context's pinned slots and their events, grown to what a call needs.
int need_stage(mag_ctx c, size_t bytes, size_t events) {
  if (bytes > c->stage_cap) {
    if (c->stage) (void)hipHostFree(c->stage);
    c->stage = nullptr;
    c->stage_cap = 0;
    if (hipHostMalloc((void**)&c->stage, bytes, hipHostMallocDefault) != hipSuccess) {
      c->stage = nullptr;
      (void)hipGetLastError();
      return fail(c, MAG_ERR_OOM, "pinned staging allocation failed");
    }
    c->stage_cap = bytes;
  }
  while (c->stage_ev.size() < events) {
    hipEvent_t e;
    if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess)
      return fail(c, MAG_ERR_DEVICE, "staging event creation failed");
    c->stage_ev.push_back(e);
  }
  return MAG_OK;
}

// Momenta and forces of few sites: the field as it is stored through a pinned
// slot, converted by this thread. Their host layout has 2.25 (FP64) or 4.5 times
// the bytes, all of which the conversion kernels move over the link. Behind a force
// kernel, through those kernels -> here, up / down:
//   FP32  4^4 30 / 25 -> 22 / 22 us, 6^4 57 / 49 -> 32 / 31, 8^4 118 / 107 -> 63 / 58, 13,824 sites 248 / 264 -> 170 / 152
//   FP64  4^4 30 / 25 -> 22 / 24, 6^4 57 / 49 -> 37 / 38, 8^4 122 / 105 -> 79 / 108
// Links and one real per link gain nothing here.
constexpr int HERE_SITES32 = 16384, HERE_SITES64 = 4096;
bool convert_here(mag_field f) {
  return f->kind == MAG_ALG8 && f->g.V <= (f->prec == MAG_F64 ? HERE_SITES64 : HERE_SITES32);
}
template <class TS>
void alg_here(TS* raw, double* host, int V, bool down) {
  constexpr int W = Packed<TS, 8>::W, NG = 8 / W;
  // FP64: 32 sites at a time by direction, where the sixteen groups of all four
  // directions would share cache sets (8^4 down 100 -> 77 us; 6^4, whose groups
  // do not, 29 site by site and 40 so)
  const int run = NG == 2 || (down && (size_t)V * W * sizeof(TS) % 4096 != 0) ? 1 : 32;
  for (int s0 = 0; s0 < V; s0 += run)
    for (int mu = 0; mu < 4; ++mu)
      for (int s = s0; s < std::min(s0 + run, V); ++s) {
        double* m = host + ((size_t)s * 4 + mu) * 18;
        TS* r = raw + ((size_t)mu * NG * V + s) * W;
        const size_t group = (size_t)V * W;
        double h[8];
        M3<double> M;
        if (down) {
          for (int k = 0; k < 8; ++k) h[k] = double(r[(k / W) * group + k % W]);
          M = alg_to_mat(h);
          for (int k = 0; k < 9; ++k) {
            m[2 * k] = M.e[k].r;
            m[2 * k + 1] = M.e[k].i;
          }
        } else {
          for (int k = 0; k < 9; ++k) M.e[k] = {m[2 * k], m[2 * k + 1]};
          mat_to_alg(M, h);
          for (int k = 0; k < 8; ++k) r[(k / W) * group + k % W] = TS(h[k]);
        }
      }
}
// A kernel, not the copy engine: alone that is 3 us faster, but behind work still in
// flight, as a result that is read back, it is 7 us slower (it waits in a queue of
// its own).
__global__ __launch_bounds__(TB) void k_raw(const V2* src, V2* dst, int n) {
  const int i = blockIdx.x * TB + threadIdx.x;
  if (i < n) dst[i] = src[i];
}
int transfer_raw(mag_field f, double* host, bool down) {
  mag_ctx c = f->ctx;
  int r;
  if ((r = need_stage(c, f->bytes, 0))) return r;
  auto convert = [&] {
    if (f->prec == MAG_F64) alg_here((double*)c->stage, host, f->g.V, down);
    else alg_here((float*)c->stage, host, f->g.V, down);
  };
  if (!down) convert();
  int n = (int)(f->bytes / sizeof(V2));  // whole: 32 V bytes or more
  void *src = down ? f->p : c->stage, *dst = down ? c->stage : f->p;
  void* args[] = {&src, &dst, &n};
  HIPCHK(c, hipLaunchKernel((const void*)k_raw, dim3((n + TB - 1) / TB), dim3(TB), args, 0, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  if (down) convert();
  return MAG_OK;
}

}  // namespace

namespace mag {

int field_transfer(mag_field f, double* host, bool down) {
  mag_ctx c = f->ctx;
  const std::lock_guard<std::mutex> hold(c->stage_mu);
  const OnDevice here(c->device);
  HIPCHK(c, here.status);
  if (convert_here(f)) return transfer_raw(f, host, down);
  const size_t per = (f->kind == MAG_REAL1 ? 4 : ROW) * sizeof(double), total = per * (size_t)f->g.V;
  // about eight chunks, 512 KiB (35 GB/s over the link; less is latency) to 4 MiB (50 GB/s) each
  const size_t want = std::min(std::max(total / 8, CHUNK_MIN), CHUNK_MAX);
  const int step = (int)(std::min((want / per + 63) / 64, CHUNK_MAX / per / 64) * 64);  // whole blocks of 64 sites
  const int nchunk = (f->g.V + step - 1) / step;
  // one more thread (11 us to start) per 2 MiB: two slots each
  const int workers = (int)std::min<size_t>({(size_t)WORKERS_MAX, (total + (2 << 20) - 1) / (2 << 20), (size_t)nchunk});
  const size_t slot_bytes = per * (size_t)std::min(step, f->g.V);
  int r;
  if ((r = need_stage(c, slot_bytes * 2 * workers, 2 * (size_t)workers))) return r;
  std::atomic<int> bad{(int)hipSuccess};
  std::atomic<int> next{0};
  auto work = [&](int w) {
    if (w) {  // a new thread starts on device 0
      const hipError_t e = hipSetDevice(c->device);
      if (e != hipSuccess) bad = (int)e;
    }
    char* slot[2] = {c->stage + slot_bytes * (2 * w), c->stage + slot_bytes * (2 * w + 1)};
    const hipEvent_t ev[2] = {c->stage_ev[2 * w], c->stage_ev[2 * w + 1]};
    int held[2] = {-1, -1};  // chunk in flight in each slot
    auto finish = [&](int k) {
      if (held[k] < 0) return;
      const hipError_t e = hipEventSynchronize(ev[k]);
      if (e != hipSuccess) {
        bad = (int)e;
      } else if (down) {
        const size_t s0 = (size_t)held[k] * step, ns = std::min<size_t>(step, f->g.V - s0);
        std::memcpy((char*)host + s0 * per, slot[k], ns * per);
      }
      held[k] = -1;
    };
    int k = 0;
    for (int i = next++; i < nchunk && bad == (int)hipSuccess; i = next++, k ^= 1) {
      finish(k);
      const size_t s0 = (size_t)i * step, ns = std::min<size_t>(step, f->g.V - s0);
      if (!down) std::memcpy(slot[k], (const char*)host + s0 * per, ns * per);
      hipError_t e = launch_chunk(f, down, (int)s0, (int)ns, (double*)slot[k]);
      if (e == hipSuccess) {
        held[k] = i;
        e = hipEventRecord(ev[k], c->stream);
      }
      if (e != hipSuccess) bad = (int)e;
    }
    finish(k);
    finish(k ^ 1);
  };
  std::vector<std::thread> pool;
  try {
    for (int w = 1; w < workers; ++w) pool.emplace_back(work, w);
  } catch (const std::exception&) {  // no more threads: those that run take all chunks
  }
  work(0);
  for (auto& t : pool) t.join();
  if (bad != (int)hipSuccess) {
    (void)hipStreamSynchronize(c->stream);  // no kernel is left in the slots
    return fail(c, MAG_ERR_DEVICE, std::string("field transfer: ") + hipGetErrorString((hipError_t)bad.load()));
  }
  return MAG_OK;
}

void free_stage(mag_ctx c) {
  for (auto e : c->stage_ev) (void)hipEventDestroy(e);
  c->stage_ev.clear();
  if (c->stage) (void)hipHostFree(c->stage);
  c->stage = nullptr;
  c->stage_cap = 0;
}

}  // namespace mag
