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
// Momenta and one-real-per-link fields of few sites cross as they are stored and
// are converted by the calling thread (convert_here).
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

// Momenta, forces and one-real-per-link fields of few sites: the field as it is
// stored through a pinned slot, converted by this thread. Their host layout has
// up to 4.5 times the bytes, all of which the kernels move over the link, and a
// launch and an event cost as much as a small copy. Through the kernels -> here,
// up / down (us):
//   FP32 momenta  4^4 20.6 / 21.6 -> 14.6 / 15.1, 8^4 102 / 104 -> 60 / 63, 13,824 sites 249 / 260 -> 169 / 190
//   FP64 momenta  4^4 20.9 / 21.8 -> 14.8 / 18.3, 8^4 104 / 104 -> 67 / 99, 6,144 sites 139 / 145 -> 91 / 160
//   one real      6^4 17.4 / 17.0 -> 12.8 / 13.5, 8^4 19.6 / 20.2 -> 15.4 / 17.1, 13,824 sites 30 / 33 -> 27 / 33
// Links go through the kernels from 4^4 on.
constexpr int HERE_SITES = 16384, HERE_SITES_ALG64 = 4096;
bool convert_here(mag_field f) {
  if (f->kind == MAG_REAL1) return f->g.V <= HERE_SITES;
  return f->kind == MAG_ALG8 && f->g.V <= (f->prec == MAG_F64 ? HERE_SITES_ALG64 : HERE_SITES);
}
template <class TS>
void alg_here(TS* raw, double* host, int V, bool down) {
  constexpr int W = Packed<TS, 8>::W, NG = 8 / W;
  constexpr int RUN = 32;  // sites at a time by direction: the groups of all four directions would share cache sets
  for (int s0 = 0; s0 < V; s0 += RUN)
    for (int mu = 0; mu < 4; ++mu)
      for (int s = s0; s < std::min(s0 + RUN, V); ++s) {
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
void real_here(double* raw, double* host, int V, bool down) {
  for (int s = 0; s < V; ++s)
    for (int mu = 0; mu < 4; ++mu) {
      double &r = raw[(size_t)mu * V + s], &h = host[(size_t)s * 4 + mu];
      if (down) h = r;
      else r = h;
    }
}
int transfer_raw(mag_field f, double* host, bool down) {
  mag_ctx c = f->ctx;
  int r;
  if ((r = need_stage(c, f->bytes, 0))) return r;
  auto convert = [&] {
    if (f->kind == MAG_REAL1) real_here((double*)c->stage, host, f->g.V, down);
    else if (f->prec == MAG_F64) alg_here((double*)c->stage, host, f->g.V, down);
    else alg_here((float*)c->stage, host, f->g.V, down);
  };
  if (!down) convert();
  HIPCHK(c, down ? hipMemcpyAsync(c->stage, f->p, f->bytes, hipMemcpyDeviceToHost, c->stream)
                 : hipMemcpyAsync(f->p, c->stage, f->bytes, hipMemcpyHostToDevice, c->stream));
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
