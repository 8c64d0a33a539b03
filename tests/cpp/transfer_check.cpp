// Host-side check of field transfers (transfer.hip) over a HIP runtime that
// this program stands in for: two devices, a current device per thread,
// streams and events that belong to a device (recording an event on another
// device's stream is refused, as by the runtime), and kernels that are emulated
// for one-real-per-link fields and write the site number for link fields. argv[1] names the check; prints "ok" lines and exits
// non-zero on the first violation.
#include "../../mag_amd/csrc/transfer.hip"

#include <cstdio>
#include <cstdlib>
#include <map>

struct FakeStream {
  int device;
};
struct FakeEvent {
  int device;
};

static thread_local int t_device = 0;  // a new thread starts on device 0
static hipError_t g_last = hipSuccess;    // what an earlier call, of the library or not, left as the last error
static hipError_t g_launch = hipSuccess;  // what a launch returns
static std::mutex g_mu;
static std::map<void*, size_t> g_pinned;
static size_t g_pinned_now = 0, g_pinned_max = 0;
static int g_bad_alloc = 0, g_bad_event = 0, g_bad_launch = 0, g_launches = 0;
static std::vector<int> g_sites;  // times each site was moved

extern "C" {
hipError_t hipGetDevice(int* d) { return *d = t_device, hipSuccess; }
hipError_t hipSetDevice(int d) {
  if (d < 0 || d > 1) return hipErrorInvalidDevice;
  return t_device = d, hipSuccess;
}
hipError_t hipGetLastError() { return g_last; }
const char* hipGetErrorString(hipError_t) { return "refused"; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned int) {
  std::lock_guard<std::mutex> l(g_mu);
  *p = std::malloc(n);
  g_pinned[*p] = n;
  g_pinned_now += n;
  g_pinned_max = std::max(g_pinned_max, g_pinned_now);
  g_bad_alloc += t_device != 1;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::lock_guard<std::mutex> l(g_mu);
  g_pinned_now -= g_pinned[p];
  g_pinned.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = (hipEvent_t) new FakeEvent{t_device};
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { return delete (FakeEvent*)e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (((FakeEvent*)e)->device == ((FakeStream*)s)->device) return hipSuccess;
  std::lock_guard<std::mutex> l(g_mu);
  ++g_bad_event;
  return hipErrorInvalidHandle;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }

hipError_t hipLaunchKernel(const void* k, dim3, dim3, void** args, size_t, hipStream_t s) {
  if (g_launch != hipSuccess) return g_launch;
  if (k == (const void*)k_raw) {  // a whole field
    std::memcpy(*(void**)args[1], *(void**)args[0], (size_t)*(int*)args[2] * sizeof(V2));
    std::lock_guard<std::mutex> l(g_mu);
    g_bad_launch += t_device != ((FakeStream*)s)->device;
    for (int& n : g_sites) ++n;
    return hipSuccess;
  }
  const int V = *(int*)args[1], s0 = *(int*)args[2], ns = *(int*)args[3];
  double* p = *(double**)args[0];
  double* slot = *(double**)args[4];
  {
    std::lock_guard<std::mutex> l(g_mu);
    ++g_launches;
    g_bad_launch += t_device != ((FakeStream*)s)->device;
    for (int i = s0; i < s0 + ns; ++i) ++g_sites.at((size_t)i);
  }
  const bool real_down = k == (const void*)k_real_to_host, real_up = k == (const void*)k_real_from_host;
  if (real_down || real_up) {
    for (int i = 0; i < 4 * ns; ++i) {
      double& f = p[(size_t)(i & 3) * V + s0 + (i >> 2)];
      if (real_down) slot[i] = f;
      else f = slot[i];
    }
  } else {
    for (size_t i = 0; i < (size_t)ns * ROW; ++i) slot[i] = (double)(s0 + (int)(i / ROW));
  }
  return hipSuccess;
}
}

struct Rig {
  FakeStream stream{1};
  mag_ctx_s ctx;
  Rig() {
    ctx.device = 1;
    ctx.stream = (hipStream_t)&stream;
  }
  ~Rig() { free_stage(&ctx); }
};

#define REQUIRE(cond, ...)                                            \
  do {                                                                \
    if (!(cond)) {                                                    \
      std::printf("FAIL " __VA_ARGS__);                               \
      std::printf(" (%s, line %d)\n", #cond, __LINE__);               \
      return 1;                                                       \
    }                                                                 \
  } while (0)

static mag_field_s field(Rig& rig, const int L[4], int kind, std::vector<double>& store) {
  mag_field_s f;
  f.ctx = &rig.ctx;
  std::memcpy(f.dims, L, sizeof f.dims);
  f.kind = kind;
  f.prec = MAG_F64;
  f.g = make_geom(L);
  store.resize(kind == MAG_REAL1 ? (size_t)f.g.V * 4 : kind == MAG_ALG8 ? (size_t)f.g.V * 32 : 1);  // link values are not looked at
  f.p = store.data();
  f.bytes = store.size() * sizeof(double);
  g_sites.assign((size_t)f.g.V, 0);
  return f;
}

static int moved_once(const mag_field_s& f) {
  for (int s = 0; s < f.g.V; ++s) REQUIRE(g_sites[(size_t)s] == 1, "site %d of %d moved %d times", s, f.g.V, g_sites[(size_t)s]);
  return 0;
}

// One field down and (one real per link) up again, from a caller on `current`.
static int round_trip(Rig& rig, const int L[4], int kind, int current) {
  std::vector<double> store;
  mag_field_s f = field(rig, L, kind, store);
  const size_t n = (size_t)f.g.V * (kind == MAG_REAL1 ? 4 : ROW);
  for (size_t i = 0; i < store.size(); ++i) store[i] = (double)i;
  std::vector<double> host(n, -1.);
  t_device = current;
  const int r = field_transfer(&f, host.data(), true);
  REQUIRE(r == MAG_OK, "download of %d sites, kind %d, caller on device %d: status %d", f.g.V, kind, current, r);
  REQUIRE(t_device == current, "the caller was left on device %d", t_device);
  if (moved_once(f)) return 1;
  if (kind == MAG_ALG8) return 0;  // values: the GPU tests
  for (size_t i = 0; i < n; ++i) {
    const double want = kind == MAG_REAL1 ? (double)((i & 3) * (size_t)f.g.V + i / 4) : (double)(i / ROW);
    REQUIRE(host[i] == want, "value %zu is %g", i, host[i]);
  }
  if (kind != MAG_REAL1) return 0;
  const std::vector<double> before = store;
  std::fill(store.begin(), store.end(), 0.);
  g_sites.assign((size_t)f.g.V, 0);
  REQUIRE(field_transfer(&f, host.data(), false) == MAG_OK, "upload refused");
  REQUIRE(t_device == current, "the caller was left on device %d", t_device);
  if (moved_once(f)) return 1;
  REQUIRE(store == before, "upload of %d sites", f.g.V);
  return 0;
}

static const int SHAPES[][4] = {{4, 4, 4, 4}, {5, 7, 4, 9}, {8, 8, 8, 8}, {9, 7, 11, 13}, {16, 16, 16, 20}, {32, 32, 32, 8}};

// A context of device 1, called from threads whose current device is 0 or 1.
static int check_device() {
  for (const auto& L : SHAPES)
    for (int kind : {(int)MAG_REAL1, (int)MAG_LINK18, (int)MAG_ALG8})
      for (int current : {0, 1}) {
        Rig rig;
        if (round_trip(rig, L, kind, current)) return 1;
        REQUIRE(!g_bad_alloc && !g_bad_event && !g_bad_launch, "%d allocations, %d events, %d launches off the device",
                g_bad_alloc, g_bad_event, g_bad_launch);
      }
  std::printf("ok device\n");
  return 0;
}

// A transfer answers for its own launches: an error that an earlier call left
// behind is none of its, a launch that fails is.
static int check_error() {
  for (const auto& L : SHAPES)
    for (int kind : {(int)MAG_REAL1, (int)MAG_LINK18, (int)MAG_ALG8}) {
      Rig rig;
      g_last = hipErrorOutOfMemory;
      if (round_trip(rig, L, kind, 1)) return 1;
      g_last = hipSuccess;
      g_launch = hipErrorInvalidValue;
      std::vector<double> store, host((size_t)L[0] * L[1] * L[2] * L[3] * ROW);
      mag_field_s f = field(rig, L, kind, store);
      REQUIRE(field_transfer(&f, host.data(), true) == MAG_ERR_DEVICE, "a failed launch went unseen");
      REQUIRE(field_transfer(&f, host.data(), false) == MAG_ERR_DEVICE, "a failed launch went unseen");
      g_launch = hipSuccess;
    }
  std::printf("ok error\n");
  return 0;
}

// The pinned memory that a context holds after fields of any size.
static int check_bound() {
  const int shapes[][4] = {{4, 4, 4, 4}, {9, 7, 11, 13}, {16, 16, 16, 20}, {24, 24, 24, 32}, {32, 32, 32, 32}};
  for (const auto& L : shapes)
    for (int kind : {(int)MAG_REAL1, (int)MAG_LINK18, (int)MAG_ALG8}) {
      Rig rig;
      std::vector<double> store;
      mag_field_s f = field(rig, L, kind, store);
      std::unique_ptr<double[]> host(new double[(size_t)f.g.V * (kind == MAG_REAL1 ? 4 : ROW)]);
      g_pinned_max = 0;
      REQUIRE(field_transfer(&f, host.get(), true) == MAG_OK, "download refused");
      if (moved_once(f)) return 1;
      REQUIRE(g_pinned_max <= (size_t)32 << 20, "%zu bytes pinned for %d sites of kind %d", g_pinned_max, f.g.V, kind);
    }
  std::printf("ok bound\n");
  return 0;
}

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "device") return check_device();
  if (what == "error") return check_error();
  if (what == "bound") return check_bound();
  return 2;
}
