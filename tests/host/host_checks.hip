// The host side of libwrfdc on the CPU: the library's source compiled for the
// host alone, over a HIP runtime of its own below, which holds memory,
// streams, events and graphs as plain objects, logs launches without running
// them and can make a chosen call fail.  Anything used after it was
// destroyed, destroyed twice or never destroyed is an error.
//
//   host_checks <check>     runs one check of the table at the end
#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include <hip/hip_runtime.h>

// ---- allocation failures -----------------------------------------------------
static std::atomic<long> g_alloc_left{-1};  // the allocation that throws (counted down), -1 none
static thread_local int t_inside = 0;           // in the runtime below, whose own allocations do not count
void *operator new(size_t n) {
  if (!t_inside && g_alloc_left.load() >= 0 && g_alloc_left.fetch_sub(1) == 0) throw std::bad_alloc();
  if (void *p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

// ---- the runtime ---------------------------------------------------------------
namespace rt {
struct Launch {
  std::string name, mangled;
  hipStream_t s;
  dim3 block;
};
std::recursive_mutex mu;
struct Guard {
  Guard() { mu.lock(), t_inside++; }
  ~Guard() { t_inside--, mu.unlock(); }
};
std::map<const void *, std::string> kernels;  // mangled names
std::vector<Launch> log_;
std::map<void *, std::string> live;      // device and pinned memory, streams, events, graphs
std::set<hipStream_t> capturing, busy;   // busy: work that nothing has waited for
std::map<hipEvent_t, hipStream_t> recorded;
std::vector<std::string> errors;
hipError_t last = hipSuccess;
std::string fail_name;  // the call (or kernel) that fails ...
long fail_left = -1;    // ... after this many successes
long fail_times = 1;    // ... this many times
long fail_any = -1;     // any call at all, after this many

void error(const std::string &s) { errors.push_back(s); }
bool fails(const std::string &name) {
  bool f = false;
  if (fail_left >= 0 && name == fail_name) {
    f = fail_left == 0;
    if (fail_left > 0 || --fail_times <= 0) fail_left--;
  }
  if (fail_any >= 0 && fail_any-- == 0) f = true;
  return f;
}
hipError_t fail(hipError_t e = hipErrorOutOfMemory) { return last = e; }
template <class T>
hipError_t make(T *out, const char *what) {
  void *p = std::calloc(1, 64);
  live[p] = what;
  *out = reinterpret_cast<T>(p);
  return hipSuccess;
}
template <class T>
hipError_t drop(T h, const char *what) {
  auto it = live.find((void *)h);
  if (it == live.end() || it->second != what) {
    error(std::string(what) + " destroyed twice or never created");
    return fail(hipErrorInvalidHandle);
  }
  live.erase(it);
  std::free((void *)h);
  return hipSuccess;
}
bool alive(const void *h, const char *what) {
  auto it = live.find(const_cast<void *>(h));
  if (it != live.end() && it->second == what) return true;
  error(std::string(what) + " used after it was destroyed");
  return false;
}
bool stream_ok(hipStream_t s) { return !s || alive(s, "stream"); }
std::string base(const char *mangled) {  // the kernel's name out of its mangled one
  std::string m = mangled;
  size_t best = m.find("k_");
  size_t end = best;
  int len = 0;
  for (size_t q = best; q > 0 && isdigit(m[q - 1]); q--) end = q - 1;
  len = atoi(m.substr(end, best - end).c_str());
  return len > 0 ? m.substr(best, len) : m;
}
long count(const std::string &name, hipStream_t s) {
  return std::count_if(log_.begin(), log_.end(), [&](const Launch &l) { return l.name == name && l.s == s; });
}
}  // namespace rt
#define RT(name)   \
  rt::Guard guard; \
  if (rt::fails(name)) return rt::fail()

extern "C" {
void **__hipRegisterFatBinary(const void *) {
  static void *h;
  return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *, int *) {
  rt::kernels[f] = name;
}
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}
static thread_local struct { dim3 g, b; size_t lds; hipStream_t s; } g_cfg;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
  g_cfg = {g, b, lds, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
  *g = g_cfg.g;
  *b = g_cfg.b;
  *lds = g_cfg.lds;
  *s = g_cfg.s;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **, size_t, hipStream_t s) {
  rt::Guard guard;
  const std::string mangled = rt::kernels.at(f), name = rt::base(mangled.c_str());
  if (rt::fails(name)) return rt::fail(hipErrorLaunchFailure);
  if (!rt::stream_ok(s)) return rt::fail(hipErrorInvalidHandle);
  if (!g.x || !g.y || !g.z) return rt::fail(hipErrorInvalidConfiguration);
  rt::log_.push_back({name, mangled, s, b});
  if (!rt::capturing.count(s)) rt::busy.insert(s);
  return hipSuccess;
}
hipError_t hipGetLastError(void) {
  rt::Guard guard;
  const hipError_t e = rt::last;
  rt::last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t) { return "failed"; }
hipError_t hipGetDevice(int *d) {
  RT("hipGetDevice");
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { RT("hipSetDevice"); return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { RT("hipFuncSetAttribute"); return hipSuccess; }
hipError_t hipGetSymbolAddress(void **, const void *) { return rt::fail(); }
hipError_t hipMalloc(void **p, size_t n) {
  RT("hipMalloc");
  rt::live[*p = std::calloc(1, n ? n : 1)] = "device memory";
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  rt::Guard guard;
  return p ? rt::drop(p, "device memory") : hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  RT("hipHostMalloc");
  rt::live[*p = std::calloc(1, n)] = "pinned memory";
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  rt::Guard guard;
  return rt::drop(p, "pinned memory");
}
hipError_t hipMemcpyAsync(void *d, const void *h, size_t n, hipMemcpyKind, hipStream_t s) {
  RT("hipMemcpyAsync");
  if (!rt::stream_ok(s)) return rt::fail();
  std::memcpy(d, h, n);
  rt::busy.insert(s);
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { RT("hipStreamCreateWithFlags"); return rt::make(s, "stream"); }
hipError_t hipStreamDestroy(hipStream_t s) {
  rt::Guard guard;
  if (rt::busy.count(s)) rt::error("stream destroyed with work in flight");
  if (rt::capturing.count(s)) rt::error("stream destroyed while it captures");
  const hipError_t e_ = rt::drop(s, "stream");
  return rt::fails("hipStreamDestroy") ? rt::fail() : e_;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  rt::Guard guard;
  rt::busy.erase(s);
  if (rt::fails("hipStreamSynchronize")) return rt::fail();
  if (rt::capturing.count(s)) rt::error("synchronised a stream that captures");
  return rt::stream_ok(s) ? hipSuccess : rt::fail();
}
hipError_t hipDeviceSynchronize(void) {
  rt::Guard guard;
  rt::busy.clear();
  return rt::fails("hipDeviceSynchronize") ? rt::fail() : hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st) {
  RT("hipStreamIsCapturing");
  *st = rt::capturing.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return rt::stream_ok(s) ? hipSuccess : rt::fail();
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
  RT("hipStreamBeginCapture");
  rt::capturing.insert(s);
  return rt::stream_ok(s) ? hipSuccess : rt::fail();
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g) {
  rt::Guard guard;
  if (!rt::capturing.count(s)) rt::error("ended a capture that was not begun");
  rt::capturing.clear();  // the streams that joined too
  *g = nullptr;
  if (rt::fails("hipStreamEndCapture")) return rt::fail();
  return rt::make(g, "graph");
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  RT("hipStreamWaitEvent");
  if (!rt::stream_ok(s) || !rt::alive(e, "event")) return rt::fail();
  auto it = rt::recorded.find(e);
  if (it != rt::recorded.end() && rt::capturing.count(it->second)) rt::capturing.insert(s);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { RT("hipEventCreateWithFlags"); return rt::make(e, "event"); }
hipError_t hipEventDestroy(hipEvent_t e) {
  rt::Guard guard;
  rt::recorded.erase(e);
  const hipError_t e_ = rt::drop(e, "event");
  return rt::fails("hipEventDestroy") ? rt::fail() : e_;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  RT("hipEventRecord");
  if (!rt::stream_ok(s) || !rt::alive(e, "event")) return rt::fail();
  rt::recorded[e] = s;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  RT("hipEventSynchronize");
  if (!rt::alive(e, "event")) return rt::fail();
  rt::busy.erase(rt::recorded[e]);
  return hipSuccess;
}
hipError_t hipGraphGetNodes(hipGraph_t g, hipGraphNode_t *, size_t *n) {
  RT("hipGraphGetNodes");
  *n = rt::log_.size();
  return rt::alive(g, "graph") ? hipSuccess : rt::fail();
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t g, hipGraphNode_t *, char *, size_t) {
  RT("hipGraphInstantiate");
  return rt::alive(g, "graph") ? rt::make(x, "graph exec") : rt::fail();
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t s) {
  RT("hipGraphLaunch");
  if (!rt::alive(x, "graph exec") || !rt::stream_ok(s)) return rt::fail();
  rt::busy.insert(s);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x) {
  rt::Guard guard;
  if (!rt::busy.empty()) rt::error("graph exec destroyed with work in flight");
  const hipError_t e_ = rt::drop(x, "graph exec");
  return rt::fails("hipGraphExecDestroy") ? rt::fail() : e_;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  rt::Guard guard;
  const hipError_t e_ = rt::drop(g, "graph");
  return rt::fails("hipGraphDestroy") ? rt::fail() : e_;
}
}  // extern "C"

#include "../../wrf-jax_amd/csrc/wrfdc.hip"

// ---- the checks ------------------------------------------------------------------
namespace {
int g_bad = 0;
#define CHECK(c)                                                            \
  do {                                                                      \
    if (!(c)) g_bad++, std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c); \
  } while (0)

float g_field[64];  // stands for every field: nothing here runs a kernel
wrfdc_ctx *make_ctx(int nx, int ny, int nz, int nmoist = 3, int nscalar = 1) {
  wrfdc_config c;
  std::memset(&c, 0, sizeof(c));
  c.nx = nx;
  c.ny = ny;
  c.nz = nz;
  c.ip = (nx + 16) / 16 * 16;
  c.nmoist = nmoist;
  c.nscalar = nscalar;
  c.spec_zone = 1;
  c.relax_zone = 4;
  c.spec_bdy_width = 5;
  c.pd_moist = c.pd_scalar = 1;
  c.dx = c.dy = 3000.0;
  c.dt = 18.0;
  wrfdc_ctx *x = nullptr;
  if (wrfdc_create(&c, &x) != WRFDC_OK) return nullptr;
  for (int f = 0; f < wrfdc_field_count(); f++) wrfdc_bind(x, wrfdc_field_name(f), g_field);
  return x;
}

// The kernels' context in device memory: uploaded when it changed, on the stream
// that reads it, and again after an upload that could not be launched.
void context_upload() {
  wrfdc_ctx *x = make_ctx(24, 20, 10);
  hipStream_t other;
  CHECK(hipStreamCreateWithFlags(&other, hipStreamNonBlocking) == hipSuccess);
  auto uploads = [&](hipStream_t s) {
    rt::log_.clear();
    const int rc = wrfdc_step(x, 1, 0.0);
    const bool first = !rt::log_.empty() && rt::log_[0].name == "k_put_ctx";
    const long n = rt::count("k_put_ctx", s);
    CHECK(n == 0 || first);
    return rc == WRFDC_OK ? n : -1;
  };
  CHECK(uploads(nullptr) == 2);
  CHECK(uploads(nullptr) == 0);
  wrfdc_bind(x, "t_2", g_field + 1);
  CHECK(uploads(nullptr) == 2);
  for (long n : {0, 1}) {  // the first or the second of the two
    wrfdc_bind(x, "t_2", g_field + 2 + n);
    rt::fail_name = "k_put_ctx";
    rt::fail_left = n;
    rt::fail_times = 1;
    CHECK(uploads(nullptr) == -1);
    CHECK(rt::count("k_uv_first", nullptr) == 0);  // nothing ran on the stale context
    CHECK(uploads(nullptr) == 2);
  }
  CHECK(wrfdc_set_stream(x, other) == WRFDC_OK);
  CHECK(uploads(other) == 2);
  CHECK(wrfdc_set_stream(x, other) == WRFDC_OK);
  CHECK(uploads(other) == 0);
  CHECK(wrfdc_set_stream(x, nullptr) == WRFDC_OK);
  CHECK(uploads(nullptr) == 2);
  CHECK(hipStreamSynchronize(other) == hipSuccess && hipStreamDestroy(other) == hipSuccess);
  wrfdc_destroy(x);
}

// The phi tendency's index arithmetic takes blocks of four waves, whatever the
// rows of the face blocks it shares its launch with (WRFDC_FACE_ROWS).
void phi_tendency_blocks() {
  for (int nx : {24, 300}) {
    wrfdc_ctx *x = make_ctx(nx, 200, 40);
    rt::log_.clear();
    CHECK(wrfdc_step(x, 1, 0.0) == WRFDC_OK);
    int phi = 0;
    for (auto &l : rt::log_)
      if (l.name == "k_tendencies" || l.mangled.find("k_tendencyILi4E") != std::string::npos) {
        phi++;
        CHECK(l.block.x == 64 && l.block.y == 4);
      } else if (l.name == "k_tendency") {
        CHECK(l.block.x == 64 && (int)l.block.y == kFaceRows);
      }
    CHECK(phi == 3);
    wrfdc_destroy(x);
  }
}

// The transfers of host arrays: whatever fails, the call returns an error or
// does without, nothing is in flight when it returns, and the next call works.
struct Arrays {
  std::vector<std::vector<float>> a;
  std::vector<int> fields;
  std::vector<void *> p;
  Arrays(wrfdc_ctx *x) {
    for (const char *name : {"moist", "u_2", "mu_2", "c1h", "t_bxs"})
      for (int f = 0; f < wrfdc_field_count(); f++)
        if (name == std::string(wrfdc_field_name(f))) {
          const LayoutSeg g = layout_of(x, f);
          fields.push_back(f);
          a.emplace_back((size_t)g.ni * g.si);
        }
    for (auto &v : a) p.push_back(v.data());
  }
  int put(wrfdc_ctx *x) { return wrfdc_put_reference(x, (int)p.size(), fields.data(), p.data()); }
  int get(wrfdc_ctx *x) { return wrfdc_get_reference(x, (int)p.size(), fields.data(), p.data()); }
};
void transfer_call_failures() {
  for (int up = 0; up < 2; up++)
    for (long n = 0;; n++) {
      wrfdc_ctx *x = make_ctx(400, 90, 33, 6, 1);  // 35 MB of moist: a chunk for each worker
      Arrays A(x);
      rt::busy.clear();
      rt::fail_any = n;
      const int rc = up ? A.put(x) : A.get(x);
      const bool failed = rt::fail_any < 0;
      rt::fail_any = -1;
      rt::last = hipSuccess;
      CHECK(rc == WRFDC_OK || (failed && rc == WRFDC_EHIP));
      CHECK(rt::busy.empty());
      CHECK(A.put(x) == WRFDC_OK && A.get(x) == WRFDC_OK);
      wrfdc_destroy(x);
      if (!failed || n > 1000) break;
    }
}
// No pinned memory, memory for one worker, memory for one small chunk: the
// transfers work all the same; none at all: an error.
void transfer_short_memory() {
  const struct {
    const char *call;
    long after;
    int rc;
  } kinds[] = {{"hipHostMalloc", 0, WRFDC_OK}, {"hipMalloc", 1, WRFDC_OK}, {"hipMalloc", 0, WRFDC_OK}, {"hipMalloc", -1, WRFDC_EHIP}};
  for (auto &k : kinds) {
    wrfdc_ctx *x = make_ctx(400, 90, 33, 6, 1);
    Arrays A(x);
    rt::fail_name = k.call;
    rt::fail_left = std::max(k.after, 0L);
    rt::fail_times = k.after < 0 ? 2 : k.call == std::string("hipHostMalloc") ? 4 : 1;
    CHECK(A.put(x) == k.rc);
    rt::fail_left = -1;
    rt::fail_times = 1;
    rt::last = hipSuccess;
    CHECK(A.put(x) == WRFDC_OK && A.get(x) == WRFDC_OK);
    wrfdc_destroy(x);
  }
}
// Every allocation of a transfer failing in turn, those of its threads among
// them: an error or fewer threads, and no way out but the return.
void transfer_allocation_failures() {
  wrfdc_ctx *x = make_ctx(400, 90, 33, 6, 1);
  Arrays A(x);
  for (long n = 0;; n++) {
    g_alloc_left = n;
    const int rc = n % 2 ? A.put(x) : A.get(x);
    const bool failed = g_alloc_left < 0;
    g_alloc_left = -1;
    CHECK(rc == WRFDC_OK || (failed && rc == WRFDC_EHIP));
    CHECK(rt::busy.empty());
    if (!failed || n > 1000) break;
  }
  wrfdc_destroy(x);
}

// An ensemble's streams, events and graph: each created once, used while
// it lives, destroyed once, after its work has been waited for.
void ensemble_lifecycle() {
  std::vector<wrfdc_ctx *> m;
  for (int q = 0; q < 4; q++) m.push_back(make_ctx(24 + q, 20, 10));
  const size_t base = rt::live.size();
  for (int round = 0; round < 7; round++) {  // as a search over layouts does
    const int nb = round % 3 == 0 ? 1 : round % 3 == 1 ? 2 : 4;
    for (auto x : m) wrfdc_set_tile(x, "face_levels", round);
    wrfdc_ensemble *e = nullptr;
    CHECK(wrfdc_ensemble_create(m.data(), 4, nullptr, nb, &e) == WRFDC_OK);
    CHECK(wrfdc_ensemble_step(e, 3, 5.0) == WRFDC_OK);
    CHECK(wrfdc_ensemble_sync(e) == WRFDC_OK);
    for (auto x : m) CHECK(x->s == nullptr && !x->capturing);
    CHECK(wrfdc_ensemble_destroy(e) == WRFDC_OK);
    CHECK(rt::live.size() == base);
  }
  for (auto x : m) wrfdc_destroy(x);
}

// A destruction that fails is reported, and the rest is destroyed all the same;
// replays that cannot be waited for leave everything as it is.
void ensemble_destroy_failures() {
  wrfdc_ctx *x = make_ctx(24, 20, 10);
  const auto before = rt::live;
  for (const char *call : {"hipStreamSynchronize", "hipGraphExecDestroy", "hipGraphDestroy", "hipEventDestroy", "hipStreamDestroy"}) {
    wrfdc_ensemble *e = nullptr;
    CHECK(wrfdc_ensemble_create(&x, 1, nullptr, 2, &e) == WRFDC_OK);
    const size_t all = rt::live.size();
    CHECK(wrfdc_ensemble_step(e, 1, 0.0) == WRFDC_OK && wrfdc_ensemble_sync(e) == WRFDC_OK);
    rt::fail_name = call;
    rt::fail_left = 0;
    rt::fail_times = 1;
    CHECK(wrfdc_ensemble_destroy(e) == WRFDC_EHIP);
    rt::last = hipSuccess;
    if (call == std::string("hipStreamSynchronize")) {
      CHECK(rt::live.size() == all);
      for (auto &l : rt::live)
        if (!before.count(l.first)) std::free(l.first);
      rt::live = before;
    }
    CHECK(rt::live.size() == before.size());
  }
  CHECK(wrfdc_ensemble_destroy(nullptr) == WRFDC_OK);
  wrfdc_destroy(x);
}

// Every runtime call of the creation failing in turn: an error, the members
// as they were, nothing left behind, and a creation after it succeeds.
void ensemble_create_failures() {
  std::vector<wrfdc_ctx *> m;
  for (int q = 0; q < 3; q++) m.push_back(make_ctx(24 + q, 20, 10));
  const size_t base = rt::live.size();
  for (long n = 0;; n++) {
    wrfdc_ensemble *e = nullptr;
    rt::fail_any = n;
    const int rc = wrfdc_ensemble_create(m.data(), 3, nullptr, 2, &e);
    const bool failed = rt::fail_any < 0;
    rt::fail_any = -1;
    rt::last = hipSuccess;
    for (auto x : m) CHECK(x->s == nullptr && !x->capturing);
    if (rc == WRFDC_OK) {
      CHECK(!failed);
      CHECK(wrfdc_ensemble_step(e, 1, 0.0) == WRFDC_OK && wrfdc_ensemble_sync(e) == WRFDC_OK);
      wrfdc_ensemble_destroy(e);
    } else {
      CHECK(rc == WRFDC_EHIP && e == nullptr);
    }
    CHECK(rt::live.size() == base);
    CHECK(rt::capturing.empty());
    if (!failed || n > 5000) break;
  }
  for (auto x : m) wrfdc_destroy(x);
}

const struct {
  const char *name;
  void (*fn)();
} kChecks[] = {{"context_upload", context_upload},
               {"phi_tendency_blocks", phi_tendency_blocks},
               {"transfer_call_failures", transfer_call_failures},
               {"transfer_short_memory", transfer_short_memory},
               {"transfer_allocation_failures", transfer_allocation_failures},
               {"ensemble_lifecycle", ensemble_lifecycle},
               {"ensemble_destroy_failures", ensemble_destroy_failures},
               {"ensemble_create_failures", ensemble_create_failures}};
}  // namespace

int main(int argc, char **argv) {
  for (auto &c : kChecks)
    if (argc > 1 && c.name == std::string(argv[1])) {
      c.fn();
      for (auto &e : rt::errors) g_bad++, std::printf("%s\n", e.c_str());
      for (auto &l : rt::live) g_bad++, std::printf("%s never destroyed\n", l.second.c_str());
      std::printf("%s: %d\n", c.name, g_bad);
      return g_bad ? 1 : 0;
    }
  return 2;
}
