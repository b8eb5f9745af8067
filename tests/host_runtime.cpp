// A HIP runtime of host memory for CPU tests of the engine's host code.
// Loaded ahead of libmpci_tdse.so, it takes the place of the runtime calls
// the library makes: device memory is malloc'ed, copies are done at once,
// and a kernel launch is counted by name.  Of the kernels only what the host
// code reads back is carried out: the step control (every attempt accepted,
// every accepted step adds 1 to each component of the state), the state
// copies and the save at the start of a persistent launch.
#include <hip/hip_runtime.h>

#include <chrono>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "../mp-citdse_amd/csrc/kernels.hpp"

using namespace mpci;

namespace {
std::recursive_mutex mu;
std::map<const void *, std::string> names;   // kernel stubs
std::map<void *, size_t> live;               // allocations
size_t fail_above = ~(size_t)0, fail_from = 1, fail_to = 0, alloc_us = 0,
       fail_unit = 0, fail_most = 0;
int abort_after = -1;                        // persistent launches give up
std::vector<std::string> launched;
std::vector<int> attempts;                   // of each persistent launch
size_t lds = 0;                              // dynamic LDS of the last one
long long stored = 0;                        // stages that kept their input
struct Cost {
  std::string what;
  double us, once;
  int nth, seen;
};
std::vector<Cost> costs;
double now_us = 0.0;                         // the device's clock
struct Rec {
  std::vector<std::function<void()>> work;
};
Rec *capture = nullptr;
struct Config {
  dim3 g, b;
  size_t lds;
  hipStream_t st;
};
thread_local std::vector<Config> config;

void step(Ctl &c, int p, const double *hs) {
  c.accept = 0;
  if (c.done) return;
  c.attempts++;
  c.accept = 1;
  c.accepted++;
  c.nlog++;
  c.hacc = c.hc;
  c.nrm = 1.0;
  if (c.mode == kModeAdaptive) {
    if (c.last) {
      c.t = c.t_end;
      c.done = 1;
    } else {
      c.t += c.hc;
    }
    if (!c.done && c.attempts >= c.max_attempts) {
      c.done = 1;
      c.status = -1;
    }
    c.last = c.t + c.h >= c.t_end;
    c.hc = c.last ? c.t_end - c.t : c.h;
  } else {
    c.t += c.hc;
    c.step++;
    if (c.step >= c.nsteps)
      c.done = 1;
    else if (c.mode == kModeSchedule)
      c.hc = hs[(long long)p * c.hstride + c.step];
  }
}

void apply(double2 *X, Ctl &c, LogEnt *log, int logcap, int track, int N,
           int P, int p) {
  if (!c.accept) return;
  for (int i = 0; i < N; ++i) {
    X[(long long)i * P + p].x += 1.0;
    X[(long long)i * P + p].y += 1.0;
  }
  const double2 x = X[(long long)track * P + p];
  if (c.nlog <= logcap)
    log[(long long)(c.nlog - 1) * P + p] = LogEnt{c.t, c.hacc, x.x};
}

template <class A>
void persistent(const A &a, int P) {
  const int n = abort_after >= 0 ? std::min(abort_after, a.attempts) : a.attempts;
  if (a.limit_ms < 0) {
    *a.abort_flag = 1;
    return;
  }
  for (int p = 0; p < P; ++p)
    for (int k = 0; k < n && !a.ctl[p].done; ++k) {
      step(a.ctl[p], p, a.hs);
      apply(a.X, a.ctl[p], a.log, a.logcap, a.track, a.N, P, p);
    }
  if (abort_after >= 0) *a.abort_flag = 1;
}

template <class T>
T arg(void **args, int i) {
  return *static_cast<T *>(args[i]);
}

hipError_t launch(const void *fn, void **args) {
  std::lock_guard<std::recursive_mutex> lk(mu);
  const std::string name = names.count(fn) ? names[fn] : "?";
  auto is = [&](const char *s) { return name.find(s) != std::string::npos; };
  std::function<void()> f = [] {};
  if (is("k_rows_begin")) {
    const auto X = arg<const double2 *>(args, 6);
    const int NP = arg<int>(args, 7), P = arg<int>(args, 10);
    const auto Xs = arg<double2 *>(args, 8);
    const auto ctl = arg<Ctl *>(args, 9);
    const auto flag = arg<int *>(args, 11);
    f = [=] {
      std::memcpy(Xs, X, sizeof(double2) * NP);
      for (int p = 0; p < P; ++p) ctl[P + p] = ctl[p];
      *flag = 0;
    };
  } else if (is("k_rows_run")) {
    // of several batches, or of one
    RowRuns r{};
    if (is("ELb1E")) {
      r = arg<RowRuns>(args, 0);
    } else {
      r.n = 1;
      r.run[0] = arg<RowRun>(args, 0);
    }
    attempts.push_back(r.run[0].attempts);
    lds = config.back().lds;
    f = [=] {
      for (int i = 0; i < r.n; ++i) persistent(r.run[i], r.run[i].P);
    };
  } else if (is("k_tiles_run")) {
    const auto a = arg<TileRun>(args, 0);
    attempts.push_back(a.attempts);
    lds = config.back().lds;
    f = [=] { persistent(a, 1); };
  } else if (is("k_finalize_g") || is("k_apply_g")) {
    const auto m = arg<const GroupMember *>(args, 0);
    const int nm = arg<int>(args, 1);
    const bool fin = is("k_finalize_g");
    f = [=] {
      for (int i = 0; i < nm; ++i)
        for (int p = 0; p < m[i].P; ++p)
          if (fin)
            step(m[i].sa.ctl[p], p, m[i].hs);
          else
            apply(m[i].X, m[i].sa.ctl[p], m[i].log, m[i].logcap, m[i].track,
                  m[i].N, m[i].P, p);
    };
  } else if (is("k_finalize")) {
    const auto ctl = arg<Ctl *>(args, 0);
    const int P = arg<int>(args, 3);
    const auto hs = arg<const double *>(args, 4);
    f = [=] {
      for (int p = 0; p < P; ++p) step(ctl[p], p, hs);
    };
  } else if (is("k_apply")) {
    const auto X = arg<double2 *>(args, 0);
    const auto Y = arg<double2 *>(args, 1);
    const auto ctl = arg<Ctl *>(args, 2);
    const auto log = arg<LogEnt *>(args, 3);
    const int cap = arg<int>(args, 4), track = arg<int>(args, 5),
              N = arg<int>(args, 6), P = arg<int>(args, 7);
    f = [=] {
      for (int p = 0; p < P; ++p) apply(X, ctl[p], log, cap, track, N, P, p);
      // the candidate state, which is not the committed one
      for (long long i = 0; i < (long long)N * P; ++i) Y[i].x = Y[i].y = -1.0;
    };
  } else if (is("k_copy_strided")) {
    const auto dst = arg<double2 *>(args, 0);
    const int ds = arg<int>(args, 1), dp = arg<int>(args, 2);
    const auto src = arg<const double2 *>(args, 3);
    const int ss = arg<int>(args, 4), sp = arg<int>(args, 5),
              n = arg<int>(args, 6), np = (int)config.back().g.y;
    f = [=] {
      for (long long y = 0; y < np; ++y)
        for (long long i = 0; i < n; ++i)
          dst[y * dp + i * ds] = src[y * sp + i * ss];
    };
  } else if (is("k_small_stage") || is("k_stage1") || is("7k_stageI")) {
    const auto a = arg<StageArgs>(args, 0);
    f = [=] { stored += a.xs_store != nullptr && !a.ctl[0].done; };
  }
  auto run = [=] {
    launched.push_back(name);
    double us = 10.0;
    for (Cost &c : costs)
      if (name.find(c.what) != std::string::npos)
        us = ++c.seen == c.nth ? c.once : c.us;
    now_us += us;
    f();
  };
  if (capture)
    capture->work.push_back(run);
  else
    run();
  return hipSuccess;
}
}  // namespace

extern "C" {
// ---- controls for the tests ---------------------------------------------
void rt_fail_above(size_t bytes) { fail_above = bytes; }
void rt_fail_at(size_t from, size_t to) {
  fail_from = from;
  fail_to = to;
}
// multiples of unit, more than `most` of it
void rt_fail_multiples(size_t unit, size_t most) {
  fail_unit = unit;
  fail_most = most;
}
void rt_alloc_us(size_t us) { alloc_us = us; }
void rt_abort_after(int n) { abort_after = n; }
size_t rt_live() { return live.size(); }
size_t rt_live_bytes() {
  size_t n = 0;
  for (auto &a : live) n += a.second;
  return n;
}
void rt_cost(const char *what, double us, double once, int nth) {
  costs.push_back({what, us, once, nth, 0});
}
int rt_launched(const char *what) {
  int n = 0;
  for (auto &s : launched) n += s.find(what) != std::string::npos;
  return n;
}
void rt_clear() {
  launched.clear();
  attempts.clear();
  stored = 0;
}
int rt_attempts(int *out, int cap) {
  for (int i = 0; i < cap && i < (int)attempts.size(); ++i)
    out[i] = attempts[i];
  return (int)attempts.size();
}
long long rt_stored() { return stored; }
size_t rt_lds() { return lds; }

// ---- the runtime ----------------------------------------------------------
void **__hipRegisterFatBinary(const void *) {
  static void *h;
  return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name,
                           unsigned, void *, void *, dim3 *, dim3 *, int *) {
  names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int,
                      int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds,
                                      hipStream_t st) {
  config.push_back({g, b, lds, st});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds,
                                     hipStream_t *st) {
  *g = config.back().g;
  *b = config.back().b;
  *lds = config.back().lds;
  *st = config.back().st;
  config.pop_back();
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3 g, dim3 b, void **args,
                           size_t lds, hipStream_t st) {
  config.push_back({g, b, lds, st});
  const hipError_t e = launch(fn, args);
  config.pop_back();
  return e;
}
hipError_t hipLaunchCooperativeKernel(const void *fn, dim3 g, dim3 b,
                                      void **args, unsigned lds,
                                      hipStream_t st) {
  return hipLaunchKernel(fn, g, b, args, lds, st);
}
hipError_t hipExtLaunchKernel(const void *fn, dim3 g, dim3 b, void **args,
                              size_t lds, hipStream_t st, hipEvent_t,
                              hipEvent_t, int) {
  return hipLaunchKernel(fn, g, b, args, lds, st);
}
hipError_t hipMalloc(void **p, size_t n) {
  if (alloc_us)
    std::this_thread::sleep_for(std::chrono::microseconds(alloc_us));
  std::lock_guard<std::recursive_mutex> lk(mu);
  *p = nullptr;
  if (n > fail_above || (n >= fail_from && n <= fail_to) ||
      (fail_unit && n % fail_unit == 0 && n / fail_unit > fail_most))
    return hipErrorOutOfMemory;
  *p = std::calloc(n, 1);
  live[*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  std::lock_guard<std::recursive_mutex> lk(mu);
  live.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = std::calloc(n, 1);
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind,
                          hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpy2D(void *d, size_t dp, const void *s, size_t sp, size_t w,
                       size_t h, hipMemcpyKind) {
  for (size_t i = 0; i < h; ++i)
    std::memcpy((char *)d + i * dp, (const char *)s + i * sp, w);
  return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
  return hipMemset(d, v, n);
}
hipError_t hipMemsetD32Async(hipDeviceptr_t d, int v, size_t n, hipStream_t) {
  for (size_t i = 0; i < n; ++i) static_cast<int *>(d)[i] = v;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
  static char scratch[10 << 20];
  *p = scratch;
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int) {
  *v = a == hipDeviceAttributeMultiprocessorCount         ? 256
       : a == hipDeviceAttributeMaxSharedMemoryPerBlock ? 160 << 10
                                                        : 1;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = (hipStream_t)std::malloc(1);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  std::free(s);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = (hipEvent_t) new double(0.0);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  delete (double *)e;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  *(double *)e = now_us;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) {
  *ms = (float)((*(double *)b - *(double *)a) * 1e-3);
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  capture = new Rec;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
  *g = (hipGraph_t)capture;
  capture = nullptr;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t g,
                               hipGraphNode_t *, char *, size_t) {
  *x = (hipGraphExec_t) new Rec(*(Rec *)g);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t) {
  for (auto &w : ((Rec *)x)->work) w();
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  delete (Rec *)g;
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x) {
  delete (Rec *)x;
  return hipSuccess;
}
}  // extern "C"
