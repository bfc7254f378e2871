// The library's host code (swe_api.cpp and what it calls) over a device that
// is host memory: HIP's calls and the kernel launches are replaced by host
// stand-ins, which record, simulate the parts a check looks at, and fail or
// wait where it asks for that.  Built with g++ into a shared library by
// tests/test_api_host.py; launches that no check reaches stay undefined.
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <thread>

#include "../../swe_fvm_amd/csrc/swe_api.cpp"

namespace fake {

std::mutex m;
std::map<void*, size_t> held;  // device allocations
size_t held_bytes = 0;
std::function<hipError_t()> on_malloc;  // called before an allocation
std::function<void(void*)> on_free;     // called in every hipFree
std::vector<std::function<void()>>* capture = nullptr;
std::vector<std::vector<std::function<void()>>> graphs;
const char* fail_launch = nullptr;  // the launch that fails, once
int launches = 0;                   // kernels so far
int flux_items = 0;                 // edges per thread of the last flux pass
int64_t listed = 0;                 // cells a reconstruction lists for pass 2
int64_t list_max = 0;               // the longest the list has been

hipError_t launch(const char* name, std::function<void()> f) {
  if (fail_launch && std::string(fail_launch) == name) {
    fail_launch = nullptr;
    return hipErrorLaunchFailure;
  }
  if (std::strcmp(name, "memcpy") != 0) launches += 1;
  if (capture) capture->push_back(std::move(f));
  else f();
  return hipSuccess;
}

}  // namespace fake

extern "C" {
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error of the stand-in device"; }
hipError_t hipMalloc(void** p, size_t n) {
  if (fake::on_malloc)
    if (const hipError_t e = fake::on_malloc(); e != hipSuccess) return e;
  *p = std::malloc(n);
  std::lock_guard<std::mutex> lock(fake::m);
  fake::held[*p] = n;
  fake::held_bytes += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (fake::on_free) fake::on_free(p);
  {
    std::lock_guard<std::mutex> lock(fake::m);
    if (!fake::held.count(p)) std::abort();
    fake::held_bytes -= fake::held[p];
    fake::held.erase(p);
  }
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  return fake::launch("memcpy", [=] { std::memcpy(d, s, n); });
}
hipError_t hipMemset(void* d, int v, size_t n) { std::memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return fake::launch("memset", [=] { std::memset(d, v, n); }); }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = nullptr; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  fake::graphs.emplace_back();
  fake::capture = &fake::graphs.back();
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  fake::capture = nullptr;
  *g = (hipGraph_t)fake::graphs.size();  // number + 1
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
  *e = (hipGraphExec_t)g;
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
  for (auto& f : fake::graphs[size_t(e) - 1]) f();
  return hipSuccess;
}
}

namespace swe {

bool fused_fits(const DevTiles&) { return true; }
hipError_t scratch_address(double** p) {
  static double scratch[1];
  *p = scratch;
  return hipSuccess;
}
hipError_t launch_setup_geometry(const DevMesh&, const DevGeomOut&, const DevTiles*, bool, hipStream_t) { return hipSuccess; }
hipError_t launch_rows_in(const double* rows, const DevOut& O, int64_t T, int64_t Tpad, hipStream_t) {
  return fake::launch("rows_in", [=] {
    for (int64_t i = 0; i < Tpad; ++i) {
      const int64_t a = O.at(i);
      O.w[a] = i < T ? rows[3 * i] : 0.;
      O.u[a] = i < T ? rows[3 * i + 1] : 0.;
      O.v[a] = i < T ? rows[3 * i + 2] : 0.;
    }
  });
}
hipError_t launch_rows_out(const DevState& S, double* rows, int64_t T, hipStream_t) {
  return fake::launch("rows_out", [=] {
    for (int64_t i = 0; i < T; ++i) {
      rows[3 * i] = S.w[S.at(i)];
      rows[3 * i + 1] = S.u[S.at(i)];
      rows[3 * i + 2] = S.v[S.at(i)];
    }
  });
}
hipError_t launch_relayout(const DevState& S, const DevOut& O, int64_t T, hipStream_t) {
  return fake::launch("relayout", [=] {
    for (int64_t i = 0; i < T; ++i) {
      O.w[O.at(i)] = S.w[S.at(i)];
      O.u[O.at(i)] = S.u[S.at(i)];
      O.v[O.at(i)] = S.v[S.at(i)];
    }
  });
}
// pass 1 appends `listed` cells to pass 2's list
hipError_t launch_recon1(const DevMesh&, const DevState&, const DevWork& W, int, hipStream_t, bool zero_count,
                         unsigned long long*, const DevTiles*) {
  return fake::launch("recon1", [=] {
    if (zero_count) *W.pw_count = 0u;
    *W.pw_count += unsigned(fake::listed);
    fake::list_max = std::max<int64_t>(fake::list_max, *W.pw_count);
  });
}
hipError_t launch_recon2(const DevMesh&, const DevState&, const DevWork&, int, hipStream_t) {
  return fake::launch("recon2", [] {});
}
hipError_t launch_zero_count(unsigned int* c, hipStream_t) { return fake::launch("zero_count", [=] { *c = 0u; }); }
hipError_t launch_flux(const DevMesh&, const DevState&, const DevWork&, int, int, double, unsigned long long*, int items,
                       int, hipStream_t, CflMode) {
  fake::flux_items = items;
  return fake::launch("flux", [] {});
}
hipError_t launch_drain(const DevMesh&, const DevState&, const DevWork&, int, hipStream_t) {
  return fake::launch("drain", [] {});
}
// a stage: a0 U0 + a1 S + coef, or S + 1
static void stage(const DevMesh& M, const DevState& S, const DevState& U0, const DevOut& O, const StageArgs& A) {
  for (int64_t i = M.c0; i < M.c1; ++i) {
    const double w = S.w[S.at(i)];
    O.w[O.at(i)] = A.a0 != 0. ? A.a0 * U0.w[U0.at(i)] + A.a1 * w + A.coef : w + 1.;
    O.u[O.at(i)] = S.u[S.at(i)];
    O.v[O.at(i)] = S.v[S.at(i)];
  }
  if (A.pw_clear) *A.pw_clear = 0u;
}
hipError_t launch_update(const DevMesh& M, const DevState& S, const DevState& U0, const DevOut& O, const DevWork&,
                         const StageArgs& A, int, int, hipStream_t) {
  return fake::launch("update", [=] { stage(M, S, U0, O, A); });
}
hipError_t launch_fused(const DevMesh& M, const DevTiles&, const DevState& S, const DevState& U0, const DevOut& O,
                        const DevWork&, const StageArgs& A, int, int, int, hipStream_t, bool, bool) {
  return fake::launch("fused", [=] { stage(M, S, U0, O, A); });
}
hipError_t launch_batch_reset_r(const DevBatch&, int, hipStream_t) { return fake::launch("batch_reset_r", [] {}); }
hipError_t launch_batch_advance(const DevBatch& B, double, double, hipStream_t) {
  return fake::launch("batch_advance", [=] {
    for (int k = 0; k < B.n; ++k) B.steps[k] += 1;
  });
}

}  // namespace swe

namespace {

struct Mesh {
  swe_topology* t = nullptr;
  double* xyz = nullptr;
  int64_t nn = 0;
  explicit Mesh(int64_t n) { swe_mesh_struct(n, n, 0.1, 0., 0., &xyz, &nn, &t); }
  ~Mesh() {
    swe_free(xyz);
    swe_topology_destroy(t);
  }
};

swe_solver* ensemble(const Mesh& m, int members) {
  std::vector<const swe_topology*> t(size_t(members), m.t);
  std::vector<const double*> x(size_t(members), m.xyz);
  swe_solver* s = nullptr;
  if (swe_batch_create(members, t.data(), x.data(), 1, 2, 0., 0., 0, 0, &s) != SWE_OK) return nullptr;
  return s;
}

}  // namespace

// An ensemble step whose launch fails leaves pass 2's list to be emptied
// before the next run: the list (T entries) never holds more than one
// reconstruction's cells.  Returns the longest it has been, or -1.
extern "C" int64_t list_after_failed_launch(const char* launch, int scheme, int fused, int graph, int64_t* cells) {
  Mesh m(4);
  swe_solver* s = ensemble(m, 3);
  if (!s) return -1;
  *cells = s->T;
  int64_t done, act;
  swe_set_fused(s, fused, nullptr);
  fake::listed = s->T;
  fake::list_max = 0;
  int rc = swe_batch_run(s, scheme, 0.15, 1e9, 3, graph, &done, &act);
  fake::fail_launch = launch;
  const int failed = swe_batch_run(s, scheme, 0.2, 1e9, 3, graph, &done, &act);
  fake::fail_launch = nullptr;
  fake::capture = nullptr;
  rc |= swe_batch_run(s, scheme, 0.2, 1e9, 3, graph, &done, &act);
  swe_destroy(s);
  return rc == SWE_OK && failed == SWE_ERR_DEVICE ? fake::list_max : -1;
}

// Euler steps of an ensemble after `layouts` changes of the state layout:
// every step adds 1 to w.  Returns the steps that the state shows, or -1.
extern "C" int64_t euler_steps_after_layouts(int layouts, int graph, int runs, int64_t steps) {
  Mesh m(4);
  swe_solver* s = ensemble(m, 3);
  if (!s) return -1;
  std::vector<double> prim(size_t(3 * s->T), 0.);
  int rc = swe_set_state(s, prim.data());
  for (int k = 0; k < layouts; ++k) rc |= swe_set_layout(s, k % 2 == 0 ? 64 : 0);
  int64_t done, act;
  for (int k = 0; k < runs; ++k) rc |= swe_batch_run(s, SWE_SCHEME_EULER, 0.15, 1e9, steps, graph, &done, &act);
  rc |= swe_get_state(s, prim.data());
  const int64_t T = s->T;
  swe_destroy(s);
  for (int64_t i = 0; i < T; ++i)
    if (prim[size_t(3 * i)] != prim[0]) rc = SWE_ERR_ARG;
  return rc == SWE_OK ? int64_t(prim[0]) : -1;
}

namespace fake {
std::function<void()> in_stats;  // called by swe_state_stats while it holds its memory
}
namespace swe {
int64_t integrals_blocks(const DevMesh&) { return 1; }
hipError_t launch_stats(const DevMesh&, const DevState&, double*, double*, hipStream_t) {
  if (fake::in_stats) fake::in_stats();
  return hipSuccess;
}
}  // namespace swe

namespace {

// a thread's call that waits in a device call until it is let go
struct Gate {
  std::mutex m;
  std::condition_variable cv;
  bool reached = false, open = false;
  void wait() {
    std::unique_lock<std::mutex> l(m);
    reached = true;
    cv.notify_all();
    cv.wait(l, [&] { return open; });
  }
  void until_reached() {
    std::unique_lock<std::mutex> l(m);
    cv.wait(l, [&] { return reached; });
  }
  void let_go() {
    std::lock_guard<std::mutex> l(m);
    open = true;
    cv.notify_all();
  }
};

}  // namespace

// While one thread waits in the device (0: hipMalloc of a workspace, 1: hipFree
// of a destroyed solver's, 2: hipFree of a given-back one), another solver's
// call on another thread goes through.  1 if it does within 10 s.
extern "C" int other_solver_goes_on(int kind) {
  Mesh m(4);
  swe_solver *a = nullptr, *b = nullptr;
  if (swe_create(m.t, m.xyz, 1, 2, 0., 0., 0, 0, &a) || swe_create(m.t, m.xyz, 1, 2, 0., 0., 0, 0, &b)) return -1;
  double out[5];
  if (kind != 0 && swe_state_stats(a, out)) return -1;
  Gate gate;
  std::thread::id slow;
  std::mutex id;
  auto hook = [&] {
    bool here;
    {
      std::lock_guard<std::mutex> l(id);
      here = std::this_thread::get_id() == slow;
    }
    if (here) gate.wait();
  };
  if (kind == 0) fake::on_malloc = [&] { hook(); return hipSuccess; };
  else fake::on_free = [&, kept = (void*)a->work.p](void* p) { if (p == kept) hook(); };
  std::thread ta([&] {
    {
      std::lock_guard<std::mutex> l(id);
      slow = std::this_thread::get_id();
    }
    double o[5];
    if (kind == 0) swe_state_stats(a, o);
    else if (kind == 1) swe_destroy(a);
    else swe_release_workspaces();
  });
  gate.until_reached();
  std::atomic<bool> done{false};
  std::thread tb([&] {
    double o[5];
    if (swe_state_stats(b, o) == SWE_OK) done = true;
  });
  for (int k = 0; k < 1000 && !done; ++k) std::this_thread::sleep_for(std::chrono::milliseconds(10));
  const int ok = done ? 1 : 0;
  gate.let_go();
  ta.join();
  tb.join();
  fake::on_malloc = nullptr;
  fake::on_free = nullptr;
  if (kind != 1) swe_destroy(a);
  swe_destroy(b);
  return ok;
}

// Device bytes that n solvers keep after a call each, after they are given back
// in the middle of one solver's call (which keeps its own), after that, and
// after another call each
extern "C" int kept_bytes(int n, int64_t* kept) {
  Mesh m(4);
  std::vector<swe_solver*> s(size_t(n), nullptr);
  for (auto& x : s)
    if (swe_create(m.t, m.xyz, 1, 2, 0., 0., 0, 0, &x)) return -1;
  const size_t base = fake::held_bytes;
  auto call = [&] {
    double o[5];
    for (auto x : s)
      if (swe_state_stats(x, o)) return -1;
    return 0;
  };
  int rc = call();
  kept[0] = int64_t(fake::held_bytes - base);
  fake::in_stats = [] { swe_release_workspaces(); };
  double o[5];
  rc |= swe_state_stats(s[0], o);
  fake::in_stats = nullptr;
  kept[1] = int64_t(fake::held_bytes - base);
  swe_release_workspaces();
  kept[2] = int64_t(fake::held_bytes - base);
  rc |= call();
  kept[3] = int64_t(fake::held_bytes - base);
  // an allocation that fails takes them back and is tried again
  int fails = 1;
  fake::on_malloc = [&] { return fails-- > 0 ? hipErrorOutOfMemory : hipSuccess; };
  std::vector<double> wp(size_t(s[0]->V));
  swe_solver* x = nullptr;
  rc |= swe_create(m.t, m.xyz, 1, 2, 0., 0., 0, 0, &x);
  fake::on_malloc = nullptr;
  if (x) swe_destroy(x);
  kept[4] = int64_t(fake::held_bytes - base);
  for (auto y : s) swe_destroy(y);
  return rc;
}

// Edges per thread of the flux passes of a solver of n x n squares: as created,
// after its tuning is read and set again, and after the settings 4, 2 and 1;
// got: what the getter says after each
extern "C" int flux_items_launched(int n, int* items, int* got) {
  Mesh m(n);
  swe_solver* s = nullptr;
  if (swe_create(m.t, m.xyz, 1, 2, 0., 0., 0, 0, &s)) return -1;
  int rc = 0;
  auto pass = [&](int k) {
    double r;
    int u;
    rc |= swe_compute_fluxes(s, &r) | swe_get_tuning(s, &got[k], &u);
    items[k] = fake::flux_items;
    return u;
  };
  const int u = pass(0);
  rc |= swe_set_tuning(s, got[0], u);
  pass(1);
  const int set[3] = {4, 2, 1};
  for (int k = 0; k < 3; ++k) {
    rc |= swe_set_tuning(s, set[k], u);
    pass(2 + k);
  }
  swe_destroy(s);
  return rc;
}

// A state set and read again on n x n squares in a layout: the launches that
// it took, or -1 where the state differs or a padding cell is not zero
extern "C" int launches_of_a_crossing(int n, int layout) {
  Mesh m(n);
  swe_solver* s = nullptr;
  if (swe_create(m.t, m.xyz, 1, 2, 0., 0., 0, 0, &s)) return -1;
  int rc = swe_set_layout(s, layout);
  std::vector<double> a(size_t(3 * s->T)), b(a.size());
  for (size_t k = 0; k < a.size(); ++k) a[k] = double(k + 1);
  std::memset(s->sbuf[s->cur], 0xff, sizeof(double) * size_t(3 * s->Tpad));
  const int before = fake::launches;
  rc |= swe_set_state(s, a.data());
  const int set = fake::launches - before;
  const DevState S = state_of(s, s->cur);
  for (int64_t i = s->T; i < s->Tpad; ++i)
    if (S.w[S.at(i)] != 0. || S.u[S.at(i)] != 0. || S.v[S.at(i)] != 0.) rc = SWE_ERR_ARG;
  rc |= swe_get_state(s, b.data());
  const int all = fake::launches - before;
  if (a != b || set * 2 != all) rc = SWE_ERR_ARG;
  swe_destroy(s);
  return rc ? -1 : all;
}
