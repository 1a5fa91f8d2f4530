// The library's use of HIP resources and host memory: what it does when an allocation or a launch fails, and how
// much it allocates.  The program defines some HIP entry points itself; the library's calls reach these first, which
// count them, fail the one that a check asks for, and pass the others on to the runtime.
#include <dlfcn.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include <random>
#include <vector>

#include "qmcx.h"

typedef void* handle;   // hipStream_t, hipEvent_t
static int fail_malloc = 0, fail_launch = 0;   // the n-th call from now fails (0: none)
static std::map<handle, handle> recorded;      // event -> stream of its latest record that no other stream waited for
static size_t device_bytes = 0;   // allocated since it was last set to zero
static int pinned_calls = 0;      // pinned allocations since it was last set to zero
static size_t pinned_largest = 0; // the largest of them
static const int kOutOfMemory = 2;

static bool no_memory = false;    // operator new fails where the library itself calls it
static int refused = 0;
__attribute__((noinline)) void* operator new(std::size_t n) {
  Dl_info at;
  if (no_memory && dladdr(__builtin_return_address(0), &at) && std::strstr(at.dli_fname, "libqmcx")) {
    ++refused;
    throw std::bad_alloc();
  }
  void* p = std::malloc(n);
  if (!p) throw std::bad_alloc();
  return p;
}
__attribute__((noinline)) void operator delete(void* p) noexcept { std::free(p); }
__attribute__((noinline)) void operator delete(void* p, std::size_t) noexcept { std::free(p); }

template <typename F>
static F next(const char* name) {
  F f = (F)dlsym(RTLD_NEXT, name);
  if (!f) std::printf("no %s\n", name);
  return f;
}
extern "C" {
int hipMalloc(void** p, size_t bytes) {
  static auto f = next<int (*)(void**, size_t)>("hipMalloc");
  if (fail_malloc > 0 && --fail_malloc == 0) return kOutOfMemory;
  device_bytes += bytes;
  return f(p, bytes);
}
int hipHostMalloc(void** p, size_t bytes, unsigned flags) {
  static auto f = next<int (*)(void**, size_t, unsigned)>("hipHostMalloc");
  ++pinned_calls;
  pinned_largest = bytes > pinned_largest ? bytes : pinned_largest;
  return f(p, bytes, flags);
}
int hipGetLastError() {
  static auto f = next<int (*)()>("hipGetLastError");
  const int e = f();
  if (fail_launch > 0 && --fail_launch == 0) return kOutOfMemory;
  return e;
}
int hipEventRecord(handle ev, handle st) {
  static auto f = next<int (*)(handle, handle)>("hipEventRecord");
  recorded[ev] = st;
  return f(ev, st);
}
int hipStreamWaitEvent(handle st, handle ev, unsigned flags) {
  static auto f = next<int (*)(handle, handle, unsigned)>("hipStreamWaitEvent");
  auto it = recorded.find(ev);
  if (it != recorded.end() && it->second != st) recorded.erase(it);
  return f(st, ev, flags);
}
}

static int failures = 0;
static void check(bool ok, const char* what) {
  std::printf("%s: %s\n", ok ? "ok" : "FAILED", what);
  std::fflush(stdout);
  failures += ok ? 0 : 1;
}
static void must(int rc, const char* what) {
  if (rc == 0) return;
  std::printf("%s: %s\n", what, qmcx_last_error());
  std::fflush(stdout);
  ++failures;
}

// 2n electrons, n orbitals and nions ions in a cube
struct Model {
  int n, nions;
  double cell = 10.0;
  qmcx_system_t sys = nullptr;
  std::mt19937 gen{7};
  double uniform(double a, double b) { return std::uniform_real_distribution<double>(a, b)(gen); }
  Model(int orbitals, int ions) : n(orbitals), nions(ions) {
    const double lattice[9] = {cell, 0, 0, 0, cell, 0, 0, 0, cell};
    std::vector<double> ion(3 * (size_t)nions);
    for (double& x : ion) x = uniform(0, cell);
    std::vector<int> species(nions, 0);
    must(qmcx_system_create(&sys, lattice, nions, ion.data(), species.data(), 1, n, n), "qmcx_system_create");
    double p[8];
    for (double& x : p) x = uniform(-0.2, 0.2);
    must(qmcx_system_set_j1(sys, 0, 8, 2.5, 0.0, p), "qmcx_system_set_j1");
    for (int s = 0; s < 2; ++s) must(qmcx_system_set_j2(sys, s, 8, 3.0, 0.0, p), "qmcx_system_set_j2");
    const int ng[3] = {10, 10, 10}, npad = (n + 15) / 16 * 16;
    std::vector<float> coefs(13 * 13 * 13 * (size_t)npad);
    for (float& x : coefs) x = (float)uniform(-1, 1);
    must(qmcx_system_set_spline(sys, ng, n, npad, coefs.data(), lattice, 3), "qmcx_system_set_spline");
  }
  ~Model() { qmcx_system_destroy(sys); }
  std::vector<double> positions(int walkers) {
    std::vector<double> r((size_t)walkers * 2 * n * 3);
    for (double& x : r) x = uniform(0, cell);
    return r;
  }
};

// evaluateLog of enough electrons for them to be ordered by place: without the memory for that it evaluates
// them in their own order, and an error leaves no work of the side stream behind
static void evaluate_log() {
  Model m(160, 10);
  const int W = 26;
  const std::vector<double> R = m.positions(W);
  for (int precision : {QMCX_FP64, QMCX_FP32}) {
    qmcx_batch_t a, b;
    must(qmcx_batch_create(&a, m.sys, W, 1, precision), "qmcx_batch_create");
    must(qmcx_batch_create(&b, m.sys, W, 1, precision), "qmcx_batch_create");
    must(qmcx_batch_set_positions(a, R.data()), "qmcx_batch_set_positions");
    must(qmcx_batch_set_positions(b, R.data()), "qmcx_batch_set_positions");
    std::vector<double> la(W), lb(W);
    must(qmcx_evaluate_log(a, la.data()), "qmcx_evaluate_log");
    fail_malloc = 1;
    const int rc = qmcx_evaluate_log(b, lb.data());
    check(fail_malloc == 0, "evaluateLog asks for memory to order its electrons");
    fail_malloc = 0;
    check(rc == 0 && la == lb, "evaluateLog without that memory gives the same log|Psi|");
    int errors = 0;
    for (int k = 2; k < 12; ++k) {
      recorded.clear();
      fail_launch = k;
      if (qmcx_evaluate_log(a, la.data()) != 0) {
        ++errors;
        // ev_start, recorded on the batch's stream, was waited for by the side stream; the side
        // stream's own event must have been waited for by the batch's
        check(recorded.empty(), "a failed evaluateLog has joined the side stream");
      }
      fail_launch = 0;
    }
    check(errors > 0, "launches failed");
    must(qmcx_evaluate_log(a, la.data()), "qmcx_evaluate_log");
    check(la == lb, "evaluateLog after the errors");
    qmcx_batch_destroy(a);
    qmcx_batch_destroy(b);
  }
}

// device memory of a NonLocalPP evaluation: per slot of a walker's electrons' lists, the slot's index, its
// pair's distance and displacement, and for each of its twelve knots a ratio and a place in the order
static void nlpp_device_memory() {
  Model m(48, 10);
  const int W = 64, slots = 64;
  const std::vector<double> R = m.positions(W), spheres((size_t)W * 12 * 3, 0.5);
  qmcx_batch_t b;
  must(qmcx_batch_create(&b, m.sys, W, 1, QMCX_FP32), "qmcx_batch_create");
  must(qmcx_batch_set_positions(b, R.data()), "qmcx_batch_set_positions");
  must(qmcx_evaluate_log(b, nullptr), "qmcx_evaluate_log");
  std::vector<int> pairs((size_t)W * 2 * m.n);
  device_bytes = 0;
  must(qmcx_nlpp_evaluate(b, 2.0, spheres.data(), slots, nullptr, pairs.data()), "qmcx_nlpp_evaluate");
  const double per_slot = (double)device_bytes / ((double)W * 2 * m.n * slots);
  std::printf("%.1f bytes per slot\n", per_slot);
  check(per_slot <= 4 + 32 + 12 * (8 + 4) + 4, "device memory of a NonLocalPP evaluation");
  qmcx_batch_destroy(b);
}

// pinned host memory of NonLocalPP evaluations and virtual ratios
static void nlpp_pinned_memory() {
  const int slots = 64, N = 96;
  Model m(N / 2, 60);
  const int W = 64, part = 8;
  const std::vector<double> R = m.positions(W);
  std::vector<double> spheres((size_t)W * 12 * 3);
  for (double& x : spheres) x = m.uniform(-0.5, 0.5);
  auto batch = [&](int first, int walkers) {
    qmcx_batch_t b;
    must(qmcx_batch_create(&b, m.sys, walkers, 1, QMCX_FP32), "qmcx_batch_create");
    must(qmcx_batch_set_positions(b, R.data() + (size_t)first * N * 3), "qmcx_batch_set_positions");
    must(qmcx_evaluate_log(b, nullptr), "qmcx_evaluate_log");
    return b;
  };
  std::vector<double> ratios((size_t)W * N * slots * 12), parts(ratios);
  std::vector<int> pairs((size_t)W * N);
  auto evaluate = [&](qmcx_batch_t b, double rmax, double* out) {
    must(qmcx_nlpp_evaluate(b, rmax, spheres.data(), slots, out, pairs.data()), "qmcx_nlpp_evaluate");
  };
  // lists that grow from call to call
  qmcx_batch_t b = batch(0, W);
  pinned_calls = 0;
  for (int i = 0; i < 20; ++i) evaluate(b, 1.5 + 0.05 * i, ratios.data());
  std::printf("%d pinned allocations in 20 evaluations\n", pinned_calls);
  check(pinned_calls <= 6, "lists that grow seldom need larger pinned buffers");
  qmcx_batch_destroy(b);
  // a small request leaves a large block to the next batch that needs it
  b = batch(0, W);
  const double point[3] = {1.0, 2.0, 3.0};
  double ratio = 0;
  qmcx_batch_t one = batch(0, 1);
  must(qmcx_flex_evaluate_ratios(one, 0, 1, point, &ratio), "qmcx_flex_evaluate_ratios");
  pinned_calls = 0;
  evaluate(b, 2.4, ratios.data());
  check(pinned_calls == 0, "a batch takes the blocks that one like it gave back");
  qmcx_batch_destroy(one);
  // every ion is in reach: the list is longer than the buffers, which stay as they are
  pinned_largest = 0;
  evaluate(b, 9.0, ratios.data());
  std::printf("pinned allocation of %.1f MB for %.1f MB of ratios\n", 1e-6 * pinned_largest, 96e-6 * W * N * 60);
  check(pinned_largest <= size_t(14) << 20, "the pinned buffers do not grow with the list");
  qmcx_batch_destroy(b);
  const std::vector<double> all = spheres;
  for (int w = 0; w < W; w += part) {
    b = batch(w, part);
    std::copy(all.begin() + w * 36, all.begin() + (w + part) * 36, spheres.begin());
    evaluate(b, 9.0, parts.data() + (size_t)w * N * slots * 12);
    qmcx_batch_destroy(b);
  }
  check(ratios == parts, "the ratios of a long list are those of its parts");
}

// a batch given back when the host has no memory for the list of free pinned blocks
static void destroy_without_memory() {
  Model m(48, 10);
  const double point[3] = {1.0, 2.0, 3.0};
  std::vector<qmcx_batch_t> batches(40);
  const std::vector<double> R = m.positions(1);
  for (qmcx_batch_t& b : batches) {
    must(qmcx_batch_create(&b, m.sys, 1, 1, QMCX_FP64), "qmcx_batch_create");
    must(qmcx_batch_set_positions(b, R.data()), "qmcx_batch_set_positions");
    must(qmcx_evaluate_log(b, nullptr), "qmcx_evaluate_log");
    double ratio;
    must(qmcx_flex_evaluate_ratios(b, 0, 1, point, &ratio), "qmcx_flex_evaluate_ratios");
  }
  int rc = 0;
  no_memory = true;   // the list of the blocks has to grow for some of them
  for (qmcx_batch_t b : batches) rc |= qmcx_batch_destroy(b);
  no_memory = false;
  check(rc == 0 && refused > 0, "batches destroyed without host memory");
}

int main() {
  evaluate_log();
  nlpp_device_memory();
  nlpp_pinned_memory();
  destroy_without_memory();
  std::printf(failures == 0 ? "All checks passed\n" : "%d checks failed\n", failures);
  return failures == 0 ? 0 : 1;
}
