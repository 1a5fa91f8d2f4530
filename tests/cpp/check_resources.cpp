// The library's use of HIP resources: what it does when an allocation fails.  The program
// defines some HIP entry points itself; the library's calls reach these first, which fail the one that a check
// asks for and pass the others on to the runtime.
#include <dlfcn.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "qmcx.h"

static int fail_malloc = 0;   // the n-th call from now fails (0: none)
static const int kOutOfMemory = 2;

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
  return f(p, bytes);
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
// them in their own order
static void evaluate_log() {
  Model m(48, 10);
  const int W = 91;
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
    qmcx_batch_destroy(a);
    qmcx_batch_destroy(b);
  }
}

int main() {
  evaluate_log();
  std::printf(failures == 0 ? "All checks passed\n" : "%d checks failed\n", failures);
  return failures == 0 ? 0 : 1;
}
