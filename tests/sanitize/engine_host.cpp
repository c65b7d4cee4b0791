// Host side of the engine and the solvers over the stand-in HIP runtime
// (hip_stub.cpp): built with AddressSanitizer and UndefinedBehaviorSanitizer and
// run by tests/test_host_runtime.py, one scenario per run.  Kernels do nothing
// there, so no result is checked, only what the host does around them.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <string>
#include <utility>
#include <vector>

#include "../../include/avionic.h"
#include "hip_stub.hpp"

#define CHECK(cond)                                                              \
  do {                                                                           \
    if (!(cond)) {                                                               \
      std::fprintf(stderr, "engine_host: line %d: %s\n", __LINE__, #cond);       \
      std::exit(1);                                                              \
    }                                                                            \
  } while (0)

// Host allocations of the library: the one that `fail_new` counts down to throws.
static long fail_new = 0;
void *operator new(size_t n) {
  if (fail_new > 0 && !stub_inside() && --fail_new == 0) throw std::bad_alloc();
  if (void *p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void *operator new(size_t n, const std::nothrow_t &) noexcept { return std::malloc(n ? n : 1); }
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

namespace {

constexpr size_t kMiB = size_t(1) << 20;

float *dev(size_t floats) {
  void *p = nullptr;
  CHECK(hipMalloc(&p, sizeof(float) * floats) == hipSuccess);
  for (size_t i = 0; i < floats; ++i) static_cast<float *>(p)[i] = 1.f;
  return static_cast<float *>(p);
}
// A request of a method (AVIONIC_*), its inputs allocated here.
struct Req {
  avionic_request_desc d{};
  avionic_params p{};
  Req(int method, unsigned T, unsigned H, unsigned W, unsigned C, unsigned its, int dual) {
    CHECK(avionic_default_params((avionic_method)method, &p) == 0);
    p.maxIt = its;
    p.dualStorage = dual;
    p.adaptLambda = 0;
    p.lambda = 1.0;
    if (method == AVIONIC_TVTEMP) p.dt = 0.8;
    d.method = (avionic_method)method;
    d.width = W, d.height = H, d.coils = C, d.frames = T;
    const size_t n = (size_t)T * H * W;
    mask = dev(n), data = dev(2 * n * C), b1 = dev((size_t)2 * C * H * W), out = dev(2 * n);
    d.mask = mask, d.data = data, d.b1 = b1;
  }
  Req(Req &&o) : d(o.d), p(o.p), mask(o.mask), data(o.data), b1(o.b1), out(o.out) { o.mask = nullptr; }
  ~Req() {
    if (!mask) return;
    for (float *f : {mask, data, b1, out}) (void)hipFree(f);
  }
  int submit(avionic_engine *e, long long *id) {
    d.params = &p;
    return avionic_engine_submit(e, &d, id);
  }
  float *mask, *data, *b1, *out;
};
avionic_engine_config config(int graphs, int tick) {
  avionic_engine_config c{};
  c.use_graphs = graphs;
  c.iterations_per_tick = tick;
  c.max_queue = -1;
  return c;
}
avionic_engine *engine(const avionic_engine_config &c) {
  avionic_engine *e = nullptr;
  CHECK(avionic_engine_create(&c, &e) == 0);
  return e;
}
avionic_engine_counts counts(const avionic_engine *e) {
  avionic_engine_counts c{};
  CHECK(avionic_engine_counters(e, &c) == 0);
  return c;
}
// Submits every request and steps the engine until each was polled.
void run_all(avionic_engine *e, std::vector<Req> &reqs) {
  std::vector<long long> id(reqs.size());
  for (size_t i = 0; i < reqs.size(); ++i) CHECK(reqs[i].submit(e, &id[i]) == 0);
  size_t left = reqs.size();
  for (int steps = 0; left > 0; ++steps) {
    CHECK(steps < 10000 && avionic_engine_step(e, nullptr) >= 0);
    for (size_t i = 0; i < reqs.size(); ++i)
      if (id[i] >= 0) {
        const int r = avionic_engine_poll(e, id[i], reqs[i].out, nullptr);
        CHECK(r >= 0);
        if (r == 1) id[i] = -1, --left;
      }
  }
}

// Requests of every method and plan kind in one engine, with a cancel, in-loop
// gaps and a cap on the running ones; the step log of an unfinished request.
void mixed() {
  for (int graphs : {1, 0}) {
    avionic_engine_config c = config(graphs, 3);
    c.max_batch = 4;
    avionic_engine *e = engine(c);
    std::vector<Req> r;
    r.emplace_back(2, 4, 32, 32, 4, 60, 0);
    r.emplace_back(0, 3, 24, 40, 3, 45, 0);
    r.emplace_back(1, 5, 16, 16, 2, 70, 0);
    r.emplace_back(2, 3, 20, 28, 3, 30, 1);
    r.emplace_back(3, 4, 24, 24, 3, 50, 0);
    r.emplace_back(4, 3, 24, 32, 2, 50, 2);
    r.emplace_back(1, 3, 39, 55, 3, 50, 2);
    r.emplace_back(0, 2, 300, 250, 2, 30, 0);
    r[2].d.debug = 1;
    r[2].d.debugstep = 7;
    r[0].p.stopPDGap = 1e-9;
    Req gone(2, 2, 32, 32, 5, 55, 0);
    long long id = 0;
    CHECK(gone.submit(e, &id) == 0);
    CHECK(avionic_engine_step(e, nullptr) >= 0);
    double sig[64], tau[64];
    size_t n = 64;
    CHECK(avionic_engine_get_step_log(e, id, sig, tau, &n) == 0 && n == 3);
    CHECK(avionic_engine_cancel(e, id) == 0);
    run_all(e, r);
    CHECK(counts(e).held == 0 && counts(e).bytes_held == 0);
    CHECK(counts(e).launch_tunings == 0);  // variants are timed on request only
    CHECK(avionic_engine_destroy(e) == 0);
  }
}

// A launch set whose variants are timed while its iterations are replayed from
// graphs: the executables of the variants that lose are destroyed only once
// their stream has been waited for.
void variants() {
  for (int tick : {1, 13}) {
    avionic_engine_config c = config(1, tick);
    c.fixed_launch = -1;
    avionic_engine *e = engine(c);
    std::vector<Req> r;
    r.emplace_back(2, 4, 32, 48, 3, 120, 2);
    r.emplace_back(2, 4, 32, 48, 3, 120, 2);
    run_all(e, r);
    CHECK(counts(e).launch_tunings == 1);
    run_all(e, r);  // the same launch set: the decision is reused
    CHECK(counts(e).launch_tunings == 1);
    CHECK(avionic_engine_destroy(e) == 0);
  }
}

// A launch that fails anywhere in the first iterations, their captures among
// them: the step reports it, no stream is left in a capture, and the engine goes
// on.
void capture_error() {
  avionic_engine *e = engine(config(1, 1));
  long n = 1;
  for (bool failed = true; failed; ++n) {
    Req r(1, 3, 24, 32, 2, 15, 0);
    long long id = 0;
    CHECK(r.submit(e, &id) == 0);
    stub_fail_launch(n);
    int rc = 0, steps = 0;
    do rc = avionic_engine_step(e, nullptr);
    while (rc >= 0 && ++steps < 13);
    stub_fail_launch(0);
    failed = rc < 0;
    CHECK(avionic_engine_cancel(e, id) == 0);
    std::vector<Req> again;
    again.emplace_back(1, 3, 24, 32, 2, 15, 0);
    run_all(e, again);
    CHECK(stub_graphs() == 0);
  }
  CHECK(n > 15);  // the launches and instantiations of two iteration graphs
  CHECK(avionic_engine_destroy(e) == 0);
}

// Position of the first launch of a kernel among `v`.
size_t first_of(const std::vector<std::string> &v, const char *kernel) {
  size_t i = 0;
  while (i < v.size() && v[i].find(kernel) == std::string::npos) ++i;
  CHECK(i < v.size());
  return i;
}
// The column pass is submitted before the dual update in small and large launch
// sets; sets whose row or column grids differ decide on their variants apart.
void launch_sets() {
  for (const auto &[frames, requests] : {std::pair{8u, 1}, {128u, 49}}) {
    avionic_engine *e = engine(config(0, 1));
    std::vector<Req> r;
    for (int i = 0; i < requests; ++i) r.emplace_back(0, frames, 16, 16, 1, 1, 0);
    long long id = 0;
    for (Req &q : r) CHECK(q.submit(e, &id) == 0);
    stub_take_launches();
    CHECK(avionic_engine_step(e, nullptr) >= 0);
    const std::vector<std::string> v = stub_take_launches();
    CHECK(first_of(v, "kt_col_forward") < first_of(v, "kt_dual"));
    CHECK(avionic_engine_destroy(e) == 0);
  }
  avionic_engine_config c = config(1, 1);
  c.fixed_launch = -1;
  avionic_engine *e = engine(c);
  for (unsigned coils : {1u, 8u}) {  // the same voxels, eight times the rows
    std::vector<Req> r;
    r.emplace_back(1, 8, 32, 32, coils, 60, 0);
    run_all(e, r);
  }
  CHECK(counts(e).launch_tunings == 2);
  CHECK(avionic_engine_destroy(e) == 0);
}

// Smaller requests after larger ones: blocks that they take over from the pool
// count with their whole size, so the memory held stays within the budget, and as
// many requests fit as in an engine that never held the larger ones.
void budget() {
  auto big = [] { return Req(0, 14, 128, 128, 1, 1, 0); };
  auto small = [] { return Req(0, 10, 128, 128, 1, 1, 0); };
  size_t accepted[2];
  for (bool larger_first : {false, true}) {
    std::vector<Req> r, rb;
    for (int i = 0; i < 8; ++i) r.push_back(small());
    for (int i = 0; i < 4; ++i) rb.push_back(big());
    const size_t inputs = stub_memory_held();
    avionic_engine_config c = config(0, 1);
    c.hbm_budget_bytes = 4 * avionic_request_footprint(&rb[0].d) + kMiB;
    avionic_engine *e = engine(c);
    if (larger_first) run_all(e, rb);
    stub_reset_peak();
    size_t n = 0;
    for (long long id; n < r.size(); ++n) {
      const int rc = r[n].submit(e, &id);
      CHECK(rc == 0 || rc == AVIONIC_E_CAPACITY);
      if (rc) break;
    }
    accepted[larger_first] = n;
    CHECK(n > 0 && n < r.size());
    CHECK(counts(e).bytes_held <= c.hbm_budget_bytes);
    // with the pool, but without the operators' tables (5% of a request's state)
    CHECK(stub_memory_peak() - inputs <= c.hbm_budget_bytes / 100 * 106);
    CHECK(avionic_engine_destroy(e) == 0);
  }
  CHECK(accepted[1] == accepted[0]);
}

// Idle blocks of the pool give way to every allocation of the library, and to the
// caller's after avionic_release_memory.
void out_of_memory() {
  const unsigned W = 48, H = 40, C = 4, T = 6;
  const size_t n = (size_t)W * H * T;
  float *data = dev(2 * n * C), *x = dev(2 * n), *b1 = dev((size_t)2 * W * H * C), *mask = dev(n);
  float *many = dev((size_t)2 * W * H * 4096);
  avionic_params p;
  CHECK(avionic_default_params(AVIONIC_TGV2, &p) == 0);
  p.maxIt = 2;
  p.lambda = 1.0;
  avionic_operator *op = nullptr, *op2 = nullptr;
  avionic_recon *r = nullptr;
  CHECK(avionic_cartesian_operator_create(W, H, C, T, nullptr, 0, &op) == 0);
  CHECK(avionic_recon_create(AVIONIC_TGV2, W, H, C, T, &p, op, &r) == 0);
  // after each run an idle block is kept, and the device is full
  auto fill = [&] {
    stub_set_memory(4096 * kMiB);
    const size_t before = stub_memory_held();
    CHECK(avionic_recon_run(r, data, x, b1, nullptr) == 0);
    stub_set_memory(stub_memory_held());
    return stub_memory_held() - before;
  };
  fill();
  CHECK(avionic_cartesian_operator_create(W, H, C, T, mask, 0, &op2) == 0);
  CHECK(avionic_operator_destroy(op2) == 0);
  fill();
  CHECK(avionic_cartesian3d_operator_create(W, H, T, 1, nullptr, &op2) == 0);
  CHECK(avionic_operator_destroy(op2) == 0);
  fill();
  CHECK(avionic_fft2(many, H, W, 16, -1, 0, 1, nullptr) == 0);
  // the FP64 operator norm, with memory for it that lacks ever more of the block
  // (its kernels do nothing: the norm itself comes out as zero, an error)
  const size_t block = fill();
  auto norm_fits = [&] {
    double norm = 0.0;
    avionic_recon_operator_norm(r, b1, 2, &norm, nullptr);
    return std::strstr(avionic_last_error(), "memory") == nullptr;
  };
  stub_set_memory(4096 * kMiB);
  stub_reset_peak();
  const size_t held = stub_memory_held();
  CHECK(block > 0 && norm_fits());
  const size_t need = stub_memory_peak() - held;
  for (size_t lack = 0; lack <= block; lack += block / 64) {
    fill();
    stub_set_memory(stub_memory_held() + need - lack);
    CHECK(norm_fits());
  }
  fill();
  const size_t all = stub_memory_held();
  CHECK(avionic_release_memory() == 0);
  CHECK(all - stub_memory_held() >= 16 * n * sizeof(float));
  CHECK(avionic_recon_destroy(r) == 0);
  CHECK(avionic_operator_destroy(op) == 0);
  for (float *f : {data, x, b1, mask, many}) (void)hipFree(f);
  stub_set_memory(4096 * kMiB);
}

// A host allocation that fails anywhere in a reconstruction or a request is an
// error of that call (or of none): nothing aborts, nothing is lost, and the next
// call runs.
void host_memory() {
  Req q(1, 3, 24, 32, 2, 12, 0);
  const size_t held = stub_memory_held();
  long failures = 0;
  for (long n = 1;; ++n) {
    avionic_operator *op = nullptr;
    avionic_recon *r = nullptr;
    avionic_engine *e = nullptr;
    avionic_engine_config c = config(1, 4);
    int rc = 0;
    fail_new = n;
    if (!rc) rc = avionic_cartesian_operator_create(32, 24, 2, 3, nullptr, 0, &op);
    if (!rc) rc = avionic_recon_create(AVIONIC_TGV2, 32, 24, 2, 3, &q.p, op, &r);
    if (!rc) rc = avionic_recon_run(r, q.data, q.out, q.b1, nullptr);
    if (!rc) rc = avionic_engine_create(&c, &e);
    long long id = 0;
    if (!rc) rc = q.submit(e, &id);
    while (!rc && avionic_engine_poll(e, id, q.out, nullptr) == 0)
      rc = std::min(0, avionic_engine_step(e, nullptr));
    const bool reached = fail_new == 0;
    fail_new = 0;
    failures += rc != 0;
    CHECK(reached || rc == 0);
    if (r) {  // the solver is as good as before
      CHECK(avionic_recon_run(r, q.data, q.out, q.b1, nullptr) == 0);
      CHECK(avionic_recon_destroy(r) == 0);
    }
    if (e) CHECK(avionic_engine_destroy(e) == 0);
    if (op) CHECK(avionic_operator_destroy(op) == 0);
    CHECK(stub_memory_held() == held && stub_graphs() == 0);
    if (!reached) break;
  }
  CHECK(failures > 20);
  // blocks given back with no host memory to note them
  avionic_engine *e = engine(config(0, 1));
  std::vector<long long> id(60);
  for (long long &i : id) CHECK(q.submit(e, &i) == 0);
  for (long long i : id) {
    fail_new = 1;
    avionic_engine_cancel(e, i);
    fail_new = 0;
  }
  CHECK(counts(e).held == 0);
  CHECK(avionic_engine_destroy(e) == 0);
}

}  // namespace

int main(int argc, char **argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  stub_set_memory(4096 * kMiB);
  if (what == "mixed") mixed();
  else if (what == "variants") variants();
  else if (what == "capture_error") capture_error();
  else if (what == "launch_sets") launch_sets();
  else if (what == "budget") budget();
  else if (what == "out_of_memory") out_of_memory();
  else if (what == "host_memory") host_memory();
  else CHECK(!"a scenario");
  CHECK(stub_launches() > 0);
  CHECK(stub_faults() == 0);
  // the FP64 transforms' tables are kept for the process
  CHECK(stub_memory_held() <= (what == "out_of_memory" ? 4096 : 0));
  std::printf("engine_host: %s ok\n", what.c_str());
  return 0;
}
