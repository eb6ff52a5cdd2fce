// librkdg.so when a HIP call fails on the host's side: the launch and allocation
// entry points are defined here, in front of the runtime's, and return an error
// without calling it when they are told to.
//
//   hip_faults batch       a read-back of the wave speeds fails between its two launches;
//                          the ensemble's next steps must not see the abandoned speeds
//   hip_faults records     memory runs out while an adjoint solve allocates its records,
//                          or they are more than a quarter of what is free; it must take
//                          checkpoints instead, give back what it took and return the
//                          same bits
#include <dlfcn.h>
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstring>
#include <vector>

#include "smoke_case.h"

static int g_launches = 0;        // launches since the last reset
static int g_fail_launch = -1;    // index of the launch that fails
static hipError_t g_pending = hipSuccess;
static size_t g_fail_size = 0;    // of the allocations of this size, counted from 0,
static int g_fail_alloc = -1;     // the one that fails
static int g_allocs = 0, g_failed = 0;
static size_t g_free = 0;         // the free memory to report (0: what there is)

template <typename F>
static F real(const char* name) {
  return reinterpret_cast<F>(dlsym(RTLD_NEXT, name));
}

extern "C" {

hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t s) {
  static auto fn = real<hipError_t (*)(const void*, dim3, dim3, void**, size_t, hipStream_t)>("hipLaunchKernel");
  if (g_launches++ == g_fail_launch) return g_pending = hipErrorLaunchFailure;
  return fn(f, grid, block, args, lds, s);
}
hipError_t hipGetLastError() {
  static auto fn = real<hipError_t (*)()>("hipGetLastError");
  const hipError_t e = g_pending;
  g_pending = hipSuccess;
  return e != hipSuccess ? e : fn();
}
hipError_t hipMalloc(void** p, size_t n) {
  static auto fn = real<hipError_t (*)(void**, size_t)>("hipMalloc");
  if (n == g_fail_size && g_allocs++ == g_fail_alloc) {
    g_failed++;
    return hipErrorOutOfMemory;
  }
  return fn(p, n);
}
hipError_t hipMemGetInfo(size_t* avail, size_t* total) {
  static auto fn = real<hipError_t (*)(size_t*, size_t*)>("hipMemGetInfo");
  const hipError_t e = fn(avail, total);
  if (g_free) *avail = g_free;
  return e;
}
}

#define CHECK(x)                                                                    \
  do {                                                                              \
    if (!(x)) {                                                                     \
      std::printf("line %d: %s (%s)\n", __LINE__, #x, rkdg_last_error());           \
      return 1;                                                                     \
    }                                                                               \
  } while (0)

static const double kA[3] = {1.0, 0.25, 0.25}, kB[3] = {1.0 / 6.0, 1.0 / 6.0, 2.0 / 3.0}, kC[3] = {0.0, 1.0, 0.5};
static smoke_case g_case;

// a smooth state on the nodes of `copies` copies of the case's mesh
static std::vector<double> state(rkdg_ctx* c, double energy) {
  rkdg_info in;
  (void)rkdg_get_info(c, &in);
  const int64_t n = in.num_dofs;
  std::vector<double> xy((size_t)n * 2), u((size_t)in.state_size);
  (void)rkdg_node_coords(c, xy.data());
  for (int64_t i = 0; i < n; i++) {
    const double x = xy[2 * i], y = xy[2 * i + 1], rho = 1.0 + 0.2 * std::sin(3.0 * x) * std::cos(2.0 * y);
    u[i] = rho;
    u[n + i] = rho * (0.4 + 0.1 * y);
    u[2 * n + i] = 0.05 * rho * x;
    u[3 * n + i] = energy * (2.5 + 0.3 * x) + 0.5 * rho * 0.25;
  }
  return u;
}

static double* device(const std::vector<double>& u) {
  double* d = nullptr;
  if (hipMalloc(reinterpret_cast<void**>(&d), sizeof(double) * u.size()) != hipSuccess) return nullptr;
  return hipMemcpy(d, u.data(), sizeof(double) * u.size(), hipMemcpyHostToDevice) == hipSuccess ? d : nullptr;
}
static std::vector<double> host(const double* d, size_t n) {
  std::vector<double> u(n);
  (void)hipMemcpy(u.data(), d, sizeof(double) * n, hipMemcpyDeviceToHost);
  return u;
}

// six steps of a two-instance ensemble; between the first and the last three a read of the wave speeds
// of a hotter state, failing at its read-back where `fault`
static int ensemble(bool fault, std::vector<double>& x, std::vector<double>& dt) {
  rkdg_mesh_desc m[2] = {g_case.mesh, g_case.mesh};
  rkdg_scheme_desc s[2] = {g_case.scheme, g_case.scheme};
  rkdg_ctx* c = nullptr;
  CHECK(rkdg_batch_create(m, s, 2, &c) == RKDG_OK);
  const std::vector<double> u = state(c, 1.0), hot = state(c, 100.0);
  double *xd = device(u), *hd = device(hot), *yd = device(hot);
  CHECK(xd && hd && yd);
  const double t0[2] = {0.0, 0.0}, tf[2] = {1e3, 1e3};
  CHECK(rkdg_batch_init(c, xd, t0, tf, 0.2, 0) == RKDG_OK);
  CHECK(rkdg_batch_advance(c, xd, 3, kA, kB, kC, 3, nullptr) == RKDG_OK);
  double lam = 0.0;
  g_launches = 0;
  g_fail_launch = fault ? 1 : -1;  // the right-hand side runs, publishing its wave speeds fails
  const int rc = rkdg_rhs(c, hd, yd, &lam);
  CHECK(g_launches == 2);
  g_fail_launch = -1;
  CHECK(rc == (fault ? RKDG_E_HIP : RKDG_OK));
  CHECK(rkdg_batch_advance(c, xd, 3, kA, kB, kC, 3, nullptr) == RKDG_OK);
  dt.assign(2, 0.0);
  CHECK(rkdg_batch_status(c, nullptr, dt.data(), nullptr, nullptr) == RKDG_OK);
  x = host(xd, u.size());
  (void)hipFree(xd);
  (void)hipFree(hd);
  (void)hipFree(yd);
  CHECK(rkdg_destroy(c) == RKDG_OK);
  return 0;
}

static int batch() {
  std::vector<double> x0, dt0, x1, dt1;
  if (ensemble(false, x0, dt0) || ensemble(true, x1, dt1)) return 1;
  CHECK(dt0 == dt1);
  CHECK(x0 == x1);
  return 0;
}

// gradient through 30 steps; the allocation of record `fail` (-1: none) fails; the records of `room`
// steps (0: any number) are a quarter of the free memory
static int gradient(int fail, int room, std::vector<double>& out) {
  rkdg_ctx* c = nullptr;
  CHECK(rkdg_create_ex(&g_case.mesh, &g_case.scheme, RKDG_CREATE_DENSE, &c) == RKDG_OK);
  rkdg_info in;
  CHECK(rkdg_get_info(c, &in) == RKDG_OK);
  double *x = device(state(c, 1.0)), *xbar = device(state(c, 1.0));
  CHECK(x && xbar);
  CHECK(rkdg_limit(c, x, nullptr) == RKDG_OK);
  const int steps = 30;
  std::vector<double> dts(steps, 1e-4);
  double J = 0.0, pbar[RKDG_MAX_BC * 8];
  g_fail_size = sizeof(double) * in.state_size * 7;  // one recorded step of three stages
  g_fail_alloc = fail;
  g_free = 4 * g_fail_size * room;
  g_allocs = g_failed = 0;
  const int rc = rkdg_adjoint_solve(c, x, steps, dts.data(), 3, kA, kB, kC, 0, 0, &J, xbar, pbar, nullptr);
  const int allocs = g_allocs, failed = g_failed;
  g_fail_size = g_free = 0;
  CHECK(rc == RKDG_OK);
  CHECK(failed == (fail >= 0));
  // every step's record, or those of one segment of six steps, at once or after the failure
  CHECK(allocs == (room > 0 && room < steps ? 6 : fail >= 0 ? fail + 1 + 6 : steps));
  out = host(xbar, (size_t)in.state_size);
  out.push_back(J);
  (void)hipFree(x);
  (void)hipFree(xbar);
  CHECK(rkdg_destroy(c) == RKDG_OK);
  return 0;
}

static int records() {
  std::vector<double> want, got;
  if (gradient(-1, 0, want)) return 1;
  for (int fail : {0, 1, 7, 29}) {
    if (gradient(fail, 0, got)) return 1;
    CHECK(got == want);
  }
  for (int room : {1, 29, 30}) {
    if (gradient(-1, room, got)) return 1;
    CHECK(got == want);
  }
  return 0;
}

int main(int argc, char** argv) {
  if (argc < 2) return 2;
  smoke_setup(&g_case, 1);
  const int rc = std::strcmp(argv[1], "batch") == 0 ? batch() : std::strcmp(argv[1], "records") == 0 ? records() : 2;
  std::printf("%s: %s\n", argv[1], rc ? "failed" : "ok");
  return rc;
}
