// The Rusanov flux from both elements of a face: of random pairs of states, the
// flux with the sides exchanged and the normal turned must be the negative of the
// flux, bit by bit, and the wave speeds the same. On the host in a build that may
// contract products into sums as the device build does (77: no fused multiply-add
// on this processor), with --gpu on the device.
//
//   flux_pairs [--gpu]         prints: dimension, gamma, covolume, pairs, mismatches
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "../../rkdg_amd/csrc/rkdg_physics.hpp"

using namespace rkdg;

static constexpr int kPairs = 1 << 16;

// in: left, right state and unit normal of each pair, component-major
template <int DIM>
RKDG_HD bool pair_differs(const SchemeParams& g, const double* in, int n, int i, bool face_norm) {
  constexpr int NE = DIM + 2;
  double L[NE], R[NE], a[DIM], b[DIM], f[NE], h[NE], nn = 0.0;
  for (int k = 0; k < NE; k++) {
    L[k] = in[k * n + i];
    R[k] = in[(NE + k) * n + i];
  }
  for (int d = 0; d < DIM; d++) {
    a[d] = in[(2 * NE + d) * n + i];
    b[d] = -a[d];
    nn += a[d] * a[d];
  }
  const double inm = face_norm ? 0.5 * recip(sqrt_ws(nn)) : 0.0;  // as the element kernels pass it
  bool ok1 = true, ok2 = true;
  const double l1 = riemann_t<DIM, RKDG_RS_RUSANOV>(g, L, R, a, f, ok1, inm);
  const double l2 = riemann_t<DIM, RKDG_RS_RUSANOV>(g, R, L, b, h, ok2, inm);
  bool same = ok1 && ok2 && l1 == l2;
  for (int k = 0; k < NE; k++) same = same && f[k] == -h[k];
  return !same;
}

template <int DIM>
__global__ void pairs_kernel(SchemeParams g, const double* in, int n, int* out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = pair_differs<DIM>(g, in, n, i, i % 2 == 0);
}

template <int DIM>
static int count(const SchemeParams& g, bool gpu, unsigned seed) {
  constexpr int NE = DIM + 2, n = kPairs;
  std::mt19937_64 rng(seed);
  std::uniform_real_distribution<double> u(-1.0, 1.0);
  std::vector<double> in((size_t)(2 * NE + DIM) * n);
  for (int i = 0; i < n; i++) {
    for (int s = 0; s < 2; s++) {
      const double rho = 1.0 + 0.9 * u(rng), p = 1.0 + 0.9 * u(rng);
      double m2 = 0.0;
      in[(size_t)(s * NE) * n + i] = rho;
      for (int d = 0; d < DIM; d++) {
        const double m = 2.0 * rho * u(rng);
        in[(size_t)(s * NE + 1 + d) * n + i] = m;
        m2 += m * m;
      }
      in[(size_t)(s * NE + 1 + DIM) * n + i] = p / (g.gamma - 1.0) + 0.5 * m2 / rho;
    }
    double v[DIM], q = 0.0;
    for (int d = 0; d < DIM; d++) {
      v[d] = u(rng) + (d == 0 ? 1.5 : 0.0);
      q += v[d] * v[d];
    }
    for (int d = 0; d < DIM; d++) in[(size_t)(2 * NE + d) * n + i] = v[d] / std::sqrt(q);
  }
  int bad = 0;
  if (!gpu) {
    for (int i = 0; i < n; i++) bad += pair_differs<DIM>(g, in.data(), n, i, i % 2 == 0);
    return bad;
  }
  double* din = nullptr;
  int* dout = nullptr;
  std::vector<int> out(n);
  if (hipMalloc(&din, sizeof(double) * in.size()) != hipSuccess || hipMalloc(&dout, sizeof(int) * n) != hipSuccess ||
      hipMemcpy(din, in.data(), sizeof(double) * in.size(), hipMemcpyHostToDevice) != hipSuccess)
    return -1;
  pairs_kernel<DIM><<<n / 256, 256>>>(g, din, n, dout);
  if (hipGetLastError() != hipSuccess ||
      hipMemcpy(out.data(), dout, sizeof(int) * n, hipMemcpyDeviceToHost) != hipSuccess)
    return -1;
  (void)hipFree(din);
  (void)hipFree(dout);
  for (int v : out) bad += v;
  return bad;
}

int main(int argc, char** argv) {
  const bool gpu = argc > 1 && std::strcmp(argv[1], "--gpu") == 0;
  if (!gpu && !__builtin_cpu_supports("fma")) return 77;
  int total = 0;
  for (int k = 0; k < 4; k++) {
    SchemeParams g{};
    g.gamma = k % 2 ? 5.0 / 3.0 : 1.4;
    g.covolume = k / 2 ? 0.05 : 0.0;
    derive_params(g);
    const int b2 = count<2>(g, gpu, 11 + k), b3 = count<3>(g, gpu, 31 + k);
    std::printf("2 %.3f %.2f %d %d\n3 %.3f %.2f %d %d\n", g.gamma, g.covolume, kPairs, b2, g.gamma, g.covolume, kPairs, b3);
    if (b2 < 0 || b3 < 0) return 2;
    total += b2 + b3;
  }
  return total ? 1 : 0;
}
