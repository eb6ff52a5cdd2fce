// Toro's two-rarefaction speeds of states that separate faster than their
// rarefactions, for gammas whose 1/z is no integer: the estimate's power then has no
// value and the speeds are the acoustic ones, bit by bit, whatever the ratio of the
// pressures. On the host, with --gpu on the device.
//
//   toro_base [--gpu]          prints: dimension, gamma, pairs, mismatches
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "../../rkdg_amd/csrc/rkdg_physics.hpp"

using namespace rkdg;

static constexpr int kPairs = 1 << 14;

// in: left and right state of each pair (rotated: the normal is x), component-major
template <int DIM>
RKDG_HD bool pair_differs(const SchemeParams& g, const double* in, int n, int i) {
  constexpr int NE = DIM + 2;
  double L[NE], R[NE];
  for (int k = 0; k < NE; k++) {
    L[k] = in[k * n + i];
    R[k] = in[(NE + k) * n + i];
  }
  const SidePrim<DIM> q1 = side_prim<DIM>(L, g), q2 = side_prim<DIM>(R, g);
  double lo, hi;
  wave_speeds<DIM>(L, R, q1, q2, g, lo, hi);
  const double a = L[1] * q1.inv - sqrt_ws(side_sound2<DIM>(L, q1, g));
  const double b = R[1] * q2.inv + sqrt_ws(side_sound2<DIM>(R, q2, g));
  return !(lo == a && hi == b);
}

template <int DIM>
__global__ void pairs_kernel(SchemeParams g, const double* in, int n, int* out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = pair_differs<DIM>(g, in, n, i);
}

template <int DIM>
static int count(const SchemeParams& g, bool gpu, unsigned seed) {
  constexpr int NE = DIM + 2, n = kPairs;
  std::mt19937_64 rng(seed);
  std::uniform_real_distribution<double> u(0.0, 1.0);
  std::vector<double> in((size_t)(2 * NE) * n);
  for (int i = 0; i < n; i++) {
    const double p[2] = {std::pow(10.0, 9.0 * u(rng) - 4.5), std::pow(10.0, 9.0 * u(rng) - 4.5)};
    const double rho[2] = {0.1 + 5.0 * u(rng), 0.1 + 5.0 * u(rng)};
    const double c = std::sqrt(g.gamma * p[0] / rho[0]) + std::sqrt(g.gamma * p[1] / rho[1]);
    const double apart = (1.2 + 3.0 * u(rng)) * 2.0 * c / (g.gamma - 1.0);
    const int still = p[0] < p[1] ? 0 : 1;  // the lower pressure is at rest: its energy resolves it
    for (int s = 0; s < 2; s++) {
      double v2 = 0.0;
      for (int d = 0; d < DIM; d++) {
        const double v = d > 0 || s == still ? 0.1 * std::sqrt(p[s]) * (u(rng) - 0.5) : (s ? apart : -apart);
        in[(size_t)(s * NE + 1 + d) * n + i] = rho[s] * v;
        v2 += v * v;
      }
      in[(size_t)(s * NE) * n + i] = rho[s];
      in[(size_t)(s * NE + 1 + DIM) * n + i] = p[s] / (g.gamma - 1.0) + 0.5 * rho[s] * v2;
    }
  }
  int bad = 0;
  if (!gpu) {
    for (int i = 0; i < n; i++) bad += pair_differs<DIM>(g, in.data(), n, i);
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
  const double gammas[5] = {1.09, 1.3, 2.6, 4.0, 6.0};
  int total = 0;
  for (int k = 0; k < 5; k++) {
    SchemeParams g{};
    g.gamma = gammas[k];
    derive_params(g);
    if (g.toro_n) return 2;  // 1/z is an integer: there is a power
    const int b2 = count<2>(g, gpu, 11 + k), b3 = count<3>(g, gpu, 31 + k);
    std::printf("2 %.3f %d %d\n3 %.3f %d %d\n", g.gamma, kPairs, b2, g.gamma, kPairs, b3);
    if (b2 < 0 || b3 < 0) return 2;
    total += b2 + b3;
  }
  return total ? 1 : 0;
}
