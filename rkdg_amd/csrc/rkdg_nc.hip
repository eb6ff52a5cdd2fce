// rkdg_nc.hip — gfx950 kernel for the non-conforming faces of tensor meshes
// (MFEM NCMesh slave faces, as the reference's face loop sees them:
// face_integrator.cpp:11-276 over an interior face whose Elem1 is the fine
// (slave) element and whose Elem2 is the coarser (master) element, Loc2 being
// the slave's point matrix in the master).
//
// One workgroup of four wavefronts per element that has such faces; each
// wavefront takes every fourth slave face touching the element. Per face: both
// states through LDS; tensor Lagrange interpolation at the face points (the
// slave face's Gauss-Legendre rule, the order of the conforming faces), the two
// sides and halves of the variables on different lanes; the Riemann flux with
// the arguments ordered (slave state, master state, slave normal), so the two
// elements of the face see bitwise identical fluxes; and the element's signed
// share flux * w * |n|. Node lanes then lift the shares with their basis at the
// element's own reference points. The partial sums of the wavefronts are added
// in a fixed order and written before the inverse mass; the element kernels add
// them to their face terms.
//
// The faces are few (the interfaces between refinement levels), so the launch is
// a chain of dependent loads and arithmetic, not throughput. A wavefront that
// took an element's faces one after the other, formed every 1D basis value by
// N(N-1) divisions and formed them again for each node and point of the lift
// needed 251 us of the 285 us of a stage on 3032 Q2 hexahedra (802 of them with
// such faces). With the denominators inverted once, the 1D values kept in LDS
// and the faces spread over four wavefronts the three-stage step takes 161
// instead of 862 us.
#include "rkdg_kernels.hpp"

namespace rkdg {

// LDS of one wavefront is written and read by its own lanes only, in order: the
// compiler must keep that order, the hardware does
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <int DIM, int P>
__global__ __launch_bounds__(256) void nc_face_kernel(const NcArgs A, const SchemeParams g,
                                                      const TensorTables* __restrict__ gtb) {
  constexpr int N = P + 1;
  constexpr int ND = DIM == 3 ? N * N * N : N * N;
  constexpr int NEQ = DIM + 2;
  constexpr int NQ = DIM == 3 ? P + 2 : P + 1;
  constexpr int NP = DIM == 3 ? NQ * NQ : NQ;
  constexpr int PR = 3 * DIM + 1;  // per point: slave xi, master xi, w |n|, unit normal
  constexpr int RG = NP * PR;
  constexpr int NW = 4;                        // wavefronts
  constexpr int VS = 4 * NP <= 64 ? 2 : 1;     // lanes per (side, point): the variables in VS parts
  constexpr int NV = (NEQ + VS - 1) / VS;
  constexpr int QS = 2 * ND <= 64 ? 2 : 1;     // lanes per node in the lift: the points in QS parts
  static_assert(ND <= 64 && 2 * NP <= 64, "one lane per node and per side and face point");

  __shared__ double s_x[N], s_den[N];              // nodes, 1 / prod_b (x_a - x_b)
  __shared__ double s_u[NW][2][NEQ][ND];           // slave and master states
  __shared__ double s_t[NW][2][NP][NEQ];           // their traces; [0] then the element's share of flux * w * |n|
  __shared__ double s_L[NW][NP][DIM][N];           // the element's 1D basis values at the points
  __shared__ double s_z[NW * QS][NEQ][ND];

  const int wave = threadIdx.x / 64, tid = threadIdx.x % 64;
  const int64_t slot = blockIdx.x;
  const int64_t NDOFS = A.NE * ND;
  if (threadIdx.x < N) {
    const double xa = gtb->x[threadIdx.x];
    double d = 1.0;
#pragma unroll
    for (int b = 0; b < N; b++) d *= b == (int)threadIdx.x ? 1.0 : xa - gtb->x[b];
    s_x[threadIdx.x] = xa;
    s_den[threadIdx.x] = 1.0 / d;
  }
  __syncthreads();
  // 1D Lagrange basis on the Gauss-Legendre nodes at t
  auto lagrange = [&](double t, double* L) {
#pragma unroll
    for (int a = 0; a < N; a++) {
      double v = s_den[a];
#pragma unroll
      for (int b = 0; b < N; b++)
        if (b != a) v *= t - s_x[b];
      L[a] = v;
    }
  };
  double z[NEQ];
#pragma unroll
  for (int v = 0; v < NEQ; v++) z[v] = 0.0;
  double lmax = 0.0;
  const int i0 = A.ptr[slot], i1 = A.ptr[slot + 1];
  for (int c0 = i0; c0 < i1; c0 += 64) {
    // the items of this chunk and their elements, one per lane
    const int cn = i1 - c0 < 64 ? i1 - c0 : 64;
    const int item_l = tid < cn ? A.item[c0 + tid] : 0;
    const int es_l = A.rec[3 * (item_l >> 1)], em_l = A.rec[3 * (item_l >> 1) + 1];
    for (int it = wave; it < cn; it += NW) {
      const int item = __builtin_amdgcn_readlane(item_l, it);
      const int es = __builtin_amdgcn_readlane(es_l, it), em = __builtin_amdgcn_readlane(em_l, it);
      const int r = item >> 1, side = item & 1;
      constexpr int UP = (NEQ * ND + 63) / 64;
      double us[UP], um[UP];
#pragma unroll
      for (int p = 0; p < UP; p++) {
        const int k = tid + 64 * p;
        const int v = k / ND, i = k - v * ND;
        us[p] = k < NEQ * ND ? A.x[v * NDOFS + (int64_t)es * ND + i] : 0.0;
        um[p] = k < NEQ * ND ? A.x[v * NDOFS + (int64_t)em * ND + i] : 0.0;
      }
      // lane -> (side h, part of the variables, point)
      const int h = tid / (NP * VS), part = (tid / NP) % VS, q = tid % NP;
      const bool tl = h < 2;
      const double* gq = A.geo + (int64_t)r * RG + q * PR;
      double xi[DIM], wn = 0.0, nrm[DIM];
#pragma unroll
      for (int d = 0; d < DIM; d++) xi[d] = tl ? gq[h * DIM + d] : 0.0;
      if (tid < NP) {
        wn = gq[2 * DIM] * (side == 0 ? -1.0 : 1.0);
#pragma unroll
        for (int d = 0; d < DIM; d++) nrm[d] = gq[2 * DIM + 1 + d];
      }
      wave_sync();  // the previous face's LDS reads are done
#pragma unroll
      for (int p = 0; p < UP; p++) {
        const int k = tid + 64 * p;
        if (k < NEQ * ND) {
          (&s_u[wave][0][0][0])[k] = us[p];
          (&s_u[wave][1][0][0])[k] = um[p];
        }
      }
      wave_sync();
      if (tl) {
        double L[3][N];
#pragma unroll
        for (int d = 0; d < DIM; d++) lagrange(xi[d], L[d]);
        if (h == side && part == 0) {
#pragma unroll
          for (int d = 0; d < DIM; d++)
#pragma unroll
            for (int a = 0; a < N; a++) s_L[wave][q][d][a] = L[d][a];
        }
#pragma unroll
        for (int k = 0; k < NV; k++) {
          const int v = part * NV + k;
          if (v < NEQ) {
            const double* u = &s_u[wave][h][v][0];
            double acc = 0.0;
#pragma unroll
            for (int c = 0; c < (DIM == 3 ? N : 1); c++) {
              double tc = 0.0;
#pragma unroll
              for (int b = 0; b < N; b++) {
                double tb = 0.0;
#pragma unroll
                for (int a = 0; a < N; a++) tb += u[a + N * (b + N * c)] * L[0][a];
                tc += tb * L[1][b];
              }
              acc += DIM == 3 ? tc * L[2][c] : tc;
            }
            s_t[wave][h][q][v] = acc;
          }
        }
      }
      wave_sync();
      if (tid < NP) {
        double ul[NEQ], ur[NEQ], fl[NEQ];
#pragma unroll
        for (int v = 0; v < NEQ; v++) {
          ul[v] = s_t[wave][0][tid][v];
          ur[v] = s_t[wave][1][tid][v];
        }
        bool ok = true;
        const double lam = riemann<DIM>(g, ul, ur, nrm, fl, ok);
        if (!ok || lam < 0.0) {
          const bool nf = nonfinite_nodes(A.x, NDOFS, es, ND, NEQ) || nonfinite_nodes(A.x, NDOFS, em, ND, NEQ);
          flag_error(A.err, es, em, A.rec[3 * r + 2], nf ? kErrNonFinite : kErrUnphysical);
#pragma unroll
          for (int v = 0; v < NEQ; v++) fl[v] = 0.0;
        } else {
          lmax = lam > lmax ? lam : lmax;
        }
#pragma unroll
        for (int v = 0; v < NEQ; v++) s_t[wave][0][tid][v] = fl[v] * wn;
      }
      wave_sync();
      if (tid < QS * ND) {
        const int i = tid % ND, qp = tid / ND;
        const int a = i % N, b = (i / N) % N, c = i / (N * N);
        for (int p = qp; p < NP; p += QS) {
          double phi = s_L[wave][p][0][a] * s_L[wave][p][1][b];
          if (DIM == 3) phi *= s_L[wave][p][DIM - 1][c];
#pragma unroll
          for (int v = 0; v < NEQ; v++) z[v] += s_t[wave][0][p][v] * phi;
        }
      }
    }
  }
  if (tid < QS * ND) {
#pragma unroll
    for (int v = 0; v < NEQ; v++) s_z[wave * QS + tid / ND][v][tid % ND] = z[v];
  }
  __syncthreads();
  for (int k = threadIdx.x; k < NEQ * ND; k += 64 * NW) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < NW * QS; w++) t += (&s_z[w][0][0])[k];
    A.out[slot * NEQ * ND + k] = t;
  }
  if (!A.no_lambda) {
    for (int off = 32; off > 0; off >>= 1) {
      const double o = __shfl_xor(lmax, off, 64);
      lmax = o > lmax ? o : lmax;
    }
    if (tid == 0) atomic_max_pos(lam_slot(A.lam, A.lam_ld), lmax);
  }
}

hipError_t launch_nc_faces(int dim, int p, const NcArgs& a, const SchemeParams& g, const TensorTables* t,
                           hipStream_t s) {
  if (a.n_elem <= 0) return hipSuccess;
#define X(D, PP)                                                                 \
  if (dim == D && p == PP) {                                                     \
    nc_face_kernel<D, PP><<<(unsigned)a.n_elem, 256, 0, s>>>(a, g, t);            \
    return hipGetLastError();                                                    \
  }
  X(2, 1) X(2, 2) X(2, 3) X(2, 4) X(2, 5) X(3, 1) X(3, 2) X(3, 3)
#undef X
  return hipErrorInvalidValue;
}

}  // namespace rkdg
