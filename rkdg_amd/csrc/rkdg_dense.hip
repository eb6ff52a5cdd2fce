// rkdg_dense.hip — gfx950 kernels for small 2D elements whose reference
// operators are kept as dense matrices: affine triangles P_p (the
// L2_TriangleElement nodal basis) and non-affine (bilinear) quadrilaterals Q_p.
// Same path as rkdg_tensor.hip: FE_Evolution::Mult
// (src/fe_evolution/fe_evolution.cpp:102-216) fused with the RK-stage epilogue,
// element means (src/averager/averager.cpp:84-109) and the limiter
// (src/limiter/limiter.cpp:22-94, src/indicator/indicator_bj.cpp:15-200,
// src/limiter/limiter_multiplier.cpp:12-99, src/limiter/limiter_findiff.cpp:3-33).
//
// Volume term: z_j += sum_r sum_k K_r(j,k) G^r_k with G^r_k = adj(J)(r,:) . F(u_k)
// (nodal flux, GetFlux fe_evolution.cpp:219-245) and K_r(j,k) the exact integral
// of phi_k d_r phi_j (triangles; DomainIntegrator with intorder 2p is exact) or
// the collocated w_k d_r phi_j(x_k) with adj(J) taken at node k (Q_p on
// Gauss-Legendre nodes). Faces: the neighbour's trace is evaluated at the
// mirrored point of its own face. Mass: M^-1 = Mhat^-1 / det J (affine
// triangles); on a bilinear quadrilateral det J is linear in each coordinate, so
// the p+1 point Gauss-Legendre rule integrates phi_i phi_j det J exactly and the
// mass matrix is diagonal, w_j det J(x_j).
#include "rkdg_dense.hpp"

namespace rkdg {

// Right-hand side. One lane per face point: T = NF * NQ lanes per element and
// 64 / T elements per wavefront (P2 triangles: 7 elements fill 63 lanes, where a
// power-of-two team of 16 lanes left 28 of 64 idle in the Riemann solves, the
// longest phase). The neighbours' states are read one (face, variable) row per
// lane, contiguous and once, instead of whole by each face point; quadrilaterals
// interpolate a row to the face points in registers (sum-factorised, tables read
// once per lane), triangles stage it in LDS. Geometry is formed from the edge
// normals alone (adj(J) and det J are polynomials in the edge vectors), so an
// element reads 2 NF doubles of its record, and the inverse mass is folded into
// the volume and lift tables (triangles) or diagonal (quadrilaterals).
//
// Bound by VALU issue (Q1 quadrilaterals: 69 % busy, LDS 47 %) or latency (P2
// triangles 45 % and 53 %) at four waves per SIMD, three at order 3 and five for P1
// triangles: the LDS of a wave (8.9 to 15.5 KB) sets it. Limited steps, at
// first (power-of-two teams, every point reading the whole neighbour, dense
// inverse mass and a full geometry record per element, the persistent loop) and
// now, with the limiter's own change: 27,467 bilinear Q2 quadrilaterals, two
// stages, HLLC 229 -> 70 us; 120,540 P2 triangles, three stages, HLLC 488 -> 187
// us; 472,000 Q1 quadrilaterals in 64 instances, eight steps of three stages, HLL
// 12.9 -> 4.4 ms.
template <int GEOM, int P>
struct RC : DC<GEOM, P> {
  using D = DC<GEOM, P>;
  static constexpr int N = P + 1;
  static constexpr int T = D::NPT;
  static constexpr int EPB = D::BLOCK / T;
  static constexpr int ROWS = D::NF * D::NEQ;       // neighbour rows (face, variable)
  static constexpr int RP = (ROWS + T - 1) / T;     // rows per lane
};

// Keeps the scheduler from moving loads across this point: the unrolled
// contractions would otherwise have every LDS read in flight at once (255 VGPRs
// and spills on P2 triangles).
__device__ __forceinline__ void hold() { __builtin_amdgcn_sched_barrier(0); }

// Keeps a contraction in its basic block: the compiler otherwise sinks the
// arithmetic below the branches of the epilogue and leaves its LDS reads, all
// of them live, above (spills).
template <int n>
__device__ __forceinline__ void pin(double* y) {
#pragma unroll
  for (int v = 0; v < n; v++) asm volatile("" : "+v"(y[v]));
}

// one work block (EPB elements, one wavefront) of the right-hand side
template <int GEOM, int P, int RS, bool BC>
__device__ __forceinline__ void dense_rhs_block(const RhsArgs& A, const SchemeParams& g, int64_t vb,
                                                DenseRhsTab<GEOM, P>& tb) {
  using C = RC<GEOM, P>;
  constexpr int N = C::N, ND = C::ND, NEQ = C::NEQ, NF = C::NF, NQ = C::NQ, NPT = C::NPT;
  constexpr int T = C::T, EPB = C::EPB, BLOCK = C::BLOCK, RP = C::RP;
  constexpr bool TRI = C::TRI;
  // traces: quadrilaterals hold the values at the face points, own and the
  // neighbour's (index along the axis), triangles the neighbours' node values
  constexpr int TR = TRI ? NF * NEQ * ND : 2 * NF * NQ * NEQ;

  __shared__ __attribute__((aligned(16))) double s_u[EPB][NEQ][ND];
  __shared__ __attribute__((aligned(16))) double s_g[EPB][2][NEQ][ND];  // contravariant nodal fluxes, then the means
  __shared__ __attribute__((aligned(16))) double s_t[EPB][TR];
  __shared__ __attribute__((aligned(16))) double s_f[EPB][NPT][NEQ];    // weighted face fluxes
  __shared__ double s_nrm[EPB][2 * NF];
  __shared__ int s_nb[EPB][NF], s_code[EPB][NF];

  // opaque to the compiler, so that the persistent form (LOOP) does not keep the LDS
  // addresses formed from it over its loop (they held 160 registers and spilled)
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int team = tid / T, lane = tid - team * T;
  const int64_t NE = A.NE;
  const int64_t NDOFS = NE * ND;
  const int64_t e0 = vb * EPB;
  const int64_t e = e0 + team;
  const bool in = team < EPB && e < NE;
  const int ins = (A.inst && in) ? A.inst[e] : 0;
  const bool active = in && (!A.active || A.active[ins]);

  // every load of the block's setup is issued before the first LDS store; the
  // neighbours' rows, which need the connectivity, follow in one more round trip
  static_assert(2 * NF <= T && ND <= T, "one lane per normal component and node");
  StateRegs<EPB, NEQ, ND, BLOCK> str;
  str.load(A.x, NDOFS, e0, NE, tid);
  const double nv = (active && lane < 2 * NF) ? A.geo[(int64_t)(C::G_NRM + lane) * NE + e] : 0.0;
  const bool face_lane = active && lane < NF;
  const int nb0 = face_lane ? A.nbr[lane * NE + e] : -1;
  const int cd0 = face_lane ? A.fcode[lane * NE + e] : 0;
  int rnb[RP];
#pragma unroll
  for (int p = 0; p < RP; p++) {
    const int it = lane + p * T;
    rnb[p] = (active && it < C::ROWS) ? A.nbr[(it / NEQ) * NE + e] : -1;
  }
  double row[RP][ND];
#pragma unroll
  for (int p = 0; p < RP; p++) {
    if (rnb[p] >= 0) {
      const double* xn = A.x + (int64_t)((lane + p * T) % NEQ) * NDOFS + (int64_t)rnb[p] * ND;
#pragma unroll
      for (int k = 0; k < ND; k++) row[p][k] = xn[k];
    }
  }
  str.store(s_u, tid);
  if (face_lane) {
    s_nb[team][lane] = nb0;
    s_code[team][lane] = nb0 >= 0 ? cd0 : 0;
  }
  if (active && lane < 2 * NF) s_nrm[team][lane] = nv;
  __syncthreads();

  const int j = lane;
  const bool node_lane = active && lane < ND;
  const int jx = TRI ? 0 : j % N, jy = TRI ? 0 : j / N;
  double lmax = 0.0;
  double idet = 0.0;  // inverse mass at this node: 1 / det J (triangles), 1 / (w_j det J)
  double mk = 0.0;    // the node's weight in the element mean, up to a factor per element

  // ---- volume: nodal flux, contravariant components. Edge f runs along
  // (-n_1, n_0) of its area normal n.
  if (!A.face_only && node_lane) {
    const double* n = s_nrm[team];
    double J0, J1, J2, J3;  // dx/dxi, dx/deta, dy/dxi, dy/deta
    double wj = 1.0;
    if constexpr (TRI) {
      mk = tb.mhat[j];
      J0 = -n[1];
      J2 = n[0];
      J1 = n[5];
      J3 = -n[4];
    } else {
      const double x = tb.x[jx], y = tb.x[jy];
      wj = tb.w[jx] * tb.w[jy];
      J0 = (1 - y) * -n[1] + y * n[5];
      J2 = (1 - y) * n[0] + y * -n[4];
      J1 = (1 - x) * n[7] + x * -n[3];
      J3 = (1 - x) * -n[6] + x * n[2];
    }
    const double det = J0 * J3 - J1 * J2;
    idet = recip(wj * det);
    if constexpr (!TRI) mk = wj * det;
    const double adj[4] = {wj * J3, wj * -J1, wj * -J2, wj * J0};
    double st[NEQ];
#pragma unroll
    for (int v = 0; v < NEQ; v++) st[v] = s_u[team][v][j];
    const SidePrim<2> q = side_prim<2>(st, g);
    if (!A.no_lambda) lmax = sqrt_ws(q.m2) * q.inv + side_sound<2>(st, q, g);
#pragma unroll
    for (int r = 0; r < 2; r++) {
      const double a0 = adj[r * 2 + 0], a1 = adj[r * 2 + 1];
      const double ma = st[1] * a0 + st[2] * a1;
      const double mai = ma * q.inv;
      s_g[team][r][0][j] = ma;
      s_g[team][r][1][j] = mai * st[1] + q.p * a0;
      s_g[team][r][2][j] = mai * st[2] + q.p * a1;
      s_g[team][r][3][j] = mai * (st[3] + q.p);
    }
  }
  // ---- traces
  if constexpr (TRI) {
#pragma unroll
    for (int p = 0; p < RP; p++) {
      if (rnb[p] >= 0) {
#pragma unroll
        for (int k = 0; k < ND; k++) s_t[team][(lane + p * T) * ND + k] = row[p][k];
      }
    }
  } else {
    // local faces 0..3: bottom, right, top, left; face f is normal to axis
    // r = (f + 1) % 2, on its side c
#pragma unroll
    for (int p = 0; p < RP; p++) {
      const int it = lane + p * T;
      if (active && it < C::ROWS) {
        const int f = it / NEQ, v = it % NEQ;
        const double* uo = &s_u[team][v][0];
#pragma unroll
        for (int s = 0; s < 2; s++) {
          if (s == 1 && rnb[p] < 0) break;
          const int fs = s == 0 ? f : (s_code[team][f] & 7);
          const bool along_x = (fs & 1) == 0;  // the face runs along x (normal to y)
          const int c = (fs == 1 || fs == 2) ? 1 : 0;
          double tr[N];
#pragma unroll
          for (int a = 0; a < N; a++) {
            double t = 0.0;
#pragma unroll
            for (int k = 0; k < N; k++) {
              const double uv = s == 0 ? uo[along_x ? a + N * k : k + N * a]
                                       : (along_x ? row[p][a + N * k] : row[p][k + N * a]);
              t += tb.E[c][k] * uv;
            }
            tr[a] = t;
          }
#pragma unroll
          for (int i = 0; i < NQ; i++) {
            double t = 0.0;
#pragma unroll
            for (int a = 0; a < N; a++) t += tb.B[i][a] * tr[a];
            s_t[team][((s * NF + f) * NQ + i) * NEQ + v] = t;
          }
        }
      }
    }
  }
  __syncthreads();

  // ---- face points: Riemann solve, weighted flux; one lane per point. The
  // point index i counts along the face's axis (quadrilaterals) or edge
  if (active) {
    const int f = lane / NQ, i = lane - f * NQ;
    const int nb = s_nb[team][f], code = s_code[team][f];
    const int fn = code & 7;
    // edge parameter, mirrored on the neighbour when its edge runs the other way
    const int q = TRI || f < 2 ? i : NQ - 1 - i;
    const int q2 = ((code >> 3) & 2) ? NQ - 1 - q : q;
    double um[NEQ], up[NEQ], fl[NEQ];
    if constexpr (TRI) {
      double ph[ND];
#pragma unroll
      for (int k = 0; k < ND; k++) ph[k] = tb.Phi[f][q][k];
#pragma unroll
      for (int v = 0; v < NEQ; v++) {
        double t = 0.0;
#pragma unroll
        for (int k = 0; k < ND; k++) t += s_u[team][v][k] * ph[k];
        um[v] = t;
      }
    } else {
#pragma unroll
      for (int v = 0; v < NEQ; v++) um[v] = s_t[team][(f * NQ + i) * NEQ + v];
    }
    const bool elem1 = nb < 0 || ((code >> 6) & 1);
    double an[2];
    if (elem1 || A.aligned) {
      // Elem1's normal; where every shared edge has the same two end points the
      // neighbour's is the exact negative of the own one
      an[0] = elem1 ? s_nrm[team][2 * f] : -s_nrm[team][2 * f];
      an[1] = elem1 ? s_nrm[team][2 * f + 1] : -s_nrm[team][2 * f + 1];
    } else {
      an[0] = A.geo[(int64_t)(C::G_NRM + 2 * fn) * NE + nb];
      an[1] = A.geo[(int64_t)(C::G_NRM + 2 * fn + 1) * NE + nb];
    }
    const double normag = sqrt_ws(an[0] * an[0] + an[1] * an[1]);
    const double inv = recip(normag);
    const double nrm[2] = {an[0] * inv, an[1] * inv};
    bool ok = true;
    double lam = 0.0;
    if (!BC || nb >= 0) {
      if constexpr (TRI) {
        double ph[ND];
#pragma unroll
        for (int k = 0; k < ND; k++) ph[k] = tb.Phi[fn][q2][k];
#pragma unroll
        for (int v = 0; v < NEQ; v++) {
          double t = 0.0;
#pragma unroll
          for (int k = 0; k < ND; k++) t += s_t[team][(f * NEQ + v) * ND + k] * ph[k];
          up[v] = t;
        }
      } else {
        const int i2 = fn < 2 ? q2 : NQ - 1 - q2;
#pragma unroll
        for (int v = 0; v < NEQ; v++) up[v] = s_t[team][((NF + f) * NQ + i2) * NEQ + v];
      }
      double sL[NEQ], sR[NEQ];
#pragma unroll
      for (int v = 0; v < NEQ; v++) {
        sL[v] = elem1 ? um[v] : up[v];
        sR[v] = elem1 ? up[v] : um[v];
      }
      lam = riemann_t<2, RS>(g, sL, sR, nrm, fl, ok);
    } else if constexpr (BC) {
      const int slot = -1 - nb;
      if (slot < g.num_bc) {
        const double* Pover = A.bcp ? A.bcp + ((int64_t)ins * RKDG_MAX_BC + slot) * 8 : nullptr;
        bc_state<2>(g, slot, um, nrm, up, Pover);
        if (g.bc_type[slot] == RKDG_BC_CHAR_OUTLET) lam = char_outlet_flux<2>(g, up, nrm, fl);
        else lam = riemann_t<2, RS>(g, um, up, nrm, fl, ok);
      } else {
#pragma unroll
        for (int v = 0; v < NEQ; v++) fl[v] = 0.0;
      }
    }
    if (!ok || lam < 0.0) {
      const int64_t other = nb >= 0 ? (int64_t)nb : -1;
      const bool nf = nonfinite_nodes(A.x, NDOFS, e, ND, NEQ) || nonfinite_nodes(A.x, NDOFS, other, ND, NEQ);
      flag_error(A.err, elem1 ? e : other, elem1 ? other : e, f, nf ? kErrNonFinite : kErrUnphysical);
    } else {
      lmax = lam > lmax ? lam : lmax;
    }
    double wgt = elem1 ? -normag : normag;
    if constexpr (!TRI) wgt *= tb.wq[i];
#pragma unroll
    for (int v = 0; v < NEQ; v++) s_f[team][lane][v] = fl[v] * wgt;
  }

  if (!A.face_only) {
    __syncthreads();
    // ---- node lanes: volume contraction, lift, inverse mass and stage epilogue
    double outv[NEQ];
    if (node_lane) {
      // every base is loaded before the first store (an output may be its own
      // base) and in flight during the contraction; without one the base is the
      // stage input
      const int64_t i0 = e * ND + j;
      const double dtm = A.dt_inst ? A.dt_inst[ins] : 1.0;
      double base[4][NEQ];
#pragma unroll
      for (int m = 0; m < 4; m++) {
        const double* bp = m < A.nout ? A.outs[m].base : nullptr;
        if (bp) {
          bp += i0;
#pragma unroll
          for (int v = 0; v < NEQ; v++) base[m][v] = bp[v * NDOFS];
        }
      }
      double y[NEQ];
#pragma unroll
      for (int v = 0; v < NEQ; v++) y[v] = 0.0;
      if constexpr (TRI) {
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
          for (int k = 0; k < ND; k++) {
            const double kk = tb.KM[r][j][k];
#pragma unroll
            for (int v = 0; v < NEQ; v++) y[v] += kk * s_g[team][r][v][k];
            if (k % 2 == 1) hold();
          }
#pragma unroll
        for (int pt = 0; pt < NPT; pt++) {
          const double ph = tb.LM[pt][j];
#pragma unroll
          for (int v = 0; v < NEQ; v++) y[v] += s_f[team][pt][v] * ph;
          if (pt % 3 == 2) hold();
        }
      } else {
#pragma unroll
        for (int a = 0; a < N; a++) {
          const double dx = tb.D[a][jx], dy = tb.D[a][jy];
#pragma unroll
          for (int v = 0; v < NEQ; v++)
            y[v] += dx * s_g[team][0][v][a + N * jy] + dy * s_g[team][1][v][jx + N * a];
          hold();
        }
#pragma unroll
        for (int f = 0; f < NF; f++) {
          const int c = (f == 1 || f == 2) ? 1 : 0;
          const int ja = (f & 1) == 0 ? jx : jy;  // the node's index along the face, and across it
          const double ec = tb.E[c][(f & 1) == 0 ? jy : jx];
          double L[NEQ];
#pragma unroll
          for (int v = 0; v < NEQ; v++) L[v] = 0.0;
#pragma unroll
          for (int i = 0; i < NQ; i++) {
            const double b = tb.B[i][ja];
#pragma unroll
            for (int v = 0; v < NEQ; v++) L[v] += s_f[team][f * NQ + i][v] * b;
          }
#pragma unroll
          for (int v = 0; v < NEQ; v++) y[v] += L[v] * ec;
          hold();
        }
      }
#pragma unroll
      for (int v = 0; v < NEQ; v++) y[v] *= idet;
      pin<NEQ>(y);
#pragma unroll
      for (int v = 0; v < NEQ; v++) outv[v] = 0.0;
#pragma unroll
      for (int m = 0; m < 4; m++) {
        if (m < A.nout) {
          double* op = A.outs[m].out + i0;
          const double cf = A.outs[m].coef * dtm;
          const double wb = A.outs[m].wb, wi = A.outs[m].wi;
          const bool own = A.outs[m].base == nullptr;
#pragma unroll
          for (int v = 0; v < NEQ; v++) {
            const double u0 = s_u[team][v][j], b = own ? u0 : base[m][v];
            const double o = wi == 0.0 ? b + cf * y[v] : wb * b + wi * (u0 + cf * y[v]);
            op[v * NDOFS] = o;
            if (m == A.means_of) outv[v] = o;
          }
        }
      }
      if (A.k) {
        double* kp = A.k + i0;
#pragma unroll
        for (int v = 0; v < NEQ; v++) kp[v * NDOFS] = y[v];
      }
    }
    if (A.means) {
      __syncthreads();  // the contraction's reads of s_g are done
      if (node_lane) {
#pragma unroll
        for (int v = 0; v < NEQ; v++) s_g[team][1][v][j] = outv[v];
        s_g[team][0][0][j] = mk;
      }
      __syncthreads();
      if (active && lane < NEQ) {
        double s = 0.0, ms = 0.0;
#pragma unroll
        for (int k = 0; k < ND; k++) {
          const double w = s_g[team][0][0][k];
          s += w * s_g[team][1][lane][k];
          ms += w;
        }
        A.means[lane * NE + e] = s / ms;
      }
    }
  }
  // ---- max wave speed: one atomic per wave, or per lane where the block's
  // elements belong to different instances
  if (!A.no_lambda) {
    const int64_t elast = e0 + EPB - 1 < NE ? e0 + EPB - 1 : NE - 1;
    const int i0 = A.inst ? A.inst[e0] : 0;
    if (!A.inst || i0 == A.inst[elast]) {
      for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(lmax, off, 64);
        lmax = o > lmax ? o : lmax;
      }
      if (tid == 0) atomic_max_pos(lam_slot(A.lam, A.lam_ld) + i0, lmax);
    } else if (active) {
      atomic_max_pos(lam_slot(A.lam, A.lam_ld) + ins, lmax);
    }
  }
  __syncthreads();  // LDS is reused by the next work block
}

// One workgroup per work block, or (LOOP, when a grid cap below the number of
// blocks is set) persistent: the grid strides over the work blocks. The loop keeps
// the kernel's arguments in registers over its body, 143 to 165 VGPRs and 140 to
// 175 spilled SGPRs against 90 to 99 (131 for P3 triangles) and 16 to 22 without
// it, and a wave's tables are now too small for sharing them to pay: without it
// the eight ensemble steps above take 4.4 instead of 5.5 ms, the Q2 step 70
// instead of 83 us, the P2 step 187 instead of 207 us.
template <int GEOM, int P, int RS, bool BC, bool LOOP>
__global__ __launch_bounds__(64, 3) void dense_rhs_kernel(const RhsArgs A, const SchemeParams g,
                                                       const double* __restrict__ gtab, int64_t nvb) {
  __shared__ __attribute__((aligned(16))) DenseRhsTab<GEOM, P> tb;
  CopyRegs<sizeof(DenseRhsTab<GEOM, P>) / sizeof(double), 64> tbr;
  tbr.load(gtab, threadIdx.x);
  tbr.store(reinterpret_cast<double*>(&tb), threadIdx.x);
  __syncthreads();
  if constexpr (!LOOP) {
    dense_rhs_block<GEOM, P, RS, BC>(A, g, xcd_remap_d(blockIdx.x, nvb), tb);
    return;
  }
  for (int64_t vb = blockIdx.x; vb < nvb; vb += gridDim.x) {
    // keep table reads inside the iteration (hoisted, they would hold registers across the loop)
    asm volatile("" ::: "memory");
    dense_rhs_block<GEOM, P, RS, BC>(A, g, vb, tb);
  }
}

template <int GEOM, int P>
__global__ __launch_bounds__(256) void dense_means_kernel(const MeansArgs A, const double* __restrict__ gtab) {
  using C = DC<GEOM, P>;
  constexpr int ND = C::ND, NEQ = C::NEQ;
  const DenseTab<GEOM, P>* tb = reinterpret_cast<const DenseTab<GEOM, P>*>(gtab);
  const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (e >= A.NE) return;
  const int64_t NDOFS = A.NE * ND;
  double s[NEQ], ms = 0.0;
#pragma unroll
  for (int v = 0; v < NEQ; v++) s[v] = 0.0;
  for (int k = 0; k < ND; k++) {
    const double mk = C::TRI ? tb->mhat[k] * A.geo[(int64_t)C::G_DET * A.NE + e]
                             : A.geo[(int64_t)(C::G_MW + k) * A.NE + e];
    ms += mk;
#pragma unroll
    for (int v = 0; v < NEQ; v++) s[v] += mk * A.x[v * NDOFS + e * ND + k];
  }
#pragma unroll
  for (int v = 0; v < NEQ; v++) A.means[v * A.NE + e] = s[v] / ms;
}

// Limiter. Only the deciding variable's indicator is formed (density for the
// multiplier, indicator_bj.cpp:193; the last variable for FinDiff,
// limiter_findiff.cpp:7-8).
//
// One lane per vertex: lane f of an element's T = 3 or 4 evaluates vertex f and
// the two indicator points of edge f from the nodes staged in LDS, 21 triangles or
// 16 quadrilaterals per wavefront. Teams sized for the right-hand side's points
// (16 lanes for a P2 triangle) worked on 6 points and 3 vertices with 4 elements
// per wavefront (120,540 P2 triangles: 23.5 -> 10.7 us; 473,000 Q1 quadrilaterals:
// 44 -> 25 us; 27,467 Q2: 11.1 -> 6.6 us). An element whose factor is exactly 1 is
// not written in place.
template <int GEOM, int P>
struct LDC : DC<GEOM, P> {
  using D = DC<GEOM, P>;
  static constexpr int T = D::NV;
  static constexpr int EPB = 64 / T;
  static constexpr int ROW = D::ND + (D::ND & 1);
  // LDS stride of an element: the elements of a wavefront, which read the same
  // node at once, start on different banks
  static constexpr int ES = D::NEQ * ROW + (32 + 2 - (D::NEQ * ROW) % 32) % 32;
  static constexpr int NTAB = (2 * D::NF + D::NV) * D::ND;  // PhiI, PhiV: the end of DenseTab
};

// minimum over the T lanes of an element (lane: its index)
template <int T>
__device__ __forceinline__ double vertex_min(double x, int lane) {
  const int base = (int)(threadIdx.x % 64) - lane;
  const double x0 = x;
#pragma unroll
  for (int k = 1; k < T; k++) {
    const int src = lane + k < T ? lane + k : lane + k - T;
    const double o = __shfl(x0, base + src, 64);
    x = o < x ? o : x;
  }
  return x;
}

template <int GEOM, int P>
__global__ __launch_bounds__(64, 4) void dense_limit_kernel(const LimitArgs A, const SchemeParams g,
                                                         const double* __restrict__ gtab) {
  using C = LDC<GEOM, P>;
  constexpr int ND = C::ND, NEQ = C::NEQ, NF = C::NF, T = C::T, EPB = C::EPB;
  constexpr int ROW = C::ROW, ES = C::ES, NTAB = C::NTAB;

  __shared__ __attribute__((aligned(16))) double s_u[EPB * ES];  // [element][variable][node]
  __shared__ double s_tab[NTAB];
  __shared__ double s_mean[EPB][NEQ];
  __shared__ double s_f[EPB];
  __shared__ int s_on[EPB];

  const int tid = threadIdx.x;
  const int team = tid / T, lane = tid - team * T;
  const int64_t NE = A.NE;
  const int64_t NDOFS = NE * ND;
  const int64_t e0 = xcd_remap_d(blockIdx.x, gridDim.x) * EPB;
  const int64_t e = e0 + team;
  const bool in = team < EPB && e < NE;
  const bool active = in && (!A.active || A.active[A.inst[e]]);
  const bool multi = g.limiter == RKDG_LIM_MULTI, findiff = g.limiter == RKDG_LIM_FINDIFF;
  const int vsel = findiff ? NEQ - 1 : 0;

  // every load of the setup is issued before the first LDS store
  constexpr int LP = (EPB * ND + 63) / 64;
  const int nn = (int)((NE - e0 < EPB ? NE - e0 : EPB) * ND);  // nodes of this block's elements
  double st[LP][NEQ];
#pragma unroll
  for (int p = 0; p < LP; p++) {
    const int i = tid + 64 * p;
#pragma unroll
    for (int v = 0; v < NEQ; v++) st[p][v] = i < nn ? sbase(A.x + (v * NDOFS + e0 * ND))[(unsigned)i] : 1.0;
  }
  CopyRegs<NTAB, 64> tbr;
  tbr.load(gtab + (sizeof(DenseTab<GEOM, P>) / sizeof(double) - NTAB), tid);
  // the element's means (lane v; three lanes hold four variables) and the
  // deciding variable's mean across edge f = lane
  static_assert(NF == T && NEQ <= T + 1, "one lane per vertex and edge");
  const bool ind_bj = g.indicator == RKDG_IND_BJ;
  const bool venkat = g.phi == RKDG_PHI_VENKAT && g.venkat_k > 0.0;
  const double mown = active ? A.means[lane * NE + e] : 0.0;
  const double mlast = (NEQ > T && active && lane == 0) ? A.means[T * NE + e] : 0.0;
  const int nbl = (active && ind_bj) ? A.nbr[lane * NE + e] : -1;
  const double nml = nbl >= 0 ? A.means[vsel * NE + nbl] : 0.0;
  double eps2 = 0.0;
  if (active && venkat) {
    // (K h)^3 with h = |element|^(1/2); a quadrilateral's area from its edges,
    // edge f running along (-n_1, n_0) of its area normal n
    double area;
    if (C::TRI) {
      area = 0.5 * A.geo[(int64_t)C::G_DET * NE + e];
    } else {
      double n[6];
#pragma unroll
      for (int k = 0; k < 6; k++) n[k] = A.geo[(int64_t)(C::G_NRM + k) * NE + e];
      const double d0 = n[0] + n[2], d1 = n[1] + n[3];  // the normal of the diagonal
      area = 0.5 * ((n[0] * n[3] - n[1] * n[2]) + (d0 * n[5] - d1 * n[4]));
    }
    const double kh = g.venkat_k * sqrt(area);
    eps2 = kh * kh * kh;
  }
#pragma unroll
  for (int p = 0; p < LP; p++) {
    const int i = tid + 64 * p;
    if (i < EPB * ND) {
      const int el = i / ND, k = i - el * ND;
#pragma unroll
      for (int v = 0; v < NEQ; v++) s_u[el * ES + v * ROW + k] = st[p][v];
    }
  }
  tbr.store(s_tab, tid);
  if (team < EPB) {
    s_mean[team][lane] = mown;
    if (NEQ > T && lane == 0) s_mean[team][NEQ - 1] = mlast;
  }
  __syncthreads();
  double mean[NEQ];
#pragma unroll
  for (int v = 0; v < NEQ; v++) mean[v] = s_mean[team < EPB ? team : 0][v];
  const double msel = findiff ? mean[NEQ - 1] : mean[0];
  double mI = 1e9, MI = -1e9;
  if (ind_bj) {
    // stencil bounds of the means: the cell and its edge neighbours
    const double a = nbl >= 0 ? nml : msel;
    mI = vertex_min<T>(a < msel ? a : msel, lane);
    MI = -vertex_min<T>(-(a > msel ? a : msel), lane);
  }
  const double* ue = &s_u[(team < EPB ? team : 0) * ES];
  const double* pv = &s_tab[2 * NF * ND + lane * ND];
  double vs[NEQ];  // the state at the vertex
  double yr = 1e9;
  if (ind_bj) {
    const double* p0 = &s_tab[2 * lane * ND];
    const double* u = ue + vsel * ROW;
    double pt[2] = {0.0, 0.0}, V = 0.0;
#pragma unroll
    for (int k = 0; k < ND; k++) {
      const double x = u[k];
      pt[0] += x * p0[k];
      pt[1] += x * p0[ND + k];
      V += x * pv[k];
    }
    vs[0] = V;
    if (nbl >= 0) {
#pragma unroll
      for (int ip = 0; ip < 2; ip++) {
        const double diff = pt[ip] - msel;
        const double y = indicator_y(diff, msel, mI, MI);
        double yc;
        if (g.phi == RKDG_PHI_BJ) {
          yc = y < 1.0 ? y : 1.0;
        } else if (g.phi == RKDG_PHI_VENKAT) {
          if (g.venkat_k > 0.0) {
            const double d2 = diff * diff;
            yc = (d2 * (y * y + 2.0 * y) + eps2) / (d2 * (y * y + y + 2.0) + eps2);
          } else {
            yc = (y * y + 2.0 * y) / (y * y + y + 2.0);
          }
        } else {
          const double yStar = 1.5;
          const double yRel = y / yStar;
          yc = y < 1.0 ? y + (3.0 - 2.0 * yStar) * yRel * yRel + (yStar - 2.0) * yRel * yRel * yRel : 1.0;
        }
        yr = yc < yr ? yc : yr;
      }
    }
    yr = vertex_min<T>(yr, lane);
  }
  if (g.indicator == RKDG_IND_NOWHERE) yr = 1.0;
  else if (g.indicator == RKDG_IND_EVERYWHERE) yr = 0.0;

  const bool linear = P == 1 && !C::TRI && g.linearize && multi;
  if constexpr (P == 1 && !C::TRI) {
    // linearize: the multiplier and the last hope work on the element's linear
    // reconstruction (triangles are skipped, limiter_multiplier.cpp:29); lane = node
    if (linear) {
      double lin[NEQ];
#pragma unroll
      for (int v = 0; v < NEQ; v++) lin[v] = linearize_q1<2>(ue + v * ROW, mean[v], lane);
      __syncthreads();
#pragma unroll
      for (int v = 0; v < NEQ; v++) s_u[team * ES + v * ROW + lane] = lin[v];
      __syncthreads();
    }
  }
  int trouble = 0;
  double f = 1.0;  // the factor of the limited state mean + f (u - mean)
  if (multi) {
    if (yr < 1.0) trouble = 1;
    f = yr;
    if (g.pow_nd) {
      double acc = 1.0, b = yr;
#pragma unroll
      for (int e2 = ND; e2 > 0; e2 >>= 1) {
        if (e2 & 1) acc *= b;
        b *= b;
      }
      f = acc;
    }
    if (g.last_hope) {
#pragma unroll
      for (int v = 0; v < NEQ; v++) {
        if (v > 0 || !ind_bj || linear) {
          double V = 0.0;
#pragma unroll
          for (int k = 0; k < ND; k++) V += ue[v * ROW + k] * pv[k];
          vs[v] = V;
        }
        vs[v] = mean[v] + f * (vs[v] - mean[v]);
      }
      // any unphysical vertex of the team's element (one ballot, no barrier)
      const unsigned long long bm = __ballot(active && !physical<2>(vs, g));
      if (active && ((bm >> (team * T)) & ((1ull << T) - 1ull))) {
        trouble |= 2;
        f = 0.0;
      }
    }
    // an element with a mean that is not finite is written also where the factor is 1:
    // mean + f (u - mean) leaves no node of that variable finite
    double t = 0.0;
#pragma unroll
    for (int v = 0; v < NEQ; v++) t += 0.0 * mean[v];
    if (f == 1.0 && !(t == 0.0)) f = 0x1.fffffffffffffp-1;
  } else if (findiff) {
    if (yr < 0.999) {
      trouble = 1;
      f = 0.0;
    }
  }
  if (A.troubled && active && lane == 0) A.troubled[e] = (int8_t)trouble;
  if (team < EPB && lane == 0) {
    s_f[team] = f;
    s_on[team] = active && (A.out || f != 1.0 || linear);
  }
  __syncthreads();
  double* dst = A.out ? A.out : A.x;
#pragma unroll
  for (int p = 0; p < LP; p++) {
    const int i = tid + 64 * p;
    if (i < nn) {
      const int el = i / ND, k = i - el * ND;
      if (s_on[el]) {
        const double fe = s_f[el];
#pragma unroll
        for (int v = 0; v < NEQ; v++) {
          const double m = s_mean[el][v], u = s_u[el * ES + v * ROW + k];
          sbase(dst + (v * NDOFS + e0 * ND))[(unsigned)i] = fe == 1.0 ? u : m + fe * (u - m);
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
bool dense_supported(int geom, int p) {
#define X(G, PP) \
  if (geom == G && p == PP) return true;
  RKDG_DENSE_CASES(X)
#undef X
  return false;
}

int dense_table_size(int geom, int p) {
#define X(G, PP) \
  if (geom == G && p == PP) return (int)(sizeof(DenseTab<G, PP>) / sizeof(double));
  RKDG_DENSE_CASES(X)
#undef X
  return 0;
}

int dense_rhs_table_size(int geom, int p) {
#define X(G, PP) \
  if (geom == G && p == PP) return (int)(sizeof(DenseRhsTab<G, PP>) / sizeof(double));
  RKDG_DENSE_CASES(X)
#undef X
  return 0;
}

int dense_geo_size(int geom, int p) {
#define X(G, PP) \
  if (geom == G && p == PP) return DC<G, PP>::GSIZE;
  RKDG_DENSE_CASES(X)
#undef X
  return 0;
}

template <int G, int PP, int RS>
hipError_t dense_rhs_rs(const RhsArgs& a, const SchemeParams& g, const double* t, bool bc, hipStream_t s) {
  using C = RC<G, PP>;
  const int64_t nvb = (a.NE + C::EPB - 1) / C::EPB;
  const int64_t grid = a.grid_cap > 0 && a.grid_cap < nvb ? a.grid_cap : nvb;
  auto launch = [&](auto kernel) {
    kernel<<<(unsigned)grid, C::BLOCK, 0, s>>>(a, g, t, nvb);
    return hipGetLastError();
  };
  if (grid < nvb) return launch(bc ? dense_rhs_kernel<G, PP, RS, true, true> : dense_rhs_kernel<G, PP, RS, false, true>);
  return launch(bc ? dense_rhs_kernel<G, PP, RS, true, false> : dense_rhs_kernel<G, PP, RS, false, false>);
}


template <int G, int PP>
hipError_t dense_rhs_gp(const RhsArgs& a, const SchemeParams& g, const double* t, bool bc, hipStream_t s) {
  switch (g.riemann) {
    case RKDG_RS_RUSANOV: return dense_rhs_rs<G, PP, RKDG_RS_RUSANOV>(a, g, t, bc, s);
    case RKDG_RS_LLF: return dense_rhs_rs<G, PP, RKDG_RS_LLF>(a, g, t, bc, s);
    case RKDG_RS_HLL: return dense_rhs_rs<G, PP, RKDG_RS_HLL>(a, g, t, bc, s);
    default: return dense_rhs_rs<G, PP, RKDG_RS_HLLC>(a, g, t, bc, s);
  }
}

hipError_t launch_dense_rhs(int geom, int p, const RhsArgs& a, const SchemeParams& g, const double* t,
                            bool has_bdr, hipStream_t s) {
#define X(G, PP) \
  if (geom == G && p == PP) return dense_rhs_gp<G, PP>(a, g, t, has_bdr, s);
  RKDG_DENSE_CASES(X)
#undef X
  return hipErrorInvalidValue;
}

hipError_t launch_dense_limit(int geom, int p, const LimitArgs& a, const SchemeParams& g, const double* t,
                              hipStream_t s) {
#define X(G, PP)                                                                \
  if (geom == G && p == PP) {                                                   \
    using C = LDC<G, PP>;                                                       \
    const int64_t nb = (a.NE + C::EPB - 1) / C::EPB;                            \
    dense_limit_kernel<G, PP><<<(unsigned)nb, 64, 0, s>>>(a, g, t);             \
    return hipGetLastError();                                                   \
  }
  RKDG_DENSE_CASES(X)
#undef X
  return hipErrorInvalidValue;
}

hipError_t launch_dense_means(int geom, int p, const MeansArgs& a, const double* t, hipStream_t s) {
#define X(G, PP)                                                                         \
  if (geom == G && p == PP) {                                                            \
    dense_means_kernel<G, PP><<<(unsigned)((a.NE + 255) / 256), 256, 0, s>>>(a, t);    \
    return hipGetLastError();                                                            \
  }
  RKDG_DENSE_CASES(X)
#undef X
  return hipErrorInvalidValue;
}

}  // namespace rkdg
