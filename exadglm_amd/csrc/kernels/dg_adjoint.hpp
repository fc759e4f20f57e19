// Discrete adjoint of the DGLM RHS and of one LSRK4(5) stage (FP64).
//
// Forward stage (see dg_fp64.hpp):  r = R(u; tau) = A B(u; tau),
//   A = [WDr | WDs | WDt | -LIFT],  B = stacked volume fluxes and LM surface
//   fluxes;  k' = a k + dt r;  u' = u + b k'.
// Reverse stage, given the adjoints (ubar, kbar) of (u', k'):
//   kb = kbar + b ubar;  rbar = dt kb;  kbar <- a kb;
//   ubar <- ubar + J_B(u)^T (A^T rbar),   taubar_f += dB/dtau_f . (A^T rbar)
// J_B^T has three parts:
//   volume   B[d*Np+j] = sum_x metric[d][x] F^x(u_j): pointwise transposed
//            Jacobians of F, G, H at node j;
//   own face fLM(m) = (n.F(ub) - tau (ub - u-)) Fscale, ub = (u- + u+)/2:
//            d/du- = Fscale (J_n(ub)/2 + tau/2), added at the face node's
//            volume node;
//   partner  the same flux seen from the neighbour element depends on this
//            element's node through its u+:  d/du+ = Fscale_nbr (J_nbr(ub)/2
//            - tau/2).  The neighbour's pass A forms it beside its own-side
//            term (the same ub, normal, h and tau) and stores it at its face
//            slot; each element PULLS these terms through the partner slot
//            (exact by the involution of the face connectivity) -- no
//            atomics, so the adjoint is bitwise deterministic.
// Pass A (dg_adjoint_euler.hpp, dg_adjoint_adv.hpp) computes A^T rbar, the volume
// and own-face terms and tau-bar, and stores the partner-side face terms; the
// next pass A adds them to ubar before anything else, and after the last one
// pass B does.
#pragma once
#include "dg_adjoint_args.hpp"
#include "dg_fp64.hpp"

namespace dglm {

// w += J_n(U)^T h, J_n = d(n.F)/dU of the Euler flux at U (5 conserved vars).
__device__ inline void euler_jt(const double U[5], double nx, double ny, double nz, const double h[5], double g,
                                double w[5]) {
  const double inv = 1.0 / U[0];
  const double v[3] = {U[1] * inv, U[2] * inv, U[3] * inv};
  const double n[3] = {nx, ny, nz};
  const double q2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
  const double p = (g - 1.0) * (U[4] - 0.5 * U[0] * q2);
  const double H = (U[4] + p) * inv;
  const double vn = nx * v[0] + ny * v[1] + nz * v[2];
  const double gm = g - 1.0;
  // rho column
  double w0 = h[4] * vn * (gm * 0.5 * q2 - H);
  double hn = 0.0, hv = 0.0;  // sum_c h_c n_c, sum_c h_c v_c
  for (int c = 0; c < 3; c++) {
    w0 += h[1 + c] * (-v[c] * vn + n[c] * gm * 0.5 * q2);
    hn += h[1 + c] * n[c];
    hv += h[1 + c] * v[c];
  }
  w[0] += w0;
  // momentum columns j: h0 n_j + sum_c h_c (v_c n_j + d_cj vn - n_c gm v_j) + h4 (H n_j - gm v_j vn)
  for (int j = 0; j < 3; j++)
    w[1 + j] += h[0] * n[j] + hv * n[j] + h[1 + j] * vn - hn * gm * v[j] + h[4] * (H * n[j] - gm * v[j] * vn);
  // energy column
  w[4] += hn * gm + h[4] * g * vn;
}

// Pass B: one thread per volume node; pull the partner-side terms of the
// (at most 3) faces the node lies on.  The partner element's pass A formed
// them (same ub, normal, h and tau as its own-side term) and stored them at
// its face-node slot, so only the connectivity, that slot and ubar are read.
template <int N, int PHYS>
__global__ __launch_bounds__(256) void adjoint_pass_b(AdjArgs a) {
  using O = Ord<N>;
  constexpr int Np = O::Np, Nfp = O::Nfp, NFF = O::NFF;
  constexpr int NV = NVar<PHYS>::value;
  __shared__ int s_slots[Np * 3], s_pslot[16 * Nfp];
  for (int i = threadIdx.x; i < Np * 3; i += 256) s_slots[i] = a.node_slots[i];
  for (int i = threadIdx.x; i < 16 * Nfp; i += 256) s_pslot[i] = a.pslot[i];
  __syncthreads();
  const int K = a.K;
  const size_t KNp = (size_t)K * Np;
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= K * Np) return;
  const int e = idx / Np, i = idx - e * Np;
  // all loads of the (at most 3) partner slots first, then the sums
  double t[3][NV];
#pragma unroll
  for (int q = 0; q < 3; q++) {
    const int ms = s_slots[i * 3 + q];
#pragma unroll
    for (int v = 0; v < NV; v++) t[q][v] = 0.0;
    if (ms >= 0) {
      const int f = ms / Nfp, j = ms - f * Nfp;
      const int c = a.conn[(size_t)e * 4 + f];
      const double *gs = &a.gsur[((size_t)conn_nbr(c) * NFF + s_pslot[(conn_face(c) * 4 + conn_code(c)) * Nfp + j]) * NV];
#pragma unroll
      for (int v = 0; v < NV; v++) t[q][v] = gs[v];
    }
  }
  for (int v = 0; v < NV; v++) {
    double w = 0.0;
#pragma unroll
    for (int q = 0; q < 3; q++) w += t[q][v];
    a.ubar[v * KNp + idx] += w;
  }
}

// Wave-speed adjoint of one step (Euler): lambda_f enters tau of both sides
// of face f and, for the face attaining max(lambda*Fscale), dt.  The
// derivative of lambda = sqrt(max v^2) + sqrt(max |gamma p/rho|) follows the
// argmax nodes the forward picked (first strict maximum, as calc_maxv).
// A block takes LAM_ADJ_EB(Np) elements: |v|^2 and |gamma p/rho| of their
// nodes are formed with coalesced loads into LDS (the arithmetic of the
// forward wave-speed kernel, so the same argmax), then one thread per face side
// scans its face nodes and forms the ubar increments at the argmax nodes into
// LDS, and four threads per element (one or two variables each) add them in
// face order, so the accumulation order per node is fixed and the result
// deterministic.
__host__ __device__ constexpr int lam_adj_elems(int Np) { return Np <= 35 ? 64 : (Np <= 84 ? 32 : 16); }

template <int N>
__global__ __launch_bounds__(4 * lam_adj_elems(Ord<N>::Np)) void lambda_adjoint_kernel(
    int K, const double *__restrict__ u, const double *__restrict__ lam, const double *__restrict__ taubar,
    const int *__restrict__ conn, const int *__restrict__ fmx, const double *dt_seq, const int *fstar_seq, int step,
    const double *scal, double tau_scale, double gamma, double *ubar) {
  using O = Ord<N>;
  constexpr int Np = O::Np, Nfp = O::Nfp;
  constexpr int EB = lam_adj_elems(Np), NT = 4 * EB;
  __shared__ double s_v2[EB * Np], s_c2[EB * Np];
  __shared__ int s_fm[4 * Nfp];
  __shared__ int s_nv[NT], s_nc[NT];  // argmax volume nodes (-1: none)
  __shared__ double s_dv[4][NT];      // increments of rho, rho v at the |v|^2 argmax
  __shared__ double s_dc[5][NT];      // increments of all five at the c^2 argmax
  const size_t KNp = (size_t)K * Np;
  const int t = threadIdx.x;
  const int e0 = blockIdx.x * EB;
  const int ne = min(EB, K - e0);
  for (int i = t; i < 4 * Nfp; i += NT) s_fm[i] = fmx[((i / Nfp) * 4 + 3) * Nfp + i % Nfp];
  for (int i = t; i < ne * Np; i += NT) {
    const size_t idx = (size_t)e0 * Np + i;
    node_speeds(u[idx], u[KNp + idx], u[2 * KNp + idx], u[3 * KNp + idx], u[4 * KNp + idx], gamma, s_v2[i], s_c2[i]);
  }
  __syncthreads();
  const int el = t >> 2, f = t & 3, e = e0 + el;
  int nv = -1, nc = -1;
  if (el < ne) {
    const double dtbar = scal[1], dt = dt_seq[step];
    const int o = e * 4 + f;
    const int c = conn[o];
    const int nbf = conn_nbr(c) * 4 + conn_face(c);
    double lb = 0.25 * tau_scale * (taubar[o] + taubar[nbf]);
    if (o == fstar_seq[step]) lb += -dtbar * dt / lam[o];
    if (lb != 0.0) {
      double mv2 = 0.0, mc2 = 0.0;
      int jv = -1, jc = -1;
      for (int j = 0; j < Nfp; j++) {
        const int q = el * Np + s_fm[f * Nfp + j];
        const double v2 = s_v2[q], c2 = s_c2[q];
        if (v2 > mv2) {
          mv2 = v2;
          jv = j;
        }
        if (c2 > mc2) {
          mc2 = c2;
          jc = j;
        }
      }
      if (jv >= 0) {
        nv = s_fm[f * Nfp + jv];
        const size_t idx = (size_t)e * Np + nv;
        const double r = u[idx], v[3] = {u[KNp + idx] / r, u[2 * KNp + idx] / r, u[3 * KNp + idx] / r};
        const double s = lb / (2.0 * sqrt(mv2));
        s_dv[0][t] = s * (-2.0 * mv2 / r);
        for (int q = 0; q < 3; q++) s_dv[1 + q][t] = s * (2.0 * v[q] / r);
      }
      if (jc >= 0) {
        nc = s_fm[f * Nfp + jc];
        const size_t idx = (size_t)e * Np + nc;
        const double r = u[idx], v[3] = {u[KNp + idx] / r, u[2 * KNp + idx] / r, u[3 * KNp + idx] / r};
        const double v2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
        const double gm = gamma - 1.0;
        const double p = gm * (u[4 * KNp + idx] - 0.5 * r * v2);
        const double sg = gamma * p / r >= 0.0 ? 1.0 : -1.0;
        const double s = sg * lb / (2.0 * sqrt(mc2));
        s_dc[0][t] = s * gamma * (gm * 0.5 * v2 / r - p / (r * r));
        for (int q = 0; q < 3; q++) s_dc[1 + q][t] = s * gamma * (-gm * v[q]) / r;
        s_dc[4][t] = s * gamma * gm / r;
      }
    }
  }
  s_nv[t] = nv;
  s_nc[t] = nc;
  __syncthreads();
  // thread (element el, k) adds variable k (and variable 4 for k = 0) over
  // the element's four faces in face order; distinct variables never alias
  if (el < ne) {
    const int k = f;
#pragma unroll
    for (int x = 0; x < 2; x++) {
      const int v = x == 0 ? k : 4;
      if (x == 1 && k != 0) break;
      for (int ff = 0; ff < 4; ff++) {
        const int q = 4 * el + ff;
        if (v < 4 && s_nv[q] >= 0) ubar[v * KNp + (size_t)e * Np + s_nv[q]] += s_dv[v][q];
        if (s_nc[q] >= 0) ubar[v * KNp + (size_t)e * Np + s_nc[q]] += s_dc[v][q];
      }
    }
  }
}

}  // namespace dglm
