// Pass A of the discrete Euler adjoint on FP64 MFMA (gfx950), every order.
//
// Mathematics in dg_adjoint.hpp.  As in the packed-column stage kernel
// (dg_cols.hpp) the columns of g = A^T rbar are the (variable, element) pairs of
// EB elements, its rows go to the waves as 16-row tiles and 4-row units, and the
// operator is streamed from the L2 in 16-byte loads.  Per workgroup:
//   0. nodes in memory order: u, ubar, kbar; ubar takes the partner-side face
//      terms the pass A before it left (when given: that pass's pass B); kbar is
//      updated and rbar = dt (kbar + b ubar) goes to LDS.  The exterior traces
//      are gathered and stay in registers;
//   1. g = A^T rbar on MFMA into LDS, [column][row];
//   2. face-node slots in memory order: the transposed flux Jacobian at the face
//      state, own-side term (into g's row of the slot), partner-side term
//      (stored for the next pass), tau-bar partial;
//   3. nodes: transposed volume Jacobians, the node's own-side terms, ubar.
// One thread per face-node slot and not per (node, face): at N = 4 an element
// has 60 slots and 35 nodes on up to three faces each, so a node-wise face part
// issues 105 masked evaluations.
// The dt partial sum_nodes kb . r comes from the homogeneity of the Euler flux,
// F(U) = J(U) U: sum over rows of g . B(u) is, at a node, (sum_x J_x^T h^x) . U
// and, at slot m, 2 (J_n(ub)^T h_m) . ub + tau tc_m.
#pragma once
#include "adjoint_ops.h"
#include "dg_adjoint.hpp"
#include "dg_cols.hpp"

namespace dglm {

template <int N>
struct EulAdjShape {
  using O = Ord<N>;
  static constexpr int Np = O::Np, Nfp = O::Nfp, NFF = O::NFF, KD = O::KD;
  static constexpr int G = (Np + 3) / 4, NS = 4 * (G | 1);  // k-steps; column stride of rbar and the state (dg_cols.hpp)
  static constexpr int U = (KD + 3) / 4, GS = 4 * (U | 1);  // row units of A^T; column stride of g
  // Elements and waves.  At N = 1 six elements are 24 nodes and 72 slots, a third of
  // four waves' threads at best, so there one wave takes eight elements (us per four
  // steps recorded and swept back, [elements, waves], the last at four waves a SIMD
  // and the others at three):
  //   K        [6,4]   [6,1]  [10,1]   [8,1]   [8,1]
  //   750        625     651     647     670     620
  //   3072       690     721     722     735     685
  //   16,464    1170     989     937     981     929
  //   48,000    2653    1935    1965    1926    1846
  //   444,528  20384   11540   11645   11442   10554   ([8,2] 12500, [16,1] 11937)
  static constexpr int EB = N == 1 ? 8 : N <= 4 ? 6 : (N <= 9 ? 3 : 2);
  static constexpr int NW = N == 1 ? 1 : N <= 7 ? 4 : 8, NT = 64 * NW;
  static constexpr int WPE = N == 1 ? 4 : N <= 6 ? 3 : 2;  // waves per SIMD (3: three workgroups a CU)
  static constexpr int NC = 5 * EB, CT = (NC + 15) / 16;
  static constexpr int KB = (G + 1) / 2;  // blocks of two k-steps
  static constexpr ColRoles<NW> roles = cols_roles<U, CT, NW>();
  // operator stream of wave w: per block a lane's 2 na values as 16-byte pairs,
  // [row set][lane][k-step of the block]
  static constexpr size_t stream(int w) {
    size_t o = 0;
    for (int i = 0; i < w; i++) o += (size_t)KB * 2 * roles.r[i].na() * 64;
    return o;
  }
};

template <int N>
inline void eul_adj_arrange(const double *opT, double *out) {
  using S = EulAdjShape<N>;
  for (int w = 0; w < S::NW; w++) {
    const ColRole r = S::roles.r[w];
    const int na = r.na();
    double *o = out + S::stream(w);
    for (int b = 0; b < S::KB; b++)
      for (int x = 0; x < na; x++)
        for (int l = 0; l < 64; l++)
          for (int s = 0; s < 2; s++) {
            const int i = 4 * (2 * b + s) + (l >> 4);
            const int k = x < r.nt ? 16 * (r.tile0 + x) + 4 * (l & 3) + ((l >> 2) & 3)
                          : x == r.nt && r.xt >= 0
                              ? 16 * r.xt + 4 * (l & 3) + ((l >> 2) & 3)
                              : 4 * (r.q0 + x - r.nt - (r.xt >= 0 ? 1 : 0)) + (l & 3);
            o[(((size_t)b * na + x) * 64 + l) * 2 + s] = i < S::Np && k < S::KD ? opT[(size_t)k * S::Np + i] : 0.0;
          }
  }
}

template <int N>
__global__ __launch_bounds__(EulAdjShape<N>::NT, EulAdjShape<N>::WPE) void adjoint_euler_kernel(AdjArgs a,
                                                                             const double *__restrict__ afragT) {
  using S = EulAdjShape<N>;
  constexpr int Np = S::Np, Nfp = S::Nfp, NFF = S::NFF, G = S::G, NS = S::NS, GS = S::GS, EB = S::EB, NT = S::NT;
  constexpr int NC = S::NC, CT = S::CT;
  // rbar, then the state: [variable][element][node]; then the tau-bar partials [element][slot]
  __shared__ __align__(16) double s_r[NC * NS];
  static_assert(EB * NFF <= NC * NS, "tau-bar partials fit");
  __shared__ __align__(16) double s_g[NC * GS];  // A^T rbar [variable][element][row]
  __shared__ double s_geo[EB * GEO_STRIDE];
  __shared__ double s_tau[EB * 4];
  __shared__ double red[S::NW];
  __shared__ int s_conn[EB * 4];
  __shared__ unsigned short s_fmx[16 * Nfp], s_pslot[16 * Nfp];
  __shared__ short s_slots[Np * 3];

  const int K = a.K;
  const size_t KNp = (size_t)K * Np;
  const int batch = xcd_batch(a.order, (K + EB - 1) / EB);
  if (batch < 0) return;
  const int e0 = batch * EB;
  const int ne = min(EB, K - e0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const size_t n0 = (size_t)e0 * Np;

  // ---- 0. stage in (elements past the end of a short batch: a state at rest) ----
  constexpr int RN = (EB * Np + NT - 1) / NT, RF = (EB * NFF + NT - 1) / NT;
  static_assert(4 * EB <= NT, "one face per thread");
  double lam_own = 0.0, lam_nbr = 0.0;
  if (tid < 4 * EB) {
    const int c = tid < 4 * ne ? a.conn[(size_t)e0 * 4 + tid] : 0;
    s_conn[tid] = c;
    if (tid < 4 * ne) {
      lam_own = a.maxv[(size_t)e0 * 4 + tid];
      lam_nbr = a.maxv[(size_t)conn_nbr(c) * 4 + conn_face(c)];
    }
  }
  double U[RN][5], UB[RN][5], R[RN][5];
#pragma unroll
  for (int r = 0; r < RN; r++) {
    const int i = tid + NT * r;
    const bool live = i < ne * Np;
#pragma unroll
    for (int v = 0; v < 5; v++) {
      U[r][v] = v == 0 ? 1.0 : 0.0;
      UB[r][v] = R[r][v] = 0.0;
      if (live) {
        const size_t gi = v * KNp + n0 + i;
        U[r][v] = a.u[gi];
        if (a.mode == 0) {
          UB[r][v] = a.ubar[gi];
          if (!a.first) R[r][v] = a.kbar[gi];
        } else {
          R[r][v] = a.rbar[gi];
        }
      }
    }
  }
  for (int i = tid; i < 16 * Nfp; i += NT) {
    s_fmx[i] = a.fmx[i];
    s_pslot[i] = a.pslot[i];
  }
  for (int i = tid; i < Np * 3; i += NT) s_slots[i] = a.node_slots[i];
  for (int i = tid; i < EB * GEO_STRIDE; i += NT) s_geo[i] = i < ne * GEO_STRIDE ? a.geo[(size_t)e0 * GEO_STRIDE + i] : 0.0;
  if constexpr (Np % 4 != 0) {  // nodes Np..4G-1
    for (int i = tid; i < NC * (4 * G - Np); i += NT) s_r[i / (4 * G - Np) * NS + Np + i % (4 * G - Np)] = 0.0;
  }
  lds_barrier();
  const double dt = a.mode == 0 ? *a.dtp : 0.0;
  if (a.gsur_in) {
#pragma unroll
    for (int r = 0; r < RN; r++) {
      const int i = tid + NT * r, e = i / Np, j = i - e * Np;
      double t[3][5];
#pragma unroll
      for (int q = 0; q < 3; q++) {
        const int ms = i < ne * Np ? s_slots[j * 3 + q] : -1;
#pragma unroll
        for (int v = 0; v < 5; v++) t[q][v] = 0.0;
        if (ms >= 0) {
          const int f = ms / Nfp, c = s_conn[e * 4 + f];
          const double *gs = &a.gsur_in[((size_t)conn_nbr(c) * NFF +
                                         s_pslot[(conn_face(c) * 4 + conn_code(c)) * Nfp + ms - f * Nfp]) * 5];
          const f64x2a8 t01 = *reinterpret_cast<const f64x2a8 *>(gs), t23 = *reinterpret_cast<const f64x2a8 *>(gs + 2);
          t[q][0] = t01[0];
          t[q][1] = t01[1];
          t[q][2] = t23[0];
          t[q][3] = t23[1];
          t[q][4] = gs[4];
        }
      }
#pragma unroll
      for (int v = 0; v < 5; v++) UB[r][v] += t[0][v] + t[1][v] + t[2][v];
    }
  }
  // exterior traces of this thread's slots, in flight until phase 2
  double uP[RF][5];
#pragma unroll
  for (int r = 0; r < RF; r++) {
    const int i = min(tid + NT * r, EB * NFF - 1), e = i / NFF, m = i - e * NFF, f = m / Nfp;
    const int c = s_conn[e * 4 + f];
    const size_t pi = (size_t)conn_nbr(c) * Np + s_fmx[(conn_face(c) * 4 + conn_code(c)) * Nfp + m - f * Nfp];
#pragma unroll
    for (int v = 0; v < 5; v++) uP[r][v] = a.u[v * KNp + pi];
  }
#pragma unroll
  for (int r = 0; r < RN; r++) {
    const int i = tid + NT * r;
    if (a.mode == 0) {
#pragma unroll
      for (int v = 0; v < 5; v++) {
        const double kb = R[r][v] + a.b * UB[r][v];
        R[r][v] = dt * kb;
        if (a.a != 0.0 && i < ne * Np) a.kbar[v * KNp + n0 + i] = a.a * kb;
      }
    }
    if (i < EB * Np) {
      const int e = i / Np, o = e * NS + i - e * Np;
#pragma unroll
      for (int v = 0; v < 5; v++) s_r[v * EB * NS + o] = R[r][v];
    }
  }
  if (tid < 4 * EB) s_tau[tid] = 0.25 * (lam_own + lam_nbr) * a.tau_scale;
  lds_barrier();

  // ---- 1. g = A^T rbar ----
  const int kk = lane >> 4, cl = lane & 15;
  auto contract = [&](auto role_, size_t stream, int tile0, int xt, int c0, int q0) {
    constexpr ColRole role = decltype(role_)::value;
    constexpr int T = role.nt, XT = role.xt >= 0 ? 1 : 0, Q = role.nq, NA = role.na();
    constexpr int T1 = T > 0 ? T : 1, Q1 = Q > 0 ? Q : 1;
    if constexpr (NA > 0) {
      const double *ap = afragT + stream + 2 * lane;
      f64x4 acc[T1][CT], acx = {0.0, 0.0, 0.0, 0.0};
      double acq[Q1][CT];
      int col[CT];
      const double *rb[CT];
#pragma unroll
      for (int t = 0; t < CT; t++) {
#pragma unroll
        for (int i = 0; i < T1; i++) acc[i][t] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int i = 0; i < Q1; i++) acq[i][t] = 0.0;
        // local column tile t is tile (c0 + t) % CT; dead columns repeat 0
        col[t] = 16 * (c0 + t < CT ? c0 + t : c0 + t - CT) + cl;
        rb[t] = &s_r[(col[t] < NC ? col[t] : 0) * NS + kk];
      }
      f64x2 A[2][NA];
      auto load = [&](f64x2 (&Ad)[NA], int b) {
#pragma unroll
        for (int x = 0; x < NA; x++) Ad[x] = *reinterpret_cast<const f64x2 *>(ap + ((size_t)b * NA + x) * 128);
      };
      auto block = [&](const f64x2 (&Ad)[NA], int b, int n) {
#pragma unroll
        for (int s = 0; s < 2; s++) {
          if (s >= n) continue;
          double B[CT];
#pragma unroll
          for (int t = 0; t < CT; t++) B[t] = rb[t][4 * (2 * b + s)];
#pragma unroll
          for (int i = 0; i < T; i++)
#pragma unroll
            for (int t = 0; t < CT; t++)
              acc[i][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(Ad[i][s], B[t], acc[i][t], 0, 0, 0);
          if constexpr (XT) acx = __builtin_amdgcn_mfma_f64_16x16x4f64(Ad[T][s], B[0], acx, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < Q; i++)
#pragma unroll
            for (int t = 0; t < CT; t++)
              acq[i][t] = __builtin_amdgcn_mfma_f64_4x4x4f64(Ad[T + XT + i][s], B[t], acq[i][t], 0, 0, 0);
        }
      };
      constexpr int KB = S::KB, LAST = G - 2 * (KB - 1);
      load(A[0], 0);
#pragma unroll 1
      for (int b = 0; b + 2 < KB; b += 2) {
        load(A[1], b + 1);
        __builtin_amdgcn_sched_barrier(0);
        block(A[0], b, 2);
        load(A[0], b + 2);
        __builtin_amdgcn_sched_barrier(0);
        block(A[1], b + 1, 2);
      }
      if constexpr (KB % 2 == 0) {
        load(A[1], KB - 1);
        block(A[0], KB - 2, 2);
        block(A[1], KB - 1, LAST);
      } else {
        block(A[0], KB - 1, LAST);
      }
      auto out = [&](int t, int row0, const f64x4 &c) {
        if (col[t] < NC) {
          f64x2 *d = reinterpret_cast<f64x2 *>(&s_g[col[t] * GS + row0 + 4 * kk]);
          d[0] = f64x2{c[0], c[1]};
          d[1] = f64x2{c[2], c[3]};
        }
      };
#pragma unroll
      for (int t = 0; t < CT; t++) {
#pragma unroll
        for (int i = 0; i < T; i++) out(t, 16 * (tile0 + i), acc[i][t]);
#pragma unroll
        for (int i = 0; i < Q; i++)
          if (col[t] < NC) s_g[col[t] * GS + 4 * (q0 + i) + kk] = acq[i][t];
      }
      if constexpr (XT) out(0, 16 * xt, acx);
    }
  };
  cols_dispatch<S, 0>(w, contract);
  lds_barrier();
#pragma unroll
  for (int r = 0; r < RN; r++) {
    const int i = tid + NT * r;
    if (i < EB * Np) {
      const int e = i / Np, o = e * NS + i - e * Np;
#pragma unroll
      for (int v = 0; v < 5; v++) s_r[v * EB * NS + o] = U[r][v];
    }
  }
  lds_barrier();

  // ---- 2. face-node slots ----
  double rdot = 0.0, tcs[RF];
#pragma unroll
  for (int r = 0; r < RF; r++) {
    tcs[r] = 0.0;
    const int i = tid + NT * r;
    if (i < ne * NFF) {
      const int e = i / NFF, m = i - e * NFF, f = m / Nfp;
      const int o = e * NS + s_fmx[(f * 4 + 3) * Nfp + m - f * Nfp];
      const double *g = &s_geo[e * GEO_STRIDE + 9 + f * 4];
      const double tau = s_tau[e * 4 + f];
      double *gm = &s_g[e * GS + 3 * Np + m];
      double ub[5], h[5], ww[5] = {0, 0, 0, 0, 0};
      double tc = 0.0, fw = 0.0;
#pragma unroll
      for (int v = 0; v < 5; v++) {
        const double um = s_r[v * EB * NS + o], gv = gm[v * EB * GS];
        ub[v] = 0.5 * (um + uP[r][v]);
        h[v] = 0.5 * g[3] * gv;
        tc += gv * (-(ub[v] - um) * g[3]);
      }
      tcs[r] = tc;
      euler_jt(ub, g[0], g[1], g[2], h, a.gamma, ww);
      double pt[5];
#pragma unroll
      for (int v = 0; v < 5; v++) {
        gm[v * EB * GS] = ww[v] + tau * h[v];  // own side
        pt[v] = ww[v] - tau * h[v];            // what the partner's node gets
        fw += ww[v] * ub[v];
      }
      rdot += 2.0 * fw + tau * tc;
      double *gs = &a.gsur[((size_t)e0 * NFF + i) * 5];
      *reinterpret_cast<f64x2a8 *>(gs) = f64x2a8{pt[0], pt[1]};
      *reinterpret_cast<f64x2a8 *>(gs + 2) = f64x2a8{pt[2], pt[3]};
      gs[4] = pt[4];
    }
  }

  // ---- 3. nodes: sum_x J_x(u_j)^T h^x,  h^x_v = sum_d metric[d][x] g[d*Np+j][v] ----
#pragma unroll
  for (int r = 0; r < RN; r++) {
    const int i = tid + NT * r;
    if (i < ne * Np) {
      const int e = i / Np, j = i - e * Np;
      const double *m = &s_geo[e * GEO_STRIDE], *g = &s_g[e * GS + j];
      double wv[5] = {0, 0, 0, 0, 0};
#pragma unroll
      for (int x = 0; x < 3; x++) {
        double h[5];
#pragma unroll
        for (int v = 0; v < 5; v++)
          h[v] = m[x] * g[v * EB * GS] + m[3 + x] * g[v * EB * GS + Np] + m[6 + x] * g[v * EB * GS + 2 * Np];
        euler_jt(U[r], x == 0 ? 1.0 : 0.0, x == 1 ? 1.0 : 0.0, x == 2 ? 1.0 : 0.0, h, a.gamma, wv);
      }
#pragma unroll
      for (int v = 0; v < 5; v++) {
        rdot += wv[v] * U[r][v];
        UB[r][v] += wv[v];
      }
    }
  }
  const bool want_dt = a.mode == 0 && a.dtpart && dt != 0.0;
  if (want_dt) {
    // deterministic block sum of rdot / dt = sum_nodes kb . r: a fixed shuffle
    // tree in each wave, then the wave sums in order
    double s = rdot / dt;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0) red[w] = s;
  }
  lds_barrier();  // own-side terms, wave sums; the state is read
#pragma unroll
  for (int r = 0; r < RF; r++)
    if (tid + NT * r < EB * NFF) s_r[tid + NT * r] = tcs[r];
#pragma unroll
  for (int r = 0; r < RN; r++) {
    const int i = tid + NT * r;
    if (i < ne * Np) {
      const int e = i / Np, j = i - e * Np;
#pragma unroll
      for (int q = 0; q < 3; q++) {
        const int ms = s_slots[j * 3 + q];
        if (ms >= 0) {
#pragma unroll
          for (int v = 0; v < 5; v++) UB[r][v] += s_g[(v * EB + e) * GS + 3 * Np + ms];
        }
      }
#pragma unroll
      for (int v = 0; v < 5; v++) a.ubar[v * KNp + n0 + i] = UB[r][v];
    }
  }
  if (a.mode == 0 && a.dtpart && tid == 0) {
    double t = 0.0;
    if (want_dt)
      for (int q = 0; q < S::NW; q++) t += red[q];
    a.dtpart[batch] = a.first ? t : a.dtpart[batch] + t;
  }
  lds_barrier();
  if (a.taubar && tid < 4 * ne) {
    double t = 0.0;
    for (int j = 0; j < Nfp; j++) t += s_r[tid * Nfp + j];
    const size_t o = (size_t)e0 * 4 + tid;
    a.taubar[o] = a.mode == 1 || a.first ? t : a.taubar[o] + t;
  }
}

template <int N>
struct EulAdjImpl {
  using S = EulAdjShape<N>;
  static void fill(const double *opT, std::vector<double> &out) {
    out.assign(S::stream(S::NW), 0.0);
    eul_adj_arrange<N>(opT, out.data());
  }
  static void launch(hipStream_t stream, const AdjArgs &a, const double *afragT) {
    hipLaunchKernelGGL((adjoint_euler_kernel<N>), dim3(((a.K + S::EB - 1) / S::EB + 7) / 8 * 8), dim3(S::NT), 0, stream, a, afragT);
  }
};

}  // namespace dglm
