// Pass A of the discrete advection adjoint on FP64 MFMA (gfx950), every order.
//
// Advection is linear: the reverse stage needs no forward state (the trace
// averages enter only taubar, which only the RHS adjoint reports).  Per
// workgroup of EB elements (the MFMA columns):
//   0. node values in memory order: ubar takes the partner-side face terms the
//      pass A before it left (when given: that pass's pass B), kbar is updated
//      and rbar = dt (kbar + b ubar) goes to LDS beside the velocity;
//   1. g = A^T rbar in 16-row tiles: a wave forms the three volume rows of its
//      16 nodes together, so w_j = sum_x vel_x sum_d metric[d][x] g_d(j) closes
//      in registers; the surface rows go to LDS;
//   2. face-node slots in memory order: own-side term Fscale (vn + tau)/2 g (to
//      LDS), partner-side term Fscale (vn - tau)/2 g (stored for the next pass);
//   3. ubar += w + the node's own-side terms, in memory order.
// N = 5, K = 48,000 moves 226 MB a pass (ubar, kbar in and out, velocity, face
// terms out and in) in 92 us, 2.5 TB/s: half of a copy's rate (phase 0 begins with
// the gather of the partner terms, which depends on connectivity and slot).
#pragma once
#include "adjoint_ops.h"
#include "dg_cols.hpp"

namespace dglm {

template <int N>
struct AdvAdjShape {
  using O = Ord<N>;
  static constexpr int Np = O::Np, Nfp = O::Nfp, NFF = O::NFF;
  static constexpr int G = (Np + 3) / 4, NS = 4 * (G | 1);  // k-steps over the nodes; element stride (dg_cols.hpp)
  static constexpr int GS = NFF + 1;                        // element stride of the surface rows
  static constexpr int EB = N <= 8 ? 16 : 8;                // (above N = 8 sixteen elements exceed the LDS)
  static constexpr int NW = N <= 2 ? 2 : (N <= 6 ? 4 : 8), NT = 64 * NW;
  static constexpr int TN = (Np + 15) / 16, TF = (NFF + 15) / 16;  // node tiles (three rows of A^T a node), surface tiles
  static constexpr int KB = (G + 1) / 2;                           // blocks of two k-steps
  // operator streams: per node tile 3 values of a k-step, per surface tile 1; a
  // lane's values of a block as 16-byte pairs [pair][lane][2]
  static constexpr size_t tile_n = (size_t)KB * 6 * 64, tile_f = (size_t)KB * 2 * 64;
  static constexpr size_t size = TN * tile_n + TF * tile_f;
  static constexpr int R = EB * NS > EB * NFF ? EB * NS : EB * NFF;  // rbar, then the taubar partials
};

// Tile row of lane l (so that a lane's four results are consecutive rows).
__host__ __device__ constexpr int tile_row(int l) { return 4 * (l & 3) + ((l >> 2) & 3); }

template <int N>
inline void adv_adj_arrange(const double *opT, double *out) {
  using S = AdvAdjShape<N>;
  auto at = [&](int k, int i) { return i < S::Np && k >= 0 ? opT[(size_t)k * S::Np + i] : 0.0; };
  for (int b = 0; b < S::KB; b++)
    for (int l = 0; l < 64; l++)
      for (int s = 0; s < 2; s++) {
        const int i = 4 * (2 * b + s) + (l >> 4);
        for (int t = 0; t < S::TN; t++)
          for (int d = 0; d < 3; d++) {
            const int j = 16 * t + tile_row(l), x = 3 * s + d;
            out[t * S::tile_n + ((size_t)b * 3 + x / 2) * 128 + 2 * l + (x & 1)] = at(j < S::Np ? d * S::Np + j : -1, i);
          }
        for (int t = 0; t < S::TF; t++) {
          const int m = 16 * t + tile_row(l);
          out[S::TN * S::tile_n + t * S::tile_f + (size_t)b * 128 + 2 * l + s] =
              at(m < S::NFF ? 3 * S::Np + m : -1, i);
        }
      }
}

template <int N>
__global__ __launch_bounds__(AdvAdjShape<N>::NT, 2) void adjoint_adv_kernel(AdjArgs a,
                                                                           const double *__restrict__ afragT) {
  using S = AdvAdjShape<N>;
  constexpr int Np = S::Np, Nfp = S::Nfp, NFF = S::NFF, G = S::G, NS = S::NS, GS = S::GS, EB = S::EB, NT = S::NT;
  constexpr int VW = Np % 2 == 0 ? 2 : 1;
  typedef typename std::conditional<VW == 2, f64x2a8, double>::type vec;
  __shared__ __align__(16) double s_r[S::R];           // rbar [element][node]; then taubar partials [element][slot]
  __shared__ __align__(16) double s_vel[3][EB * NS];
  __shared__ __align__(16) double s_w[EB * NS];        // volume part
  __shared__ double s_g[EB * GS];                      // surface rows of A^T rbar, then the own-side terms
  __shared__ double s_geo[EB * GEO_STRIDE];
  __shared__ double s_tau[EB * 4];
  __shared__ int s_conn[EB * 4];
  __shared__ int s_fmx[16 * Nfp], s_pslot[16 * Nfp];
  __shared__ int s_slots[Np * 3];

  const int K = a.K;
  const size_t KNp = (size_t)K * Np;
  const int batch = xcd_batch(a.order, (K + EB - 1) / EB);
  if (batch < 0) return;
  const int e0 = batch * EB;
  const int ne = min(EB, K - e0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const size_t n0 = (size_t)e0 * Np;

  // ---- 0. stage in ----
  constexpr int RN = (EB * Np / VW + NT - 1) / NT;
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
  vec ub[RN], kb[RN], vl[RN][3];
#pragma unroll
  for (int r = 0; r < RN; r++) {
    const int i = (tid + NT * r) * VW;
    ub[r] = kb[r] = vl[r][0] = vl[r][1] = vl[r][2] = vec(0.0);
    if (i < ne * Np) {
      if (a.mode == 0) {
        ub[r] = *reinterpret_cast<const vec *>(a.ubar + n0 + i);
        if (!a.first) kb[r] = *reinterpret_cast<const vec *>(a.kbar + n0 + i);
      } else {
        kb[r] = *reinterpret_cast<const vec *>(a.rbar + n0 + i);
      }
#pragma unroll
      for (int d = 0; d < 3; d++) vl[r][d] = *reinterpret_cast<const vec *>(a.vel + d * KNp + n0 + i);
    }
  }
  for (int i = tid; i < 16 * Nfp; i += NT) {
    s_fmx[i] = a.fmx[i];
    s_pslot[i] = a.pslot[i];
  }
  for (int i = tid; i < Np * 3; i += NT) s_slots[i] = a.node_slots[i];
  for (int i = tid; i < EB * GEO_STRIDE; i += NT) s_geo[i] = i < ne * GEO_STRIDE ? a.geo[(size_t)e0 * GEO_STRIDE + i] : 0.0;
  if constexpr (Np % 4 != 0) {  // nodes Np..4G-1
    for (int i = tid; i < EB * (4 * G - Np); i += NT) s_r[i / (4 * G - Np) * NS + Np + i % (4 * G - Np)] = 0.0;
  }
  lds_barrier();
  const double dt = a.mode == 0 ? *a.dtp : 0.0;
  double pend[RN][VW][3];
  if (a.gsur_in) {
#pragma unroll
    for (int r = 0; r < RN; r++)
#pragma unroll
      for (int x = 0; x < VW; x++) {
        const int i = (tid + NT * r) * VW + x, e = i / Np, j = i - e * Np;
#pragma unroll
        for (int q = 0; q < 3; q++) {
          pend[r][x][q] = 0.0;
          const int ms = i < ne * Np ? s_slots[j * 3 + q] : -1;
          if (ms >= 0) {
            const int f = ms / Nfp, c = s_conn[e * 4 + f];
            pend[r][x][q] = a.gsur_in[(size_t)conn_nbr(c) * NFF +
                                      s_pslot[(conn_face(c) * 4 + conn_code(c)) * Nfp + ms - f * Nfp]];
          }
        }
      }
  }
#pragma unroll
  for (int r = 0; r < RN; r++) {
    const int i = (tid + NT * r) * VW;
    if (a.gsur_in) {
      if constexpr (VW == 2) {
        ub[r][0] += pend[r][0][0] + pend[r][0][1] + pend[r][0][2];
        ub[r][1] += pend[r][1][0] + pend[r][1][1] + pend[r][1][2];
      } else {
        ub[r] += pend[r][0][0] + pend[r][0][1] + pend[r][0][2];
      }
    }
    vec rb = kb[r];
    if (a.mode == 0) {
      const vec kn = kb[r] + a.b * ub[r];
      rb = dt * kn;
      if (a.a != 0.0 && i < ne * Np) *reinterpret_cast<vec *>(a.kbar + n0 + i) = a.a * kn;
    }
    if (i < EB * Np) {
      const int e = i / Np, o = e * NS + i - e * Np;
      *reinterpret_cast<vec *>(&s_r[o]) = rb;
#pragma unroll
      for (int d = 0; d < 3; d++) *reinterpret_cast<vec *>(&s_vel[d][o]) = vl[r][d];
    }
  }
  if (tid < 4 * EB) s_tau[tid] = 0.25 * (lam_own + lam_nbr) * a.tau_scale;
  lds_barrier();

  // ---- 1. g = A^T rbar ----
  const int kk = lane >> 4, cl = lane & 15;
  const int ec = cl < EB ? cl : 0;  // this lane's column (EB < 16: the rest repeats column 0)
  const double *rb = &s_r[ec * NS + kk];
  for (int t = w; t < S::TN; t += S::NW) {
    const double *ap = afragT + t * S::tile_n + 2 * lane;
    f64x4 acc[3] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
    auto block = [&](int b, int n) {
      f64x2 A[3];
#pragma unroll
      for (int p = 0; p < 3; p++) A[p] = *reinterpret_cast<const f64x2 *>(ap + ((size_t)b * 3 + p) * 128);
#pragma unroll
      for (int s = 0; s < 2; s++) {
        if (s >= n) continue;
        const double B = rb[4 * (2 * b + s)];
#pragma unroll
        for (int d = 0; d < 3; d++)
          acc[d] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[(3 * s + d) / 2][(3 * s + d) % 2], B, acc[d], 0, 0, 0);
      }
    };
#pragma unroll 4
    for (int b = 0; b < G / 2; b++) block(b, 2);
    if constexpr (G % 2) block(G / 2, 1);
    if (cl < EB) {
      const double *m = &s_geo[ec * GEO_STRIDE];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int j = 16 * t + 4 * kk + r;
        if (j < Np) {
          double wv = 0.0;
#pragma unroll
          for (int x = 0; x < 3; x++)
            wv += s_vel[x][ec * NS + j] * (m[x] * acc[0][r] + m[3 + x] * acc[1][r] + m[6 + x] * acc[2][r]);
          s_w[ec * NS + j] = wv;
        }
      }
    }
  }
  // (dealt from the last wave: the first ones may have one node tile more)
  for (int t = S::NW - 1 - w; t < S::TF; t += S::NW) {
    const double *ap = afragT + S::TN * S::tile_n + t * S::tile_f + 2 * lane;
    f64x4 acc = {0.0, 0.0, 0.0, 0.0};
    auto block = [&](int b, int n) {
      const f64x2 A = *reinterpret_cast<const f64x2 *>(ap + (size_t)b * 128);
#pragma unroll
      for (int s = 0; s < 2; s++)
        if (s < n) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(A[s], rb[4 * (2 * b + s)], acc, 0, 0, 0);
    };
#pragma unroll 8
    for (int b = 0; b < G / 2; b++) block(b, 2);
    if constexpr (G % 2) block(G / 2, 1);
    if (cl < EB) {
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int m = 16 * t + 4 * kk + r;
        if (m < NFF) s_g[ec * GS + m] = acc[r];
      }
    }
  }
  lds_barrier();

  // ---- 2. face-node slots ----
  for (int i = tid; i < ne * NFF; i += NT) {
    const int e = i / NFF, m = i - e * NFF, f = m / Nfp, j = m - f * Nfp;
    const int o = s_fmx[(f * 4 + 3) * Nfp + j];
    const double *g = &s_geo[e * GEO_STRIDE + 9 + f * 4];
    const double tau = s_tau[e * 4 + f], gg = s_g[e * GS + m];
    const double vn = g[0] * s_vel[0][e * NS + o] + g[1] * s_vel[1][e * NS + o] + g[2] * s_vel[2][e * NS + o];
    s_g[e * GS + m] = g[3] * (0.5 * vn + 0.5 * tau) * gg;
    a.gsur[(size_t)e0 * NFF + i] = g[3] * (0.5 * vn - 0.5 * tau) * gg;
    if (a.taubar) {
      const int c = s_conn[e * 4 + f];
      const double um = a.u[n0 + e * Np + o];
      const double up = a.u[(size_t)conn_nbr(c) * Np + s_fmx[(conn_face(c) * 4 + conn_code(c)) * Nfp + j]];
      s_r[i] = gg * (-(0.5 * (um + up) - um) * g[3]);
    }
  }
  lds_barrier();
  if (a.taubar && tid < 4 * ne) {
    const int e = tid >> 2, f = tid & 3;
    double t = 0.0;
    for (int j = 0; j < Nfp; j++) t += s_r[e * NFF + f * Nfp + j];
    const size_t o = (size_t)e0 * 4 + tid;
    a.taubar[o] = a.mode == 1 || a.first ? t : a.taubar[o] + t;
  }

  // ---- 3. ubar ----
#pragma unroll
  for (int r = 0; r < RN; r++) {
    const int i = (tid + NT * r) * VW;
    if (i < ne * Np) {
      vec out;
#pragma unroll
      for (int x = 0; x < VW; x++) {
        const int e = (i + x) / Np, j = i + x - e * Np;
        double v = s_w[e * NS + j];
        if constexpr (VW == 2) v += ub[r][x];
        else v += ub[r];
#pragma unroll
        for (int q = 0; q < 3; q++) {
          const int ms = s_slots[j * 3 + q];
          if (ms >= 0) v += s_g[e * GS + ms];
        }
        if constexpr (VW == 2) out[x] = v;
        else out = v;
      }
      *reinterpret_cast<vec *>(a.ubar + n0 + i) = out;
    }
  }
}

template <int N>
struct AdvAdjImpl {
  using S = AdvAdjShape<N>;
  static void fill(const double *opT, std::vector<double> &out) {
    out.assign(S::size, 0.0);
    adv_adj_arrange<N>(opT, out.data());
  }
  static void launch(hipStream_t stream, const AdjArgs &a, const double *afragT) {
    hipLaunchKernelGGL((adjoint_adv_kernel<N>), dim3(((a.K + S::EB - 1) / S::EB + 7) / 8 * 8), dim3(S::NT), 0, stream, a, afragT);
  }
};

}  // namespace dglm
