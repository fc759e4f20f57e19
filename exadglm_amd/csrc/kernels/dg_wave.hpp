// FP64 Euler stage kernel for large meshes of order 3 and 4 (gfx950): one
// persistent workgroup per CU, every wave on batches of its own.
//
// The contraction and its tiles are those of the packed-column kernel
// (dg_cols.hpp: columns are (variable, element) pairs, rows go in tiles of
// sixteen and units of four).  Here the operator (16 KB at N = 3, 48 KB at N =
// 4) stays in LDS for the whole launch, and a wave takes EB elements at a time
// through all phases alone, in LDS of its own: no workgroup barrier after the
// operator is staged, so the waves of a SIMD drift apart and one's MFMAs run
// beside the others' other phases (which the SIMD's scheduler prefers: 386 ->
// 375 us at N = 4, K = 196,608).  While a batch is contracted its exterior
// traces, later its LSRK registers, and the next batch's node values, geometry
// and connectivity are in flight.
#pragma once
#include "dg_cols.hpp"
#include "wave_ops.h"

namespace dglm {

template <int N, int EB_, int NW_>
struct WaveShape {
  using O = Ord<N>;
  static constexpr int Np = O::Np, Nfp = O::Nfp, NFF = O::NFF;
  static constexpr int G = (Np + 3) / 4, T = G / 4, Q = G % 4;  // tiles of sixteen rows and units of four
  static constexpr int KS = 3 * G + Nfp;                        // k-steps
  static constexpr int SB = (Nfp + 2) / 3, SLAST = Nfp - 3 * (SB - 1);  // surface blocks, k-steps of the last
  static constexpr int NS = 4 * (G | 1);  // element stride of the node arrays (as in ColShape)
  static constexpr int EB = EB_, NW = NW_, NT = 64 * NW;
  static constexpr int NC = 5 * EB, CT = (NC + 15) / 16;
  static constexpr int CS = NC | 1;  // row stride of the surface fluxes (odd; the unused columns of a tile
                                     // read on into the next row)
  static constexpr int AK = 64 * T + 16 * Q;  // operator values of a k-step
  static constexpr int U = 5 * EB * NS;
  static constexpr int VOL = 4 * EB * NS, SUR = (NFF - 1) * CS + 16 * CT, OUT = NC * NS;
  static constexpr int X = ((VOL > SUR ? (VOL > OUT ? VOL : OUT) : (SUR > OUT ? SUR : OUT)) + 1) / 2 * 2;
  static constexpr int GEO = (EB * GEO_STRIDE + 1) / 2 * 2;
  static constexpr int WAVE = U + X + GEO + 4 * EB;  // doubles of a wave (+ 4 EB of int2 and int)
};

// Operator values of order N as the kernel reads them: [k-step][tile rows
// (64), unit rows (16)], k-steps as in cols_arrange.
template <class S>
inline void wave_arrange(const double *opT /*[KD][Np]*/, double *out) {
  for (int ks = 0; ks < S::KS; ks++)
    for (int i = 0; i < S::T + S::Q; i++)
      for (int l = 0; l < (i < S::T ? 64 : 16); l++) {
        const int kk = i < S::T ? l >> 4 : l >> 2;
        const int row = i < S::T ? 16 * i + 4 * (l & 3) + ((l >> 2) & 3) : 16 * S::T + 4 * (i - S::T) + (l & 3);
        int k = -1;
        if (ks < 3 * S::G) {
          const int node = 4 * (ks / 3) + kk;
          if (node < S::Np) k = (ks % 3) * S::Np + node;
        } else {
          k = 3 * S::Np + 4 * (ks - 3 * S::G) + kk;
        }
        *out++ = k >= 0 && row < S::Np ? opT[(size_t)k * S::Np + row] : 0.0;
      }
}

// Global value at a byte offset from a wave-uniform address.  The address stays
// in scalar registers: a use the compiler cannot see through keeps it from
// adding the offset in vector registers, one instruction for every access.
#define DGLM_GLOBAL __attribute__((address_space(1)))
template <class V>
__device__ inline DGLM_GLOBAL V &global_at(const double *base, unsigned off) {
  unsigned long long b = reinterpret_cast<unsigned long long>(base);
  asm("" : "+s"(b));
  return *reinterpret_cast<DGLM_GLOBAL V *>(reinterpret_cast<DGLM_GLOBAL char *>(b) + off);
}

//   MODE 0: LSRK update; MODE 1: write the RHS only.
template <int N, int EB, int NW, int MODE>
__global__ __launch_bounds__(64 * NW, NW / 4) void stage_wave_kernel(StageArgs a, const double *__restrict__ op,
                                                                    const int *__restrict__ order, int nbatch) {
  using S = WaveShape<N, EB, NW>;
  constexpr int Np = S::Np, Nfp = S::Nfp, NFF = S::NFF, G = S::G, NS = S::NS, NT = S::NT, T = S::T, Q = S::Q;
  constexpr int NC = S::NC, CT = S::CT, CS = S::CS, NV = 5;
  constexpr int VW = Np % 2 == 0 ? 2 : 1;
  typedef typename std::conditional<VW == 2, f64x2a8, double>::type vec;
  static_assert(4 * EB <= 64, "one face per lane");

  __shared__ __align__(16) double s_op[S::KS * S::AK];
  __shared__ __align__(16) double s_wave[NW][S::WAVE];
  __shared__ int2 s_cn[NW][4 * EB];
  __shared__ int s_dmw[NW][4 * EB];
  __shared__ int s_fmx[16 * Nfp];
  __shared__ int4 s_fn[EB * NFF];  // a batch's face nodes: face, node of it, own trace in s_u, first flux in s_x

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int K = a.K;
  const size_t KNp = (size_t)K * Np;

  // this wave's batches: every stride-th of its XCD's eighth of the visiting order
  const int xcd = blockIdx.x & 7, first = (int)((long)nbatch * xcd / 8), last = (int)((long)nbatch * (xcd + 1) / 8);
  const int stride = (int)(gridDim.x >> 3) * NW;
  int slot = first + (int)(blockIdx.x >> 3) * NW + w;
  int ids = 0, at = 0;  // the next 64 of them, one a lane; the current one
  auto refill = [&]() {
    const int s = slot + lane * stride;
    ids = -1;
    if (s < last) ids = order ? order[s] : s;
    at = 0;
  };
  refill();
  auto batch_at = [&](int i) { return __builtin_amdgcn_readlane(ids, i); };

  constexpr int RN = (EB * Np / VW + 63) / 64, RF = (EB * NFF + 63) / 64, RG = (EB * GEO_STRIDE + 63) / 64;
  vec un[RN][NV];
  double gx[RG], lam_own = 0.0;
  int cw = 0, dm = -1;
  auto fetch = [&](int b) {
    const int e0 = b * EB, ne = min(EB, K - e0);
    const size_t n0 = (size_t)e0 * Np;
    cw = 0;
    dm = -1;
    if (lane < 4 * ne) {
      cw = a.conn[(size_t)e0 * 4 + lane];
      lam_own = a.maxv[(size_t)e0 * 4 + lane];
      if (a.dmap) dm = a.dmap[(size_t)e0 * 4 + lane];
    }
#pragma unroll
    for (int r = 0; r < RG; r++)
      gx[r] = lane + 64 * r < ne * GEO_STRIDE ? a.geo[(size_t)e0 * GEO_STRIDE + lane + 64 * r] : 0.0;
#pragma unroll
    for (int r = 0; r < RN; r++) {
      const unsigned off = 8u * min((lane + 64 * r) * VW, ne * Np - VW);
#pragma unroll
      for (int v = 0; v < NV; v++) un[r][v] = global_at<vec>(a.u_in + (v * KNp + n0), off);
    }
  };
  // a use of what fetch() loads
  auto arrived = [&]() {
    asm volatile("" : "+v"(cw), "+v"(dm), "+v"(lam_own));
#pragma unroll
    for (int r = 0; r < RG; r++) asm volatile("" : "+v"(gx[r]));
#pragma unroll
    for (int r = 0; r < RN; r++)
#pragma unroll
      for (int v = 0; v < NV; v++) asm volatile("" : "+v"(un[r][v]));
  };
  int b = batch_at(0);
  if (b >= 0) fetch(b);
  for (int i = tid; i < S::KS * S::AK; i += NT) s_op[i] = op[i];
  for (int i = tid; i < 16 * Nfp; i += NT) s_fmx[i] = a.fmx[i];
  for (int i = tid; i < EB * NFF; i += NT) {
    const int e = i / NFF, m = i - e * NFF, f = m / Nfp, j = m - f * Nfp;
    s_fn[i] = make_int4(e * 4 + f, j, e * NS + a.fmx[(f * 4 + 3) * Nfp + j], m * CS + e);
  }

  double *s_u = s_wave[w], *s_x = s_u + S::U, *s_geo = s_x + S::X, *s_tau = s_geo + S::GEO;
  int2 *s_conn = s_cn[w];
  int *s_dm = s_dmw[w];
  if constexpr (Np % 4 != 0)  // nodes Np..4G-1 of the state: zero for good
    for (int i = lane; i < 5 * EB * (4 * G - Np); i += 64)
      s_u[i / (4 * G - Np) * NS + Np + i % (4 * G - Np)] = 0.0;
  double dt = 0.0;
  const bool active = MODE == 1 || begin_stage(a, dt);
  __syncthreads();
  arrived();

  const int kk = lane >> 4, cl = lane & 15;
  int cv[CT], ce[CT];
#pragma unroll
  for (int t = 0; t < CT; t++) {
    const int c = 16 * t + cl;
    cv[t] = c < NC ? c / EB : 0;
    ce[t] = c < NC ? c - cv[t] * EB : 0;
  }
  const double *a_tile = s_op + lane, *a_unit = s_op + 64 * T + 4 * kk + (lane & 3);

  while (b >= 0) {
    const int e0 = b * EB, ne = min(EB, K - e0);
    const size_t n0 = (size_t)e0 * Np;
    if (!active) {  // past tmax: the stage is the identity on u
      for (int v = 0; v < NV; v++)
        for (int i = lane; i < ne * Np; i += 64) a.u_out[v * KNp + n0 + i] = a.u_in[v * KNp + n0 + i];
    } else {
      // ---- 1. the batch's values to LDS; exterior traces on their way ----
      double lam_nbr = 0.0;
      if (lane < 4 * EB) {
        s_conn[lane] = make_int2(conn_nbr(cw), (conn_face(cw) * 4 + conn_code(cw)) * Nfp);
        s_dm[lane] = dm;
        if (lane < 4 * ne) lam_nbr = a.maxv[(size_t)conn_nbr(cw) * 4 + conn_face(cw)];
      }
      const double lam = lam_own;
#pragma unroll
      for (int r = 0; r < RG; r++)
        if (lane + 64 * r < EB * GEO_STRIDE) s_geo[lane + 64 * r] = gx[r];
      wave_lds_sync();
      double uP[RF][NV];
#pragma unroll
      for (int r = 0; r < RF; r++) {
        const int4 fn = s_fn[min(lane + 64 * r, EB * NFF - 1)];
        const int2 c = s_conn[fn.x];
        const size_t pi = (size_t)c.x * Np + s_fmx[c.y + fn.y];
#pragma unroll
        for (int v = 0; v < NV; v++) uP[r][v] = a.u_in[v * KNp + pi];
      }
      if (a.dmap) {  // Dirichlet faces: the prescribed state instead
#pragma unroll
        for (int r = 0; r < RF; r++) {
          const int4 fn = s_fn[min(lane + 64 * r, EB * NFF - 1)];
          const int ds = s_dm[fn.x];
          if (ds >= 0) {
#pragma unroll
            for (int v = 0; v < NV; v++) uP[r][v] = dirichlet_value(a, v, ds, fn.y, Nfp);
          }
        }
      }
      if constexpr (Np % 4 != 0)
        for (int i = lane; i < 4 * EB * (4 * G - Np); i += 64)
          s_x[i / (4 * G - Np) * NS + Np + i % (4 * G - Np)] = 0.0;
#pragma unroll
      for (int r = 0; r < RN; r++) {
        const int i = (lane + 64 * r) * VW;
        if (i < EB * Np) {
          const int e = i / Np, o = e * NS + i - e * Np;
          const double *g = &s_geo[e * GEO_STRIDE];
          vec inv;
          if constexpr (VW == 2)
            inv = vec{rcp_refined(un[r][0][0]), rcp_refined(un[r][0][1])};
          else
            inv = rcp_refined(un[r][0]);
          const vec p = (a.gamma - 1.0) *
                        (un[r][4] - 0.5 * (un[r][1] * un[r][1] + un[r][2] * un[r][2] + un[r][3] * un[r][3]) * inv);
          const vec vx = un[r][1] * inv, vy = un[r][2] * inv, vz = un[r][3] * inv;
#pragma unroll
          for (int d = 0; d < 3; d++)
            *reinterpret_cast<vec *>(&s_x[d * EB * NS + o]) = g[3 * d] * vx + g[3 * d + 1] * vy + g[3 * d + 2] * vz;
          *reinterpret_cast<vec *>(&s_x[3 * EB * NS + o]) = p;
#pragma unroll
          for (int v = 0; v < NV; v++) *reinterpret_cast<vec *>(&s_u[v * EB * NS + o]) = un[r][v];
        }
      }
      wave_lds_sync();
      // the next batch's values
      if (at + 1 < 64) {
        const int nb = batch_at(at + 1);
        if (nb >= 0) fetch(nb);
      }

      __builtin_amdgcn_s_setprio(0);
      f64x4 acc[T > 0 ? T : 1][CT];
      double acq[Q > 0 ? Q : 1][CT];
#pragma unroll
      for (int t = 0; t < CT; t++) {
#pragma unroll
        for (int i = 0; i < T; i++) acc[i][t] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int i = 0; i < Q; i++) acq[i][t] = 0.0;
      }
      double A[2][3][T + Q];
      auto load_op = [&](double (&Ad)[3][T + Q], int ks, int n) {
#pragma unroll
        for (int d = 0; d < 3; d++) {
          if (d >= n) continue;
#pragma unroll
          for (int i = 0; i < T; i++) Ad[d][i] = a_tile[(ks + d) * S::AK + 64 * i];
#pragma unroll
          for (int i = 0; i < Q; i++) Ad[d][T + i] = a_unit[(ks + d) * S::AK + 16 * i];
        }
      };
      auto contract = [&](const double (&Ad)[3][T + Q], const double (&Bd)[3][CT], int n) {
#pragma unroll
        for (int d = 0; d < 3; d++) {
          if (d >= n) continue;
#pragma unroll
          for (int t = 0; t < CT; t++) {
#pragma unroll
            for (int i = 0; i < T; i++)
              acc[i][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(Ad[d][i], Bd[d][t], acc[i][t], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < Q; i++)
              acq[i][t] = __builtin_amdgcn_mfma_f64_4x4x4f64(Ad[d][T + i], Bd[d][t], acq[i][t], 0, 0, 0);
          }
        }
      };

      // ---- 2. volume k-steps ----
      {
        int oe[CT], ou[CT];
        double gv[CT][3], fe[CT];
#pragma unroll
        for (int t = 0; t < CT; t++) {
          oe[t] = ce[t] * NS + kk;
          ou[t] = cv[t] * EB * NS + oe[t];
          const bool mom = cv[t] >= 1 && cv[t] <= 3;
#pragma unroll
          for (int d = 0; d < 3; d++) gv[t][d] = mom ? s_geo[ce[t] * GEO_STRIDE + 3 * d + (mom ? cv[t] - 1 : 0)] : 0.0;
          fe[t] = cv[t] == 4 ? 1.0 : 0.0;
        }
        double R[CT][5], B[3][CT];
        auto read = [&](int g) {
#pragma unroll
          for (int t = 0; t < CT; t++) {
#pragma unroll
            for (int d = 0; d < 4; d++) R[t][d] = s_x[d * EB * NS + oe[t] + 4 * g];
            R[t][4] = s_u[ou[t] + 4 * g];
          }
        };
        auto form = [&]() {
#pragma unroll
          for (int t = 0; t < CT; t++) {
            const double c = R[t][4] + fe[t] * R[t][3];
#pragma unroll
            for (int d = 0; d < 3; d++) B[d][t] = c * R[t][d] + R[t][3] * gv[t][d];
          }
        };
        auto step = [&](int g, int cur) {
          load_op(A[cur ^ 1], 3 * (g + 1), 3);
          form();
          read(g + 1);
          __builtin_amdgcn_sched_barrier(0);
          contract(A[cur], B, 3);
          __builtin_amdgcn_sched_barrier(0);
        };
        load_op(A[0], 0, 3);
        read(0);
        constexpr int G2 = (G - 1) / 2 * 2;
#pragma unroll 1
        for (int g = 0; g < G2; g += 2) {
          step(g, 0);
          step(g + 1, 1);
        }
        if constexpr (G2 < G - 1) step(G2, 0);
        form();
        contract(A[(G - 1) & 1], B, 3);
      }
      if (lane < 4 * EB) s_tau[lane] = 0.25 * (lam + lam_nbr) * a.tau_scale;
      wave_lds_sync();  // the volume arrays are read: their LDS takes the surface fluxes

      // ---- 3. surface fluxes ----
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int r = 0; r < RF; r++) {
        const int i = lane + 64 * r;
        const int4 fn = s_fn[min(i, EB * NFF - 1)];
        const bool dir = a.dmap && s_dm[fn.x] >= 0;
        double uM[5], fl[5];
#pragma unroll
        for (int v = 0; v < 5; v++) uM[v] = s_u[v * EB * NS + fn.z];
        cols_surface_flux5(uM, uP[r], dir, &s_geo[(fn.x >> 2) * GEO_STRIDE + 9 + (fn.x & 3) * 4], s_tau[fn.x], a.flux,
                           a.gamma, fl);
        if (i < EB * NFF) {
#pragma unroll
          for (int v = 0; v < NV; v++) s_x[fn.w + v * EB] = fl[v];
        }
      }
      wave_lds_sync();

      __builtin_amdgcn_s_setprio(0);
      // ---- 4. surface k-steps; the LSRK registers arrive meanwhile ----
      vec kr[RN][NV];
#pragma unroll
      for (int r = 0; r < RN; r++)
#pragma unroll
        for (int v = 0; v < NV; v++) kr[r][v] = vec(0.0);
      if (MODE == 0 && a.rka != 0.0) {
#pragma unroll
        for (int r = 0; r < RN; r++)
#pragma unroll
          for (int v = 0; v < NV; v++)
            kr[r][v] = global_at<vec>(a.k + (v * KNp + n0), 8u * min((lane + 64 * r) * VW, ne * Np - VW));
      }
      {
        constexpr int SB = S::SB;
        double B[2][3][CT];
        auto read = [&](double (&Bd)[3][CT], int s, int n) {
#pragma unroll
          for (int d = 0; d < 3; d++)
            if (d < n)
#pragma unroll
              for (int t = 0; t < CT; t++) Bd[d][t] = s_x[(4 * (3 * s + d) + kk) * CS + 16 * t + cl];
        };
        auto step = [&](int s, int cur, int n) {  // n: k-steps of block s + 1
          load_op(A[cur ^ 1], 3 * (G + s + 1), n);
          read(B[cur ^ 1], s + 1, n);
          __builtin_amdgcn_sched_barrier(0);
          contract(A[cur], B[cur], 3);
          __builtin_amdgcn_sched_barrier(0);
        };
        load_op(A[0], 3 * G, SB > 1 ? 3 : S::SLAST);
        read(B[0], 0, SB > 1 ? 3 : S::SLAST);
        constexpr int M = SB > 1 ? SB - 2 : 0, M2 = M / 2 * 2;  // steps whose next block is full
#pragma unroll 1
        for (int s = 0; s < M2; s += 2) {
          step(s, 0, 3);
          step(s + 1, 1, 3);
        }
        if constexpr (M2 < M) step(M2, 0, 3);
        if constexpr (SB > 1) step(SB - 2, M & 1, S::SLAST);
        contract(A[(SB - 1) & 1], B[(SB - 1) & 1], S::SLAST);
      }
      wave_lds_sync();  // the surface fluxes are read: their LDS takes the contraction
#pragma unroll
      for (int t = 0; t < CT; t++) {
        const int col = 16 * t + cl;
        if (col < NC) {
#pragma unroll
          for (int i = 0; i < T; i++) {
            f64x2 *d = reinterpret_cast<f64x2 *>(&s_x[col * NS + 16 * i + 4 * kk]);
            d[0] = f64x2{acc[i][t][0], acc[i][t][1]};
            d[1] = f64x2{acc[i][t][2], acc[i][t][3]};
          }
#pragma unroll
          for (int i = 0; i < Q; i++) s_x[col * NS + 16 * T + 4 * i + kk] = acq[i][t];
        }
      }
      wave_lds_sync();

      // The next batch's values and the LSRK registers are waited for here,
      // before this batch's stores go out behind them: at the head of the loop
      // the wait would be for the stores as well.
      arrived();
#pragma unroll
      for (int r = 0; r < RN; r++)
#pragma unroll
        for (int v = 0; v < NV; v++) asm volatile("" : "+v"(kr[r][v]));

      // ---- LSRK update, in memory order ----
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int r = 0; r < RN; r++) {
        const int i = (lane + 64 * r) * VW;
        if (i < ne * Np) {
          const int e = i / Np, o = e * NS + i - e * Np;
          vec x[NV];
#pragma unroll
          for (int v = 0; v < NV; v++) x[v] = *reinterpret_cast<const vec *>(&s_x[v * EB * NS + o]);
          if (MODE == 1) {
#pragma unroll
            for (int v = 0; v < NV; v++) global_at<vec>(a.rhs + (v * KNp + n0), 8u * i) = x[v];
          } else {
#pragma unroll
            for (int v = 0; v < NV; v++) x[v] = a.rka * kr[r][v] + dt * x[v];
            if (a.k_out) {
#pragma unroll
              for (int v = 0; v < NV; v++) global_at<vec>(a.k + (v * KNp + n0), 8u * i) = x[v];
            }
#pragma unroll
            for (int v = 0; v < NV; v++)
              global_at<vec>(a.u_out + (v * KNp + n0), 8u * i) =
                  *reinterpret_cast<const vec *>(&s_u[v * EB * NS + o]) + a.rkb * x[v];
          }
        }
      }
      wave_lds_sync();  // the arrays are read: the next batch takes their place
    }

    slot += stride;
    if (++at == 64) {
      refill();
      b = batch_at(0);
      if (b >= 0) fetch(b);
      arrived();
    } else {
      b = batch_at(at);
    }
  }
}

template <int N, int EB, int NW>
struct WaveImpl {
  using S = WaveShape<N, EB, NW>;
  static void fill(const double *opT, std::vector<double> &out) {
    out.assign((size_t)S::KS * S::AK, 0.0);
    wave_arrange<S>(opT, out.data());
  }
  static void launch(int mode, int cus, hipStream_t stream, const StageArgs &a, const double *op, const int *order) {
    const int nbatch = (a.K + EB - 1) / EB;
    const int full = cus >= 8 ? cus / 8 * 8 : 8, need = ((nbatch + NW - 1) / NW + 7) / 8 * 8;
    const dim3 grid(need < full ? need : full), block(S::NT);
    if (mode == 1)
      hipLaunchKernelGGL((stage_wave_kernel<N, EB, NW, 1>), grid, block, 0, stream, a, op, order, nbatch);
    else
      hipLaunchKernelGGL((stage_wave_kernel<N, EB, NW, 0>), grid, block, 0, stream, a, op, order, nbatch);
  }
};

}  // namespace dglm
