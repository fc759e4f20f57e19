// FP64 stage kernel on MFMA with packed columns (gfx950): Euler and advection,
// every order, any mesh size.
//
// The stage contraction  rhs[v][e][i] = sum_k A[i][k] B[k][(v, e)]  (update_rhs,
// dim3/src/cpp/euler_dglm.cpp:254-302; A = [WDr|WDs|WDt|-LIFT]) has as columns
// every (variable, element) pair.  A workgroup takes EB elements, packs their
// EB*NV columns into CT tiles of 16, and goes through
//   1. node values -> LDS, with the primitives the volume fluxes are formed
//      from (pressure and contravariant velocity; for advection the three
//      contravariant fluxes); the gathers of the exterior traces are issued
//      and stay in registers;
//   2. the volume k-steps (three directions of four nodes at a time), whose
//      B-fragments are formed in registers, f_d = c V_d + p g_d,v-1;
//   3. the surface flux of all variables at every face node, once, into the
//      LDS the primitives held;
//   4. the surface k-steps and the LSRK update.
//
// Rows: sixteen at a time on v_mfma_f64_16x16x4f64, what is left of Np in
// units of four on v_mfma_f64_4x4x4f64 with the unit's A in all four blocks,
// which then is a 4 x 16 tile: the same flops per cycle (64.2 against 68.1
// TF/s measured, 256 CUs) and the same B-fragment, so Np rows cost ceil(Np/4)
// units and not 4 ceil(Np/16).  The operator is streamed from the L2 in the
// order each wave uses it.
//
// What the layout is for: every vector memory instruction of a wave takes the
// CU's L1 at least 16 cycles (64 where each lane is on a line of its own), and
// no VALU instruction overlaps an FP64 MFMA.  Hence 16-byte operator loads
// that serve a whole block of k-steps, the new state written through LDS in
// memory order, and as many columns per operator load as the LDS holds.
#pragma once
#include <type_traits>

#include "cols_ops.h"
#include "dg_mfma.hpp"

namespace dglm {

// Rows of one wave: nt tiles from tile0 with every column tile; one column
// tile (c0) of tile xt (-1: none); nq units of four rows from unit q0 with
// every column tile.
struct ColRole {
  int tile0, nt, xt, c0, q0, nq;
  constexpr int na() const { return nt + (xt >= 0 ? 1 : 0) + nq; }
  constexpr bool same(const ColRole &o) const { return nt == o.nt && (xt >= 0) == (o.xt >= 0) && nq == o.nq; }
};

template <int NW>
struct ColRoles {
  ColRole r[NW];
};

// Deal the G row units (G / 4 tiles, G % 4 single units) and CT column tiles
// to NW waves: equal numbers of tiles first; of the tiles left over, whole
// ones while there are more (tile, column) items than waves, then one item to
// a wave; each single unit to the wave with the least work.
template <int G, int CT, int NW>
constexpr ColRoles<NW> cols_roles() {
  ColRoles<NW> R{};
  const int tiles = G / 4, base = tiles / NW, rt = tiles % NW;
  int n = CT == 1 ? rt : 0;
  while ((rt - n) * CT > NW - n) n++;
  int load[NW] = {}, t = 0;
  for (int w = 0; w < NW; w++) {
    R.r[w] = ColRole{t, base + (w < n ? 1 : 0), -1, 0, 4 * tiles, 0};
    t += R.r[w].nt;
    load[w] = 4 * CT * R.r[w].nt;
  }
  for (int i = 0; i < (rt - n) * CT; i++) {
    R.r[n + i].xt = t + i / CT;
    R.r[n + i].c0 = i % CT;
    load[n + i] += 4;
  }
  for (int q = 4 * tiles; q < G; q++) {
    int b = NW - 1;
    for (int w = NW - 1; w >= 0; w--)
      if (load[w] + (R.r[w].nq ? -1 : 0) < load[b] + (R.r[b].nq ? -1 : 0)) b = w;
    // a wave's units are consecutive: the rest of the units of a wave that has some
    if (R.r[b].nq && R.r[b].q0 + R.r[b].nq != q) {
      b = 0;
      for (int w = 0; w < NW; w++)
        if (R.r[w].nq && R.r[w].q0 + R.r[w].nq == q) b = w;
    }
    if (!R.r[b].nq) R.r[b].q0 = q;
    R.r[b].nq++;
    load[b] += CT;
  }
  return R;
}

template <int N, int PHYS, int EB_, int NW_>
struct ColShape {
  using O = Ord<N>;
  static constexpr int NV = NVar<PHYS>::value;
  static constexpr int Np = O::Np, Nfp = O::Nfp, NFF = O::NFF;
  static constexpr int G = (Np + 3) / 4;  // groups of four nodes: blocks of three k-steps, and row units
  static constexpr int KSS = Nfp;         // surface k-steps
  static constexpr int SB = (KSS + 2) / 3, SLAST = KSS - 3 * (SB - 1);  // their blocks; k-steps of the last one
  static constexpr int NBLK = G + SB;
  static constexpr int NS = 4 * (G | 1);  // element stride of the node arrays: an odd number of groups of four, so
                                          // that the 16 columns x 4 nodes of a fragment read fall on the 32 LDS
                                          // bank pairs twice each (nodes Np..4G-1 are zero)
  static constexpr int EB = EB_, NW = NW_, NT = 64 * NW;
  static constexpr int NC = EB * NV, CT = (NC + 15) / 16;
  static constexpr int CS = 16 * CT + 1;                 // row stride of the surface fluxes (odd: a wave writes
                                                         // consecutive face nodes of one column)
  static constexpr int NA = PHYS == PHYS_EULER ? 4 : 3;  // volume arrays: V_0..2 and p, or f_0..2
  static constexpr int VOL = NA * EB * NS, SUR = NFF * CS, OUT = NC * NS;
  static constexpr int X = VOL > SUR ? (VOL > OUT ? VOL : OUT) : (SUR > OUT ? SUR : OUT);
  static constexpr ColRoles<NW> roles = cols_roles<G, CT, NW>();
  // operator stream of wave w: blocks of 3 k-steps, each lane's 3 na values of a
  // block as 16-byte pairs [pair][lane][2] and, where 3 na is odd, [lane] doubles
  static constexpr size_t stream(int w) {
    size_t o = 0;
    for (int i = 0; i < w; i++) o += (size_t)NBLK * 3 * roles.r[i].na() * 64;
    return o;
  }
};

// Host side: the operator streams of all waves (ColShape::stream(NW) doubles).
// Value x of a lane in a block is k-step x / na, row set x % na: its tiles,
// then xt, then its units.  A tile's lane l holds tile row 4 (l % 4) + (l / 4) % 4,
// so that a lane's four results are consecutive rows; a unit's lane l holds
// row l % 4; both column l / 16 of the k-step.
template <class S>
inline void cols_arrange(const double *opT /*[KD][Np]*/, double *out) {
  for (int w = 0; w < S::NW; w++) {
    const ColRole r = S::roles.r[w];
    const int na = r.na();
    double *o = out + S::stream(w);
    for (int b = 0; b < S::NBLK; b++)
      for (int x = 0; x < 3 * na; x++)
        for (int l = 0; l < 64; l++) {
          const int d = x / na, i = x % na, kk = l >> 4;
          int row, k;
          if (i < r.nt)
            row = 16 * (r.tile0 + i) + 4 * (l & 3) + ((l >> 2) & 3);
          else if (i == r.nt && r.xt >= 0)
            row = 16 * r.xt + 4 * (l & 3) + ((l >> 2) & 3);
          else
            row = 4 * (r.q0 + i - r.nt - (r.xt >= 0 ? 1 : 0)) + (l & 3);
          if (b < S::G) {
            const int j = 4 * b + kk;
            k = j < S::Np ? d * S::Np + j : -1;
          } else {
            const int m = 4 * (3 * (b - S::G) + d) + kk;
            k = m < S::NFF ? 3 * S::Np + m : -1;
          }
          const size_t at = x < 3 * na / 2 * 2 ? ((size_t)(x / 2) * 64 + l) * 2 + (x & 1) : (size_t)(3 * na - 1) * 64 + l;
          o[(size_t)b * 3 * na * 64 + at] = row < S::Np && k >= 0 ? opT[(size_t)k * S::Np + row] : 0.0;
        }
  }
}

// Two doubles at an 8-byte aligned address: one 16-byte memory instruction.
typedef double f64x2a8 __attribute__((ext_vector_type(2), aligned(8)));
typedef double f64x2 __attribute__((ext_vector_type(2)));

// Surface flux of the five variables times Fscale at one face node, g = (nx,
// ny, nz, Fscale): LM, whose face state ub is the mean of the traces (on a
// Dirichlet face the prescribed state uP), or Rusanov.
__device__ inline void cols_surface_flux5(const double uM[5], const double uP[5], bool dirichlet, const double *g,
                                          double tau, int flux, double gamma, double fl[5]) {
  auto normal = [&](const double U[5], double &lam, double F[5]) {
    const double inv = rcp_refined(U[0]);
    const double p = (gamma - 1.0) * (U[4] - 0.5 * (U[1] * U[1] + U[2] * U[2] + U[3] * U[3]) * inv);
    const double mn = g[0] * U[1] + g[1] * U[2] + g[2] * U[3], vn = mn * inv;
    lam = flux == 1 ? fabs(vn) + sqrt_refined(fabs(gamma * p * inv)) : 0.0;
    F[0] = mn;
    F[1] = U[1] * vn + g[0] * p;
    F[2] = U[2] * vn + g[1] * p;
    F[3] = U[3] * vn + g[2] * p;
    F[4] = (U[4] + p) * vn;
  };
  double lm;
  if (flux == 1) {
    double fm[5], fp[5], lp;
    normal(uM, lm, fm);
    normal(uP, lp, fp);
    const double lam = fmax(lm, lp);
#pragma unroll
    for (int v = 0; v < 5; v++) fl[v] = (0.5 * (fm[v] + fp[v]) + 0.5 * lam * (uM[v] - uP[v])) * g[3];
  } else {
    double ub[5], nF[5];
#pragma unroll
    for (int v = 0; v < 5; v++) ub[v] = dirichlet ? uP[v] : 0.5 * (uM[v] + uP[v]);
    normal(ub, lm, nF);
#pragma unroll
    for (int v = 0; v < 5; v++) fl[v] = (nF[v] - tau * (ub[v] - uM[v])) * g[3];
  }
}

// Workgroup barrier over LDS: waits for this wave's LDS operations only, so
// that the gathers, the LSRK registers and the stores stay in flight across it
// (nothing in a launch reads global memory that the launch writes).
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Value at a byte offset from a wave-uniform address.
template <class V>
__device__ inline V &at_offset(double *base, unsigned off) {
  return *reinterpret_cast<V *>(reinterpret_cast<char *>(base) + off);
}
template <class V>
__device__ inline V at_offset(const double *base, unsigned off) {
  return *reinterpret_cast<const V *>(reinterpret_cast<const char *>(base) + off);
}

// A lane's operator values of one block.
template <int NA>
struct ColA {
  f64x2 p[3 * NA / 2 > 0 ? 3 * NA / 2 : 1];
  double o;
  __device__ inline void load(const double *__restrict__ b, int lane) {
#pragma unroll
    for (int i = 0; i < 3 * NA / 2; i++) p[i] = *reinterpret_cast<const f64x2 *>(b + 128 * i + 2 * lane);
    if constexpr (NA % 2) o = b[(3 * NA - 1) * 64 + lane];
  }
  __device__ inline double at(int x) const { return NA % 2 && x == 3 * NA - 1 ? o : p[x / 2][x % 2]; }
};

// Calls body with wave w's role: one instantiation for each distinct shape.
template <class S, int I>
struct ColRoleAt {
  static constexpr ColRole value = S::roles.r[I];
};
template <class S, int I>
constexpr bool cols_first() {
  for (int j = 0; j < I; j++)
    if (S::roles.r[j].same(S::roles.r[I])) return false;
  return true;
}
template <class S, int I, class F>
__device__ inline void cols_dispatch(int w, F &body) {
  if constexpr (I < S::NW) {
    if constexpr (cols_first<S, I>()) {
      bool mine = false;
      size_t stream = 0;
      int tile0 = 0, xt = 0, c0 = 0, q0 = 0;
#pragma unroll
      for (int j = I; j < S::NW; j++)
        if (w == j && S::roles.r[j].same(S::roles.r[I])) {
          mine = true;
          stream = S::stream(j);
          tile0 = S::roles.r[j].tile0;
          xt = S::roles.r[j].xt;
          c0 = S::roles.r[j].c0;
          q0 = S::roles.r[j].q0;
        }
      if (mine) {
        body(ColRoleAt<S, I>{}, stream, tile0, xt, c0, q0);
        return;
      }
    }
    cols_dispatch<S, I + 1>(w, body);
  }
}

// Batch of this workgroup (-1: none): workgroup i of XCD x (workgroups go to the
// XCDs round-robin) takes entry i of the x-th eighth of the visiting order, so
// neighbouring batches share an L2.  The grid is nbatch rounded up to a multiple
// of 8.
__device__ inline int xcd_batch(const int *order, int nbatch) {
  const int xcd = blockIdx.x & 7;
  const int slot = (int)((long)nbatch * xcd / 8) + (int)(blockIdx.x >> 3);
  if (slot >= (int)((long)nbatch * (xcd + 1) / 8)) return -1;
  return order ? order[slot] : slot;
}

//   MODE 0: LSRK update; MODE 1: write the RHS only.
template <int N, int PHYS, int EB, int NW, int MODE>
__global__ __launch_bounds__(64 * NW, 2) void stage_cols_kernel(StageArgs a, const double *__restrict__ afrag,
                                                                  const int *__restrict__ order, int nbatch) {
  using S = ColShape<N, PHYS, EB, NW>;
  constexpr int Np = S::Np, Nfp = S::Nfp, NFF = S::NFF, G = S::G, NS = S::NS, NT = S::NT, NV = S::NV;
  constexpr int NC = S::NC, CT = S::CT, CS = S::CS;
  constexpr bool EUL = PHYS == PHYS_EULER;
  constexpr int VW = Np % 2 == 0 ? 2 : 1;  // nodes a thread takes at a time
  typedef typename std::conditional<VW == 2, f64x2a8, double>::type vec;
  static_assert(4 * EB <= NT, "one face per thread");

  __shared__ __align__(16) double s_u[NV * EB * NS];
  // volume arrays [V_0, V_1, V_2(, p)][element][node], then the surface
  // fluxes [face node][column], then the contraction [column][row]
  __shared__ __align__(16) double s_x[S::X];
  __shared__ double s_geo[EB * GEO_STRIDE];
  __shared__ double s_tau[EB * 4];
  __shared__ int2 s_conn[EB * 4];  // exterior element, row of its trace in s_fmx
  __shared__ int s_dm[EB * 4];
  __shared__ int s_fmx[16 * Nfp];

  double dt = 0.0;
  const int batch = xcd_batch(order, nbatch);
  if (batch < 0) {
    if (MODE == 0) begin_stage(a, dt);
    return;
  }
  const int e0 = batch * EB;
  const int K = a.K;
  const size_t KNp = (size_t)K * Np;
  const int ne = min(EB, K - e0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const size_t n0 = (size_t)e0 * Np;

  // ---- 1. stage in: every load before the first wait.  Threads past the end of
  // a short batch repeat its last node; the columns of elements past it are
  // computed and not written ----
  constexpr int RN = (EB * Np / VW + NT - 1) / NT;  // nodes (or pairs) per thread
  constexpr int RF = (EB * NFF + NT - 1) / NT;      // face nodes per thread
  constexpr int RX = (16 * Nfp + NT - 1) / NT, RG = (EB * GEO_STRIDE + NT - 1) / NT;
  double lam_own = 0.0, lam_nbr = 0.0;
  int cw = 0, dm = -1;
  if (tid < 4 * ne) {
    cw = a.conn[(size_t)e0 * 4 + tid];
    if (a.dmap) dm = a.dmap[(size_t)e0 * 4 + tid];
    lam_own = a.maxv[(size_t)e0 * 4 + tid];
  }
  // waves that the last round leaves without a node skip it
  auto some = [&](int r) { return (NT * (r + 1) - 64) * VW < EB * Np || (64 * w + NT * r) * VW < EB * Np; };
  vec un[RN][NV], vl[EUL ? 1 : RN][3];
#pragma unroll
  for (int r = 0; r < RN; r++) {
    const unsigned off = 8u * min((tid + NT * r) * VW, ne * Np - VW);
    if (some(r)) {
#pragma unroll
      for (int v = 0; v < NV; v++) un[r][v] = at_offset<vec>(a.u_in + (v * KNp + n0), off);
      if constexpr (!EUL) {
#pragma unroll
        for (int d = 0; d < 3; d++) vl[r][d] = at_offset<vec>(a.vel + (d * KNp + n0), off);
      }
    }
  }
  int fx[RX];
  double gx[RG];
#pragma unroll
  for (int r = 0; r < RX; r++) fx[r] = tid + NT * r < 16 * Nfp ? a.fmx[tid + NT * r] : 0;
#pragma unroll
  for (int r = 0; r < RG; r++)
    gx[r] = tid + NT * r < ne * GEO_STRIDE ? a.geo[(size_t)e0 * GEO_STRIDE + tid + NT * r] : 0.0;
  if (MODE == 0 && !begin_stage(a, dt)) {
    // Past tmax: the stage is the identity on u (k untouched).
    for (int v = 0; v < NV; v++)
      for (int i = tid; i < ne * Np; i += NT) a.u_out[v * KNp + n0 + i] = a.u_in[v * KNp + n0 + i];
    return;
  }
  if (tid < 4 * EB) {
    s_conn[tid] = make_int2(conn_nbr(cw), (conn_face(cw) * 4 + conn_code(cw)) * Nfp);
    s_dm[tid] = dm;
    if (tid < 4 * ne) lam_nbr = a.maxv[(size_t)conn_nbr(cw) * 4 + conn_face(cw)];
  }
#pragma unroll
  for (int r = 0; r < RX; r++)
    if (tid + NT * r < 16 * Nfp) s_fmx[tid + NT * r] = fx[r];
#pragma unroll
  for (int r = 0; r < RG; r++)
    if (tid + NT * r < EB * GEO_STRIDE) s_geo[tid + NT * r] = gx[r];
  if constexpr (Np % 4 != 0) {  // nodes Np..4G-1
    for (int i = tid; i < EB * (4 * G - Np); i += NT) {
      const int o = i / (4 * G - Np) * NS + Np + i % (4 * G - Np);
#pragma unroll
      for (int v = 0; v < NV; v++) s_u[v * EB * NS + o] = 0.0;
#pragma unroll
      for (int d = 0; d < S::NA; d++) s_x[d * EB * NS + o] = 0.0;
    }
  }
  lds_barrier();

  // exterior traces (and, for advection, the velocity) at this thread's face
  // nodes; in flight until phase 3
  double uP[RF][NV], vf[EUL ? 1 : RF][3];
#pragma unroll
  for (int r = 0; r < RF; r++) {
    const int idx = min(tid + NT * r, EB * NFF - 1), e = idx / NFF, m = idx - e * NFF;
    const int f = m / Nfp, j = m - f * Nfp;
    const int2 c = s_conn[e * 4 + f];
    const int n = s_fmx[c.y + j];
    const size_t pi = (size_t)c.x * Np + n;
#pragma unroll
    for (int v = 0; v < NV; v++) uP[r][v] = a.u_in[v * KNp + pi];
    if constexpr (!EUL) {
      const unsigned o = e < ne ? 8u * (e * Np + s_fmx[(f * 4 + 3) * Nfp + j]) : 0;
#pragma unroll
      for (int d = 0; d < 3; d++) vf[r][d] = at_offset<double>(a.vel + (d * KNp + n0), o);
    }
  }
  if (a.dmap) {  // Dirichlet faces: the prescribed state instead
#pragma unroll
    for (int r = 0; r < RF; r++) {
      const int idx = min(tid + NT * r, EB * NFF - 1), e = idx / NFF, m = idx - e * NFF;
      const int f = m / Nfp, ds = s_dm[e * 4 + f];
      if (ds >= 0) {
#pragma unroll
        for (int v = 0; v < NV; v++) uP[r][v] = dirichlet_value(a, v, ds, m - f * Nfp, Nfp);
      }
    }
  }
  // Pressure and contravariant velocity (fluxes) of this thread's nodes.  In a
  // closure because the compiler then keeps its index arithmetic out of the
  // phases after it: 158 VGPRs for N = 3 [6,1] and 85 for N = 5 [3,4], written
  // inline 160 and 93 (5 to 6% slower stages).
  auto primitives = [&]() {
#pragma unroll
  for (int r = 0; r < RN; r++) {
    const int i = (tid + NT * r) * VW;
    if (i < EB * Np) {
      const int e = i / Np, o = e * NS + i - e * Np;
      const double *g = &s_geo[e * GEO_STRIDE];
      vec V[3];
      if constexpr (EUL) {
        vec inv;
        if constexpr (VW == 2)
          inv = vec{rcp_refined(un[r][0][0]), rcp_refined(un[r][0][1])};
        else
          inv = rcp_refined(un[r][0]);
        const vec p = (a.gamma - 1.0) *
                      (un[r][4] - 0.5 * (un[r][1] * un[r][1] + un[r][2] * un[r][2] + un[r][3] * un[r][3]) * inv);
        const vec vx = un[r][1] * inv, vy = un[r][2] * inv, vz = un[r][3] * inv;
#pragma unroll
        for (int d = 0; d < 3; d++) V[d] = g[3 * d] * vx + g[3 * d + 1] * vy + g[3 * d + 2] * vz;
        *reinterpret_cast<vec *>(&s_x[3 * EB * NS + o]) = p;
      } else {
        const vec F = vl[r][0] * un[r][0], H = vl[r][1] * un[r][0], L = vl[r][2] * un[r][0];
#pragma unroll
        for (int d = 0; d < 3; d++) V[d] = g[3 * d] * F + g[3 * d + 1] * H + g[3 * d + 2] * L;
      }
#pragma unroll
      for (int d = 0; d < 3; d++) *reinterpret_cast<vec *>(&s_x[d * EB * NS + o]) = V[d];
#pragma unroll
      for (int v = 0; v < NV; v++) *reinterpret_cast<vec *>(&s_u[v * EB * NS + o]) = un[r][v];
    }
  }
  if (tid < 4 * EB) s_tau[tid] = 0.25 * (lam_own + lam_nbr) * a.tau_scale;
  lds_barrier();
  };
  primitives();

  const int kk = lane >> 4, cl = lane & 15;
  // Update: thread's nodes as in phase 1, all variables; where half the waves or
  // more would be left without a node, groups of UW waves take the variables in
  // turn (a wave has one variable at a time, so its rows' addresses are scalar)
  constexpr int UW = (EB * Np / VW + 63) / 64, UG = NW / UW > 1 ? NW / UW : 1;
  constexpr int RU = UG > 1 ? 1 : RN, RV = (NV + UG - 1) / UG;
  const int ug = UG > 1 ? w / UW : 0, ut = UG > 1 ? tid - ug * 64 * UW : tid;
  auto mine = [&](int r, int q) { return UG > 1 ? ug < UG && q * UG + ug < NV : some(r); };

  // phases 2..4 of a wave
  auto body = [&](auto role_, size_t stream, int tile0, int xt, int c0, int q0) {
    constexpr ColRole role = decltype(role_)::value;
    constexpr int T = role.nt, XT = role.xt >= 0 ? 1 : 0, Q = role.nq, NA = role.na();
    constexpr int T1 = T > 0 ? T : 1, Q1 = Q > 0 ? Q : 1;
    const double *ap = afrag + stream;
    ColA<NA> A[2];
    f64x4 acc[T1][CT], acx = {0.0, 0.0, 0.0, 0.0};
    double acq[Q1][CT];
#pragma unroll
    for (int t = 0; t < CT; t++) {
#pragma unroll
      for (int i = 0; i < T1; i++) acc[i][t] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int i = 0; i < Q1; i++) acq[i][t] = 0.0;
    }
    // local column tile t is tile (c0 + t) % CT: the extra item's is local 0.
    // This lane's column of it: (variable cv, element ce), dead ones repeat 0
    int ct[CT], cv[CT], ce[CT];
#pragma unroll
    for (int t = 0; t < CT; t++) {
      ct[t] = c0 + t < CT ? c0 + t : c0 + t - CT;
      const int c = 16 * ct[t] + cl;
      cv[t] = c < NC ? c / EB : 0;
      ce[t] = c < NC ? c - cv[t] * EB : 0;
    }
    auto contract = [&](const ColA<NA> &Ad, const double (&Bd)[3][CT], int n) {
#pragma unroll
      for (int d = 0; d < 3; d++) {
        if (d >= n) continue;
#pragma unroll
        for (int i = 0; i < T; i++)
#pragma unroll
          for (int t = 0; t < CT; t++)
            acc[i][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(Ad.at(d * NA + i), Bd[d][t], acc[i][t], 0, 0, 0);
        if constexpr (XT) acx = __builtin_amdgcn_mfma_f64_16x16x4f64(Ad.at(d * NA + T), Bd[d][0], acx, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < Q; i++)
#pragma unroll
          for (int t = 0; t < CT; t++)
            acq[i][t] = __builtin_amdgcn_mfma_f64_4x4x4f64(Ad.at(d * NA + T + XT + i), Bd[d][t], acq[i][t], 0, 0, 0);
      }
    };

    // ---- 2. volume k-steps ----
    // A block's operator values and node values are loaded while the block
    // before it is contracted; the fences keep the compiler from sinking the
    // loads to their uses.
    if constexpr (NA > 0) {
      A[0].load(ap, lane);
      int oe[CT], ou[CT];
      double gv[CT][3], fe[CT];
#pragma unroll
      for (int t = 0; t < CT; t++) {
        oe[t] = ce[t] * NS + kk;
        ou[t] = cv[t] * EB * NS + oe[t];
        if constexpr (EUL) {
          const bool mom = cv[t] >= 1 && cv[t] <= 3;
#pragma unroll
          for (int d = 0; d < 3; d++) gv[t][d] = mom ? s_geo[ce[t] * GEO_STRIDE + 3 * d + (mom ? cv[t] - 1 : 0)] : 0.0;
          fe[t] = cv[t] == 4 ? 1.0 : 0.0;
        }
      }
      constexpr int NR = EUL ? 5 : 3;  // node values of a column
      double R[CT][NR], B[3][CT];
      auto read = [&](int g) {
#pragma unroll
        for (int t = 0; t < CT; t++) {
#pragma unroll
          for (int d = 0; d < 3; d++) R[t][d] = s_x[d * EB * NS + oe[t] + 4 * g];
          if constexpr (EUL) {
            R[t][3] = s_x[3 * EB * NS + oe[t] + 4 * g];
            R[t][4] = s_u[ou[t] + 4 * g];
          }
        }
      };
      auto form = [&]() {
#pragma unroll
        for (int t = 0; t < CT; t++) {
          if constexpr (EUL) {
            const double c = R[t][4] + fe[t] * R[t][3];
#pragma unroll
            for (int d = 0; d < 3; d++) B[d][t] = c * R[t][d] + R[t][3] * gv[t][d];
          } else {
#pragma unroll
            for (int d = 0; d < 3; d++) B[d][t] = R[t][d];
          }
        }
      };
      auto step = [&](int g, int cur) {
        A[cur ^ 1].load(ap + (size_t)(g + 1) * (3 * NA * 64), lane);
        form();
        read(g + 1);
        __builtin_amdgcn_sched_barrier(0);
        contract(A[cur], B, 3);
        __builtin_amdgcn_sched_barrier(0);
      };
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
    lds_barrier();  // the volume arrays are read: their LDS takes the surface fluxes

    // ---- 3. surface fluxes ----
#pragma unroll
    for (int r = 0; r < RF; r++) {
      const int i = tid + NT * r, idx = min(i, EB * NFF - 1), e = idx / NFF, m = idx - e * NFF;
      const int f = m / Nfp, j = m - f * Nfp;
      const int o = e * NS + s_fmx[(f * 4 + 3) * Nfp + j];
      const double *g = &s_geo[e * GEO_STRIDE + 9 + f * 4];
      const double tau = s_tau[e * 4 + f];
      const bool dir = a.dmap && s_dm[e * 4 + f] >= 0;
      double fl[NV];
      if constexpr (EUL) {
        double uM[5];
#pragma unroll
        for (int v = 0; v < 5; v++) uM[v] = s_u[v * EB * NS + o];
        cols_surface_flux5(uM, uP[r], dir, g, tau, a.flux, a.gamma, fl);
      } else {
        const double uM = s_u[o], up = uP[r][0];
        const double ub = dir && a.flux != 1 ? up : 0.5 * (uM + up);
        if (a.flux == 1) {
          const double vn = g[0] * vf[r][0] + g[1] * vf[r][1] + g[2] * vf[r][2];
          fl[0] = (vn * ub + 0.5 * fabs(vn) * (uM - up)) * g[3];
        } else {
          const double nF = g[0] * (vf[r][0] * ub) + g[1] * (vf[r][1] * ub) + g[2] * (vf[r][2] * ub);
          fl[0] = (nF - tau * (ub - uM)) * g[3];
        }
      }
      if (i < EB * NFF) {
#pragma unroll
        for (int v = 0; v < NV; v++) s_x[m * CS + v * EB + e] = fl[v];
      }
    }
    lds_barrier();

    // ---- 4. surface k-steps; the LSRK registers arrive meanwhile ----
    vec kr[RU][RV];
    if (MODE == 0) {
#pragma unroll
      for (int r = 0; r < RU; r++)
#pragma unroll
        for (int q = 0; q < RV; q++) {
          kr[r][q] = vec(0.0);
          if (a.rka != 0.0 && mine(r, q))
            kr[r][q] = at_offset<vec>(a.k + ((q * UG + ug) * KNp + n0), 8u * min((ut + NT * r) * VW, ne * Np - VW));
        }
    }
    if constexpr (NA > 0) {
      constexpr int SB = S::SB;
      const double *as = ap + (size_t)G * (3 * NA * 64);
      double B[2][3][CT];
      auto read = [&](double (&Bd)[3][CT], int s, int n) {
#pragma unroll
        for (int d = 0; d < 3; d++)
          if (d < n)
#pragma unroll
            for (int t = 0; t < CT; t++) Bd[d][t] = s_x[(4 * (3 * s + d) + kk) * CS + 16 * ct[t] + cl];
      };
      auto step = [&](int s, int cur, int n) {  // n: k-steps of block s + 1
        A[cur ^ 1].load(as + (size_t)(s + 1) * (3 * NA * 64), lane);
        read(B[cur ^ 1], s + 1, n);
        __builtin_amdgcn_sched_barrier(0);
        contract(A[cur], B[cur], 3);
        __builtin_amdgcn_sched_barrier(0);
      };
      A[0].load(as, lane);
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
    lds_barrier();  // the surface fluxes are read: their LDS takes the contraction
    auto out = [&](int t, int row0, const f64x4 &c) {
      const int col = 16 * ct[t] + cl;
      if (col < NC) {
        f64x2 *d = reinterpret_cast<f64x2 *>(&s_x[col * NS + row0 + 4 * kk]);
        d[0] = f64x2{c[0], c[1]};
        d[1] = f64x2{c[2], c[3]};
      }
    };
#pragma unroll
    for (int t = 0; t < CT; t++) {
#pragma unroll
      for (int i = 0; i < T; i++) out(t, 16 * (tile0 + i), acc[i][t]);
#pragma unroll
      for (int i = 0; i < Q; i++) {
        const int col = 16 * ct[t] + cl;
        if (col < NC) s_x[col * NS + 4 * (q0 + i) + kk] = acq[i][t];
      }
    }
    if constexpr (XT) out(0, 16 * xt, acx);
    lds_barrier();

    // ---- LSRK update, in memory order ----
#pragma unroll
    for (int r = 0; r < RU; r++) {
      const int i = (ut + NT * r) * VW;
      if (i < ne * Np) {
        const int e = i / Np, o = e * NS + i - e * Np;
#pragma unroll
        for (int q = 0; q < RV; q++) {
          if (UG > 1 && !mine(r, q)) continue;
          const int v = q * UG + ug;
          const size_t row = v * KNp + n0;
          const vec rhs = *reinterpret_cast<const vec *>(&s_x[v * EB * NS + o]);
          if (MODE == 1) {
            at_offset<vec>(a.rhs + row, 8u * i) = rhs;
          } else {
            const vec kn = a.rka * kr[r][q] + dt * rhs;
            if (a.k_out) at_offset<vec>(a.k + row, 8u * i) = kn;
            vec &u = *reinterpret_cast<vec *>(&s_u[v * EB * NS + o]);
            const vec u1 = u + a.rkb * kn;
            at_offset<vec>(a.u_out + row, 8u * i) = u1;
            if (EUL && a.lam_out) u = u1;
          }
        }
      }
    }
  };

  cols_dispatch<S, 0>(w, body);

  // ---- wave speeds of the new state, in a step's last stage: the state is at
  // hand in LDS, a wave-speed kernel would read it all again ----
  if constexpr (EUL && MODE == 0) {
    if (!a.lam_out) return;
    lds_barrier();
    for (int i = tid; i < ne * Np; i += NT) {
      const int e = i / Np, o = e * NS + i - e * Np;
      node_speeds(s_u[o], s_u[EB * NS + o], s_u[2 * EB * NS + o], s_u[3 * EB * NS + o], s_u[4 * EB * NS + o], a.gamma,
                  s_x[o], s_x[EB * NS + o]);
    }
    lds_barrier();
    // four threads per face
    double lfs = 0.0;
    for (int f0 = 0; f0 < 4 * ne; f0 += NT / 4) {
      const int fi = f0 + (tid >> 2), e = fi >> 2, f = fi & 3;
      double mv2 = 0.0, mc2 = 0.0, sum = 0.0;
      if (fi < 4 * ne) {
        for (int j = tid & 3; j < Nfp; j += 4) {
          const int o = e * NS + s_fmx[(f * 4 + 3) * Nfp + j];
          const double v2 = s_x[o], c2 = s_x[EB * NS + o];
          mv2 = v2 > mv2 ? v2 : mv2;
          mc2 = c2 > mc2 ? c2 : mc2;
          sum += v2 + c2;
        }
      }
      // (a state that is not a number reaches dt as an infinite wave speed: the
      // maxima pass over a NaN, the sum of the squares does not)
      if (sum != sum) lfs = INFINITY;
#pragma unroll
      for (int q = 1; q <= 2; q <<= 1) {
        mv2 = fmax(mv2, __shfl_xor(mv2, q, 64));
        mc2 = fmax(mc2, __shfl_xor(mc2, q, 64));
      }
      if (fi < 4 * ne && (tid & 3) == 0) {
        const double lam = sqrt(mv2) + sqrt(mc2);
        a.lam_out[(size_t)e0 * 4 + fi] = lam;
        lfs = fmax(lfs, lam * s_geo[e * GEO_STRIDE + 9 + f * 4 + 3]);
      }
    }
    raise_maxfs(a.clk_out, lfs, s_tau);
  }
}

// Elements per workgroup and waves: a small-mesh and a large-mesh configuration
// of each order.  Measured in us per stage, launch included (uniform vortex
// meshes, Rusanov flux; [EB, waves]):
//   Euler, K =            1296   6000   10368  13182  20250  82944
//   N = 1   [6,2]          7.2    8.2    9.7   10.5   13.5   33.8
//           [16,1]         8.4    9.0    9.6   10.4   12.1   25.5
//   N = 2   [3,2]          8.1   11.3   15.5   18.0   23.9   78.7
//           [6,1]          9.3   11.1   14.1   16.5   20.8   56.2
//   N = 3   [3,2]          8.9   13.9   20.3   22.7   31.4    105
//           [6,1]         11.5   14.5   19.6   23.3   33.7   93.9
//   N = 4   [3,4]         11.9   24.8   36.1   45.1   66.2    206
//           [6,2]         14.3   23.1   39.0   45.0   61.7    207
//   N = 5   [3,4]         14.4   37.1   56.4   69.3    103    401
//           [6,2]         19.8   35.2   62.2   69.7   98.7    359
//   N = 6   [6,4]         21.5   59.7   93.7    116    168    617
//           [9,4]         26.2   62.6    101    118    166    617
//   advection N = 5 [16,8] 10.5  14.5   21.5          35.4    117
//                   [16,4] 10.9  14.9   20.5          32.7    106
// Few elements per workgroup while the mesh does not fill the GPU (a stage is
// then one pass of the chain load, gather, flux, contraction, store), many to a
// wave once it does: each operator load then serves more columns, and fewer
// waves meet at a barrier (Euler N = 3, K = 82,944: [9,2] 107, [6,1] 99; N = 5:
// [12,4] 371, [6,2] 356, in one run).  Nine or more elements in fewer waves
// leave two waves a SIMD (N = 5 [9,2] 444).  Above N = 7 the LDS holds three
// elements beside a second workgroup.  For advection a column tile is 16
// elements, and 32 were slower (N = 4: 84 against 63 us at K = 82,944).
struct ColConfig {
  int eb, nw;
};
constexpr ColConfig cols_config(int N, int phys, bool small) {
  if (phys == PHYS_ADV) return {16, N <= 2 ? N : (N <= 4 || (N <= 6 && !small) ? 4 : 8)};
  switch (N) {
    case 1:
      return small ? ColConfig{6, 2} : ColConfig{16, 1};
    case 2:
    case 3:
      return small ? ColConfig{3, 2} : ColConfig{6, 1};
    case 4:
    case 5:
      return small ? ColConfig{3, 4} : ColConfig{6, 2};
    case 6:
      return small ? ColConfig{6, 4} : ColConfig{9, 4};
    case 7:
      return {6, 4};
    default:
      return {3, 4};
  }
}
// Whether a mesh of K elements takes the small-mesh configuration: about where
// the lines above cross, in small batches.
constexpr bool cols_small(int N, int phys, int K) {
  const int nb = (K + cols_config(N, phys, true).eb - 1) / cols_config(N, phys, true).eb;
  return nb <= (phys == PHYS_ADV ? 512 : N >= 3 && N <= 5 ? 6144 : 2048);
}

template <int N, int PHYS, bool SMALL>
struct ColImpl {
  static constexpr ColConfig C = cols_config(N, PHYS, SMALL);
  using S = ColShape<N, PHYS, C.eb, C.nw>;
  static void fill(const double *opT, std::vector<double> &out) {
    out.assign(S::stream(S::NW), 0.0);
    cols_arrange<S>(opT, out.data());
  }
  static void launch(int mode, hipStream_t stream, const StageArgs &a, const double *afrag, const int *order) {
    const int nbatch = (a.K + C.eb - 1) / C.eb;
    const dim3 grid((nbatch + 7) / 8 * 8), block(S::NT);
    if (mode == 1)
      hipLaunchKernelGGL((stage_cols_kernel<N, PHYS, C.eb, C.nw, 1>), grid, block, 0, stream, a, afrag, order, nbatch);
    else
      hipLaunchKernelGGL((stage_cols_kernel<N, PHYS, C.eb, C.nw, 0>), grid, block, 0, stream, a, afrag, order, nbatch);
  }
};

// The entry points of one translation unit's orders.
template <int N, int PHYS>
inline ColOps cols_ops(int K) {
  if (cols_small(N, PHYS, K)) return {cols_config(N, PHYS, true).eb, ColImpl<N, PHYS, true>::fill, ColImpl<N, PHYS, true>::launch};
  return {cols_config(N, PHYS, false).eb, ColImpl<N, PHYS, false>::fill, ColImpl<N, PHYS, false>::launch};
}

}  // namespace dglm
