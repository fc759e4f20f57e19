// Wave speeds of a state (calc_maxv), in a kernel of their own: before a step
// whose predecessor did not leave them, and for the adjoint's recording.
#pragma once
#include "dg_fp64.hpp"

namespace dglm {

// --------------------------------------------------------------------------
// LDS-staged wave speed: a block converts the node values of WE elements to
// |v|^2 and |c|^2 with coalesced loads, then one thread per face takes the
// maxima over the face nodes (calc_maxv, euler_dglm.cpp:6-50,
// advec_dglm.cpp:6-35).  The largest lambda*Fscale goes to the clock;
// without one the block keeps its own with the face index (smallest index on ties),
// for the adjoint's recording.
// --------------------------------------------------------------------------
__host__ __device__ constexpr int wavespeed_elems(int Np) { return Np <= 35 ? 64 : (Np <= 84 ? 32 : 16); }

template <int N, int PHYS>
__global__ __launch_bounds__(256) void wavespeed_lds_kernel(int K, const double *__restrict__ u,
                                                            const double *__restrict__ vel,
                                                            const double *__restrict__ geo,
                                                            const int *__restrict__ fmx, double *__restrict__ maxv,
                                                            DevClock *clk,
                                                            double *__restrict__ partial,
                                                            int *__restrict__ partial_idx, double gamma) {
  using O = Ord<N>;
  constexpr int Np = O::Np, Nfp = O::Nfp, WE = wavespeed_elems(O::Np);
  __shared__ double s_v2[WE * Np];
  __shared__ double s_c2[PHYS == PHYS_EULER ? WE * Np : 1];
  __shared__ int s_fm[4 * Nfp];
  __shared__ double red[256];
  __shared__ int red_i[256];
  const int tid = threadIdx.x;
  const size_t KNp = (size_t)K * Np;
  const int e0 = blockIdx.x * WE;
  const int ne = min(WE, K - e0);
  for (int i = tid; i < 4 * Nfp; i += 256) s_fm[i] = fmx[((i / Nfp) * 4 + 3) * Nfp + i % Nfp];
  for (int i = tid; i < ne * Np; i += 256) {
    const size_t idx = (size_t)e0 * Np + i;
    if (PHYS == PHYS_EULER) {
      node_speeds(u[idx], u[KNp + idx], u[2 * KNp + idx], u[3 * KNp + idx], u[4 * KNp + idx], gamma, s_v2[i], s_c2[i]);
    } else {
      const double vx = vel[idx], vy = vel[KNp + idx], vz = vel[2 * KNp + idx];
      s_v2[i] = vx * vx + vy * vy + vz * vz;
    }
  }
  __syncthreads();
  const int fid = e0 * 4 + tid;
  double lfs = 0.0;
  if (tid < ne * 4) {
    const int e = tid >> 2, f = tid & 3;
    double mv2 = 0.0, mc2 = 0.0, sum = 0.0;
    for (int j = 0; j < Nfp; j++) {
      const int q = e * Np + s_fm[f * Nfp + j];
      const double v2 = s_v2[q];
      mv2 = v2 > mv2 ? v2 : mv2;
      sum += v2;
      if (PHYS == PHYS_EULER) {
        const double c2 = s_c2[q];
        mc2 = c2 > mc2 ? c2 : mc2;
        sum += c2;
      }
    }
    const double lam = PHYS == PHYS_EULER ? sqrt(mv2) + sqrt(mc2) : sqrt(mv2);
    maxv[fid] = lam;
    lfs = lam * geo[(size_t)(e0 + e) * GEO_STRIDE + 9 + f * 4 + 3];
    // A state that is not a number reaches dt as an infinite wave speed, and dt = 0
    // is flagged as bad on the device.  The face maxima pass over a NaN, the sum of
    // the squares (all >= 0) does not.
    if (sum != sum) lfs = INFINITY;
  }
  if (clk) {
    raise_maxfs(clk, lfs, red);
    return;
  }
  red[tid] = lfs;
  red_i[tid] = tid < ne * 4 ? fid : 0x7fffffff;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (tid < s) {
      const double o = red[tid + s];
      if (o > red[tid] || (o == red[tid] && red_i[tid + s] < red_i[tid])) {
        red[tid] = o;
        red_i[tid] = red_i[tid + s];
      }
    }
    __syncthreads();
  }
  if (tid == 0) {
    partial[blockIdx.x] = red[0];
    partial_idx[blockIdx.x] = red_i[0];
  }
}

}  // namespace dglm
