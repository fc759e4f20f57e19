// Shared device-side definitions for the DGLM kernels (gfx950).
#pragma once
#include <hip/hip_runtime.h>

namespace dglm {

constexpr int NFACE = 4;

template <int N>
struct Ord {
  static constexpr int Np = (N + 1) * (N + 2) * (N + 3) / 6;
  static constexpr int Nfp = (N + 1) * (N + 2) / 2;
  static constexpr int NFF = NFACE * Nfp;
  static constexpr int KD = 3 * Np + NFF;  // stacked contraction length [WDr|WDs|WDt|LIFT]
};

// Reciprocal and square root of the stage kernels (the adjoint's pass A, where
// they were measured no faster, divides): the hardware estimates v_rcp_f64 and
// v_rsq_f64 refined by Newton steps (two r += r (1 - x r); for the root a coupled
// step on g = x y, h = y / 2 and a correction g += h (x - g^2)), within an ulp of
// the IEEE results and equal to them on every one of 4M sampled densities in
// [1e-3, 1e3] and squared sound speeds in [1e-6, 1e6]; the IEEE division and
// square-root sequences are chains about twice as long.  For normal arguments, as
// a sound state has them.  The reciprocal of 0 or an infinity is NaN, where the
// division has an infinity or 0, so the fluxes of a state with such a density are
// NaN; zero and NaN pass through the root.
__device__ inline double rcp_refined(double x) {
  double r = __builtin_amdgcn_rcp(x);
  double e = __builtin_fma(-x, r, 1.0);
  r = __builtin_fma(r, e, r);
  e = __builtin_fma(-x, r, 1.0);
  return __builtin_fma(r, e, r);
}
__device__ inline double sqrt_refined(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  return x > 0.0 ? g : x;
}

// The step scalars live in device memory, so the step loop never reads back to
// the host (the reference copies dt to the host every step,
// euler_nopad_dglm.cu:79-96), in two slots that the steps use in turn: the first
// stage of a step forms dt from one for itself, leaves it there for the other
// stages and starts the next step's in the other slot.
constexpr int MAXFS_SLOTS = 16, MAXFS_STRIDE = 8;  // 64 bytes apart
struct DevClock {
  double t;        // start of the step (= the committed time)
  double dt;       // its size (written by its first stage)
  double last_dt;  // size of the step before (0: it was past tmax)
  int active;      // 0: the step is past tmax (written by its first stage)
  int tstep;       // steps taken
  int bad;         // a non-finite or non-positive dt was seen
  int pad[5];
  // Largest lambda * Fscale over the faces, in parts by workgroup: bits of
  // doubles >= 0, which order as integers.  One address for the whole grid's
  // atomics took the wave-speed kernel from 10 to 27 us at 697 workgroups.
  unsigned long long maxfs[MAXFS_SLOTS * MAXFS_STRIDE];
};

// Per-element geometry record: 9 metrics followed by 4x(nx,ny,nz,Fscale).
constexpr int GEO_STRIDE = 25;

// Packed face connectivity: (nbr << 4) | (nbr_face << 2) | code, where code
// 0..2 selects FmaskP[nbr_face][rot] and code 3 selects Fmask[nbr_face]
// (a boundary face whose exterior trace is the interior one).
__host__ __device__ inline int conn_nbr(int c) { return c >> 4; }
__host__ __device__ inline int conn_face(int c) { return (c >> 2) & 3; }
__host__ __device__ inline int conn_code(int c) { return c & 3; }

// The step that starts at t: dt = CFL/(2N+1) / max(lambda*Fscale), clipped so that
// the run ends exactly at tmax (euler_time.cpp:49-57); false past tmax.
__device__ inline bool step_dt(double t, double maxfs, double cfl_fac, double tmax, double &dt, bool &clipped) {
#pragma clang fp contract(off)
  dt = 0.0;
  clipped = false;
  if (!(t < tmax)) return false;
  dt = cfl_fac * (1.0 / maxfs);
  const double end = t + dt;
  if (end > tmax) {
    dt = tmax - t;
    clipped = true;
  }
  return true;
}

// Orders the compiler's LDS accesses of one wave; the LDS executes them in order.
__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Raise the workgroup's part of maxfs to its largest x.  Nothing below 0 gets there
// (Fscale of an inside-out element is negative, and a negative double's bits are
// above every positive one's).  red: LDS, one double per wave (at most 16 waves);
// every thread of the workgroup calls it.
__device__ inline void raise_maxfs(DevClock *c, double x, double *red) {
  x = fmax(x, 0.0);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x = fmax(x, __shfl_xor(x, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (unsigned w = 1; w < blockDim.x >> 6; w++) x = fmax(x, red[w]);
    atomicMax(&c->maxfs[blockIdx.x % MAXFS_SLOTS * MAXFS_STRIDE], (unsigned long long)__double_as_longlong(x));
  }
}

}  // namespace dglm
