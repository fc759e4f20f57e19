// Per-step reductions that are plain (non-template) kernels: the device-side
// dt, its adjoint and the conserved integrals.  Included by solver.hip only, so each is
// defined in one translation unit.
#pragma once
#include "dg_common.hpp"

namespace dglm {

// The adjoint's recording: the largest of the wave-speed blocks' maxima into the
// step's clock, and its face (smallest index on ties), dt and the clip flag into
// the step's entries of the tape.  One block.
__global__ __launch_bounds__(1024) void record_dt_kernel(const double *__restrict__ partial,
                                                         const int *__restrict__ partial_idx, int n, DevClock *s,
                                                         double cfl_fac, double tmax, double *dt_rec, int *fstar_rec,
                                                         int *clip_rec) {
  __shared__ double red[1024];
  __shared__ int red_i[1024];
  double m = 0.0;
  int mi = 0x7fffffff;
  for (int i = threadIdx.x; i < n; i += 1024) {
    const double o = partial[i];
    if (o > m || (o == m && partial_idx[i] < mi)) {
      m = o;
      mi = partial_idx[i];
    }
  }
  red[threadIdx.x] = m;
  red_i[threadIdx.x] = mi;
  __syncthreads();
  for (int w = 512; w > 0; w >>= 1) {
    if (threadIdx.x < w) {
      const double o = red[threadIdx.x + w];
      if (o > red[threadIdx.x] || (o == red[threadIdx.x] && red_i[threadIdx.x + w] < red_i[threadIdx.x])) {
        red[threadIdx.x] = o;
        red_i[threadIdx.x] = red_i[threadIdx.x + w];
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    s->maxfs[0] = (unsigned long long)__double_as_longlong(red[0]);
    for (int i = 1; i < MAXFS_SLOTS; i++) s->maxfs[i * MAXFS_STRIDE] = 0;
    double dt;
    bool clipped;
    step_dt(s->t, red[0], cfl_fac, tmax, dt, clipped);
    if (dt_rec) *dt_rec = dt;
    if (fstar_rec) *fstar_rec = red_i[0];
    if (clip_rec) *clip_rec = clipped;
  }
}

// Clock updates between steps: copy *src (when given), set the time (what & 1),
// clear maxfs (what & 2).  MAXFS_SLOTS threads.
__global__ void set_clock_kernel(DevClock *c, const DevClock *src, int what, double t, int tstep) {
  const int part = threadIdx.x * MAXFS_STRIDE;
  if (src || (what & 2)) c->maxfs[part] = what & 2 ? 0 : src->maxfs[part];
  if (threadIdx.x != 0) return;
  if (src) {
    c->t = src->t;
    c->last_dt = src->last_dt;
    c->tstep = src->tstep;
    c->bad = src->bad;
  }
  if (what & 1) {
    c->t = t;
    c->last_dt = 0.0;
    c->tstep = tstep;
    c->bad = 0;
  }
}

struct ClockReport {
  double t, last_dt;
  int tstep, bad;
};

// The clock and the first n dt of a step call into mapped host memory.
__global__ __launch_bounds__(256) void report_kernel(const DevClock *c, const double *dt_hist, int n,
                                                     ClockReport *c_out, double *dt_out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) dt_out[i] = dt_hist[i];
  if (i == 0) *c_out = {c->t, c->last_dt, c->tstep, c->bad};
}

// Conserved integrals sum_e J_e w^T u_e (w = column sums of M), FP64: one
// thread per element, a fixed-order block reduction, partials per block.
__global__ __launch_bounds__(256) void integrals_kernel(int K, int Np, int nvar, const double *__restrict__ u,
                                                       const double *__restrict__ J,
                                                       const double *__restrict__ w, double *partial) {
  __shared__ double red[256];
  const int e = blockIdx.x * 256 + threadIdx.x;
  const size_t KNp = (size_t)K * Np;
  for (int v = 0; v < nvar; v++) {
    double s = 0.0;
    if (e < K) {
      const double *ue = u + v * KNp + (size_t)e * Np;
      for (int i = 0; i < Np; i++) s += w[i] * ue[i];
      s *= J[e];
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int q = 128; q > 0; q >>= 1) {
      if (threadIdx.x < q) red[threadIdx.x] += red[threadIdx.x + q];
      __syncthreads();
    }
    if (threadIdx.x == 0) partial[(size_t)blockIdx.x * nvar + v] = red[0];
    __syncthreads();
  }
}

// dtbar of the step = sum of the block partials + tbar (adjoint of the time
// after the step).  If the step was clipped to end at tmax, dt = tmax - t
// does not depend on the wave speed and its adjoint flows into t instead.
// One block; scal[0] = tbar (in/out), scal[1] = dtbar seen by lambda (out).
__global__ __launch_bounds__(256) void adjoint_dt_reduce(const double *__restrict__ dtpart, int n,
                                                         const int *__restrict__ clipped, int step, double *scal) {
  __shared__ double red[256];
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) s += dtpart[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double dtbar = red[0] + scal[0];
    if (clipped[step]) {
      scal[0] -= dtbar;
      scal[1] = 0.0;
    } else {
      scal[1] = dtbar;
    }
  }
}

}  // namespace dglm
