// Host-side access to the packed-column stage kernel (dg_cols.hpp), which is
// compiled in translation units of its own, a few orders each.
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "dg_fp64.hpp"

namespace dglm {

struct ColOps {
  int eb = 0;  // elements per batch (0: order not built)
  void (*fill)(const double *opT /*[KD][Np]*/, std::vector<double> &out) = nullptr;  // the kernel's operator streams
  // one stage (mode 0: LSRK update, 1: RHS only); order: visiting order of the
  // batches (null: mesh order)
  void (*launch)(int mode, hipStream_t stream, const StageArgs &a, const double *afrag, const int *order) = nullptr;
};

ColOps cols_euler_low(int N, int K);   // N = 1..5
ColOps cols_euler_high(int N, int K);  // N = 6..10
ColOps cols_advection(int N, int K);   // N = 1..10

inline ColOps cols_find(int N, int phys, int K) {
  return phys == PHYS_ADV ? cols_advection(N, K) : (N <= 5 ? cols_euler_low(N, K) : cols_euler_high(N, K));
}

}  // namespace dglm
