// Host-side access to the packed-column adjoint kernels, which are compiled in
// translation units of their own.
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "dg_adjoint_args.hpp"

namespace dglm {

struct AdjOps {
  int eb = 0;  // elements per workgroup (0: not built)
  void (*fill)(const double *opT /*[KD][Np]*/, std::vector<double> &out) = nullptr;  // the kernel's operator streams
  void (*launch)(hipStream_t stream, const AdjArgs &a, const double *afragT) = nullptr;  // one pass A
};

AdjOps adjoint_advection(int N);  // N = 1..10
AdjOps adjoint_euler(int N);      // N = 1..10

}  // namespace dglm
