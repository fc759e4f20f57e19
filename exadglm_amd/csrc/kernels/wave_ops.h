// Entry points of the persistent one-wave-per-batch stage kernel (dg_wave.hpp).
#pragma once
#include <vector>

#include "dg_fp64.hpp"

namespace dglm {

struct WaveOps {
  int eb = 0, nw = 0;  // elements per batch (0: the order has no such kernel), waves per workgroup
  void (*fill)(const double *opT, std::vector<double> &out) = nullptr;
  void (*launch)(int mode, int cus, hipStream_t stream, const StageArgs &a, const double *op, const int *order) = nullptr;
};

// Euler, order 3 or 4.
WaveOps wave_ops(int N);

}  // namespace dglm
