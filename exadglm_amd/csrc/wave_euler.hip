// The persistent one-wave-per-batch stage kernel (kernels/dg_wave.hpp).
#include "kernels/dg_wave.hpp"

namespace dglm {

WaveOps wave_ops(int N) {
  switch (N) {
    case 3:
      return {6, 8, WaveImpl<3, 6, 8>::fill, WaveImpl<3, 6, 8>::launch};
    case 4:
      return {3, 8, WaveImpl<4, 3, 8>::fill, WaveImpl<4, 3, 8>::launch};
    default:
      return {};
  }
}

}  // namespace dglm
