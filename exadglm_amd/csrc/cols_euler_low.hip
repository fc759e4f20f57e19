// The packed-column stage kernel, Euler, orders 1..5.
#include "kernels/dg_cols.hpp"

namespace dglm {

ColOps cols_euler_low(int N, int K) {
  switch (N) {
    case 1:
      return cols_ops<1, PHYS_EULER>(K);
    case 2:
      return cols_ops<2, PHYS_EULER>(K);
    case 3:
      return cols_ops<3, PHYS_EULER>(K);
    case 4:
      return cols_ops<4, PHYS_EULER>(K);
    case 5:
      return cols_ops<5, PHYS_EULER>(K);
    default:
      return {};
  }
}

}  // namespace dglm
