// The packed-column stage kernel, Euler, orders 6..10.
#include "kernels/dg_cols.hpp"

namespace dglm {

ColOps cols_euler_high(int N, int K) {
  switch (N) {
    case 6:
      return cols_ops<6, PHYS_EULER>(K);
    case 7:
      return cols_ops<7, PHYS_EULER>(K);
    case 8:
      return cols_ops<8, PHYS_EULER>(K);
    case 9:
      return cols_ops<9, PHYS_EULER>(K);
    case 10:
      return cols_ops<10, PHYS_EULER>(K);
    default:
      return {};
  }
}

}  // namespace dglm
