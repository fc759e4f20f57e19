// The packed-column stage kernel, advection, orders 1..10.
#include "kernels/dg_cols.hpp"

namespace dglm {

ColOps cols_advection(int N, int K) {
  switch (N) {
    case 1:
      return cols_ops<1, PHYS_ADV>(K);
    case 2:
      return cols_ops<2, PHYS_ADV>(K);
    case 3:
      return cols_ops<3, PHYS_ADV>(K);
    case 4:
      return cols_ops<4, PHYS_ADV>(K);
    case 5:
      return cols_ops<5, PHYS_ADV>(K);
    case 6:
      return cols_ops<6, PHYS_ADV>(K);
    case 7:
      return cols_ops<7, PHYS_ADV>(K);
    case 8:
      return cols_ops<8, PHYS_ADV>(K);
    case 9:
      return cols_ops<9, PHYS_ADV>(K);
    case 10:
      return cols_ops<10, PHYS_ADV>(K);
    default:
      return {};
  }
}

}  // namespace dglm
