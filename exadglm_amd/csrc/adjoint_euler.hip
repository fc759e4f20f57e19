// Pass A of the Euler adjoint, orders 1..10.
#include "kernels/dg_adjoint_euler.hpp"

namespace dglm {

AdjOps adjoint_euler(int N) {
  switch (N) {
#define DGLM_CASE(n) \
  case n:            \
    return {EulAdjShape<n>::EB, EulAdjImpl<n>::fill, EulAdjImpl<n>::launch};
    DGLM_CASE(1)
    DGLM_CASE(2)
    DGLM_CASE(3)
    DGLM_CASE(4)
    DGLM_CASE(5)
    DGLM_CASE(6)
    DGLM_CASE(7)
    DGLM_CASE(8)
    DGLM_CASE(9)
    DGLM_CASE(10)
#undef DGLM_CASE
    default:
      return {};
  }
}

}  // namespace dglm
