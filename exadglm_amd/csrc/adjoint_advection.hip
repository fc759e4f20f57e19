// Pass A of the advection adjoint, orders 1..10.
#include "kernels/dg_adjoint_adv.hpp"

namespace dglm {

AdjOps adjoint_advection(int N) {
  switch (N) {
#define DGLM_CASE(n) \
  case n:            \
    return {AdvAdjShape<n>::EB, AdvAdjImpl<n>::fill, AdvAdjImpl<n>::launch};
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
