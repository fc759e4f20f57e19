// Arguments of the adjoint's pass A and pass B (dg_adjoint.hpp).
#pragma once
#include "dg_common.hpp"

namespace dglm {

struct AdjArgs {
  int K;
  int first;           // 1: the first pass A of a reverse step (taubar and dtpart start here, kbar is zero: the
                       // forward's first stage, a = 0, takes no k; for the same reason the last pass A, a = 0,
                       // writes none)
  int mode;            // 0: reverse LSRK stage; 1: plain RHS adjoint (rbar given, ubar := J^T rbar)
  const double *u;     // forward stage state u_s
  double *ubar;        // [NV][K*Np]  in/out
  double *kbar;        // [NV][K*Np]  in/out (mode 0)
  const double *rbar;  // [NV][K*Np]  (mode 1)
  double *gsur;        // [K][NFF][NV] partner-side face terms (pass A out, pass B in)
  // partner-side face terms of the previous pass A, not yet added to ubar
  // (null: none)
  const double *gsur_in;
  double *taubar;      // [K*4] accumulated tau adjoint per face side (may be null)
  const double *vel;
  const double *geo;
  const int *conn;
  const int *fmx;
  const int *node_slots;  // [Np][3] face-node slots m = f*Nfp + j with Fmask[f][j] == node (-1 pad)
  const int *pslot;       // [4][4][Nfp] partner slot: (face, code, j) of a connectivity word -> face-node slot
                          // nf*Nfp + jp of the neighbour
  const double *maxv;     // wave speed per face at the step start (tau)
  const double *dtp;      // device dt of the step (mode 0)
  double *dtpart;         // [workgroups] dt sensitivity (exact adjoint): sum_nodes r_s . kb (may be null)
  double a, b;
  double gamma, tau_scale;
  const int *order;  // visiting order of pass A's batches (null: mesh order)
};

}  // namespace dglm
