// seqcg.hpp — the band-sequential preconditioned CG (kscg_r / kscg_c) as fused launches without
// host round trips (seqcg.hip).
#pragma once
#include "bloch.hpp"
#include "solvers.hpp"

namespace kukan {

template <class T>  // double, or double2 for the complex path
struct SeqCgArgs {
  int M, northo, nkscg, nsdmax, nprecon_cg, ns;
  bool recompute;  // <p|psi> and S psi afresh before a band is orthonormalised
  double epssd;
  const double *veff;
  T *psi, *spsi, *hpsi, *cps;  // spsi may be psi (S = 1)
  double *sval, *resid;
  int *ksconv, *ksitmax;
};
void seq_cg(Ctx &c, const SeqCgArgs<double> &a);
void seq_cg(ZCtx &z, const SeqCgArgs<double2> &a);

}  // namespace kukan
