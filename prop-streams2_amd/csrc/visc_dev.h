// visc_dev.h — arguments of the viscous / diffusive fluxes, shared by the per-direction
// viscous kernels and the fused convective+viscous sweeps.
#pragma once
#include "common.h"

namespace streams {

struct ViscArgs {
  const double *w_aux, *coord, *rgas;
  double *fl;
  Thermo th;
  double r_univ;
  int n;
};

}  // namespace streams
