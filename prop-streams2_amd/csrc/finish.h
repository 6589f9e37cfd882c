// finish.h — arguments of the pointwise tail of an RK substep (finish.hip).
#pragma once
#include "kinpack.h"

namespace streams {

struct FinishArgs {
  const double *cd1, *dcsidx, *detady, *dzitdz;
  const int *mask;
  const double *mw;
  KinPacked K;
  int lmax, reduced, chem;
  double gamdt;
  // fold = 1: the next substep's init_flux is done here (fln = -rhodt_next * fl, written in
  // place of fl, which then needs no store: the next x sweep overwrites it with init = 2)
  int fold;
  double rhodt_next;
};

// chemistry source and RK update of the species (finish_species_kernel)
int finish_species_launch(int n_s, const Box &b, double *w, const double *w_aux, double *fl, double *fln,
                          const FinishArgs &F, hipStream_t st);

}  // namespace streams
