// rosenbrock.hip — the implicit chemistry of a field's cells, a 16-lane row of a wave per cell.
#include "reactors_ref_dev.h"

namespace streams {
int rosenbrock_rows(int n_s, const Box &b, double *w, double *w_aux, const Kin &K, const Thermo &th,
                    double tol_iter_nr, double dttry, double time_start, double time_end, int maxsteps, int maxtry,
                    double tol, const Pasr &pasr, hipStream_t st) {
  RefArgs A{};
  A.R.w = w;
  A.R.maxsteps = maxsteps;
  A.R.maxtry = maxtry;
  A.R.tol = tol;
  A.R.tol_iter_nr = tol_iter_nr;
  A.R.mw = K.mw;
  A.R.K = KinPacked{nullptr, K.kc_tab, K.nr, K.num_t_tab, K.t_min_tab, K.dt_tab, K.r_univ};
  A.R.th = th;
  A.b = b;
  A.w_aux = w_aux;
  A.D = K;
  A.pasr = pasr;
  A.dttry = dttry;
  A.time_start = time_start;
  A.time_end = time_end;
  A.ncells = (unsigned)b.fstride();
  const int g = reactor_grid(device_cus(), 8, 8, REF_BS / GROW, b.fstride());
  const long bytes = (long)K.nr * KREC * 8;
  STREAMS_DISPATCH_NS(n_s, STREAMS_DISPATCH_NASA(th.lo, th.hi,
                                                 (reactor_ref_kernel<NS, LO, false, true><<<g, REF_BS, bytes, st>>>(A))));
  return hip_status();
}
}  // namespace streams
