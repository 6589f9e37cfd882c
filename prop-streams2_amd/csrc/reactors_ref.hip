// reactors_ref.hip — the constant-volume plain FP64 form of the reactor batch.
#include "reactors_ref_dev.h"

namespace streams {
int reactor_ref_cv(int n_s, int indx_cp_l, int indx_cp_r, const ReactorArgs &A, int ncu, int wg_per_cu,
                   hipStream_t st) {
  return reactor_ref_dispatch<false>(n_s, indx_cp_l, indx_cp_r, A, ncu, wg_per_cu, st);
}
}  // namespace streams
