// reactors_group_cp.hip — the constant-pressure species-block forms of the reactor batch.
#include "reactors_group_dev.h"

namespace streams {
int reactor_group_cp(int n_s, int indx_cp_l, int indx_cp_r, const ReactorArgs &A, int ncu, int wg_per_cu,
                     hipStream_t st) {
  return reactor_group_dispatch<true>(n_s, indx_cp_l, indx_cp_r, A, ncu, wg_per_cu, st);
}
}  // namespace streams
