// reactors_lanes_wide_cp.hip — one lane per reactor: constant pressure, larger batches.
#include "reactors_lanes_dev.h"

namespace streams {
int reactor_lanes_cp_wide(int n_s, int indx_cp_l, int indx_cp_r, const ReactorArgs &A, int ncu, int wg_per_cu,
                          hipStream_t st) {
  return reactor_lanes_dispatch<true, false>(n_s, indx_cp_l, indx_cp_r, A, ncu, wg_per_cu, st);
}
}  // namespace streams
