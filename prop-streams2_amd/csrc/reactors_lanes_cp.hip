// reactors_lanes_cp.hip — one lane per reactor: constant pressure, batches of up to LANES_NARROW reactors.
#include "reactors_lanes_dev.h"

namespace streams {
int reactor_lanes_cp(int n_s, int indx_cp_l, int indx_cp_r, const ReactorArgs &A, int ncu, int wg_per_cu,
                     hipStream_t st) {
  return reactor_lanes_dispatch<true, true>(n_s, indx_cp_l, indx_cp_r, A, ncu, wg_per_cu, st);
}
}  // namespace streams
