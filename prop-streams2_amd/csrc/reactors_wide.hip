// reactors_wide.hip — the wide (two waves per SIMD) instance of the plain FP64 reactor
// kernel, in its own translation unit so that its device code gets its own register budget.
#include "reactors_dev.h"

namespace streams {
int reactor_dispatch_wide(int n_s, const ReactorArgs &A, int ncu, int wg_per_cu, hipStream_t st) {
  return reactor_dispatch<true>(n_s, A, ncu, wg_per_cu, st);
}
}  // namespace streams
