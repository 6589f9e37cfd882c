// reactors.hip — batched stiff chemistry: millions of independent 0-D reactors (constant
// volume, or constant pressure) integrated in one persistent launch.
//
// Each reactor is one cell of the reference's rosenbrock_kernel (kernels_gpu.F90:8928-9193):
// adaptive 4-stage Rosenbrock (Numerical-Recipes ROS4 constants), error scaled by
// max(1,|w|).  Three forms of it (the `mixed` argument):
//  0  the plain FP64 integrator, the yardstick of the other two: central-difference
//     Jacobian over all N_S + 4 variables, FP64 Crout LU with implicit pivoting, and
//     rosenbrock_rhs (:9249-9339) in the reference's own arithmetic forms (reference-form
//     kinetics from the packed records);
//  1  mixed precision on the species block: one-sided species Jacobian, FP32 LU refined
//     against the FP64 residual, fast-form kinetics and the NASA tables staged in LDS;
//  2  form 1 with the LU in FP64 (no refinement): the like-for-like FP64 counterpart of 1,
//     so that the difference between 1 and 2 is the precision of the factorisation alone.
// Reactors have uneven stiffness, so a fixed
// reactor-to-thread assignment would leave lanes idle behind the stiffest reactor of their
// wave: instead every row of 16 lanes pulls its next reactor from a device-wide counter as soon as it
// is done, and the grid is sized to the resident capacity of the GPU (persistent).  In large batches of
// forms 1 and 2 one lane per reactor takes the first steps (reactors_lanes_dev.h).
#include "reactors_dev.h"

namespace streams {
// The work counter's first value, and the counters of what the lanes leave.
__global__ void set_counter_kernel(unsigned *c, unsigned v, unsigned *left) {
  *c = v;
  if (left) left[0] = left[1] = 0u;
}

// Looks at 256 reactors: starts the work counter for the lanes when half of them would cover the
// interval in their first step (of those not finished before), for the rows otherwise.
__global__ void __launch_bounds__(256) choose_kernel(ReactorArgs A) {
  const long r = (long)threadIdx.x * A.nbatch / 256;
  double t0 = 0.0, dt = A.dttry[r];
  const double end = A.time_end[r];
  if (A.t_done) {
    t0 = A.t_done[r];
    if (A.dt_next[r] > 0.0) dt = A.dt_next[r];
  }
  const int n = __syncthreads_count(t0 < end && dt * 1.5 > end - t0);
  if (threadIdx.x == 0) {
    *A.next = n >= 128 ? LANES_TAKE : 0u;
    if (A.left.n) A.left.n[0] = A.left.n[1] = 0u;
  }
}

// Who begins a batch of forms 1 and 2.  Lanes are the faster where the GPU is full of them and their
// reactors step together; what is uneven they leave to the rows, so that they may begin whatever
// large batch comes.  Times in ms, rows alone and as it is (form 2, 9 species, unless said):
//   one step:          16384 reactors 0.55, 0.41; 65536 1.11, 0.49; 524288 6.4, 2.5
//                      14 species 65536 1.50, 1.43; 524288 8.9, 7.3
//   15 even steps:     65536 7.6, 6.2; 131072 14.5, 8.9; 524288 55.7, 30.5; form 1 131072 14.5, 9.2
//                      14 species 131072 31.2, 26.4 (98304 24.0, and 24.8 if lanes began it)
//   82 steps, to 291:  65536 57.8, 55.5; 131072 98.7, 89.7
//   345 steps, to 870: 65536 223, 226; 90000 289, 290; 131072 401, 397; form 1 131072 400, 395
//                      14 species 131072 812, 831
// Form 1 beyond 9 species is the faster in rows at any size (one step of 131072: 6.0 in lanes, 2.7), form 0
// too.  A call of one step pays up to 0.05 ms for the workspace and the two empty launches that the
// other kinds need.
//   ROWS: below the sizes at which lanes win even a single step
//   LOOK: where they win a single step only: choose_kernel looks
//   LANES: above
enum class Take { ROWS, LANES, LOOK };
inline Take who_takes(int n_s, int mixed, int nbatch, bool even) {
  if (mixed == 0 || (mixed == 1 && n_s > LANES_NS) || nbatch >= (1 << 30)) return Take::ROWS;
  const bool few = n_s <= LANES_NS;
  if (even || nbatch >= (few ? 65536 : 131072)) return Take::LANES;
  return nbatch >= (few ? 12288 : 40960) ? Take::LOOK : Take::ROWS;
}

// Steps of a resumed call in which its reactors, by its budget alone, stay together enough for the
// lanes to take it to its end (budgets of 6, 60 and 200 steps: 49152 reactors 2.64 in rows, 2.46; 65536 33.4,
// 29.0; 131072 181, 136; 13 and 14 species, 60 steps of 131072: 125, 103 and 128, 128).
inline int even_steps(int n_s, int nbatch) {
  if (n_s > LANES_NS) return nbatch >= 131072 ? 60 : nbatch >= 98304 ? 20 : 0;
  return nbatch >= 131072 ? 200 : nbatch >= 65536 ? 60 : nbatch >= 49152 ? 6 : nbatch >= 24576 ? 2 : 0;
}

inline bool capturing(hipStream_t st) {
  hipStreamCaptureStatus c = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(st, &c) != hipSuccess || c != hipStreamCaptureStatusNone;
}
}  // namespace streams

using namespace streams;

// Batched integration of nbatch independent reactors (rosenbrock_kernel per reactor with
// mixed = 0, the mixed-precision species-block variant with mixed = 1, its FP64 counterpart
// with mixed = 2) from t = 0 to time_end[b]: constant volume when
// pressure is null, else constant pressure pressure[b] with the state (Y, 0, 0, 0, h).  With
// t_done / dt_next (both or neither) the call is resumable: each reactor starts at
// t_done[b] with the step dt_next[b] (dttry[b] when not positive), takes at most maxsteps
// steps, and returns the time reached and its next step there.  work points to one unsigned
// of device memory used as the shared work counter (zeroed here, on the stream);
// wg_per_cu <= 0 gives 4 workgroups per CU.
extern "C" int streams_reactor_batch(int n_s, int nbatch, double *w, double *tguess, const double *dttry,
                                     const double *time_end, const double *pressure, const double *mw,
                                     const double *rgas, const double *cp_coeff, int nreactions,
                                     const double *kin_pack, const double *kc_tab, int num_t_tab, double t_min_tab,
                                     double dt_tab, double r_univ, double tol_iter_nr, const double *cv_coeff,
                                     int nsetcv, const double *trange, int indx_cp_l, int indx_cp_r, int maxsteps,
                                     int maxtry, double tol, int *nacc, int *nrej, double *t_done, double *dt_next,
                                     unsigned *work, int wg_per_cu, int mixed, void *stream) {
  if (nbatch < 0 || nreactions < 0 || maxsteps < 1 || maxtry < 1) return STREAMS_E_DIMS;
  if (mixed < 0 || mixed > 2) return STREAMS_E_OPTION;
  if (n_s > KTB) return STREAMS_E_NSPECIES;
  if (nsetcv < 1 || nsetcv > TMAXSET) return STREAMS_E_OPTION;
  if (nbatch == 0) return 0;
  if (work == nullptr) return STREAMS_E_DIMS;
  hipStream_t st = as_stream(stream);
  if (pressure != nullptr && (rgas == nullptr || cp_coeff == nullptr)) return STREAMS_E_DIMS;
  if ((t_done == nullptr) != (dt_next == nullptr)) return STREAMS_E_DIMS;
  ReactorArgs A{w, tguess, dttry, time_end, nacc, nrej, t_done, dt_next, work, nbatch, maxsteps, maxtry, mixed, tol,
                tol_iter_nr, mw,
                rgas, pressure, KinPacked{kin_pack, kc_tab, nreactions, num_t_tab, t_min_tab, dt_tab, r_univ},
                Thermo{cv_coeff, cp_coeff, trange, nsetcv, indx_cp_l, indx_cp_r}};
  const int ncu = device_cus();
  const bool even = t_done != nullptr && maxsteps <= even_steps(n_s, nbatch);
  Take take = who_takes(n_s, mixed, nbatch, even);
  char *left = nullptr;
  if (take != Take::ROWS && !even && maxsteps > LANE_STEPS) {
    // stream-ordered, each call's own
    const size_t nb = (size_t)nbatch, head = 256;
    if (!capturing(st) && hipMallocAsync((void **)&left, head + nb * 28, st) == hipSuccess) {
      char *p = left + head;
      A.left = LaneLeft{(unsigned *)left, (unsigned *)(p + 24 * nb), (double *)p, (double *)(p + 8 * nb),
                        (int *)(p + 16 * nb), (int *)(p + 20 * nb)};
    } else {
      // the lanes would have to integrate every reactor to its end
      (void)hipGetLastError();
      left = nullptr;
      take = Take::LOOK;
    }
  }
  if (take == Take::LOOK) choose_kernel<<<1, 256, 0, st>>>(A);
  else set_counter_kernel<<<1, 1, 0, st>>>(work, take == Take::LANES ? LANES_TAKE : 0u, A.left.n);
  int rc = 0;
  if (take != Take::ROWS) {
    const bool narrow = nbatch <= LANES_NARROW;
    rc = (pressure != nullptr ? (narrow ? reactor_lanes_cp : reactor_lanes_cp_wide)
                              : (narrow ? reactor_lanes_cv : reactor_lanes_cv_wide))(n_s, indx_cp_l, indx_cp_r, A, ncu,
                                                                                    wg_per_cu, st);
  }
  if (rc == 0 && (take != Take::LANES || left != nullptr)) {
    if (mixed != 0)
      rc = pressure != nullptr ? reactor_group_cp(n_s, indx_cp_l, indx_cp_r, A, ncu, wg_per_cu, st)
                               : reactor_group_cv(n_s, indx_cp_l, indx_cp_r, A, ncu, wg_per_cu, st);
    else
      rc = pressure != nullptr ? reactor_ref_cp(n_s, indx_cp_l, indx_cp_r, A, ncu, wg_per_cu, st)
                               : reactor_ref_cv(n_s, indx_cp_l, indx_cp_r, A, ncu, wg_per_cu, st);
  }
  if (left != nullptr && hipFreeAsync(left, st) != hipSuccess && rc == 0) return hip_status();
  return rc;
}
