// reactors_lanes.hip — the FP64 species block of large constant-volume batches with one lane per
// reactor, for reactors that take one step each.
//
// A row of 16 lanes per reactor (reactors_group_dev.h) wins wherever reactors differ in their steps
// or the batch does not fill the GPU.  Where a large batch's first trial step spans the interval, as in
// the half-steps of an operator splitting, the lanes of a wave stay together, and a row's
// shared temperature iterations and solves cost more than the scratch of a lane's Jacobian: 98304
// cells of a 14-species layer 1.70 ms a lane per cell, 1.95 a row, 204800 3.35 and 3.68, 16.8 M 214 and
// 272; but 38400 cells 1.23 and 1.00, and 131072 random reactors of 14 species over 20 steps
// 78 and 61 (mixed form: 4.8 and 2.0 ms at 98304, so rows always).  Both give the same bits.
#include "reactors_dev.h"

namespace streams {

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
  if (threadIdx.x == 0) *A.next = n >= 128 ? LANES_TAKE : 0u;
}

// rosenbrock_rhs on the packed tables, a lane's own
template <int NS, int LO>
struct LaneRhs {
  const KinPacked &K;
  const ThermoLds &TL;
  const double *mw;
  double tol_iter_nr;
  __device__ inline void operator()(double *wv, double &tg, double *rhs) const {
    double yy[NS], conc[NS], acc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) wv[s] = wv[s] > 0.0 ? wv[s] : 0.0;
    double rho = wv[0];
#pragma unroll
    for (int s = 1; s < NS; ++s) rho = rho + wv[s];
    const double ri = 1.0 / rho;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      yy[s] = wv[s] * ri;
      conc[s] = rho * yy[s] / mw[s];
      acc[s] = 0.0;
    }
    const double uu = wv[NS] * ri, vv = wv[NS + 1] * ri, ww = wv[NS + 2] * ri;
    const double qq = 0.5 * (uu * uu + vv * vv + ww * ww);
    const double ee = wv[NS + 3] * ri - qq;
    int nrange[NS];
    const double tt = temperature_from_e_lds<NS, LO>(ee, tg, TL, tol_iter_nr, yy, nrange);
    tg = tt;
    chemistry_source_packed<NS>(K, tt, conc, acc);
#pragma unroll
    for (int s = 0; s < NS; ++s) rhs[s] = -acc[s];
#pragma unroll
    for (int m = NS; m < NS + 4; ++m) rhs[m] = 0.0;
  }
};

// The ROS4 cell on the species block: one-sided Jacobian, FP64 LU.
template <int NS, class Rhs>
__device__ void rosenbrock_cell_block(const Rhs &rhs_fn, double *wv, double &tg, double dttry, double time_start,
                                      double time_end, int maxsteps, int maxtry, double tol, RosStats &st) {
  constexpr int NV = NS + 4;
  const double safety = 0.9, grow = 1.5, pgrow = -0.25, shrnk = 0.5, pshrnk = -1.0 / 3.0, errcon = 0.1296;
  const double gam = 1.0 / 2.0, a21 = 2.0, a31 = 48.0 / 25.0, a32 = 6.0 / 25.0;
  const double c21 = -8.0, c31 = 372.0 / 25.0, c32 = 12.0 / 5.0;
  const double c41 = -112.0 / 125.0, c42 = -54.0 / 125.0, c43 = -2.0 / 5.0;
  const double b1 = 19.0 / 9.0, b2 = 1.0 / 2.0, b3 = 25.0 / 108.0, b4 = 125.0 / 108.0;
  const double e1 = 17.0 / 54.0, e2 = 7.0 / 36.0, e3 = 0.0, e4 = 125.0 / 108.0;
  double jac[NS * NS];
  double lu[NS * NS];
  double w_sav[NS], rhs_sav[NV], yscal[NS], rhs[NV], rp[NV];
  double g1[NS], g2[NS], g3[NS], g4[NS];
  int indx[NS];
  int finish = 0;
  double time = time_start, dt = dttry, itol = 1.0 / tol, dtnext = dt;
  if (st.resume && dt * 1.5 > time_end - time) { dt = time_end - time; finish = 1; }
  for (int iter = 1; iter <= maxsteps; ++iter) {
    const double t0 = time;
    rhs_fn(wv, tg, rhs_sav);
    for (int n = 0; n < NS; ++n) {
      const double wtmp = wv[n];
      const double h = wtmp * 1.0e-06 + 1.0e-14;
      wv[n] = wtmp + h;
      double tj = tg;
      rhs_fn(wv, tj, rp);
      wv[n] = wtmp;
      for (int m = 0; m < NS; ++m) jac[m + NS * n] = (rp[m] - rhs_sav[m]) / h;
    }
    for (int m = 0; m < NS; ++m) {
      w_sav[m] = wv[m];
      yscal[m] = fmax(1.0, fabs(w_sav[m]));
    }
    for (int jtry = 1; jtry <= maxtry; ++jtry) {
      const double gi = 1.0 / (gam * dt);
      for (int n = 0; n < NS; ++n) {
        for (int m = 0; m < NS; ++m) lu[m + NS * n] = -jac[m + NS * n];
        lu[n + NS * n] = gi - jac[n + NS * n];
      }
      ludcmp<NS>(lu, indx);
      for (int m = 0; m < NS; ++m) g1[m] = rhs_sav[m];
      lubksb<NS>(lu, indx, g1);
      for (int m = 0; m < NS; ++m) wv[m] = w_sav[m] + a21 * g1[m];
      time = t0 + dt;
      rhs_fn(wv, tg, rhs);
      for (int m = 0; m < NS; ++m) g2[m] = rhs[m] + c21 * g1[m] / dt;
      lubksb<NS>(lu, indx, g2);
      for (int m = 0; m < NS; ++m) wv[m] = w_sav[m] + a31 * g1[m] + a32 * g2[m];
      time = t0 + 3.0 / 5.0 * dt;
      rhs_fn(wv, tg, rhs);
      for (int m = 0; m < NS; ++m) g3[m] = rhs[m] + (c31 * g1[m] + c32 * g2[m]) / dt;
      lubksb<NS>(lu, indx, g3);
      for (int m = 0; m < NS; ++m) g4[m] = rhs[m] + (c41 * g1[m] + c42 * g2[m] + c43 * g3[m]) / dt;
      lubksb<NS>(lu, indx, g4);
      double errmax = 0.0;
      for (int m = 0; m < NS; ++m) {
        wv[m] = w_sav[m] + b1 * g1[m] + b2 * g2[m] + b3 * g3[m] + b4 * g4[m];
        const double err = e1 * g1[m] + e2 * g2[m] + e3 * g3[m] + e4 * g4[m];
        errmax = fmax(errmax, fabs(err / yscal[m]));
      }
      time = t0 + dt;
      errmax = errmax * itol;
      if (errmax < 1.0 || finish == 1) {
        if (errmax > errcon) dtnext = safety * dt * pow(errmax, pgrow);
        else dtnext = grow * dt;
        break;
      } else {
        st.nrej += 1;
        dtnext = safety * dt * pow(errmax, pshrnk);
        dt = copysign(fmax(fabs(dtnext), shrnk * fabs(dt)), dt);
      }
    }
    st.nacc += 1;
    const double remaining = time_end - time;
    if (finish == 1 || remaining < 1.0e-12 * time_end) { st.done = 1; break; }
    if (dtnext * 1.5 > remaining) { dt = remaining; finish = 1; }
    else { dt = dtnext; finish = 0; }
  }
  st.t_end = time;
  st.dt_next = st.done ? dtnext : dt;
}

template <int NS, class Rhs>
__device__ inline void integrate_one(const Rhs &f, const ReactorArgs &A, unsigned r) {
  constexpr int NV = NS + 4;
  const long nb = A.nbatch;
  double wv[NV];
#pragma unroll
  for (int m = 0; m < NV; ++m) wv[m] = A.w[(long)m * nb + r];
  double tg = A.tg[r];
  RosStats st;
  double t0 = 0.0, dt0 = A.dttry[r];
  if (A.t_done) {
    st.resume = true;
    t0 = A.t_done[r];
    if (A.dt_next[r] > 0.0) dt0 = A.dt_next[r];
    if (t0 >= A.time_end[r]) {                        // finished earlier: nothing to do
      if (A.nacc) A.nacc[r] = 0;
      if (A.nrej) A.nrej[r] = 0;
      return;
    }
  }
  rosenbrock_cell_block<NS>(f, wv, tg, dt0, t0, A.time_end[r], A.maxsteps, A.maxtry, A.tol, st);
#pragma unroll
  for (int m = 0; m < NV; ++m) A.w[(long)m * nb + r] = wv[m];
  A.tg[r] = tg;
  if (A.nacc) A.nacc[r] = st.nacc;
  if (A.nrej) A.nrej[r] = st.nrej;
  if (A.t_done) {
    A.t_done[r] = st.done ? A.time_end[r] : st.t_end;
    A.dt_next[r] = st.dt_next;
  }
}

// 3 waves per SIMD up to 9 species, 2 beyond: every lane spills, and more resident waves
// hide the latency (2^19 reactors of 9 species at 1, 2, 3, 4 waves: 171k, 257k, 283k, 234k solves/s).
template <int NS, int LO>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NS <= 9 ? 3 : 2)))
reactor_lane_kernel(ReactorArgs A) {
  constexpr int WHICH = TH_CV | TH_CVH;
  __shared__ double tlds[thermo_lds_doubles<NS>(WHICH)];
  if (*(volatile unsigned *)A.next < LANES_TAKE) return;   // the rows take the batch
  const ThermoLds TL = thermo_stage<NS, LO>(A.th, tlds, WHICH);
  __syncthreads();
  const long nb = A.nbatch;
  for (;;) {
    const unsigned r = atomicAdd(A.next, 1u) - LANES_TAKE;
    if ((long)r >= nb) break;
    const LaneRhs<NS, LO> f{A.K, TL, A.mw, A.tol_iter_nr};
    integrate_one<NS>(f, A, r);
  }
}

int reactor_lanes(int n_s, int indx_cp_l, int indx_cp_r, const ReactorArgs &A, int ncu, int wg_per_cu, hipStream_t st) {
  const int g = reactor_grid(ncu, wg_per_cu, 3, 256, A.nbatch);
  if (g <= 0) return STREAMS_E_DIMS;
  choose_kernel<<<1, 256, 0, st>>>(A);
  STREAMS_DISPATCH_NS(n_s, STREAMS_DISPATCH_NASA(indx_cp_l, indx_cp_r,
                                                 (reactor_lane_kernel<NS, LO><<<g, 256, 0, st>>>(A))));
  return hip_status();
}
}  // namespace streams
