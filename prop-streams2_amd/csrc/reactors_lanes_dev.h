// reactors_lanes_dev.h — the species-block forms of large batches with one lane per reactor, while
// the reactors of a wave take steps together.
//
// A row of 16 lanes per reactor (reactors_group_dev.h) wins wherever reactors differ in their steps
// or the batch does not fill the GPU.  Where the reactors of a wave take the same few steps its
// lanes stay together, and a row's shared temperature iterations and solves, and its turn at the
// work counter (12 ns), cost more than the scratch of a lane's Jacobian.  So the lanes of a large
// batch take its first steps, and leave to the rows (LaneLeft) the reactors that go on when a third of
// their wave has finished, and after LANE_STEPS steps those that are still under way.  Both give the
// same bits.  reactors.hip has the rule and the times on both sides of it.
#pragma once
#include "reactors_dev.h"

namespace streams {

// The right-hand side of the packed tables, species rows, unscaled; returns the scale (1 at
// constant volume).
template <int NS, int LO, bool CP>
struct LaneRhs {
  const KinPacked &K;
  const ThermoLds &TL;
  const double *mw, *rgas;
  double pres, tol_iter_nr;
  __device__ inline double operator()(double *wv, double &tg, double *rhs) const {
    double yy[NS], conc[NS], acc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) wv[s] = wv[s] > 0.0 ? wv[s] : 0.0;
    double rho = wv[0];
#pragma unroll
    for (int s = 1; s < NS; ++s) rho = rho + wv[s];
    const double ri = 1.0 / rho;
    int nrange[NS];
    double scale = 1.0;
    if constexpr (CP) {
      double rmix = 0.0;
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        yy[s] = wv[s] * ri;
        rmix = rmix + rgas[s] * yy[s];
      }
      tg = temperature_newton_lds<NS, LO>(wv[NS + 3], tg, TL, TL.cp, TL.cph, tol_iter_nr, yy, nrange);
      rho = pres / (rmix * tg);
      scale = 1.0 / rho;
    } else {
#pragma unroll
      for (int s = 0; s < NS; ++s) yy[s] = wv[s] * ri;
      const double uu = wv[NS] * ri, vv = wv[NS + 1] * ri, ww = wv[NS + 2] * ri;
      const double qq = 0.5 * (uu * uu + vv * vv + ww * ww);
      const double ee = wv[NS + 3] * ri - qq;
      tg = temperature_from_e_lds<NS, LO>(ee, tg, TL, tol_iter_nr, yy, nrange);
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      conc[s] = rho * yy[s] / mw[s];
      acc[s] = 0.0;
    }
    chemistry_source_packed<NS>(K, tg, conc, acc);
#pragma unroll
    for (int s = 0; s < NS; ++s) rhs[s] = -acc[s];
    return scale;
  }
};

// Solve W b = b with W = gi I - J; an FP32 factor is refined once against the FP64 residual.
template <int N, class LU>
__device__ inline void solve_block(const double *jac, const LU *lu, const int *indx, double gi, double *b) {
  if constexpr (sizeof(LU) == sizeof(double)) {
    lubksb<N, double>(lu, indx, b);
  } else {
    float x32[N];
#pragma unroll
    for (int m = 0; m < N; ++m) x32[m] = (float)b[m];
    lubksb<N, float>(lu, indx, x32);
    double x[N], r[N];
#pragma unroll
    for (int m = 0; m < N; ++m) {
      x[m] = (double)x32[m];
      r[m] = b[m] - gi * x[m];
    }
    for (int n = 0; n < N; ++n) {
      const double xn = x[n];
#pragma unroll
      for (int m = 0; m < N; ++m) r[m] = r[m] + jac[m + N * n] * xn;
    }
#pragma unroll
    for (int m = 0; m < N; ++m) x32[m] = (float)r[m];
    lubksb<N, float>(lu, indx, x32);
#pragma unroll
    for (int m = 0; m < N; ++m) b[m] = x[m] + (double)x32[m];
  }
}

// Lanes of a wave below which they leave their reactors: a step of the rows takes 1.4 to 1.9 times
// as long as one of full waves.
constexpr int LANES_FULL = 44;

// The ROS4 cell on the species block: one-sided Jacobian, LU in the type given.  steps > 0: may
// return before the end (true), after that many steps or when the wave has emptied.
template <int NS, class LU, bool CP, class Rhs>
__device__ bool rosenbrock_cell_block(const Rhs &rhs_fn, double *wv, double &tg, double dttry, double time_start,
                                      double time_end, int maxsteps, int maxtry, double tol, RosStats &st, int steps,
                                      int &finish) {
  const double safety = 0.9, grow = 1.5, pgrow = -0.25, shrnk = 0.5, pshrnk = -1.0 / 3.0, errcon = 0.1296;
  const double gam = 1.0 / 2.0, a21 = 2.0, a31 = 48.0 / 25.0, a32 = 6.0 / 25.0;
  const double c21 = -8.0, c31 = 372.0 / 25.0, c32 = 12.0 / 5.0;
  const double c41 = -112.0 / 125.0, c42 = -54.0 / 125.0, c43 = -2.0 / 5.0;
  const double b1 = 19.0 / 9.0, b2 = 1.0 / 2.0, b3 = 25.0 / 108.0, b4 = 125.0 / 108.0;
  const double e1 = 17.0 / 54.0, e2 = 7.0 / 36.0, e3 = 0.0, e4 = 125.0 / 108.0;
  double jac[NS * NS];
  LU lu[NS * NS];
  double w_sav[NS], rhs_sav[NS], yscal[NS], rhs[NS], rp[NS];
  double g1[NS], g2[NS], g3[NS], g4[NS];
  int indx[NS];
  bool left = false;
  finish = 0;
  double time = time_start, dt = dttry, itol = 1.0 / tol, dtnext = dt;
  // scale * r + x, with the roundings of the rows
  auto scaled_plus = [&](double r, double scale, double x) { return CP ? fma(r, scale, x) : r + x; };
  auto scaled = [&](double &r, double scale) {
    if constexpr (CP) {
      r = r * scale;
      opaque(r);
    }
  };
  if (st.resume && dt * 1.5 > time_end - time) { dt = time_end - time; finish = 1; }
  for (int iter = 1; iter <= maxsteps; ++iter) {
    const double t0 = time;
    double scale = rhs_fn(wv, tg, rhs_sav);
    for (int m = 0; m < NS; ++m) scaled(rhs_sav[m], scale);
    for (int n = 0; n < NS; ++n) {
      const double wtmp = wv[n];
      const double h = wtmp * 1.0e-06 + 1.0e-14;
      wv[n] = wtmp + h;
      double tj = tg;
      scale = rhs_fn(wv, tj, rp);
      wv[n] = wtmp;
      for (int m = 0; m < NS; ++m) jac[m + NS * n] = scaled_plus(rp[m], scale, -rhs_sav[m]) / h;
    }
    for (int m = 0; m < NS; ++m) {
      w_sav[m] = wv[m];
      yscal[m] = fmax(1.0, fabs(w_sav[m]));
    }
    for (int jtry = 1; jtry <= maxtry; ++jtry) {
      const double gi = 1.0 / (gam * dt);
      for (int n = 0; n < NS; ++n) {
        for (int m = 0; m < NS; ++m) lu[m + NS * n] = (LU)(-jac[m + NS * n]);
        lu[n + NS * n] = (LU)(gi - jac[n + NS * n]);
      }
      ludcmp<NS, LU>(lu, indx);
      for (int m = 0; m < NS; ++m) g1[m] = rhs_sav[m];
      solve_block<NS>(jac, lu, indx, gi, g1);
      for (int m = 0; m < NS; ++m) wv[m] = w_sav[m] + a21 * g1[m];
      time = t0 + dt;
      scale = rhs_fn(wv, tg, rhs);
      for (int m = 0; m < NS; ++m) g2[m] = scaled_plus(rhs[m], scale, c21 * g1[m] / dt);
      solve_block<NS>(jac, lu, indx, gi, g2);
      for (int m = 0; m < NS; ++m) wv[m] = w_sav[m] + a31 * g1[m] + a32 * g2[m];
      time = t0 + 3.0 / 5.0 * dt;
      scale = rhs_fn(wv, tg, rhs);
      for (int m = 0; m < NS; ++m) g3[m] = scaled_plus(rhs[m], scale, (c31 * g1[m] + c32 * g2[m]) / dt);
      solve_block<NS>(jac, lu, indx, gi, g3);
      for (int m = 0; m < NS; ++m) scaled(rhs[m], scale);
      for (int m = 0; m < NS; ++m) g4[m] = rhs[m] + (c41 * g1[m] + c42 * g2[m] + c43 * g3[m]) / dt;
      solve_block<NS>(jac, lu, indx, gi, g4);
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
    left = steps > 0 && iter < maxsteps && (iter >= steps || __popcll(__ballot(1)) < LANES_FULL);
    if (left) break;
  }
  st.t_end = time;
  st.dt_next = st.done ? dtnext : dt;
  return left;
}

template <int NS, class LU, bool CP, class Rhs>
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
  int finish;
  const bool left = rosenbrock_cell_block<NS, LU, CP>(f, wv, tg, dt0, t0, A.time_end[r], A.maxsteps, A.maxtry, A.tol, st,
                                                      A.left.n ? LANE_STEPS : 0, finish);
#pragma unroll
  for (int m = 0; m < NV; ++m) A.w[(long)m * nb + r] = wv[m];
  A.tg[r] = tg;
  if (left) {
    A.left.time[r] = st.t_end;
    A.left.dt[r] = st.dt_next;
    A.left.nacc[r] = st.nacc;
    A.left.nrej2[r] = 2 * st.nrej + finish;
    A.left.list[atomicAdd(A.left.n, 1u)] = r;
    return;
  }
  if (A.nacc) A.nacc[r] = st.nacc;
  if (A.nrej) A.nrej[r] = st.nrej;
  if (A.t_done) {
    A.t_done[r] = st.done ? A.time_end[r] : st.t_end;
    A.dt_next[r] = st.dt_next;
  }
}

// 3 waves per SIMD up to 9 species, 2 beyond: every lane spills, and more resident waves
// hide the latency (2^19 reactors of 9 species at 1, 2, 3, 4 waves: 171k, 257k, 283k, 234k solves/s).
// A batch that cannot fill them runs the narrow instance, whose lanes spill less (65536 reactors of 9
// species, 6 steps: 2.52 ms narrow, 2.66 wide; form 1 2.71 and 3.05).  The two are compiled in
// separate translation units: device functions that both called would get one register budget for
// both (2.5 times the time, wide).
template <int NS, bool NARROW>
constexpr int lane_waves() { return NARROW ? 1 : NS <= 9 ? 3 : 2; }
template <int NS, int LO, int MODE, bool CP, bool NARROW>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(lane_waves<NS, NARROW>())))
reactor_lane_kernel(ReactorArgs A) {
  using LU = std::conditional_t<MODE == 1, float, double>;
  constexpr int WHICH = CP ? (TH_CP | TH_CPH) : (TH_CV | TH_CVH);
  __shared__ double tlds[thermo_lds_doubles<NS>(WHICH)];
  if (*(volatile unsigned *)A.next < LANES_TAKE) return;   // the rows take the batch
  const ThermoLds TL = thermo_stage<NS, LO>(A.th, tlds, WHICH);
  __syncthreads();
  const long nb = A.nbatch;
  for (;;) {
    const unsigned r = atomicAdd(A.next, 1u) - LANES_TAKE;
    if ((long)r >= nb) break;
    const LaneRhs<NS, LO, CP> f{A.K, TL, A.mw, A.rgas, CP ? A.pressure[r] : 0.0, A.tol_iter_nr};
    integrate_one<NS, LU, CP>(f, A, r);
  }
}

template <int NS, int LO, int MODE, bool CP, bool NARROW>
inline void reactor_lanes_launch(const ReactorArgs &A, int ncu, int wg_per_cu, hipStream_t st) {
  if constexpr (MODE == 2 || NS <= LANES_NS) {
    // a workgroup is one wave per SIMD: an instance needs as many per CU as its waves
    const int g = reactor_grid(ncu, wg_per_cu, lane_waves<NS, NARROW>(), 256, A.nbatch);
    reactor_lane_kernel<NS, LO, MODE, CP, NARROW><<<g, 256, 0, st>>>(A);
  }
}

// The batch for any N_S and NASA range; form 1 beyond 9 species stays with the rows.
template <bool CP, bool NARROW>
int reactor_lanes_dispatch(int n_s, int indx_cp_l, int indx_cp_r, const ReactorArgs &A, int ncu, int wg_per_cu,
                           hipStream_t st) {
  if (A.mode == 2) {
    STREAMS_DISPATCH_NS(n_s, STREAMS_DISPATCH_NASA(indx_cp_l, indx_cp_r,
                                                   (reactor_lanes_launch<NS, LO, 2, CP, NARROW>(A, ncu, wg_per_cu, st))));
  } else {
    STREAMS_DISPATCH_NS(n_s, STREAMS_DISPATCH_NASA(indx_cp_l, indx_cp_r,
                                                   (reactor_lanes_launch<NS, LO, 1, CP, NARROW>(A, ncu, wg_per_cu, st))));
  }
  return hip_status();
}

}  // namespace streams
