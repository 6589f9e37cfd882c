// reactors_dev.h — device code of the batched reactor integrator (streams_reactor_batch):
// arguments, right-hand sides of the species-block forms and the persistent grid.  Included by
// reactors.hip (the entry point), reactors_group_dev.h and reactors_lanes_dev.h (the kernels).
#pragma once
#include <type_traits>

#include "chem_common.h"
#include "kinpack.h"
#include "thermo_dev.h"

namespace streams {

// rosenbrock_rhs on the packed tables, species rows: rhs returned unscaled (dw_s/dt = scale
// rhs_s; scale is 1 in this constant-volume cell)
template <int NS, int LO>
struct RosRhsPacked {
  const KinPacked &K;
  const ThermoLds &TL;
  const double *mw;
  double tol_iter_nr;
  // the temperature of state wv (species not negative), from the guess tg; density, the
  // factor ri that makes mass fractions of the state, and scale
  __device__ inline void prepare(const double *wv, double &tg, double &rho, double &ri, double &scale) const {
    double yy[NS];
    rho = wv[0];
#pragma unroll
    for (int s = 1; s < NS; ++s) rho = rho + wv[s];
    ri = 1.0 / rho;
    scale = 1.0;
#pragma unroll
    for (int s = 0; s < NS; ++s) yy[s] = wv[s] * ri;
    const double uu = wv[NS] * ri, vv = wv[NS + 1] * ri, ww = wv[NS + 2] * ri;
    const double qq = 0.5 * (uu * uu + vv * vv + ww * ww);
    const double ee = wv[NS + 3] * ri - qq;
    int nrange[NS];
    tg = temperature_from_e_lds<NS, LO>(ee, tg, TL, tol_iter_nr, yy, nrange);
  }
  // fix: tg is the state's temperature already; the lane's concentrations are also kept in
  // cbuf (species stride cst) for the products that a record's species indices pick
  __device__ inline double operator()(double *wv, double &tg, double *rhs, bool fix, double *cbuf, int cst) const {
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
      cbuf[s * cst] = conc[s];
    }
    const double uu = wv[NS] * ri, vv = wv[NS + 1] * ri, ww = wv[NS + 2] * ri;
    const double qq = 0.5 * (uu * uu + vv * vv + ww * ww);
    const double ee = wv[NS + 3] * ri - qq;
    int nrange[NS];
    const double tt = temperature_from_e_lds<NS, LO>(ee, tg, TL, tol_iter_nr, yy, nrange);
    tg = fix ? tg : tt;
    chemistry_source_from<NS, false>(K, tg, conc, acc, nullptr, [&](int s) { return cbuf[s * cst]; });
#pragma unroll
    for (int s = 0; s < NS; ++s) rhs[s] = -acc[s];
    return 1.0;
  }
};

// Constant-pressure adiabatic reactor (the serving workload; the reference's reactor is
// constant-volume).  State: wv = (Y_1..Y_NS, 0, 0, 0, h) with h the mixture enthalpy,
// constant in time; T from the Newton inversion of h on the cp tables, rho = p/(R T),
// dY_s/dt = omega_s W_s / rho: scale = 1 / rho.
template <int NS, int LO>
struct RosRhsPressure {
  const KinPacked &K;
  const ThermoLds &TL;
  const double *mw, *rgas;
  double pres, tol_iter_nr;
  __device__ inline void prepare(const double *wv, double &tg, double &rho, double &yi, double &scale) const {
    double yy[NS];
    double ysum = wv[0];
#pragma unroll
    for (int s = 1; s < NS; ++s) ysum = ysum + wv[s];
    yi = 1.0 / ysum;
    double rmix = 0.0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      yy[s] = wv[s] * yi;
      rmix = rmix + rgas[s] * yy[s];
    }
    int nrange[NS];
    tg = temperature_newton_lds<NS, LO>(wv[NS + 3], tg, TL, TL.cp, TL.cph, tol_iter_nr, yy, nrange);
    rho = pres / (rmix * tg);
    scale = 1.0 / rho;
  }
  __device__ inline double operator()(double *wv, double &tg, double *rhs, bool fix, double *cbuf, int cst) const {
    double yy[NS], conc[NS], acc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) wv[s] = wv[s] > 0.0 ? wv[s] : 0.0;
    double ysum = wv[0];
#pragma unroll
    for (int s = 1; s < NS; ++s) ysum = ysum + wv[s];
    const double yi = 1.0 / ysum;
    double rmix = 0.0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      yy[s] = wv[s] * yi;
      rmix = rmix + rgas[s] * yy[s];
    }
    int nrange[NS];
    const double tt = temperature_newton_lds<NS, LO>(wv[NS + 3], tg, TL, TL.cp, TL.cph, tol_iter_nr, yy, nrange);
    tg = fix ? tg : tt;
    const double rho = pres / (rmix * tg);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      conc[s] = rho * yy[s] / mw[s];
      acc[s] = 0.0;
      cbuf[s * cst] = conc[s];
    }
    chemistry_source_from<NS, false>(K, tg, conc, acc, nullptr, [&](int s) { return cbuf[s * cst]; });
#pragma unroll
    for (int s = 0; s < NS; ++s) rhs[s] = -acc[s];
    return 1.0 / rho;
  }
};

// Reactors that the lanes leave to the rows: r's time, next step (finish: it ends the interval) and
// steps so far, at its own place; the list of them, and two counters (how many, and how many
// the rows have taken).  n null: the lanes integrate every reactor to its end.
struct LaneLeft {
  unsigned *n, *list;
  double *time, *dt;
  int *nacc, *nrej2;              // accepted; 2 * rejected + finish
};

struct ReactorArgs {
  double *w, *tg;                 // w[m * nbatch + b] (SoA), T guess / result
  const double *dttry, *time_end; // per reactor
  int *nacc, *nrej;               // per reactor (may be null)
  double *t_done, *dt_next;       // per reactor, resumable mode (both null: from t = 0)
  unsigned *next;                 // work counter (starts at 0)
  int nbatch, maxsteps, maxtry, mode;   // mode: 0 plain FP64, 1 mixed, 2 FP64 species block
  double tol, tol_iter_nr;
  const double *mw, *rgas;
  const double *pressure;         // per reactor; null: constant volume
  KinPacked K;
  Thermo th;
  LaneLeft left;
};

// Persistent grid: wg_per_cu workgroups per CU (default 4, at least the resident capacity
// of these register-heavy kernels), never more than the batch needs at `per_wg` reactors a
// workgroup.  Any size is correct: reactors are pulled from the shared counter until it runs
// out, so workgroups queued behind the resident ones start after it has run out and exit at
// once.  The occupancy API is not used: its query has returned error 999 after many other
// kernels had been launched in the process.
inline int device_cus() {
  int dev = 0, ncu = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      ncu <= 0) {
    (void)hipGetLastError();
    ncu = 256;
  }
  return ncu;
}

inline int reactor_grid(int ncu, int wg_per_cu, int min_per_cu, int per_wg, long nbatch) {
  long per = wg_per_cu > 0 ? wg_per_cu : 4;
  per = per < min_per_cu ? min_per_cu : per;
  const long need = (nbatch + per_wg - 1) / per_wg;
  const long g = ncu * per;
  return (int)(g < need ? g : need);
}

// the plain FP64 form (reactors_ref_dev.h), compiled in reactors_ref.hip (constant volume) and
// reactors_ref_cp.hip (constant pressure)
int reactor_ref_cv(int n_s, int indx_cp_l, int indx_cp_r, const ReactorArgs &A, int ncu, int wg_per_cu, hipStream_t st);
int reactor_ref_cp(int n_s, int indx_cp_l, int indx_cp_r, const ReactorArgs &A, int ncu, int wg_per_cu, hipStream_t st);

// one lane per reactor (reactors_lanes_dev.h): form 2, and form 1 up to LANES_NS species
int reactor_lanes_cv(int n_s, int indx_cp_l, int indx_cp_r, const ReactorArgs &A, int ncu, int wg_per_cu, hipStream_t st);
int reactor_lanes_cp(int n_s, int indx_cp_l, int indx_cp_r, const ReactorArgs &A, int ncu, int wg_per_cu, hipStream_t st);
int reactor_lanes_cv_wide(int n_s, int indx_cp_l, int indx_cp_r, const ReactorArgs &A, int ncu, int wg_per_cu,
                          hipStream_t st);
int reactor_lanes_cp_wide(int n_s, int indx_cp_l, int indx_cp_r, const ReactorArgs &A, int ncu, int wg_per_cu,
                          hipStream_t st);
constexpr int LANES_NS = 9;
constexpr int LANE_STEPS = 24;                 // steps that the lanes take where they may leave a reactor
constexpr int LANES_NARROW = 65536;            // reactors that the GPU holds at one wave per SIMD
constexpr unsigned LANES_TAKE = 0x80000000u;   // the counter's first value when lanes take the batch

// the species-block forms (reactors_group_dev.h), compiled in reactors_group.hip (constant
// volume) and reactors_group_cp.hip (constant pressure)
int reactor_group_cv(int n_s, int indx_cp_l, int indx_cp_r, const ReactorArgs &A, int ncu, int wg_per_cu, hipStream_t st);
int reactor_group_cp(int n_s, int indx_cp_l, int indx_cp_r, const ReactorArgs &A, int ncu, int wg_per_cu, hipStream_t st);

}  // namespace streams
