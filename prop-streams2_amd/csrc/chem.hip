// chem.hip — finite-rate chemistry source and the per-cell Rosenbrock integrator (FP64).
//
// compute_chemistry: one thread per interior cell; the tables come in their Fortran layout
// (arr_a(nr,2), tb_eff(nr,N_S), kc_tab(num_t_tab+1,nr), ...).
// rosenbrock: rosenbrock_kernel with its central-difference Jacobian and Crout LU, a row of lanes
// per cell (rosenbrock.hip) or, for tables that do not fit its records, one thread per cell.
#include "chem_common.h"
#include "kinpack.h"
#include "thermo_dev.h"

namespace streams {

// The reference's dense tables are packed into one record per reaction in LDS (kinpack.h) once
// per workgroup, each of which takes many cells: walking the dense rows costs a uniform branch
// per species and side of every reaction (96x72x60 cells, 9 species and 21 reactions 0.29 ms dense,
// 0.17 packed; 14 species and 29 reactions 0.65 and 0.33), bounded by the exponentials and powers of the
// reference's rate forms, which both walks keep: folding b ln T into one exponential with -Ea/RT takes
// 0.04 ms off but has 1.2 to 1.4 times the error.
// PACKED = false walks the dense tables: a mechanism with more records than LDS holds, or with a
// side of more than KSIDE species, for which both are launched and each looks whether the call is its
// own (checked; 3 to 9 us in small fields).  In a kernel of its own, because its registers would halve
// the waves of the packed walk and a loop over cells its own: 160^3 cells, 14 species and 87 reactions
// 27.4 ms together, 15.0 apart; 9 species with a side of five 2.81 and 2.31.
// LO: NASA form of the tables staged in LDS, 99: any other form, from global memory.
template <int NS, int LO, bool PACKED>
__global__ void __launch_bounds__(256) chemistry_kernel(Box b, double *__restrict__ w, double *__restrict__ w_aux,
                                                        double *__restrict__ fl, Kin K, Thermo th,
                                                        double tol_iter_nr, unsigned ncells, bool checked) {
  using X = Idx<NS>;
  constexpr bool STAGED = LO != 99;
  extern __shared__ double rec[];
  __shared__ double tlds[STAGED ? thermo_lds_doubles<NS>(TH_CV | TH_CVH) : 1];
  __shared__ int flag;
  ThermoLds TL{};
  if constexpr (PACKED) {
    if (threadIdx.x == 0) flag = 1;
    __syncthreads();
    if constexpr (STAGED) TL = thermo_stage<NS, LO>(th, tlds, TH_CV | TH_CVH);
    for (int lr = threadIdx.x; lr < K.nr; lr += 256)
      if (!pack_record(rec + KREC * lr, NS, lr, K.nr, K)) flag = 0;
    __syncthreads();
    if (flag == 0) return;
  } else {
    if (checked && sides_fit(NS, K, &flag)) return;
  }
  const long ps = b.pstride(), fs_ = b.fstride(), ntab = (long)K.num_t_tab + 1;
  // the dense walk takes one cell a thread: about a loop, the constants of its exponentials
  // would be kept in registers throughout
  for (unsigned t = blockIdx.x * 256u + threadIdx.x; t < ncells; t += gridDim.x * 256u) {
    const long pt = b.p(1 + (int)(t % b.nx), 1 + (int)(t / b.nx % b.ny), 1 + (int)(t / b.nx / b.ny));
    double yy[NS], conc[NS], acc[NS];
    double rho = 0.0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      double v = w[pt + ps * s];
      if (!(v > 0.0)) { v = 0.0; w[pt + ps * s] = 0.0; }
      yy[s] = v;
      rho = (s == 0) ? v : rho + v;
    }
    const double ri = 1.0 / rho;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      yy[s] = yy[s] * ri;
      w_aux[pt + ps * s] = yy[s];
      conc[s] = rho * yy[s] / K.mw[s];
      acc[s] = PACKED ? 0.0 : fl[t + fs_ * s];
    }
    const double uu = w[pt + ps * (X::I_U - 1)] * ri, vv = w[pt + ps * (X::I_V - 1)] * ri;
    const double ww = w[pt + ps * (X::I_W - 1)] * ri, rhoe = w[pt + ps * (X::I_E - 1)];
    const double qq = 0.5 * (uu * uu + vv * vv + ww * ww);
    const double ee = rhoe * ri - qq;
    const double t0 = w_aux[pt + ps * (X::J_T - 1)];
    double tt;
    if constexpr (STAGED) {
      int nrange[NS];
      tt = temperature_from_e_lds<NS, LO>(ee, t0, TL, tol_iter_nr, yy, nrange);
    } else {
      tt = temperature_from_e<NS>(ee, t0, th, tol_iter_nr, yy);
    }
    w_aux[pt + ps * (X::J_T - 1)] = tt;
    const double Rtti = 1.0 / (K.r_univ * tt);
    int itt = (int)((tt - K.t_min_tab) / K.dt_tab) + 1;
    itt = itt < 1 ? 1 : itt;
    itt = itt > K.num_t_tab ? K.num_t_tab : itt;
    const double dtt = (tt - ((itt - 1) * K.dt_tab + K.t_min_tab)) / K.dt_tab;
    for (int lr = 0; lr < K.nr; ++lr) {
      if constexpr (PACKED) {
        const double *R = rec + KREC * lr;
        auto c = [&](int s) { return conc[s]; };
        const double q = reaction_progress<NS, true>(R, UniformInts{(const int *)R}, K.kc_tab + (itt - 1) + ntab * lr,
                                                     tt, 0.0, Rtti, dtt, c, c);
#pragma unroll
        for (int s = 0; s < NS; ++s) acc[s] = acc[s] - q * R[KD_NET + s];
      } else {
        const double q = progress_rate<NS>(K, lr, tt, Rtti, itt, dtt, conc);
#pragma unroll
        for (int s = 0; s < NS; ++s) acc[s] = acc[s] - (K.p_co[lr + K.nr * s] - K.r_co[lr + K.nr * s]) * q * K.mw[s];
      }
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) fl[t + fs_ * s] = PACKED ? fl[t + fs_ * s] + acc[s] : acc[s];
    if constexpr (!PACKED) break;
  }
}

// workgroups of the packed walk: each packs the tables once, so no more than fill the GPU
constexpr long CHEM_BLOCKS = 1024;
constexpr long CHEM_LDS = 48 * 1024;         // bytes of records at most, beside up to 8 KB of NASA tables

template <int NS, int LO>
void chemistry_launch(const Box &b, double *w, double *w_aux, double *fl, const Kin &K, const Thermo &th, double tol,
                      unsigned n, hipStream_t st) {
  const long g = ((long)n + 255) / 256, bytes = (long)K.nr * KREC * 8;
  const bool packed = K.nr > 0 && bytes <= CHEM_LDS;
  if (packed)
    chemistry_kernel<NS, LO, true><<<(unsigned)(g < CHEM_BLOCKS ? g : CHEM_BLOCKS), 256, bytes, st>>>(b, w, w_aux, fl, K,
                                                                                                     th, tol, n, true);
  chemistry_kernel<NS, 99, false><<<(unsigned)g, 256, 0, st>>>(b, w, w_aux, fl, K, th, tol, n, packed);
}

// ------------------------------------------------------------------ Rosenbrock
int rosenbrock_rows(int n_s, const Box &b, double *w, double *w_aux, const Kin &K, const Thermo &th,
                    double tol_iter_nr, double dttry, double time_start, double time_end, int maxsteps, int maxtry,
                    double tol, const Pasr &pasr, hipStream_t st);
// Cells up to which rows are no slower where every cell takes one step: the time of the rows grows with the
// cells, that of one lane per cell only once the GPU is full.  One lane -> rows, ms: 9 species 24576
// cells 2.62 -> 1.71, 40960 3.15 -> 2.77, 65536 3.41 -> 4.40; 13 species 24576 7.03 -> 6.47, 26624 7.08 ->
// 7.12, 32768 7.30 -> 8.61; 14 species 26624 8.63 -> 7.45, 32768 8.92 -> 9.06, 131072 14.1 -> 35.9.  Where cells
// differ in their steps rows win far beyond (random radical pools, 14 species, 65536 cells 1050 -> 420),
// which the call cannot know.
inline long rows_cells(int n_s) { return n_s <= 9 ? 40960 : 26624; }
constexpr long ROWS_LDS = 36 * 1024;         // bytes of records at most, beside the rows' own 24 KB

// 2 waves per SIMD (the compiler's own choice is 1, with 2.8-3.7 KB of per-lane spills):
// the extra resident wave hides the spill latency (one integration of a 128^3 box at 1500 K,
// 87.3 -> 67.2 ms; 3 waves: 92.9 ms; bit-identical).  rows: rosenbrock_rows was launched and
// takes the call if every side of the reactions fits its records.
template <int NS>
__global__ void __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(2)))
rosenbrock_kernel(Box b, double *__restrict__ w, double *__restrict__ w_aux, Kin K, Thermo th, double tol_iter_nr,
                  double dttry, double time_start, double time_end, int maxsteps, int maxtry, double tol, Pasr pasr,
                  bool rows) {
  using X = Idx<NS>;
  constexpr int NV = NS + 4;
  if (rows) {
    __shared__ int flag;
    if (sides_fit(NS, K, &flag)) return;
  }
  long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= b.fstride()) return;
  int i = 1 + (int)(t % b.nx);
  long r = t / b.nx;
  int j = 1 + (int)(r % b.ny);
  int k = 1 + (int)(r / b.ny);
  const long pt = b.p(i, j, k), ps = b.pstride();
  double wv[NV];
#pragma unroll
  for (int m = 0; m < NV; ++m) wv[m] = w[pt + ps * m];
  double tg = w_aux[pt + ps * (X::J_T - 1)];
  const double tau_k = pasr.on ? pasr.tau_k<NS>(w_aux, pt, ps, i, j, k) : 0.0;
  RosStats st;
  rosenbrock_cell<NS>(K, th, tol_iter_nr, wv, tg, dttry, time_start, time_end, maxsteps, maxtry, tol, st, tau_k);
#pragma unroll
  for (int m = 0; m < NV; ++m) w[pt + ps * m] = wv[m];
  w_aux[pt + ps * (X::J_T - 1)] = tg;
}

}  // namespace streams

using namespace streams;

extern "C" int streams_compute_chemistry(int n_s, int nx, int ny, int nz, int nv, int nv_aux, int ng,
                                         int nreactions, double *w, double *w_aux, double *fl, const double *mw,
                                         const double *arr_a, const double *arr_b, const double *arr_ea,
                                         const double *tb_eff, const double *falloff_coeffs, const int *reac_ty,
                                         const int *isrev, const double *r_coeffs, const double *p_coeffs,
                                         const double *kc_tab, int num_t_tab, double t_min_tab, double dt_tab,
                                         double r_univ, int indx_cp_l, int indx_cp_r, const double *cv_coeff,
                                         int nsetcv, const double *trange, double tol_iter_nr, void *stream) {
  if (nv != n_s + 4 || nv_aux < 2 * n_s + 13 || nreactions < 0) return STREAMS_E_DIMS;
  Box b{nx, ny, nz, ng};
  long n = b.fstride();
  if (n == 0) return 0;
  Kin K{mw, arr_a, arr_b, arr_ea, tb_eff, falloff_coeffs, r_coeffs, p_coeffs, kc_tab, reac_ty, isrev,
        nreactions, num_t_tab, t_min_tab, dt_tab, r_univ};
  Thermo th{cv_coeff, nullptr, trange, nsetcv, indx_cp_l, indx_cp_r};
  // cells are indexed with 32 bits: w, w_aux and fl of more would not fit the memory
  if (n > 0xfff00000l) return STREAMS_E_DIMS;
  const bool staged = indx_cp_r == 4 && nsetcv >= 1 && nsetcv <= TMAXSET;
  hipStream_t st = as_stream(stream);
  if (staged && indx_cp_l == 0) {
    STREAMS_DISPATCH_NS(n_s, (chemistry_launch<NS, 0>(b, w, w_aux, fl, K, th, tol_iter_nr, (unsigned)n, st)));
  } else if (staged && indx_cp_l == -2) {
    STREAMS_DISPATCH_NS(n_s, (chemistry_launch<NS, -2>(b, w, w_aux, fl, K, th, tol_iter_nr, (unsigned)n, st)));
  } else {
    STREAMS_DISPATCH_NS(n_s, (chemistry_launch<NS, 99>(b, w, w_aux, fl, K, th, tol_iter_nr, (unsigned)n, st)));
  }
  return hip_status();
}

extern "C" int streams_rosenbrock(int n_s, int nv, int nv_aux, int nx, int ny, int nz, int ng, double *w,
                                  double *w_aux, const double *fl, const double *mw, int nreactions,
                                  const double *arr_a, const double *arr_b, const double *arr_ea,
                                  const double *tb_eff, const double *falloff_coeffs, const int *reac_ty,
                                  const int *isrev, const double *r_coeffs, const double *p_coeffs,
                                  const double *kc_tab, int num_t_tab, double t_min_tab, double dt_tab,
                                  double r_univ, double tol_iter_nr, const double *cv_coeff, int nsetcv,
                                  const double *trange, int indx_cp_l, int indx_cp_r, double dttry,
                                  double time_start, double time_end, int maxsteps, int maxtry, double tol,
                                  int simpler_splitting, int enable_pasr, double les_c_yoshi, double les_c_mix,
                                  double les_c_eps, const double *dcsidx, const double *detady,
                                  const double *dzitdz, void *stream) {
  (void)fl; (void)simpler_splitting;
  if (nv != n_s + 4 || nv_aux < 2 * n_s + 13 || maxsteps < 1 || maxtry < 1) return STREAMS_E_DIMS;
  if (enable_pasr > 0 && (nv_aux < 2 * n_s + 14 || !dcsidx || !detady || !dzitdz)) return STREAMS_E_DIMS;
  const Pasr pasr{enable_pasr > 0, les_c_yoshi, les_c_mix, les_c_eps, dcsidx, detady, dzitdz};
  Box b{nx, ny, nz, ng};
  long n = b.fstride();
  if (n == 0) return 0;
  Kin K{mw, arr_a, arr_b, arr_ea, tb_eff, falloff_coeffs, r_coeffs, p_coeffs, kc_tab, reac_ty, isrev,
        nreactions, num_t_tab, t_min_tab, dt_tab, r_univ};
  Thermo th{cv_coeff, nullptr, trange, nsetcv, indx_cp_l, indx_cp_r};
  const bool rows = (indx_cp_l == 0 || indx_cp_l == -2) && indx_cp_r == 4 && nreactions >= 0 &&
                    (long)nreactions * KREC * 8 <= ROWS_LDS && n <= rows_cells(n_s);
  hipStream_t st = as_stream(stream);
  if (rows) {
    const int rc = rosenbrock_rows(n_s, b, w, w_aux, K, th, tol_iter_nr, dttry, time_start, time_end, maxsteps,
                                   maxtry, tol, pasr, st);
    if (rc) return rc;
  }
  STREAMS_DISPATCH_NS(n_s, (rosenbrock_kernel<NS><<<blocks_for(n, 128), 128, 0, st>>>(
                                b, w, w_aux, K, th, tol_iter_nr, dttry, time_start, time_end, maxsteps, maxtry,
                                tol, pasr, rows)));
  return hip_status();
}
