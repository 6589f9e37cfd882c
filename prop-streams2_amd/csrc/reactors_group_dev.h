// reactors_group_dev.h — the species-block Rosenbrock integrator of the reactor batch with a
// 16-lane row of a wave per reactor.
//
// Same method and the same operations in the same order as rosenbrock_cell_block
// (reactors_lanes_dev.h: the ROS4 cell with a one-sided species Jacobian), laid out across lanes:
//   * lane n evaluates the right-hand side perturbed in species n, lane NS the unperturbed
//     one, so a step's N_S + 1 right-hand sides run side by side;
//   * lane m holds component m of every vector (state, stages) and row m of the matrix, so
//     nothing is indexed dynamically and little spills (0.3-0.4 KB a lane): one lane per reactor
//     keeps the Jacobian, its factors and the stages in 1.2-4.5 KB of scratch per lane, whose
//     traffic bounds it (FP64 units 5-8 % busy);
//   * a component reaches the other lanes by row_newbcast DPP moves; the Jacobian is
//     transposed from columns to rows through LDS, where it stays for a retry of the step.
// Each row takes its next reactor from the work counter as soon as its own is done: the loop
// is over step attempts, so a wave waits for no reactor of another row.  Where lanes began the batch,
// the rows take the reactors that they left, from the step they had reached.
#pragma once
#include "reactors_dev.h"

namespace streams {

constexpr int GROW = 16;            // lanes per reactor

// v of row lane L.  The move is kept apart from its users by an empty asm: folded into a
// conversion it would become v_cvt_f64_f32_dpp, which does not return the conversion of lane
// L's value here.
template <int L>
__device__ inline int row_bcast(int v) {
  int r = __builtin_amdgcn_update_dpp(0, v, 0x150 + L, 0xf, 0xf, true);
  asm("" : "+v"(r));
  return r;
}
template <int L>
__device__ inline float row_bcast(float v) {
  return __builtin_bit_cast(float, row_bcast<L>(__builtin_bit_cast(int, v)));
}
template <int L>
__device__ inline double row_bcast(double v) {
  const long b = __builtin_bit_cast(long, v);
  const unsigned lo = (unsigned)row_bcast<L>((int)b), hi = (unsigned)row_bcast<L>((int)(b >> 32));
  return __builtin_bit_cast(double, (long)(((unsigned long)hi << 32) | lo));
}

// f(integral_constant) for I = B..E-1, unrolled with I a constant expression
template <int B, int E, class F>
__device__ inline void static_for(const F &f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// v of the row lane `src` (0..15, per lane)
__device__ inline float row_shuffle(float v, int src) { return __shfl(v, src, GROW); }
__device__ inline double row_shuffle(double v, int src) { return __shfl(v, src, GROW); }

// Crout LU with implicit partial pivoting (ludcmp), row l in lane l: the right-looking order
// subtracts the same products from each element in the same order.  perm returns the lane
// whose right-hand side component this row's equation takes; amax: largest magnitude of the
// row's elements beside the N columns.
template <int N, class T>
__device__ inline void row_ludcmp(T *a, int l, int &perm, T amax = 0) {
  const T tiny = (T)1.5e-16;
  perm = l;
  static_for<0, N>([&](auto J) { amax = fabs(a[J]) > amax ? fabs(a[J]) : amax; });
  const unsigned long low = __ballot(l < N && amax < tiny);
  const int sh = (int)(threadIdx.x & 48);
  if ((low >> sh) & 0xffff) return;         // ludcmp's early return on an empty row
  T vv = (T)1 / amax;
  int imax = 0;
  static_for<0, N>([&](auto K) {
    constexpr int k = K;
    const T dum = vv * fabs(a[k]);
    T big = 0;
    static_for<k, N>([&](auto I) {
      const T d = row_bcast<I>(dum);
      if (d >= big) { imax = I; big = d; }
    });
    if (imax != k) {
      const int src = l == k ? imax : (l == imax ? k : l);
      static_for<0, N>([&](auto J) { a[J] = row_shuffle(a[J], src); });
      vv = row_shuffle(vv, src);
      perm = __shfl(perm, src, GROW);
    }
    if (l == k && fabs(a[k]) < tiny) a[k] = tiny;
    if constexpr (k != N - 1) {
      const T inv = (T)1 / row_bcast<k>(a[k]);
      T u[N];
      static_for<k + 1, N>([&](auto J) { u[J] = row_bcast<k>(a[J]); });
      if (l > k) {
        a[k] = a[k] * inv;
        static_for<k + 1, N>([&](auto J) { a[J] = a[J] - a[k] * u[J]; });
      }
    }
  });
}

// lubksb on the rows: b is component l in, x the whole solution out (in every lane)
template <int N, class T>
__device__ inline void row_lubksb(const T *a, int l, int perm, T b, T *x) {
  b = row_shuffle(b, perm);
  bool on = false;
  static_for<0, N - 1>([&](auto J) {
    constexpr int j = J;
    const T bj = row_bcast<j>(b);
    on = on || bj != (T)0;
    const T t = b - a[j] * bj;
    if (l > j && on) b = t;
  });
  static_for<0, N>([&](auto Q) {
    constexpr int i = N - 1 - Q;
    T s = b;
    static_for<i + 1, N>([&](auto J) { s = s - a[J] * x[J]; });
    x[i] = row_bcast<i>(s / a[i]);
  });
}

template <int N, class T>
__device__ inline T own(const T *v, int l) {
  T r = v[0];
  static_for<1, N>([&](auto S) { r = l == S ? v[S] : r; });
  return r;
}

// Solve W g = b for component l of g.  FP32 rows: one refinement against the FP64 residual
// b - W x with W = gi I - J, J's row read from LDS (solve_refined).
template <int N, class LU>
__device__ inline double row_solve(const double *jrow, const LU *a, int l, int perm, double gi, double b) {
  if constexpr (sizeof(LU) == sizeof(double)) {
    double x[N];
    row_lubksb<N, double>(a, l, perm, b, x);
    return own<N>(x, l);
  } else {
    float x32[N];
    row_lubksb<N, float>(a, l, perm, (float)b, x32);
    const double xl = (double)own<N>(x32, l);
    double r = b - gi * xl;
    static_for<0, N>([&](auto J) { r = r + jrow[J * (GROW + 1)] * (double)x32[J]; });
    row_lubksb<N, float>(a, l, perm, (float)r, x32);
    return xl + (double)own<N>(x32, l);
  }
}

// Orders LDS accesses of a wave's lanes: what was written before it is read after it.
__device__ inline void row_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int QMAX = 64;            // reactions whose rates a row keeps at once

// The order in which a row's lanes take the reactions: fall-off forms first, then third-body
// ones, then the others, so that the lanes of a pass share their branches.  All threads call;
// the caller synchronises.  More than QMAX reactions are taken in their own order.
__device__ inline void rate_order(const KinPacked &K, int *order, int *kind) {
  const int n = K.nr < QMAX ? K.nr : QMAX;
  if ((int)threadIdx.x < n) {
    const int ty = ((const int *)(K.pack + KREC * threadIdx.x))[KI_TY];
    kind[threadIdx.x] = K.nr > QMAX ? 0 : (ty > 2 ? 2 : ty);
  }
  __syncthreads();
  if ((int)threadIdx.x < n) {
    const int k = kind[threadIdx.x];
    int rank = 0;
    for (int q = 0; q < n; ++q) rank += kind[q] > k || (kind[q] == k && q < (int)threadIdx.x) ? 1 : 0;
    order[rank] = threadIdx.x;
  }
}

// chemistry_source_packed of one state with a reaction per lane: c is species l's
// concentration, the result component l of the source.  The rates meet in LDS and lane l
// subtracts them in ascending order.
template <int NS>
__device__ inline double row_source(const KinPacked &K, double tt, double c, double *cl, double *ql, const int *order,
                                    int l) {
  const double Rtti = 1.0 / (K.r_univ * tt);
  const double lnT = log(tt);
  int itt = (int)((tt - K.t_min_tab) / K.dt_tab) + 1;
  itt = itt < 1 ? 1 : itt;
  itt = itt > K.num_t_tab ? K.num_t_tab : itt;
  const double ttleft = (itt - 1) * K.dt_tab + K.t_min_tab;
  const double dtt = (tt - ttleft) / K.dt_tab;
  const long ntab = (long)K.num_t_tab + 1;
  double acc = 0.0;
  cl[l] = c;
  for (int r0 = 0; r0 < K.nr; r0 += QMAX) {
    const int n = K.nr - r0 < QMAX ? K.nr - r0 : QMAX;
    row_sync();
    for (int i = l; i < n; i += GROW) {
      const int q = order[i], r = r0 + q;
      const double *R = K.pack + KREC * r;
      ql[q] = reaction_progress<NS>(R, (const int *)R, K.kc_tab + (itt - 1) + ntab * r, tt, lnT, Rtti, dtt,
                                    [&](int s) { return cl[s]; }, [&](int s) { return cl[s]; });
    }
    row_sync();
    const double *net = K.pack + KREC * r0 + KD_NET + l;
#pragma unroll 4
    for (int k = 0; k < n; ++k) acc = acc - ql[k] * net[KREC * k];
  }
  row_sync();
  return acc;
}

template <int NS, int LO, int MODE, bool CP>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NS <= 9 ? 3 : 2))) reactor_group_kernel(ReactorArgs A) {
  using LU = std::conditional_t<MODE == 1, float, double>;
  static_assert(NS < GROW, "a row holds the N_S columns and the base state");
  constexpr int WHICH = CP ? (TH_CP | TH_CPH) : (TH_CV | TH_CVH);
  constexpr double safety = 0.9, grow = 1.5, pgrow = -0.25, shrnk = 0.5, pshrnk = -1.0 / 3.0, errcon = 0.1296;
  constexpr double gam = 1.0 / 2.0, a21 = 2.0, a31 = 48.0 / 25.0, a32 = 6.0 / 25.0;
  constexpr double c21 = -8.0, c31 = 372.0 / 25.0, c32 = 12.0 / 5.0;
  constexpr double c41 = -112.0 / 125.0, c42 = -54.0 / 125.0, c43 = -2.0 / 5.0;
  constexpr double b1 = 19.0 / 9.0, b2 = 1.0 / 2.0, b3 = 25.0 / 108.0, b4 = 125.0 / 108.0;
  constexpr double e1 = 17.0 / 54.0, e2 = 7.0 / 36.0, e3 = 0.0, e4 = 125.0 / 108.0;
  __shared__ double tlds[thermo_lds_doubles<NS>(WHICH)];
  __shared__ double jbuf[256 / GROW][NS * (GROW + 1)];
  __shared__ double cbuf[256 / GROW][GROW + QMAX];
  __shared__ int order[QMAX], kind[QMAX];
  __shared__ double lane_conc[NS * 256];
  // What the lanes took is theirs but for the reactors they left.  Read before any row asks the
  // counter in its turn: 16384 rows asking would cost 0.2 ms.
  long nb_rows = A.nbatch;
  bool rest = false;
  if ((MODE == 2 || NS <= LANES_NS) && *(volatile unsigned *)A.next >= LANES_TAKE) {
    rest = true;
    nb_rows = A.left.n ? *(volatile unsigned *)A.left.n : 0;
    if ((long)blockIdx.x * (256 / GROW) >= nb_rows) return;
  }
  unsigned *const counter = rest ? A.left.n + 1 : A.next;
  const ThermoLds TL = thermo_stage<NS, LO>(A.th, tlds, WHICH);
  rate_order(A.K, order, kind);
  __syncthreads();
  const int l = threadIdx.x % GROW;
  double *J = jbuf[threadIdx.x / GROW];
  double *cl = cbuf[threadIdx.x / GROW], *ql = cl + GROW;
  const double mwl = A.mw[l < NS ? l : 0];
  const long nb = A.nbatch;
  const double itol = 1.0 / A.tol;
  bool active = false, fresh = true;
  unsigned r = 0;
  double w = 0.0, wsav = 0.0, rhs_sav = 0.0;       // component l
  double mom[4] = {0.0, 0.0, 0.0, 0.0};            // momentum and energy (enthalpy): constant
  double tg = 0.0, t0 = 0.0, time = 0.0, dt = 0.0, time_end = 0.0, pres = 0.0;
  int iter = 0, jtry = 0, finish = 0, nacc = 0, nrej = 0;
  auto rhs_fn = [&]() {
    if constexpr (CP) return RosRhsPressure<NS, LO>{A.K, TL, A.mw, A.rgas, pres, A.tol_iter_nr};
    else return RosRhsPacked<NS, LO>{A.K, TL, A.mw, A.tol_iter_nr};
  };
  // stage state v (component l): component l of its right-hand side, unscaled, and the scale
  auto rhs_stage = [&](double v, double &scale) {
    double wv[NS + 4], rho, ri;
    v = v > 0.0 ? v : 0.0;
    static_for<0, NS>([&](auto S) { wv[S] = row_bcast<S>(v); });
    static_for<0, 4>([&](auto S) { wv[NS + S] = mom[S]; });
    rhs_fn().prepare(wv, tg, rho, ri, scale);
    return -row_source<NS>(A.K, tg, rho * (v * ri) / mwl, cl, ql, order, l);
  };
  // scale * r + x
  auto scaled_plus = [&](double r, double scale, double x) { return CP ? fma(r, scale, x) : r + x; };
  for (;;) {
    if (!active) {
      unsigned q = 0;
      if (l == 0) q = atomicAdd(counter, 1u);
      r = (unsigned)row_bcast<0>((int)q);
      if ((long)r >= nb_rows) break;
      if (rest) r = A.left.list[r];
      if (l < NS) w = A.w[(long)l * nb + r];
      static_for<0, 4>([&](auto S) { mom[S] = A.w[(long)(NS + S) * nb + r]; });
      tg = A.tg[r];
      time_end = A.time_end[r];
      if (CP) pres = A.pressure[r];
      time = 0.0;
      dt = A.dttry[r];
      nacc = nrej = finish = 0;
      iter = 1;
      fresh = active = true;
      if (rest) {
        time = A.left.time[r];
        dt = A.left.dt[r];
        nacc = A.left.nacc[r];
        nrej = A.left.nrej2[r] >> 1;
        finish = A.left.nrej2[r] & 1;
        iter = nacc + 1;
      } else if (A.t_done) {
        time = A.t_done[r];
        if (A.dt_next[r] > 0.0) dt = A.dt_next[r];
        if (time >= time_end) {                      // finished earlier: nothing to do
          if (l == 0 && A.nacc) A.nacc[r] = 0;
          if (l == 0 && A.nrej) A.nrej[r] = 0;
          active = false;
        } else if (dt * 1.5 > time_end - time) {
          dt = time_end - time;
          finish = 1;
        }
      }
      if (!active) continue;
    }
    if (fresh) {
      t0 = time;
      w = w > 0.0 ? w : 0.0;
      double wv[NS + 4], rp[NS];
      static_for<0, NS>([&](auto S) { wv[S] = row_bcast<S>(w); });
      static_for<0, 4>([&](auto S) { wv[NS + S] = mom[S]; });
      const double h = w * 1.0e-06 + 1.0e-14;
      double rho, ri, sc;
      rhs_fn().prepare(wv, tg, rho, ri, sc);
      double tj = tg;
      static_for<0, NS>([&](auto S) { wv[S] = l == S ? w + h : wv[S]; });
      const double scale = rhs_fn()(wv, tj, rp, l >= NS, lane_conc + threadIdx.x, 256);
      static_for<0, NS>([&](auto M) {
        const double base = row_bcast<NS>(CP ? rp[M] * scale : rp[M]);
        if (l == M) rhs_sav = base;
        const double jm = (CP ? fma(rp[M], scale, -base) : rp[M] - base) / h;
        if (l < NS) J[M + (GROW + 1) * l] = jm;
      });
      row_sync();
      wsav = w;
      jtry = 1;
      fresh = false;
    }
    const double gi = 1.0 / (gam * dt);
    const double *jrow = J + (l < NS ? l : 0);
    LU a[NS];
    static_for<0, NS>([&](auto C) {
      const double j = jrow[C * (GROW + 1)];
      a[C] = l == C ? (LU)(gi - j) : (LU)(-j);
    });
    int perm;
    row_ludcmp<NS, LU>(a, l, perm);
    const double g1 = row_solve<NS>(jrow, a, l, perm, gi, rhs_sav);
    time = t0 + dt;
    double scale;
    double rhs = rhs_stage(fma(a21, g1, wsav), scale);
    const double g2 = row_solve<NS>(jrow, a, l, perm, gi, scaled_plus(rhs, scale, c21 * g1 / dt));
    rhs = rhs_stage(fma(a32, g2, fma(a31, g1, wsav)), scale);
    const double g3 = row_solve<NS>(jrow, a, l, perm, gi, scaled_plus(rhs, scale, fma(c31, g1, c32 * g2) / dt));
    if (CP) rhs = rhs * scale;
    opaque(rhs);
    const double g4 = row_solve<NS>(jrow, a, l, perm, gi, rhs + fma(c43, g3, fma(c41, g1, c42 * g2)) / dt);
    w = fma(b4, g4, fma(b3, g3, fma(b2, g2, fma(b1, g1, wsav))));
    const double err = fma(e4, g4, fma(e3, g3, fma(e1, g1, e2 * g2)));
    const double rel = fabs(err / fmax(1.0, fabs(wsav)));
    double errmax = 0.0;
    static_for<0, NS>([&](auto M) { errmax = fmax(errmax, row_bcast<M>(rel)); });
    errmax = errmax * itol;
    double dtnext;
    bool leave = false, done = false;
    if (errmax < 1.0 || finish == 1) {
      if (errmax > errcon) dtnext = safety * dt * pow(errmax, pgrow);
      else dtnext = grow * dt;
      fresh = true;
    } else {
      nrej += 1;
      dtnext = safety * dt * pow(errmax, pshrnk);
      dt = copysign(fmax(fabs(dtnext), shrnk * fabs(dt)), dt);
      if (jtry == A.maxtry) fresh = true;
      jtry += 1;
    }
    if (fresh) {
      nacc += 1;
      const double remaining = time_end - time;
      if (finish == 1 || remaining < 1.0e-12 * time_end) {
        leave = done = true;
      } else {
        if (dtnext * 1.5 > remaining) { dt = remaining; finish = 1; }
        else { dt = dtnext; finish = 0; }
        leave = iter == A.maxsteps;
      }
      iter += 1;
    }
    if (leave) {
      if (l < NS) A.w[(long)l * nb + r] = w;
      if (l == 0) {
        A.tg[r] = tg;
        if (A.nacc) A.nacc[r] = nacc;
        if (A.nrej) A.nrej[r] = nrej;
        if (A.t_done) {
          A.t_done[r] = done ? time_end : time;
          A.dt_next[r] = done ? dtnext : dt;
        }
      }
      active = false;
    }
  }
}

// Launch for any N_S, NASA range and species-block form.  A workgroup integrates 16 reactors
// at a time.
template <bool CP>
int reactor_group_dispatch(int n_s, int indx_cp_l, int indx_cp_r, const ReactorArgs &A, int ncu, int wg_per_cu,
                           hipStream_t st) {
  const int g = reactor_grid(ncu, wg_per_cu, 2, 256 / GROW, A.nbatch);
  if (g <= 0) return STREAMS_E_DIMS;
  if (A.mode == 1) {
    STREAMS_DISPATCH_NS(n_s, STREAMS_DISPATCH_NASA(indx_cp_l, indx_cp_r,
                                                   (reactor_group_kernel<NS, LO, 1, CP><<<g, 256, 0, st>>>(A))));
  } else {
    STREAMS_DISPATCH_NS(n_s, STREAMS_DISPATCH_NASA(indx_cp_l, indx_cp_r,
                                                   (reactor_group_kernel<NS, LO, 2, CP><<<g, 256, 0, st>>>(A))));
  }
  return hip_status();
}

}  // namespace streams
