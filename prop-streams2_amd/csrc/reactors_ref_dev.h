// reactors_ref_dev.h — rosenbrock_kernel (kernels_gpu.F90:8928-9193) in the reference's own
// arithmetic with a 16-lane row of a wave per cell: the plain FP64 form of the reactor batch and
// the implicit chemistry of a field.
//
// The operations of one cell and their order are those of a lane that integrates it alone
// (central differences over all N_S + 4 variables, each right-hand side's Newton iteration
// started from the temperature of the one before), laid out as in reactors_group_dev.h:
//   * the 2 (N_S + 4) + 1 states of a Jacobian are a state per lane, 16 at a time.  Each lane
//     forms its state's mixture coefficients; the Newton iterations, whose start values form a
//     chain, then run in turn on those sums in every lane; the 16 reaction sources run side by side;
//   * momentum and energy have no source: their Jacobian rows are zero and their stages are zero,
//     so the solves are those of the species block.  Their columns only enter the row maxima of
//     the implicit pivoting, and where one is not finite no component is.
// One lane per cell kept the Jacobian, its factors and the stages in 4.5 to 7 KB of scratch and
// walked 2 (N_S + 4) + 1 right-hand sides one after the other.  Measured, one lane -> a row, same
// bits: 60 constant-pressure reactors of 9 species, 12 steps 65 -> 3.4 ms, of 14 species, 8 steps
// 147 -> 7.1; 200000 reactors of 9 species, 2 steps 64 -> 41; 40000 of 14 species, 8 steps 224 -> 81.
// What bounds it: the reference's powers and exponentials (a right-hand side of 21 reactions is
// about 12000 instructions of a wave) and, in small batches, the chain of Newton iterations.
#pragma once
#include "reactors_group_dev.h"

namespace streams {

constexpr int REF_BS = 64;          // one wave: four cells at a time

struct RefArgs {
  ReactorArgs R;
  // field (FIELD): interior cells of a box
  Box b;
  double *w_aux;
  Kin D;                            // dense tables
  Pasr pasr;
  double dttry, time_start, time_end;
  unsigned ncells;
};

// Rate of progress of reaction r in the reference's forms at the concentrations c (LDS); d gets
// p - r of the species, NaN for those that take no part.
template <int NS>
__device__ inline double row_reaction(const KinPacked &K, const double *pack, int r, double tt, double Rtti, double dtt,
                                      int itt, const double *c, double *d) {
  const double *R = pack + KREC * r;
  const int *I = (const int *)R;
  const double q = reaction_progress<NS, true>(R, I, K.kc_tab + (itt - 1) + ((long)K.num_t_tab + 1) * r, tt, 0.0, Rtti,
                                               dtt, [&](int s) { return c[s]; }, [&](int s) { return c[s]; });
#pragma unroll
  for (int s = 0; s < GROW; ++s) d[s] = __builtin_nan("");
#pragma unroll
  for (int e = 0; e < KSIDE; ++e)
    if (e < I[KI_NRE]) d[I[KI_RE + e]] = -R[KD_REX + e];
#pragma unroll
  for (int e = 0; e < KSIDE; ++e)
    if (e < I[KI_NPR]) {
      const double v = d[I[KI_PR + e]];
      d[I[KI_PR + e]] = v == v ? R[KD_PEX + e] + v : R[KD_PEX + e];
    }
  return q;
}

// row_source in the reference's forms: acc_s -= ((p - r) q) W_s over the species of each reaction.
// dn: 16 x 16 doubles, p - r of species s in reaction k, NaN when it takes no part.
template <int NS>
__device__ inline double row_source_ref(const KinPacked &K, const double *pack, double tt, double c, double mwl,
                                        double *cl, double *ql, double *dn, int l) {
  const double Rtti = 1.0 / (K.r_univ * tt);
  int itt = (int)((tt - K.t_min_tab) / K.dt_tab) + 1;
  itt = itt < 1 ? 1 : itt;
  itt = itt > K.num_t_tab ? K.num_t_tab : itt;
  const double ttleft = (itt - 1) * K.dt_tab + K.t_min_tab;
  const double dtt = (tt - ttleft) / K.dt_tab;
  double acc = 0.0;
  cl[l] = c;
  for (int r0 = 0; r0 < K.nr; r0 += GROW) {
    const int r = r0 + l;
    row_sync();
    if (r < K.nr) {
      ql[l] = row_reaction<NS>(K, pack, r, tt, Rtti, dtt, itt, cl, dn + GROW * l);
    }
    row_sync();
    const int n = K.nr - r0 < GROW ? K.nr - r0 : GROW;
#pragma unroll 4
    for (int k = 0; k < n; ++k) {
      const double d = dn[GROW * k + l];
      if (d == d) acc = acc - (d * ql[k]) * mwl;
    }
  }
  row_sync();
  return acc;
}

// One state's right-hand side but for its temperature: mass fractions, density (constant
// volume) or gas constant (constant pressure) and the energy the Newton iteration inverts.
template <int NS, bool CP>
__device__ inline void ref_state(const double *wv, const double *mom, const double *rgas, double *yy, double &rho,
                                 double &ri, double &ee) {
  double sum = wv[0];
#pragma unroll
  for (int s = 1; s < NS; ++s) sum = sum + wv[s];
  ri = 1.0 / sum;
  if constexpr (CP) {
    double rmix = 0.0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      yy[s] = wv[s] * ri;
      rmix = rmix + rgas[s] * yy[s];
    }
    rho = rmix;
    ee = mom[3];
  } else {
#pragma unroll
    for (int s = 0; s < NS; ++s) yy[s] = wv[s] * ri;
    rho = sum;
    const double uu = mom[0] * ri, vv = mom[1] * ri, ww = mom[2] * ri;
    const double qq = 0.5 * (uu * uu + vv * vv + ww * ww);
    ee = mom[3] * ri - qq;
  }
}

template <int NS, int LO, bool CP, bool FIELD>
__global__ void __launch_bounds__(REF_BS) __attribute__((amdgpu_waves_per_eu(2))) reactor_ref_kernel(RefArgs A) {
  constexpr int NV = NS + 4, NL = Nasa<LO>::NL, NSTATE = 2 * NV + 1, ROWS = REF_BS / GROW, JS = GROW + 1;
  static_assert(NS <= GROW - 1 && NL + 2 <= GROW, "a row holds the species and a state's sums");
  constexpr double safety = 0.9, grow = 1.5, pgrow = -0.25, shrnk = 0.5, pshrnk = -1.0 / 3.0, errcon = 0.1296;
  constexpr double gam = 1.0 / 2.0, a21 = 2.0, a31 = 48.0 / 25.0, a32 = 6.0 / 25.0;
  constexpr double c21 = -8.0, c31 = 372.0 / 25.0, c32 = 12.0 / 5.0;
  constexpr double c41 = -112.0 / 125.0, c42 = -54.0 / 125.0, c43 = -2.0 / 5.0;
  constexpr double b1 = 19.0 / 9.0, b2 = 1.0 / 2.0, b3 = 25.0 / 108.0, b4 = 125.0 / 108.0;
  constexpr double e1 = 17.0 / 54.0, e2 = 7.0 / 36.0, e3 = 0.0, e4 = 125.0 / 108.0;
  constexpr int THCAP = (NL + 2) * NS * TMAXSET + NS * (TMAXSET + 1);
  extern __shared__ double rec[];                    // FIELD: the packed records
  __shared__ double thbuf[THCAP];
  __shared__ double jbuf[ROWS][NV * JS];
  __shared__ double nbuf[ROWS][GROW * GROW];         // a chain's sums, concentrations, or dn
  __shared__ double cbuf[ROWS][2 * GROW];
  __shared__ int flag;
  const ReactorArgs &R = A.R;
  if constexpr (FIELD) {
    if (!sides_fit(NS, A.D, &flag)) return;          // rosenbrock_kernel takes the call
    for (int lr = threadIdx.x; lr < A.D.nr; lr += REF_BS) pack_record(rec + KREC * lr, NS, lr, A.D.nr, A.D);
  }
  Thermo th = R.th;
  if (CP) th.cv_coeff = R.th.cp_coeff;
  th.cp_coeff = nullptr;
  th = thermo_to_lds<NS>(th, thbuf, THCAP);
  th.lo = LO;
  th.hi = LO + NL - 1;
  __syncthreads();
  const int l = threadIdx.x % GROW, row = threadIdx.x / GROW;
  double *J = jbuf[row], *nb_ = nbuf[row], *cl = cbuf[row], *ql = cl + GROW;
  const double *pack = FIELD ? rec : R.K.pack;
  const double mwl = R.mw[l < NS ? l : 0];
  const long nb = FIELD ? (long)A.ncells : (long)R.nbatch;
  const double itol = 1.0 / R.tol;
  bool active = false, fresh = true;
  unsigned r = 0, turn = blockIdx.x * ROWS + row;
  long pt = 0, ps = nb;
  double w = 0.0, wsav = 0.0, rhs_sav = 0.0;         // component l
  double mom[4] = {0.0, 0.0, 0.0, 0.0};              // momentum and energy (enthalpy): constant
  double tg = 0.0, t0 = 0.0, time = 0.0, dt = 0.0, time_end = 0.0, pres = 0.0, tau_k = 0.0;
  int iter = 0, jtry = 0, finish = 0, nacc = 0, nrej = 0;
  // stage state v (component l): component l of its right-hand side, unscaled, and the scale
  auto rhs_stage = [&](double v, double &scale) {
    double wv[NS], yy[NS], rho, ri, ee;
    v = v > 0.0 ? v : 0.0;
    static_for<0, NS>([&](auto S) { wv[S] = row_bcast<S>(v); });
    ref_state<NS, CP>(wv, mom, R.rgas, yy, rho, ri, ee);
    tg = temperature_from_e<NS>(ee, tg, th, R.tol_iter_nr, yy);
    if (CP) rho = pres / (rho * tg);
    double out = -row_source_ref<NS>(R.K, pack, tg, rho * (v * ri) / mwl, mwl, cl, ql, nb_, l);
    scale = CP ? 1.0 / rho : 1.0;
    if (FIELD && tau_k > DBL_MIN) {
      double all[NS];
      static_for<0, NS>([&](auto S) { all[S] = row_bcast<S>(out); });
      pasr_scale<NS>(tau_k, ri, yy, all);
      out = own<NS>(all, l);
    }
    return out;
  };
  // scale * r + x, in one rounding as the products of a lane's own right-hand side are
  auto scaled_plus = [&](double r, double scale, double x) { return CP ? fma(r, scale, x) : r + x; };
  for (;;) {
    if (!active) {
      if constexpr (FIELD) {
        r = turn;
        turn += gridDim.x * ROWS;
      } else {
        unsigned q = 0;
        if (l == 0) q = atomicAdd(R.next, 1u);
        r = (unsigned)row_bcast<0>((int)q);
      }
      if ((long)r >= nb) break;
      pt = r;
      if constexpr (FIELD) {
        using X = Idx<NS>;
        const int i = 1 + (int)(r % A.b.nx), j = 1 + (int)(r / A.b.nx % A.b.ny), k = 1 + (int)(r / A.b.nx / A.b.ny);
        pt = A.b.p(i, j, k);
        ps = A.b.pstride();
        tg = A.w_aux[pt + ps * (X::J_T - 1)];
        tau_k = A.pasr.on ? A.pasr.tau_k<NS>(A.w_aux, pt, ps, i, j, k) : 0.0;
        time = A.time_start;
        time_end = A.time_end;
        dt = A.dttry;
      } else {
        tg = R.tg[r];
        time = 0.0;
        time_end = R.time_end[r];
        dt = R.dttry[r];
        if (CP) pres = R.pressure[r];
      }
      if (l < NS) w = R.w[pt + ps * l];
      static_for<0, 4>([&](auto S) { mom[S] = R.w[pt + ps * (NS + S)]; });
      nacc = nrej = finish = 0;
      iter = 1;
      fresh = active = true;
      if (!FIELD && R.t_done) {
        time = R.t_done[r];
        if (R.dt_next[r] > 0.0) dt = R.dt_next[r];
        if (time >= time_end) {                      // finished earlier: nothing to do
          if (l == 0 && R.nacc) R.nacc[r] = 0;
          if (l == 0 && R.nrej) R.nrej[r] = 0;
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
      // the first species is differenced about its value before clipping, as the reference's
      // loop restores it after the calls that clip the others
      const double raw0 = row_bcast<0>(w);
      w = w > 0.0 ? w : 0.0;
      double wv[NS];
      static_for<0, NS>([&](auto S) { wv[S] = row_bcast<S>(w); });
#pragma unroll 1
      for (int k0 = 0; k0 < NSTATE; k0 += GROW) {
        const int k = k0 + l < NSTATE ? k0 + l : NSTATE - 1;
        const int n = k >> 1;                        // NV: the unperturbed state
        double wtmp = raw0;
        static_for<1, NS>([&](auto S) { wtmp = n == S ? wv[S] : wtmp; });
        static_for<0, 4>([&](auto S) { wtmp = n == NS + S ? mom[S] : wtmp; });
        const double h = wtmp * 1.0e-06 + 1.0e-14;
        const double moved = (k & 1) ? wtmp - h : wtmp + h;
        double ws[NS], ms[4], yy[NS], rho, ri, ee;
        static_for<0, NS>([&](auto S) { ws[S] = n == S ? (moved > 0.0 ? moved : 0.0) : wv[S]; });
        static_for<0, 4>([&](auto S) { ms[S] = n == NS + S ? moved : mom[S]; });
        ref_state<NS, CP>(ws, ms, R.rgas, yy, rho, ri, ee);
        // mixture coefficients in the temperature ranges of tg, good between tlo and thi
        double tlo = -HUGE_VAL, thi = HUGE_VAL, sumb = 0.0, cvl[NL];
        int nr[NS];
        static_for<0, NS>([&](auto S) {
          nr[S] = locate_range<NS>(tg, th, S + 1);
          if (nr[S] > 1) tlo = fmax(tlo, th.trange[S + NS * (nr[S] - 1)]);
          if (nr[S] < th.nsetcv) thi = fmin(thi, th.trange[S + NS * nr[S]]);
          sumb = sumb + cpc<NS>(th.cv_coeff, th, th.hi + 1, S + 1, nr[S]) * yy[S];
        });
        row_sync();
        static_for<0, NL>([&](auto Q) {
          double c = 0.0;
          static_for<0, NS>([&](auto S) { c = c + cpc<NS>(th.cv_coeff, th, LO + Q, S + 1, nr[S]) * yy[S]; });
          nb_[GROW * l + Q] = c;
        });
        nb_[GROW * l + NL] = sumb;
        nb_[GROW * l + NL + 1] = ee;
        row_sync();
        // temperature_from_e of the 16 states in turn
        const int last = NSTATE - k0 < GROW ? NSTATE - k0 : GROW;
        double tk = tg;
#pragma unroll 1
        for (int q = 0; q < last; ++q) {
          const double *c = nb_ + GROW * q;
          const double ebar = c[NL + 1] - c[NL];
          double t_old = tg, tt = tg;
          bool same = true;
          for (int it = 1; it <= 10; ++it) {
            if (!(t_old > tlo && t_old < thi)) { same = false; break; }
            double den = 0.0, num = 0.0;
            static_for<0, NL>([&](auto Q) {
              constexpr int p = LO + Q;
              const double t_pow = ipow(t_old, p);
              const double tnum = p == -1 ? log(t_old) : (t_old * t_pow) / (p + 1.0);
              num = num + c[Q] * tnum;
              den = den + c[Q] * t_pow;
            });
            tt = t_old + (ebar - num) / den;
            if (fabs(tt - t_old) < R.tol_iter_nr) break;
            t_old = tt;
          }
          if (!same) {                               // a range changes: the whole iteration, by its lane
            if (l == q) tt = temperature_from_e<NS>(ee, tg, th, R.tol_iter_nr, yy);
            tt = row_shuffle(tt, q);
          }
          tg = tt;
          tk = l == q ? tt : tk;
        }
        row_sync();
        if (k0 + l >= NSTATE) tk = tg;
        double conc[NS], rhs[NS];
        if (CP) rho = pres / (rho * tk);
        static_for<0, NS>([&](auto S) {
          conc[S] = rho * yy[S] / R.mw[S];
          rhs[S] = 0.0;
          nb_[GROW * S + l] = conc[S];
        });
        auto pick = [&](int s) { return nb_[GROW * s + l]; };
        chemistry_source_from<NS, true, FIELD>(R.K, tk, conc, rhs, R.mw, pick, pack);
        const double back = 1.0 / rho, minus_back = __shfl_xor(back, 1, GROW);
        static_for<0, NS>([&](auto S) { rhs[S] = -rhs[S]; });
        if (FIELD && tau_k > DBL_MIN) pasr_scale<NS>(tau_k, ri, yy, rhs);
        static_for<0, NS>([&](auto M) {
          const double minus = __shfl_xor(rhs[M], 1, GROW);
          const double plus = CP ? rhs[M] * back : rhs[M];
          const double jm = (CP ? fma(-minus, minus_back, plus) : plus - minus) / (2.0 * h);
          if (n < NV && !(k & 1)) J[M + JS * n] = jm;
          if (k0 + l == NSTATE - 1) cl[M] = plus;
        });
      }
      row_sync();
      rhs_sav = l < NS ? cl[l] : 0.0;
      row_sync();
      wsav = w;
      jtry = 1;
      fresh = false;
    }
    const double gi = 1.0 / (gam * dt);
    const double *jrow = J + (l < NS ? l : 0);
    double a[NS], amax = 0.0;
    static_for<0, NS>([&](auto C) {
      const double j = jrow[C * JS];
      a[C] = l == C ? gi - j : -j;
    });
    bool bad = false;
    static_for<NS, NV>([&](auto C) {
      const double j = fabs(jrow[C * JS]);
      amax = j > amax ? j : amax;
      bad = bad || !(j < HUGE_VAL);
    });
    int perm;
    row_ludcmp<NS, double>(a, l, perm, amax);
    // a non-finite entry of those columns makes the momentum and energy pivots, and through their
    // stages every component, not a number
    const bool lost = ((__ballot(l < NS && bad) >> (threadIdx.x & 48)) & 0xffff) != 0;
    double g1 = row_solve<NS>(jrow, a, l, perm, gi, rhs_sav);
    if (lost) g1 = __builtin_nan("");
    time = t0 + dt;
    double scale;
    double rhs = rhs_stage(fma(a21, g1, wsav), scale);
    const double g2 = row_solve<NS>(jrow, a, l, perm, gi, scaled_plus(rhs, scale, c21 * g1 / dt));
    rhs = rhs_stage(fma(a32, g2, fma(a31, g1, wsav)), scale);
    const double g3 = row_solve<NS>(jrow, a, l, perm, gi, scaled_plus(rhs, scale, fma(c31, g1, c32 * g2) / dt));
    const double g4 =
        row_solve<NS>(jrow, a, l, perm, gi, scaled_plus(rhs, scale, fma(c43, g3, fma(c41, g1, c42 * g2)) / dt));
    w = fma(b4, g4, fma(b3, g3, fma(b2, g2, fma(b1, g1, wsav))));
    const double err = fma(e4, g4, fma(e3, g3, fma(e1, g1, e2 * g2)));
    const double rel = fabs(err / fmax(1.0, fabs(wsav)));
    // a stage that is not finite makes the others' components (zero rows) not a number as well
    const double size = fabs(g1) + fabs(g2) + fabs(g3) + fabs(g4);
    if ((__ballot(l < NS && !(size < HUGE_VAL)) >> (threadIdx.x & 48)) & 0xffff)
      mom[0] = mom[1] = mom[2] = mom[3] = __builtin_nan("");
    double errmax = 0.0;
    static_for<0, NS>([&](auto M) { errmax = fmax(errmax, row_bcast<M>(rel)); });
    time = t0 + dt;
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
      if (jtry == R.maxtry) fresh = true;
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
        leave = iter == R.maxsteps;
      }
      iter += 1;
    }
    if (leave) {
      if (l < NS) R.w[pt + ps * l] = w;
      if (l == 0) {
        if (mom[0] != mom[0]) static_for<0, 4>([&](auto S) { R.w[pt + ps * (NS + S)] = mom[S]; });
        if constexpr (FIELD) {
          A.w_aux[pt + ps * (Idx<NS>::J_T - 1)] = tg;
        } else {
          R.tg[r] = tg;
          if (R.nacc) R.nacc[r] = nacc;
          if (R.nrej) R.nrej[r] = nrej;
          if (R.t_done) {
            R.t_done[r] = done ? time_end : time;
            R.dt_next[r] = done ? dtnext : dt;
          }
        }
      }
      active = false;
    }
  }
}

// The batch for any N_S and NASA range.  A wave integrates four reactors at a time, so a quarter
// of the workgroups' lanes of the other forms makes four times their number.
template <bool CP>
int reactor_ref_dispatch(int n_s, int indx_cp_l, int indx_cp_r, const ReactorArgs &R, int ncu, int wg_per_cu,
                         hipStream_t st) {
  const int g = reactor_grid(ncu, 4 * (wg_per_cu > 0 ? wg_per_cu : 4), 8, REF_BS / GROW, R.nbatch);
  if (g <= 0) return STREAMS_E_DIMS;
  RefArgs A{};
  A.R = R;
  STREAMS_DISPATCH_NS(n_s, STREAMS_DISPATCH_NASA(indx_cp_l, indx_cp_r,
                                                 (reactor_ref_kernel<NS, LO, CP, false><<<g, REF_BS, 0, st>>>(A))));
  return hip_status();
}

}  // namespace streams
