// krylov_rows.hip — the Rosenbrock-Krylov integrator with half a wave per cell.
//
// The operations of krylov_cell (krylov.hip) in their order, a component of every vector per
// lane: the right-hand sides take a reaction per lane, the small products read the other
// components from LDS, and nothing is indexed dynamically.  One lane per cell walks some nine right-hand
// sides of the dense tables per step and keeps a (N_S + 4)^2 product in scratch: an 800-cell tube's
// half step 0.49 -> 0.13 ms.  Bounded by the chain of right-hand sides of a step (temperature iteration,
// rate, sum), which no more lanes shorten.
#include "reactors_ref_dev.h"

namespace streams {

constexpr int HW = 32;              // lanes per cell
constexpr int KROWS_BS = 64;
constexpr int KM = 4, KSTAGE = 4;

template <int D>
__device__ inline void inv_block(double *a) {
  double blk[D * D], y[D * D];
  int indx[D];
#pragma unroll
  for (int c = 0; c < D; ++c)
#pragma unroll
    for (int r = 0; r < D; ++r) blk[r + D * c] = a[r + KM * c];
  ludcmp<D>(blk, indx);
#pragma unroll
  for (int c = 0; c < D; ++c) {
#pragma unroll
    for (int r = 0; r < D; ++r) y[r + D * c] = r == c ? 1.0 : 0.0;
    lubksb<D>(blk, indx, y + D * c);
  }
#pragma unroll
  for (int c = 0; c < D; ++c)
#pragma unroll
    for (int r = 0; r < D; ++r) a[r + KM * c] = y[r + D * c];
}

struct KrylovArgs {
  double *w;
  const double *w_aux, *fl_sav;
  Kin K;
  Thermo th;
  double tol_iter_nr, dttry, time_start, time_end;
  int maxsteps;
  Pasr pasr;
  unsigned ncells;
};

template <int NS, int LO>
__global__ void __launch_bounds__(KROWS_BS) __attribute__((amdgpu_waves_per_eu(2))) krylov_rows_kernel(Box b, KrylovArgs A) {
  using X = Idx<NS>;
  constexpr int NV = NS + 4, NL = Nasa<LO>::NL, THCAP = (NL + 2) * NS * TMAXSET + NS * (TMAXSET + 1);
  static_assert(NV <= HW, "a component per lane");
  constexpr double gam = 0.572816062482135, TOL = 1.0e-6, eps = 1.0e-08;
  constexpr double a21 = 0.432364435748567, a31 = -0.514211316876170, a32 = 1.382271144617360;
  constexpr double a41 = -0.514211316876170, a42 = 1.382271144617360, a43 = 0.0;
  constexpr double g21 = -0.602765307997356, g31 = -1.389195789724843, g32 = 1.072950969011413;
  constexpr double g41 = 0.992356412977094, g42 = -1.390032613873701, g43 = -0.440875890223325;
  constexpr double bs[KSTAGE] = {0.194335256262729, 0.483167813989227, 0.0, 0.322496929748044};
  constexpr double bt[KSTAGE] = {-0.217819895945721, 1.03130847478467, 0.186511421161047, 0.0};
  constexpr double alpha[KSTAGE][KSTAGE] = {{0, 0, 0, 0}, {a21, 0, 0, 0}, {a31, a32, 0, 0}, {a41, a42, a43, 0}};
  constexpr double gamc[KSTAGE][KSTAGE] = {{0, 0, 0, 0}, {g21, 0, 0, 0}, {g31, g32, 0, 0}, {g41, g42, g43, 0}};
  extern __shared__ double rec[];
  __shared__ double thbuf[THCAP];
  __shared__ double buf[KROWS_BS / HW][2 * HW];
  __shared__ double dnb[KROWS_BS / HW][HW * GROW];
  __shared__ int flag;
  if (!sides_fit(NS, A.K, &flag)) return;            // krylov_kernel takes the call
  for (int lr = threadIdx.x; lr < A.K.nr; lr += KROWS_BS) pack_record(rec + KREC * lr, NS, lr, A.K.nr, A.K);
  Thermo th = A.th;
  th.cp_coeff = nullptr;
  th = thermo_to_lds<NS>(th, thbuf, THCAP);
  th.lo = LO;
  th.hi = LO + NL - 1;
  __syncthreads();
  const KinPacked K{nullptr, A.K.kc_tab, A.K.nr, A.K.num_t_tab, A.K.t_min_tab, A.K.dt_tab, A.K.r_univ};
  const int l = threadIdx.x % HW, row = threadIdx.x / HW;
  double *vb = buf[row], *ql = vb + HW, *dn = dnb[row];
  const double mwl = A.K.mw[l < NS ? l : 0];
  const long ps = b.pstride(), fs_ = b.fstride();
  // the components of a vector in every lane
  auto gather = [&](double v, double *all) {
    row_sync();
    vb[l] = v;
    row_sync();
    static_for<0, NV>([&](auto M) { all[M] = vb[M]; });
  };
  auto norm2 = [&](const double *all) {
    double s = 0.0;
    static_for<0, NV>([&](auto M) { s = s + all[M] * all[M]; });
    return sqrt(s);
  };
  for (unsigned t = blockIdx.x * (KROWS_BS / HW) + row; t < A.ncells; t += gridDim.x * (KROWS_BS / HW)) {
    const int i = 1 + (int)(t % b.nx), j = 1 + (int)(t / b.nx % b.ny), k = 1 + (int)(t / b.nx / b.ny);
    const long pt = b.p(i, j, k);
    const double zb = A.w_aux[pt + ps * (X::J_Z - 1)];
    if (!(zb > 5.0e-4 && zb < 1.0 - 5.0e-4)) continue;
    double vec = l < NV ? A.w[pt + ps * l] : 0.0;
    const double fls = A.fl_sav && l < NV ? A.fl_sav[t + fs_ * l] : 0.0;
    const double tau_k = A.pasr.on ? A.pasr.tau_k<NS>(A.w_aux, pt, ps, i, j, k) : 0.0;
    double t_iter = A.w_aux[pt + ps * (X::J_T - 1)];
    // kry_rhs of the state with component v in this lane
    auto rhs_of = [&](double v) {
      double all[NV], yy[NS];
      gather(l < NS && !(v > 0.0) ? 0.0 : v, all);
      double rho = all[0];
      static_for<1, NS>([&](auto S) { rho = rho + all[S]; });
      const double ri = 1.0 / rho;
      static_for<0, NS>([&](auto S) { yy[S] = all[S] * ri; });
      const double uu = all[NS] * ri, vv = all[NS + 1] * ri, ww = all[NS + 2] * ri;
      const double qq = 0.5 * (uu * uu + vv * vv + ww * ww);
      const double ee = all[NS + 3] * ri - qq;
      const double tt = temperature_from_e<NS>(ee, t_iter, th, A.tol_iter_nr, yy);
      const double Rtti = 1.0 / (K.r_univ * tt);
      int itt = (int)((tt - K.t_min_tab) / K.dt_tab) + 1;
      itt = itt < 1 ? 1 : itt;
      itt = itt > K.num_t_tab ? K.num_t_tab : itt;
      const double ttleft = (itt - 1) * K.dt_tab + K.t_min_tab;
      const double dtt = (tt - ttleft) / K.dt_tab;
      row_sync();
      vb[l] = rho * own<NS>(yy, l) / mwl;
      double acc = 0.0;
      for (int r0 = 0; r0 < K.nr; r0 += HW) {
        row_sync();
        if (r0 + l < K.nr)
          ql[l] = row_reaction<NS>(K, rec, r0 + l, tt, Rtti, dtt, itt, vb, dn + GROW * l);
        row_sync();
        const int n = K.nr - r0 < HW ? K.nr - r0 : HW;
        if (l < NS)
#pragma unroll 4
          for (int q = 0; q < n; ++q) {
            const double d = dn[GROW * q + l];
            if (d == d) acc = acc + (d * ql[q]) * mwl;
          }
      }
      if (tau_k > DBL_MIN) {
        gather(acc, all);
        pasr_scale<NS>(tau_k, ri, yy, all);
        acc = l < NS ? own<NS>(all, l) : 0.0;
      }
      row_sync();
      return acc;
    };
    double time = A.time_start, dt = A.dttry, errn = 1.0;
    int it = 0;
    while (time < (A.time_end - 1.0e-12)) {
      dt = dt < A.time_end - time ? dt : A.time_end - time;
      it = it + 1;
      // Arnoldi
      double V[KM + 1], Vb[KM] = {0.0, 0.0, 0.0, 0.0}, HH[(KM + 1) * KM], H[KM * KM], inv[KM * KM], all[NV], sav[NV];
      static_for<0, (KM + 1) * KM>([&](auto Q) { HH[Q] = 0.0; });
      static_for<0, KM * KM>([&](auto Q) { H[Q] = inv[Q] = 0.0; });
      double rhs_sav = rhs_of(vec);
      if (A.fl_sav) rhs_sav = rhs_sav - fls;
      gather(rhs_sav, sav);
      const double nrm = norm2(sav);
      V[0] = rhs_sav / nrm;
      double rpr[KM] = {0.0, 0.0, 0.0, 0.0};
      bool found = false;
      static_for<1, KM + 1>([&](auto KK) {
        constexpr int kk = KK;
        if (found) return;
        double jac = rhs_of(vec + eps * V[kk - 1]);
        if (A.fl_sav) jac = jac - fls;
        jac = (jac - rhs_sav) / eps;
        static_for<1, kk + 1>([&](auto JJ) {
          double va[NV], d = 0.0;
          gather(jac, all);
          gather(V[JJ - 1], va);
          static_for<0, NV>([&](auto M) { d = d + va[M] * all[M]; });
          HH[(JJ - 1) + (KM + 1) * (kk - 1)] = d;
          jac = jac - d * V[JJ - 1];
          // V^T rhs_sav of the newest basis vector
          if constexpr (JJ == kk) {
            double r = 0.0;
            static_for<0, NV>([&](auto M) { r = r + va[M] * sav[M]; });
            rpr[kk - 1] = r;
          }
        });
        gather(jac, all);
        const double hn = norm2(all);
        HH[kk + (KM + 1) * (kk - 1)] = hn;
        V[kk] = jac / hn;
        static_for<1, kk + 1>([&](auto N) {
          static_for<1, kk + 1>([&](auto M) {
            double v = -(dt * gam * HH[(N - 1) + (KM + 1) * (M - 1)]);
            if (N == M) v = v + 1.0;
            H[(N - 1) + KM * (M - 1)] = v;
          });
        });
        static_for<kk + 1, KM + 1>([&](auto N) { H[(N - 1) + KM * (N - 1)] = 1.0; });
        if constexpr (kk == 1) H[0] = 1.0 / H[0];
        else inv_block<kk>(H);
        double lam = 0.0;
        static_for<1, KM + 1>([&](auto JJ) { lam = lam + H[(kk - 1) + KM * (JJ - 1)] * rpr[JJ - 1]; });
        if (fabs(dt * gam * hn) * fabs(lam) < TOL) {
          static_for<0, kk>([&](auto C) { Vb[C] = V[C]; });
          static_for<0, KM * KM>([&](auto Q) { inv[Q] = H[Q]; });
          found = true;
        }
      });
      // B = (Vb (I - inv)) Vb^T, this component's row
      double Am[KM], Bm[NV], Ks[KSTAGE];
      static_for<0, KM>([&](auto Q) {
        double a = Vb[0] * ((Q == 0 ? 1.0 : 0.0) - inv[0 + KM * Q]);
        static_for<1, KM>([&](auto JJ) { a = a + Vb[JJ] * ((JJ == Q ? 1.0 : 0.0) - inv[JJ + KM * Q]); });
        Am[Q] = a;
      });
      static_for<0, KM>([&](auto JJ) {
        gather(Vb[JJ], all);
        static_for<0, NV>([&](auto M) { Bm[M] = JJ == 0 ? Am[0] * all[M] : Bm[M] + Am[JJ] * all[M]; });
      });
      static_for<0, KSTAGE>([&](auto II) {
        constexpr int ii = II;
        double ys = vec, GK = 0.0;
        static_for<0, ii>([&](auto JJ) { ys = ys + dt * alpha[ii][JJ] * Ks[JJ]; });
        double F = rhs_of(ys);
        static_for<0, ii>([&](auto JJ) { GK = GK + gamc[ii][JJ] / gam * Ks[JJ]; });
        F = F + GK;
        if (A.fl_sav) F = F - fls;
        gather(F, all);
        double c = Bm[0] * all[0];
        static_for<1, NV>([&](auto M) { c = c + Bm[M] * all[M]; });
        Ks[ii] = F - c - GK;
      });
      double s = vec, tq = vec;
      static_for<0, KSTAGE>([&](auto II) {
        s = s + dt * bs[II] * Ks[II];
        tq = tq + dt * bt[II] * Ks[II];
      });
      const double e = (tq - s) / ((1.0e-4) * s + 1.0e-8);
      gather(e, all);
      double err2 = 0.0;
      static_for<0, NV>([&](auto M) { err2 = err2 + all[M] * all[M]; });
      const double errmax = sqrt(err2);
      double fac = 0.625 * pow(errn, 0.1) / pow(errmax, 0.175);
      fac = fac > 0.2 ? fac : 0.2;
      fac = fac < 5.0 ? fac : 5.0;
      const double dtnext = dt * fac;
      if (errmax < 1.0) {
        time = time + dt;
        vec = s;
        double yy[NS];
        gather(vec, all);
        double rho = all[0];
        static_for<1, NS>([&](auto S) { rho = rho + all[S]; });
        const double ri = 1.0 / rho;
        static_for<0, NS>([&](auto S) { yy[S] = all[S] * ri; });
        const double uu = all[NS] * ri, vv = all[NS + 1] * ri, ww = all[NS + 2] * ri;
        const double qq = 0.5 * (uu * uu + vv * vv + ww * ww);
        const double ee = all[NS + 3] * ri - qq;
        t_iter = temperature_from_e<NS>(ee, t_iter, th, A.tol_iter_nr, yy);
      }
      dt = dtnext;
      errn = errmax;
      if (it > A.maxsteps) break;
    }
    if (l < NV) A.w[pt + ps * l] = vec;
  }
}

int krylov_rows(int n_s, const Box &b, double *w, const double *w_aux, const Kin &K, const Thermo &th,
                double tol_iter_nr, double dttry, double time_start, double time_end, int maxsteps,
                const double *fl_sav, const Pasr &pasr, hipStream_t st) {
  const KrylovArgs A{w, w_aux, fl_sav, K, th, tol_iter_nr, dttry, time_start, time_end, maxsteps, pasr,
                     (unsigned)b.fstride()};
  const int g = reactor_grid(device_cus(), 8, 8, KROWS_BS / HW, b.fstride());
  const long bytes = (long)K.nr * KREC * 8;
  STREAMS_DISPATCH_NS(n_s, STREAMS_DISPATCH_NASA(th.lo, th.hi,
                                                 (krylov_rows_kernel<NS, LO><<<g, KROWS_BS, bytes, st>>>(b, A))));
  return hip_status();
}

}  // namespace streams
