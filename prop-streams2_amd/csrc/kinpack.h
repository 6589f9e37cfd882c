// kinpack.h — compact per-reaction records of a mechanism's kinetics.
//
// The reference keeps the kinetics as dense tables indexed (reaction, species)
// (arr_a/b/ea(nr,2), falloff_coeffs(nr,5), tb_eff/r_coeffs/p_coeffs(nr,N_S),
// reac_ty/isRev(nr); multideal.F90:2763-2926).  Every cell walks the same reactions in the
// same order, so a reaction's data is wave-uniform: the fused chemistry reads one record
// per reaction through the constant address space, which the compiler turns into scalar
// (SMEM) loads into SGPRs, and touches only the species that take part in the reaction.
//
// One record is KREC doubles (640 bytes):
//   the first 16 doubles hold 32 int32:
//     [0] reac_ty   [1] isRev   [2] n_reac   [3] n_prod
//     [5] 1 when b or Ea of the (low-pressure) rate is nonzero
//     [6] 1 when the Troe T2 term is present (falloff(4) != -3.14)
//     [8..11]  reactant species (0-based), [12..15] product species
//   doubles:
//     [16..18] A, b, Ea of the rate (the low-pressure limit of a fall-off reaction)
//     [19..21] A, b, Ea of the high-pressure limit
//     [22..26] falloff_coeffs(1..5)
//     [28..31] reactant exponents, [32..35] product exponents
//     [36..51] (p_s - r_s) * W_s of species 1..N_S (zero for species the reaction leaves
//              unchanged: subtracting q*0 leaves the accumulator as it is)
//     [52..67] third-body efficiencies of species 1..N_S
#pragma once
#include "common.h"

namespace streams {

constexpr int KREC = 80, KSIDE = 4, KTB = 16;
constexpr int KI_TY = 0, KI_REV = 1, KI_NRE = 2, KI_NPR = 3, KI_ARR = 5, KI_T2 = 6;
constexpr int KI_RE = 8, KI_PR = 12;
constexpr int KD_A = 16, KD_AINF = 19, KD_FC = 22, KD_REX = 28, KD_PEX = 32, KD_NET = 36, KD_TB = 52;

typedef __attribute__((address_space(4))) const double kdouble;
typedef __attribute__((address_space(4))) const int kint;

// The tables the fused chemistry needs beside the packed records.
struct KinPacked {
  const double *pack;     // nr records of KREC doubles
  const double *kc_tab;   // kc_tab(num_t_tab+1, nr)
  int nr, num_t_tab;
  double t_min_tab, dt_tab, r_univ;
};

// c**ex for a stoichiometric exponent.  Exponents other than 1, 2 and 3 go through
// exp(ex ln c) rather than pow: the same value to a few ulp for c > 0 and the same special
// values for c = 0 (0 or inf) and c < 0 (NaN for a fractional exponent), with a fraction of
// pow's register footprint, which the whole chemistry loop would otherwise carry.
__device__ inline double conc_power(double c, double ex) {
  if (ex == 1.0) return c;
  if (ex == 2.0) return c * c;
  if (ex == 3.0) return c * c * c;
  return exp(ex * log(c));
}

// The record's (reactant, product) exponents of species s (0 when s does not take part):
// the values of r_coeffs(lr,s) and p_coeffs(lr,s).
template <int S, class RD, class RI>
__device__ inline void record_coeffs(RD R, RI I, int nre, int npr, double &rr, double &pp) {
  rr = 0.0;
  pp = 0.0;
#pragma unroll
  for (int e = 0; e < KSIDE; ++e) {
    if (e < nre && I[KI_RE + e] == S) rr = R[KD_REX + e];
    if (e < npr && I[KI_PR + e] == S) pp = R[KD_PEX + e];
  }
}

template <int S, int NS>
struct RefSpecies {
  // acc_s -= ((p - r) q) W_s for the species of the reaction
  template <class RD, class RI>
  __device__ static inline void accumulate(RD R, RI I, int nre, int npr, double q, const double *mw, double *acc) {
    double rr, pp;
    record_coeffs<S>(R, I, nre, npr, rr, pp);
    if (rr != 0.0 || pp != 0.0) acc[S] = acc[S] - ((pp - rr) * q) * mw[S];
    RefSpecies<S + 1, NS>::accumulate(R, I, nre, npr, q, mw, acc);
  }
};
template <int NS>
struct RefSpecies<NS, NS> {
  template <class RD, class RI>
  __device__ static inline void accumulate(RD, RI, int, int, double, const double *, double *) {}
};

// Rate of progress of one reaction (REF: see chemistry_source_from).  The record and conc(s) are
// read through the caller's pointers: wave-uniform scalar loads when every lane walks the same
// reaction, vector loads when each lane takes its own.  kc points at K_c's table row.  pick(s)
// is conc(s) where s comes from the record (a register array would be indexed dynamically); a
// side's species are in ascending order.
template <int NS, bool REF = false, class RD, class RI, class Conc, class Pick>
__device__ inline double reaction_progress(RD R, RI I, const double *kc, double tt, double lnT, double Rtti, double dtt,
                                           const Conc &conc, const Pick &pick) {
  constexpr double LN10 = 2.302585092994045684;
  constexpr double ILN10 = 0.434294481903251827651;
  auto arrhenius = [&](int k) {
    if constexpr (REF) return R[k] * pow(tt, R[k + 1]) * exp(-R[k + 2] * Rtti);
    else return R[k] * exp(R[k + 1] * lnT - R[k + 2] * Rtti);
  };
  auto lg = [&](double x) {
    if constexpr (REF) return log10(x);
    else return log(x) * ILN10;
  };
  auto third_body = [&] {
    double tb = 0.0;
#pragma unroll
    for (int s = 0; s < NS; ++s) tb = tb + R[KD_TB + s] * conc(s);
    return tb;
  };
  const int ty = I[KI_TY];
  double kf, tbv = 1.0;
  if (ty <= 1) {
    kf = R[KD_A];
    if constexpr (REF) {
      if (R[KD_A + 1] != 0.0) kf = kf * pow(tt, R[KD_A + 1]);
      if (R[KD_A + 2] != 0.0) kf = kf * exp(-R[KD_A + 2] * Rtti);
    } else {
      if (I[KI_ARR]) kf = kf * exp(R[KD_A + 1] * lnT - R[KD_A + 2] * Rtti);
    }
    if (ty == 1) tbv = third_body();
  } else {
    const double k0 = arrhenius(KD_A), kinf = arrhenius(KD_AINF), tb = third_body();
    const double rpres = k0 * tb / kinf;
    if (ty == 2) {
      kf = kinf * (rpres / (1.0 + rpres));
    } else if (ty == 3) {
      if (rpres < 1e-30) {
        kf = k0 * tb;
      } else {
        double fcent = (1.0 - R[KD_FC]) * exp(-tt / R[KD_FC + 1]) + R[KD_FC] * exp(-tt / R[KD_FC + 2]);
        if (I[KI_T2]) fcent = fcent + exp(-R[KD_FC + 3] / tt);
        fcent = lg(fcent);
        const double coff = -0.4 - 0.67 * fcent;
        const double noff = 0.75 - 1.27 * fcent;
        const double lr10 = lg(rpres);
        const double fo = (lr10 + coff) / (noff - 0.14 * (lr10 + coff));
        double foff;
        if constexpr (REF) foff = pow(10.0, pow(1.0 + pow(fo, 2.0), -1.0) * fcent);
        else foff = exp(LN10 * (fcent / (1.0 + fo * fo)));
        kf = kinf * (rpres / (1.0 + rpres)) * foff;
      }
    } else {
      const double l10 = lg(rpres);
      const double sri = R[KD_FC] * exp(-R[KD_FC + 1] / tt) + exp(-tt / R[KD_FC + 2]);
      double foff;
      if constexpr (REF) foff = R[KD_FC + 3] * pow(sri, 1.0 / (1.0 + pow(l10, 2.0))) * pow(tt, R[KD_FC + 4]);
      else foff = R[KD_FC + 3] * exp(1.0 / (1.0 + l10 * l10) * log(sri)) * exp(R[KD_FC + 4] * lnT);
      kf = kinf * (rpres / (1.0 + rpres)) * foff;
    }
  }
  double kb = 0.0;
  if (I[KI_REV] == 1) {
    const DoublePair k = load_pair(kc);
    kb = kf / (k.a + (k.b - k.a) * dtt);
  }
  auto power = [&](double c, double ex) {
    if constexpr (REF) return ex == 1.0 ? c : pow(c, ex);
    else return conc_power(c, ex);
  };
  double q1 = 1.0, q2 = 1.0;
  const int nre = I[KI_NRE], npr = I[KI_NPR];
#pragma unroll
  for (int e = 0; e < KSIDE; ++e)
    if (e < nre) q1 = q1 * power(pick(I[KI_RE + e]), R[KD_REX + e]);
#pragma unroll
  for (int e = 0; e < KSIDE; ++e)
    if (e < npr) q2 = q2 * power(pick(I[KI_PR + e]), R[KD_PEX + e]);
  return tbv * (kf * q1 - kb * q2);
}

// The same for all lanes, as a scalar.
struct UniformInts {
  const int *p;
  __device__ inline int operator[](int i) const { return __builtin_amdgcn_readfirstlane(p[i]); }
};

// Species source -omega_s W_s accumulated into acc[0..NS) for one cell at temperature tt
// with molar concentrations conc (compute_chemistry_cuf's reaction loop,
// kernels_gpu.F90:9551-9649).
//  * REF = false (the fused RHS and the fast reactor paths): rate constants through
//    A exp(b ln T - Ea/RT), log10(x) = ln(x)/ln(10), 10^x = exp(x ln 10), c^2 = c*c, and the
//    net coefficient (p - r) W_s taken from the record; these identities change results in
//    the last digits only.
//  * REF = true (the plain FP64 reactor integrator, the yardstick of the others): the
//    reference's own forms and operation order (rosenbrock_rhs, :9249-9339): A T^b exp(-Ea/RT)
//    with the b = 0 and Ea = 0 cases skipped, log10, pow(10, .), pow for exponents other
//    than 1, products over the species in ascending order, acc -= ((p - r) q) W_s with
//    mw = W_s.
//  * LDSREC: the records are read from LDS (pack) instead of K.pack.
template <int NS, bool REF, bool LDSREC = false, class Pick>
__device__ inline void chemistry_source_from(const KinPacked &K, double tt, const double *conc, double *acc,
                                             const double *mw, const Pick &pick, const double *pack = nullptr) {
  static_assert(NS <= KTB, "third-body efficiencies of a record hold at most KTB species");
  const double Rtti = 1.0 / (K.r_univ * tt);
  const double lnT = log(tt);
  int itt = (int)((tt - K.t_min_tab) / K.dt_tab) + 1;
  itt = itt < 1 ? 1 : itt;
  itt = itt > K.num_t_tab ? K.num_t_tab : itt;
  const double ttleft = (itt - 1) * K.dt_tab + K.t_min_tab;
  const double dtt = (tt - ttleft) / K.dt_tab;
  const long ntab = (long)K.num_t_tab + 1;
  for (int lr = 0; lr < K.nr; ++lr) {
    auto record = [&] {
      if constexpr (LDSREC) return pack + KREC * lr;
      else return (kdouble *)K.pack + KREC * lr;
    };
    auto R = record();
    auto ints = [&] {
      if constexpr (LDSREC) return UniformInts{(const int *)R};
      else return (kint *)R;
    };
    auto I = ints();
    const double *kp = K.kc_tab + (itt - 1) + ntab * lr;
    if (REF) {
      const double q = reaction_progress<NS, true>(R, I, kp, tt, 0.0, Rtti, dtt, [&](int s) { return conc[s]; }, pick);
      RefSpecies<0, NS>::accumulate(R, I, I[KI_NRE], I[KI_NPR], q, mw, acc);
    } else {
      const double q = reaction_progress<NS>(R, I, kp, tt, lnT, Rtti, dtt, [&](int s) { return conc[s]; }, pick);
#pragma unroll
      for (int s = 0; s < NS; ++s) acc[s] = acc[s] - q * R[KD_NET + s];
    }
  }
}

template <int NS, bool REF = false>
__device__ inline void chemistry_source_packed(const KinPacked &K, double tt, const double *conc, double *acc,
                                               const double *mw = nullptr) {
  chemistry_source_from<NS, REF>(K, tt, conc, acc, mw, [&](int s) { return conc[s]; });
}

// One reaction's record from the dense tables (the layout above); false when a side has more
// than KSIDE species.
template <class Dense>
__device__ inline bool pack_record(double *R, int n_s, int lr, int nr, const Dense &K) {
  for (int q = 0; q < KREC; ++q) R[q] = 0.0;
  int *I = reinterpret_cast<int *>(R);
  I[KI_TY] = K.reac_ty[lr];
  I[KI_REV] = K.isrev[lr];
  int nre = 0, npr = 0;
  bool fits = true;
  for (int s = 0; s < n_s; ++s) {
    const double rr = K.r_co[lr + nr * s], pp = K.p_co[lr + nr * s];
    if (rr != 0.0) {
      if (nre == KSIDE) fits = false;
      else { I[KI_RE + nre] = s; R[KD_REX + nre] = rr; ++nre; }
    }
    if (pp != 0.0) {
      if (npr == KSIDE) fits = false;
      else { I[KI_PR + npr] = s; R[KD_PEX + npr] = pp; ++npr; }
    }
    R[KD_NET + s] = (pp - rr) * K.mw[s];
    R[KD_TB + s] = K.tb_eff[lr + nr * s];
  }
  I[KI_NRE] = nre;
  I[KI_NPR] = npr;
  I[KI_ARR] = (K.arr_b[lr] != 0.0 || K.arr_ea[lr] != 0.0) ? 1 : 0;
  R[KD_A] = K.arr_a[lr];
  R[KD_A + 1] = K.arr_b[lr];
  R[KD_A + 2] = K.arr_ea[lr];
  R[KD_AINF] = K.arr_a[lr + nr];
  R[KD_AINF + 1] = K.arr_b[lr + nr];
  R[KD_AINF + 2] = K.arr_ea[lr + nr];
  for (int q = 0; q < 5; ++q) R[KD_FC + q] = K.falloff[lr + nr * q];
  I[KI_T2] = K.falloff[lr + 3 * nr] != -3.14 ? 1 : 0;
  return fits;
}

// false when a side of a reaction has more than KSIDE species (all threads of the block call)
template <class Dense>
__device__ inline bool sides_fit(int n_s, const Dense &K, int *flag) {
  if (threadIdx.x == 0) *flag = 1;
  __syncthreads();
  for (int lr = threadIdx.x; lr < K.nr; lr += blockDim.x) {
    int nre = 0, npr = 0;
    for (int s = 0; s < n_s; ++s) {
      nre += K.r_co[lr + K.nr * s] != 0.0 ? 1 : 0;
      npr += K.p_co[lr + K.nr * s] != 0.0 ? 1 : 0;
    }
    if (nre > KSIDE || npr > KSIDE) *flag = 0;
  }
  __syncthreads();
  return *flag != 0;
}

}  // namespace streams
