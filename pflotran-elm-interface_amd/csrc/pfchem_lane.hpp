// pfchem_lane.hpp -- network-specialized batched reaction step: one cell per
// lane, persistent grid, lane-level work stealing.
//
// This file is device source compiled at run time (hiprtc) after a generated
// `struct Net` that holds one reaction network and its solver options as
// compile-time constants (species counts, species ids, stoichiometry, log K
// or its temperature coefficients, Debye-Hueckel parameters, mineral rate
// parameters, tolerances).  Every index into a cell's Jacobian is therefore a
// constant: the cell's Jacobian stays in registers, the complex and mineral
// loops are straight-line code, and no lane ever reads another lane's data
// (no atomics, no barriers; per-cell values the complex loop does not touch
// wait in the lane's own LDS slots).
//
// Algorithm: RStep (reaction.F90:3564-3738) / RReact (:3742-4055) with
// RTotalAqueous (:4665-4759), RTAccumulation(Derivative) (:5710-5848),
// RKineticMineral (reaction_mineral.F90:647-1078), RImmobileDecay
// (reaction_immobile.F90:244-294), RActivityCoefficients LAG per Newton
// iteration (reaction.F90:4555-4611) and RSolve (:5457-5516,
// back-substituting).  Reformulation of the linear solve (same Newton step,
// different rounding):
//   * in the log formulation the aqueous Jacobian of RReact is
//       J_log = jc (diag(x) + S^T diag(m) S) + sum_m g_m nu_m nu_m^T,
//     jc = phi s 1000 V rho/1000 / dt, with g_m = dIm/dQK QK V rho/1000 >= 0
//     for every TST rate law: symmetric positive definite.  M = J_log / jc is
//     factored as L D L^T without pivoting; the linear formulation solves
//     the same system and multiplies the step by x (J_lin = J_log diag(x)^-1);
//   * immobile rows are diagonal (accumulation + first-order decay); with the
//     SomDec sandbox (networks without complexes and minerals) the system is
//     a sparse unsymmetric one, see PFLANE_SD;
//   * JT = float: the off-diagonal entries are accumulated pre-scaled by
//     1/sqrt(x_i x_j) in FP32 (|entry| <= sqrt(D_i D_j / x_i x_j)), scaled to
//     unit diagonal in FP32 and factored in FP32; the diagonal, totals,
//     residual, log K sums, exponentials, the update and every convergence
//     test stay FP64 (the Newton iteration is the iterative refinement);
//   * a pivot below the tolerance, a non-finite entry, or (FP32) a Newton
//     iteration that does not converge hands the cell, with its inputs
//     untouched, to a later pass: status kEscalate.
// With packed FP32 off, FP32 and FP64 instructions issue at the same rate on
// gfx950, and forming an FP32 entry takes three instructions (multiply,
// convert, FMA) where an FP64 one takes an FMA.  What FP32 saves is registers,
// and only where the system is what fills them: the SomDec step takes 256
// VGPRs + 129 AGPRs against 256 + 222, the step of 15 primaries and 60
// complexes 256 + 160 against 256 + 158, neither with scratch.  There the FP32
// pass also hands over more cells (its pivot test is 1e-6), and the FP64
// kernel is the faster one.  Where the FP32 Newton iteration ends is decided
// by the rounding of its factorization in one cell of a hundred, so its
// arithmetic is left as it is rather than moved to FP64 accumulation or
// another scaling.
#pragma once

namespace pflane {

typedef long long i64;

// pflotran_constants.F90:84, 89; reactive_transport_aux.F90:19
constexpr double kLogToLn = 2.30258509299;
constexpr double kIdealGas = 8.31446;
constexpr double kRtMinSat = 1.0e-40;
constexpr int kEscalate = 16;        // per-cell status: handed to the next pass
constexpr int kClaim = 64;           // cells per refill of a wave's queue
// Waiting lanes that make a wave write back and load.  1,048,576 cells of
// the 15-primary network, 7 iterations a cell: 4.4 ms at 1, 3.7 at 16, 3.6 at
// 24 and 32 (the waiting lanes idle); uneven 262,144 cells 3.6, 3.1, 3.1 ms.
constexpr int kServe = 24;
enum : int { kOk = 0, kMaxIter = 1, kSingular = 2 };
enum : int { kFreqNewtonIter = 2 };

// kernel arguments (by value); the host defines the same layout
struct Args {
  i64 ld, ncell;
  double* pri_molal;
  double* total;
  double* immobile;
  double* sec_molal;
  double* pri_act_coef;
  double* sec_act_coef;
  double* ln_act_h2o;
  double* mnrl_volfrac;
  const double* mnrl_area;
  double* mnrl_rate;
  const double* porosity;
  const double* saturation;
  const double* den_kg;
  const double* volume;
  const double* temperature;
  int* num_iterations;
  int* num_sub_steps;
  int* status;
  unsigned long long* cursors;  // one work cursor per XCD, 128-byte stride
  double dt;
  int nxcd;
  int rescue;    // 1: only cells whose status is kEscalate
  int escalate;  // 1: hand failing cells to a later pass (status kEscalate)
  int list_min;  // with a list: the pass does nothing unless it holds more cells
  const int* list;        // NULL, or the cells to step: list[0 .. *list_count)
  const int* list_count;  // device memory, written by an earlier kernel
  int* esc_list;                  // NULL, or receives the cells handed over,
  unsigned long long* esc_count;  // in any order, and their number
  const double* sd_ft;            // SomDec: ELM temperature / moisture scalars, or NULL
  const double* sd_fw;
};
static_assert(sizeof(Args) == 240, "Args layout");

template <int V>
struct IC {
  static constexpr int value = V;
};
template <int B, int E, typename F>
__device__ __forceinline__ void sfor(F&& f) {
  if constexpr (B < E) {
    f(IC<B>{});
    sfor<B + 1, E>(f);
  }
}

// packed lower triangle, i > j (off-diagonal entries only)
__host__ __device__ constexpr int tri(int i, int j) {
  return i > j ? i * (i - 1) / 2 + j : j * (j - 1) / 2 + i;
}

// A copy of a wave-uniform value that the compiler cannot trace to its
// source: row offsets k * ld derived from it are formed where they are used
// instead of being hoisted out of the persistent loop, where 450 of them
// were spilled to vector lanes and read back in every iteration.
__device__ __forceinline__ i64 opaque(i64 v) {
#ifdef __AMDGCN__
  asm volatile("" : "+s"(v));
#endif
  return v;
}

// keeps the loads written before it ahead of the uses written after it
__device__ __forceinline__ void issue_loads() {
#ifdef __AMDGCN__
  __builtin_amdgcn_sched_barrier(0);
#endif
}

// FP64 exp / log (inlined: out-of-line calls cost more than the
// instruction-cache misses of the larger unrolled loop, measured on MI355X)
__device__ __forceinline__ double pf_exp(double v) { return exp(v); }
__device__ __forceinline__ double pf_log(double v) { return log(v); }

// exp(v) for |v| <= 600: v = n ln 2 + r with |r| <= ln 2 / 2, the Taylor series of
// exp(r) to r^13 (remainder below 5e-18) and one ldexp; without the range
// tests of exp, which the clipped Newton step does not need
__device__ __forceinline__ double exp_bounded(double v) {
  const double n = __builtin_rint(v * 1.4426950408889634074);
  double r = fma(-n, 0x1.62e42fefa3800p-1, v);  // ln 2 in two parts, the first
  r = fma(-n, 0x1.ef35793c76730p-45, r);        // short enough for n * part to be exact
  double p = 1.0 / 6227020800.0;
  p = fma(p, r, 1.0 / 479001600.0);
  p = fma(p, r, 1.0 / 39916800.0);
  p = fma(p, r, 1.0 / 3628800.0);
  p = fma(p, r, 1.0 / 362880.0);
  p = fma(p, r, 1.0 / 40320.0);
  p = fma(p, r, 1.0 / 5040.0);
  p = fma(p, r, 1.0 / 720.0);
  p = fma(p, r, 1.0 / 120.0);
  p = fma(p, r, 1.0 / 24.0);
  p = fma(p, r, 1.0 / 6.0);
  p = fma(p, r, 0.5);
  p = fma(p, r, 1.0);
  p = fma(p, r, 1.0);
  return __builtin_ldexp(p, (int)n);
}
// Mass action as products (see Acts below).  The residual and Jacobian block
// keeps the log form: it is evaluated once a cell, and its totals come from
// sums that cancel, where the form the caller had before counts.
#if PFLANE_GIRT
constexpr bool kProd = false;
#else
constexpr bool kProd = Net::ANY_PROD;
#endif
__device__ __forceinline__ double exp_step(double v) {
  if constexpr ((kProd || Net::HAS_SD) && Net::MAX_DLNC <= 600.0) return exp_bounded(v);
  else return pf_exp(v);
}
// 1/g by the hardware reciprocal estimate refined with two Newton-Raphson
// steps r <- r + r (1 - g r) (within about one ulp of the quotient; g > 0,
// normal)
__device__ __forceinline__ double rcp_nr(double g) {
  double r = __builtin_amdgcn_rcp(g);
  double e = fma(-g, r, 1.0);
  r = fma(e, r, r);
  e = fma(-g, r, 1.0);
  return fma(e, r, r);
}

// ReactionInterpolateLogK (reaction_aux.F90:1285-1312)
__device__ __forceinline__ double interp_logk(const double (&c)[5], double lnT, double tk) {
  return c[0] * lnT + c[1] + c[2] * tk + c[3] / tk + c[4] / (tk * tk);
}

// Debye-Hueckel activity coefficient (reaction.F90:4586-4592)
__device__ __forceinline__ double dh_gamma(double z, double a0, double sI, double I) {
  return pf_exp((-z * z * sI * Net::DH_A / (1.0 + a0 * Net::DH_B * sI) + Net::DH_BDOT * I) *
             kLogToLn);
}

// ln K of complex k / mineral m at the cell temperature (isothermal: the
// tabulated value; the product -logK*ln10 is formed as the reference does)
template <int K>
__device__ __forceinline__ double cplx_lnk(double lnT, double tk) {
  if constexpr (Net::ISOTHERMAL || !Net::HAS_CPLX_COEF)
    return -Net::CPLX_LOGK[K] * kLogToLn;
  else
    return -interp_logk(Net::CPLX_COEF[K], lnT, tk) * kLogToLn;
}
template <int M>
__device__ __forceinline__ double mnrl_lnk(double lnT, double tk) {
  if constexpr (Net::ISOTHERMAL || !Net::HAS_MNRL_COEF)
    return -Net::MNRL_LOGK[M] * kLogToLn;
  else
    return -interp_logk(Net::MNRL_COEF[M], lnT, tk) * kLogToLn;
}

// Mass action as products of powers.  With integer stoichiometry and a
// constant log K, K prod a^nu is formed from the activities' mantissas
// (in [1/2, 1), their reciprocals for negative nu) with the exponents summed
// as integers and applied once by ldexp, so no intermediate leaves the FP64
// range whatever the activities.  One multiplication per unit of |nu| (six
// for an average complex of the 15-primary network) replaces the exponential
// of each complex and the logarithm of each primary, which were 40 % of the
// step kernel's instructions; a product of at most 32 factors is good to
// ~1e-14, the exponential of a sum of logarithms of size 40 to the same.
// Networks of up to 8 primaries keep the log form and the arithmetic that
// goes with it (exp_step, the factorization's scaling): with 8 primaries and
// 32 complexes a cell in a hundred meets the 1e-14 residual test, and one in
// ten thousand the iteration limit, by rounding alone, so other rounding
// would move its sub-steps; their kernels are short either way.
// Rows with other stoichiometry, log K(T) or a water-activity factor keep the
// log form (Net::CPLX_PROD / MNRL_PROD).
template <int NA1>
struct Acts {
  double m[NA1], r[NA1];  // mantissa of the activity and its reciprocal
  int e[NA1];             // exponent
  double l[NA1];          // ln activity (rows in log form)
};
// ln gamma (networks without product rows) or gamma, as the kernels keep it
__device__ __forceinline__ double act_keep(double gamma) {
  if constexpr (kProd) return gamma;
  else return pf_log(gamma);
}
// activity of primary I at molality x; a <= 0 (or NaN) gives NaN, as its
// logarithm would
template <int I, int NA1>
__device__ __forceinline__ void act_set(Acts<NA1>& A, double x, double kept) {
  if constexpr (!kProd) {
    A.l[I] = pf_log(x) + kept;
    return;
  }
  const double a = x * kept;
  if constexpr (Net::NEED_PROD[I] != 0) {
    const double v = a > 0.0 ? a : __builtin_nan("");
    int e = 0;
    A.m[I] = __builtin_frexp(v, &e);
    A.e[I] = e;
    if constexpr (Net::NEED_PROD[I] > 1) A.r[I] = rcp_nr(A.m[I]);
  }
  if constexpr (Net::NEED_LN[I] != 0) A.l[I] = pf_log(a);
}
template <int P>
__device__ __forceinline__ double ipow(double b) {
  if constexpr (P == 1) return b;
  else if constexpr (P == 2) return b * b;
  else if constexpr (P == 3) return b * b * b;
  else return (b * b) * (b * b);
}
// scale K_k prod a^nu of complex K as p 2^e
template <int K, int NA1>
__device__ __forceinline__ double cplx_pe(const Acts<NA1>& A, double lnT, double tk, double ln_aw,
                                          double scale, int& e) {
  if constexpr (kProd && Net::CPLX_PROD[K] != 0) {
    double p = Net::CPLX_KM[K] * scale;
    e = Net::CPLX_KE[K];
    sfor<0, Net::CPLX_N[K]>([&](auto Q) {
      constexpr int i = Net::CPLX_ID[K][decltype(Q)::value];
      constexpr int nu = (int)Net::CPLX_NU[K][decltype(Q)::value];
      if constexpr (nu > 0) p *= ipow<nu>(A.m[i]);
      else p *= ipow<-nu>(A.r[i]);
      e += nu * A.e[i];
    });
    return p;
  } else {
    e = 0;
    double lnQK = cplx_lnk<K>(lnT, tk);
    if constexpr (Net::CPLX_H2O[K] != 0.0) lnQK += Net::CPLX_H2O[K] * ln_aw;
    sfor<0, Net::CPLX_N[K]>([&](auto Q) {
      constexpr int a = decltype(Q)::value;
      lnQK += Net::CPLX_NU[K][a] * A.l[Net::CPLX_ID[K][a]];
    });
    return pf_exp(lnQK) * scale;
  }
}
template <int K, int NA1>
__device__ __forceinline__ double cplx_q(const Acts<NA1>& A, double lnT, double tk, double ln_aw,
                                         double scale) {
  int e;
  const double p = cplx_pe<K>(A, lnT, tk, ln_aw, scale, e);
  if constexpr (kProd && Net::CPLX_PROD[K] != 0) return __builtin_ldexp(p, e);
  else return p;
}
// Q/K of kinetic mineral M
template <int M, int NA1>
__device__ __forceinline__ double mnrl_q(const Acts<NA1>& A, double lnT, double tk,
                                         double ln_aw) {
  if constexpr (kProd && Net::MNRL_PROD[M] != 0) {
    double p = Net::MNRL_KM[M];
    int e = Net::MNRL_KE[M];
    sfor<0, Net::MNRL_N[M]>([&](auto Q) {
      constexpr int i = Net::MNRL_ID[M][decltype(Q)::value];
      constexpr int nu = (int)Net::MNRL_NU[M][decltype(Q)::value];
      if constexpr (nu > 0) p *= ipow<nu>(A.m[i]);
      else p *= ipow<-nu>(A.r[i]);
      e += nu * A.e[i];
    });
    return __builtin_ldexp(p, e);
  } else {
    double lnQK = mnrl_lnk<M>(lnT, tk);
    if constexpr (Net::MNRL_H2O[M] != 0.0) lnQK += Net::MNRL_H2O[M] * ln_aw;
    sfor<0, Net::MNRL_N[M]>([&](auto Q) {
      constexpr int a = decltype(Q)::value;
      lnQK += Net::MNRL_NU[M][a] * A.l[Net::MNRL_ID[M][a]];
    });
    return pf_exp(lnQK);
  }
}

// RKineticMineral rate of mineral M (reaction_mineral.F90:729-908): Im per
// unit bulk volume and dIm/dQK per unit volume; active = the reference does
// not `cycle` past the mineral
struct MRate {
  double Im, dIm;
  bool active;
};
template <int M>
__device__ __forceinline__ MRate mineral_rate(double QK, double vf, double area, double temp) {
  MRate r{0.0, 0.0, false};
  constexpr bool temkin = Net::HAS_TEMKIN, mscale = Net::HAS_MINSCALE;
  double sig = 1.0;
  if constexpr (temkin && mscale) sig = Net::MNRL_MINSCALE[M] * Net::MNRL_TEMKIN[M];
  else if constexpr (temkin) sig = Net::MNRL_TEMKIN[M];
  else if constexpr (mscale) sig = Net::MNRL_MINSCALE[M];
  double aff;
  if constexpr (temkin || mscale) aff = 1.0 - pow(QK, 1.0 / sig);
  else aff = 1.0 - QK;
  const double sgn = copysign(1.0, aff);
  if (!(vf > 0.0 || sgn < 0.0)) return r;
  if constexpr (Net::HAS_IRREV) {
    if (Net::MNRL_IRREV[M] == 1 && sgn < 0.0) return r;
  }
  if constexpr (Net::HAS_THRESHOLD) {
    if (Net::MNRL_THRESHOLD[M] > 0.0 && sgn < 0.0 && QK < Net::MNRL_THRESHOLD[M]) return r;
  }
  constexpr double lim = Net::HAS_LIMITER ? Net::MNRL_LIMITER[M] : 0.0;
  if constexpr (lim > 0.0) aff = aff / (1.0 + (1.0 - aff) / lim);
  double kr = Net::MNRL_K[M];
  if constexpr (Net::HAS_EA) {
    if constexpr (Net::MNRL_EA[M] > 0.0)
      kr = kr * pf_exp(Net::MNRL_EA[M] / kIdealGas * (1.0 / (25.0 + 273.15) - 1.0 / (temp + 273.15)));
  }
  double Im_const = -area;
  if constexpr (mscale) Im_const = Im_const / Net::MNRL_MINSCALE[M];
  double Im;
  if constexpr (Net::HAS_AFFPOWER) Im = Im_const * sgn * pow(fabs(aff), Net::MNRL_AFFPOWER[M]) * kr;
  else Im = Im_const * sgn * fabs(aff) * kr;
  double d;
  if constexpr (Net::HAS_AFFPOWER) d = -Im * Net::MNRL_AFFPOWER[M] / fabs(aff);
  else d = -Im_const * kr;
  if constexpr (temkin || mscale) d = d * (1.0 / sig) / QK * (1.0 - aff);
  if constexpr (lim > 0.0) {
    const double den = 1.0 + (1.0 - aff) / lim;
    d = d * (1.0 + QK / lim / den) / den;
  }
  r.Im = Im;
  r.dIm = d;
  r.active = true;
  return r;
}

// secondary molality of complex K: with coefficients fixed during the step
// gi holds the inverse of each (Z^2, a0) class's; otherwise g receives the
// Debye-Hueckel coefficient at the ionic strength I
template <int K, bool NEWTON_ACT, int NA1, int NG1>
__device__ __forceinline__ double cplx_m(const Acts<NA1>& act, double lnT, double tk, double ln_aw,
                                         const double (&gi)[NG1], double sI, double I, double& g) {
  if constexpr (NEWTON_ACT) {
    g = 1.0;
    if constexpr (Net::CPLX_Z[K] > 1.0e-10 || Net::CPLX_Z[K] < -1.0e-10)
      g = dh_gamma(Net::CPLX_Z[K], Net::CPLX_A0[K], sI, I);
    return cplx_q<K>(act, lnT, tk, ln_aw, 1.0) / g;
  } else if constexpr (Net::CPLX_GCLS[K] >= 0) {
    return cplx_q<K>(act, lnT, tk, ln_aw, gi[Net::CPLX_GCLS[K]]);
  } else {
    return cplx_q<K>(act, lnT, tk, ln_aw, 1.0);
  }
}

#if PFLANE_SD
// ---------------------------------------------------------------------------
// SomDec decomposition sandbox (reaction_sandbox_somdec.F90) of one cell with
// the network's reactions as compile-time constants: residual terms R and the
// entries of d R / d c the reference assembles (the ones that are not exact
// derivatives among them), on the sparse pattern Net::JPOS (row, column ->
// entry, closed under the elimination's fill-in, -1 elsewhere).  Statements
// follow SomDecReact (:1504-1910), React1 (:1914-2418), React2 (:2423-3472)
// and SomDecNemission (:3477-3640) without oxygen and aqueous complexes.
struct SdCell {
  double dkl, theta, vol, sat, tdt, itdt;
  double ft[Net::SD_NFT], fw[Net::SD_NFW];  // response factors per class
  double em;                                // min(f_t, 1) min(f_w, 1) of the emission, 0: none
  double unc[Net::SDN];                     // upstream N:C of the variable C:N pools
  double dnc[Net::SDN][4];                  // downstream N:C of variable C:N pools
};
struct SdSum {
  double R[Net::NAQ + Net::NIMM];
  double J[Net::JNNZ];
};
template <int ROW>
__device__ __forceinline__ void sd_R(SdSum& s, double v) {
  if constexpr (ROW >= 0) s.R[ROW] += v;
}
template <int ROW, int COL>
__device__ __forceinline__ void sd_J(SdSum& s, double v) {
  if constexpr (ROW >= 0 && COL >= 0) s.J[Net::JPOS[ROW][COL]] += v;
}
// dof of an immobile species (-1: none)
constexpr int sd_row(int imm) { return imm >= 0 ? Net::NAQ + imm : -1; }
// column p of the pattern has entries below the diagonal
constexpr bool lu_eliminates(int p) {
  for (int i = p + 1; i < Net::NAQ + Net::NIMM; ++i)
    if (Net::JPOS[i][p] >= 0) return true;
  return false;
}
__device__ __forceinline__ double sd_div(double a, double b) { return a * rcp_nr(b); }
__device__ __forceinline__ double sd_monod(double c, double k) { return sd_div(c, c + k); }
__device__ __forceinline__ double sd_dmonod(double c, double k) {
  const double r = rcp_nr(c + k);
  return k * r * r;
}
// HfunctionSmooth (utility.F90:2542-2597) between x0eps and 10 x0eps; without
// x0eps the factor is 1
__device__ __forceinline__ void sd_smooth(double c, double& H, double& dH) {
  constexpr double x0 = Net::SD_X0EPS, x1 = 10.0 * Net::SD_X0EPS;
  H = 1.0;
  dH = 0.0;
  if constexpr (x0 > 0.0) {
    if constexpr (x1 - x0 < 1.0e-50) {
      H = copysign(0.5, c - x1) + 0.5;
    } else {
      constexpr double w = x1 > x0 ? 1.0 / (x1 - x0) : 0.0;  // formed for x0 = 0 too
      const double u = (c - x0) * w;
      const double xs = 1.0 - u * u;
      if (u < 0.0) {
        H = 0.0;
      } else if (u <= 1.0) {
        H = 1.0 - xs * xs;
        dH = 4.0 * xs * u * w;
      }
    }
  }
}
// GetTemperatureResponse (elm_rspfuncs.F90:61-120)
template <int TYPE>
__device__ __forceinline__ double sd_temperature(double tc, double q) {
  if constexpr (TYPE == 2) {
    if (tc > 0.0) return pow(q, (tc - 25.0) / 10.0);
    return pow(q, -25.0 / 10.0) * pow(2.0, tc / 10.0);
  } else if constexpr (TYPE == 1) {
    const double tk = tc + 273.15;
    return tk > 227.15 ? pf_exp(308.56 * (1.408054069e-2 - 1.0 / (tk - 227.13))) : 0.0;
  } else if constexpr (TYPE == 3) {
    if (tc < -5.0) return 0.0;
    if (tc >= 30.0) return 1.0;
    return pow(q, (tc - 30.0) / 10.0);
  } else {
    return pf_exp(q / kIdealGas * (1.0 / 298.15 - 1.0 / (tc + 273.15)));
  }
}
// the per-cell factors: temperature and moisture responses, the emission's,
// and the stoichiometry's Setup values
__device__ __forceinline__ void sd_load(SdCell& e, double temp, bool has_ft, double ft, bool has_fw,
                                        double fw) {
  sfor<0, Net::SD_NFT>([&](auto Q) {
    constexpr int q = decltype(Q)::value;
    if constexpr (Net::SD_FT_TYPE[q] == 0) e.ft[q] = has_ft ? ft : 1.0;
    else e.ft[q] = sd_temperature<Net::SD_FT_TYPE[q]>(temp, Net::SD_FT_PAR[q]);
  });
  sfor<0, Net::SD_NFW>([&](auto Q) {
    constexpr int q = decltype(Q)::value;
    double f = 1.0;
    if (has_fw) f = fw;
    else if constexpr (Net::SD_FW_TYPE[q] % 2 != 0)
      f = e.theta <= 0.08 ? 0.01 : pf_log(e.theta / 0.08) / pf_log(1.0 / 0.08);
    if constexpr (Net::SD_FW_TYPE[q] / 2 != 0) {  // water-filled pore space
      const double a = 1.27 - e.sat, b = e.sat - 0.0012;
      double w = 0.0;
      if (a > 0.0 && b > 0.0) w = fmin(pow(a / 0.67, 3.1777) * pow(b / 0.5988, 2.84), 1.0);
      f = f * w;
    }
    e.fw[q] = f;
  });
  e.em = 0.0;
  if constexpr (Net::SD_N2O >= 0) {
    const double et = -0.06 + 0.13 * pf_exp(0.07 * temp);
    const double ew = pow((1.27 - e.sat) / 0.67, 3.1777) * pow((e.sat - 0.0012) / 0.5988, 2.84);
    if (et > Net::SD_X0EPS && ew > Net::SD_X0EPS) e.em = fmin(et, 1.0) * fmin(ew, 1.0);
  }
#pragma unroll
  for (int r = 0; r < Net::SDN; ++r) {
    e.unc[r] = Net::SD_UNC[r];
#pragma unroll
    for (int j = 0; j < 4; ++j) e.dnc[r][j] = Net::SD_DNC[r][j];
  }
}
// Monod and inhibition factors of reaction r; SKIP: React2 takes its NH4+ and
// NO3- Monod terms apart
template <int r, bool SKIP>
__device__ __forceinline__ void sd_factors(const SdCell& e, const double (&x)[Net::NAQ + Net::NIMM],
                                           double c4, double c3, double& f, double& df,
                                           double& f4, double& d4, double& f3, double& d3) {
  constexpr int uc = Net::SD_UC[r];
  auto conc = [&](auto ID) {
    constexpr int id = decltype(ID)::value;
    if constexpr (id >= 0) return x[id] * e.dkl;
    else return x[Net::NAQ - id - 1];
  };
  sfor<0, Net::SD_NMON[r]>([&](auto Q) {
    constexpr int q = decltype(Q)::value;
    constexpr int id = Net::SD_MSP[r][q];
    constexpr double k = Net::SD_MHS[r][q], th = Net::SD_MTH[r][q];
    constexpr bool pool = Net::SD_MPN[r][q] != 0;
    if constexpr (SKIP && id >= 0 && (id == Net::SD_NH4 || id == Net::SD_NO3)) {
      double t = fmax(0.0, (id == Net::SD_NH4 ? c4 : c3) - th);
      if constexpr (pool) t = sd_div(t, x[Net::NAQ + uc]);
      if constexpr (id == Net::SD_NH4) {
        f4 = sd_monod(t, k);
        d4 = sd_dmonod(t, k);
      } else {
        f3 = sd_monod(t, k);
        d3 = sd_dmonod(t, k);
      }
    } else {
      double t = fmax(0.0, conc(IC<id>{}) - th);
      if constexpr (pool) {
        t = sd_div(t, x[Net::NAQ + uc]);
        if constexpr (id >= 0) t = t * e.theta * 1000.0;
      }
      const double fx = sd_monod(t, k);
      const double dfx = id == -uc - 1 ? sd_dmonod(t, k) : 0.0;
      df = df * fx + f * dfx;
      f = f * fx;
    }
  });
  sfor<0, Net::SD_NINH[r]>([&](auto Q) {
    constexpr int q = decltype(Q)::value;
    constexpr int id = Net::SD_ISP[r][q], ty = Net::SD_ITY[r][q];
    constexpr double k = Net::SD_IC1[r][q], k2 = Net::SD_IC2[r][q];
    const double t = conc(IC<id>{});
    double fx = 1.0, dfx = 0.0;
    if constexpr (ty == 1) {
      const double w = (t - k) * k2;
      fx = 0.5 + atan(w) / 3.14159265358979323846;
      dfx = (k2 / (1.0 + w * w)) / 3.14159265358979323846;
    } else if constexpr (ty == 3) {
      fx = sd_monod(k, t);  // k / (t + k)
      dfx = -sd_dmonod(t, k);
    } else if constexpr (ty == 4) {
      fx = sd_monod(t, k);
      dfx = sd_dmonod(t, k);
    }
    if constexpr (id != -uc - 1) dfx = 0.0;
    df = df * fx + f * dfx;
    f = f * fx;
  });
}
// reaction r: adds its terms, returns its N mineralization (> 0) or
// immobilization (< 0) rate
template <int r>
__device__ __forceinline__ double sd_reaction(SdCell& e, const double (&x)[Net::NAQ + Net::NIMM],
                                              SdSum& s) {
  constexpr int NAQ = Net::NAQ;
  constexpr int uc = Net::SD_UC[r], un = Net::SD_UN[r], nd = Net::SD_ND[r];
  constexpr bool vary = Net::SD_VARY[r] != 0;
  constexpr int ruc = NAQ + uc, run = vary ? sd_row(un) : -1;
  constexpr int nh4 = Net::SD_NH4, no3 = Net::SD_NO3, co2 = Net::SD_CO2;
  constexpr int uhr = sd_row(Net::SD_UHR[r]), hr = sd_row(Net::SD_HR);
  const double f_t = e.ft[Net::SD_TCLS[r]], f_w = e.fw[Net::SD_WCLS[r]];
  if (f_t < 1.0e-20 || f_w < 1.0e-20) return 0.0;
  double k = 0.0;
  if constexpr (Net::SD_K0[r] >= 0.0) k = Net::SD_K0[r];
  else if constexpr (Net::SD_KD[r] >= 0.0) k = (1.0 - pf_exp(-Net::SD_KD[r] * e.tdt)) * e.itdt;
  k = fmin(Net::SD_AD[r] * k, e.itdt);
  const double scaled = k * e.vol * f_t * f_w;
  const double c_uc = x[ruc];
  double h, dh;
  sd_smooth(c_uc, h, dh);
  if constexpr (!(Net::SD_X0EPS > 0.0)) {
    if (c_uc <= Net::SD_X0EPS) return 0.0;
  }
  double rate = scaled * c_uc * h;
  double drate = scaled * (h + c_uc * dh);
  // variable C:N stoichiometry
  sfor<0, nd>([&](auto Q) {
    constexpr int j = decltype(Q)::value;
    constexpr int dc = Net::SD_DC[r][j], dn = Net::SD_DN[r][j];
    if constexpr (Net::SD_DVARY[r][j] != 0 && dc >= 0 && dn >= 0) {
      if (x[NAQ + dn] >= Net::SD_X0EPS && x[NAQ + dc] >= Net::SD_X0EPS)
        e.dnc[r][j] = sd_div(x[NAQ + dn], x[NAQ + dc]);
    }
  });
  double cs = Net::SD_MCS[r], ns = Net::SD_MNS[r];
  if constexpr (vary && un >= 0) {
    if (x[NAQ + un] >= Net::SD_X0EPS && c_uc >= Net::SD_X0EPS) e.unc[r] = sd_div(x[NAQ + un], c_uc);
    cs = 1.0;
    ns = e.unc[r];
    sfor<0, nd>([&](auto Q) {
      constexpr int j = decltype(Q)::value;
      cs -= Net::SD_DS[r][j];
      ns -= Net::SD_DS[r][j] * e.dnc[r][j];
    });
  }
  const double unc = e.unc[r];
  // pools: the C row (and variable N row) of every product
  auto pools_R = [&](double v) {
    sfor<0, nd>([&](auto Q) {
      constexpr int j = decltype(Q)::value;
      sd_R<sd_row(Net::SD_DC[r][j])>(s, -Net::SD_DS[r][j] * v);
      if constexpr (Net::SD_DVARY[r][j] != 0)
        sd_R<sd_row(Net::SD_DN[r][j])>(s, -Net::SD_DS[r][j] * v * e.dnc[r][j]);
    });
  };
  auto pools_J = [&](auto C, double v) {
    constexpr int col = decltype(C)::value;
    sfor<0, nd>([&](auto Q) {
      constexpr int j = decltype(Q)::value;
      sd_J<sd_row(Net::SD_DC[r][j]), col>(s, Net::SD_DS[r][j] * v);
      if constexpr (Net::SD_DVARY[r][j] != 0)
        sd_J<sd_row(Net::SD_DN[r][j]), col>(s, Net::SD_DS[r][j] * v * e.dnc[r][j]);
    });
  };
  double f = 1.0, df = 0.0, f4 = 1.0, d4 = 0.0, f3 = 1.0, d3 = 0.0;
  if (ns >= 0.0) {  // React1
    constexpr int unmin = sd_row(Net::SD_UNMIN[r]), nmin = sd_row(Net::SD_NMIN);
    sd_factors<r, false>(e, x, 0.0, 0.0, f, df, f4, d4, f3, d3);
    drate = drate * f + rate * df;
    rate = rate * f;
    sd_R<ruc>(s, rate);
    sd_R<co2>(s, -cs * rate);
    sd_R<uhr>(s, -cs * rate);
    sd_R<hr>(s, -cs * rate);
    pools_R(rate);
    sd_R<run>(s, unc * rate);
    sd_R<nh4>(s, -ns * rate);
    sd_R<unmin>(s, -ns * rate);
    sd_R<nmin>(s, -ns * rate);
    const double dco2 = drate * cs, duc = -1.0 * drate;
    const double dnh4 = dco2 * ns;  // as the reference writes it (:2273)
    sd_J<co2, ruc>(s, -dco2);
    sd_J<uhr, ruc>(s, -dco2);
    sd_J<hr, ruc>(s, -dco2);
    sd_J<ruc, ruc>(s, -duc);
    pools_J(IC<ruc>{}, duc);
    sd_J<nh4, ruc>(s, -dnh4);
    sd_J<unmin, ruc>(s, -dnh4);
    sd_J<nmin, ruc>(s, -dnh4);
    sd_J<run, ruc>(s, -unc * duc);
    return ns * rate;
  }
  if constexpr (vary || Net::SD_MNS[r] < 0.0) {  // React2
    constexpr int unimm = sd_row(Net::SD_UNIMM[r]), unimp = sd_row(Net::SD_UNIMP[r]);
    constexpr int gimm = sd_row(Net::SD_NIMM), gimp = sd_row(Net::SD_NIMP);
    const double c4 = nh4 >= 0 ? x[nh4 >= 0 ? nh4 : 0] * e.dkl * e.theta * 1000.0 : 0.0;
    const double c3 = no3 >= 0 ? x[no3 >= 0 ? no3 : 0] * e.dkl * e.theta * 1000.0 : 0.0;
    double fin = 1.0;
    if constexpr (Net::SD_INHIB > 0.0) {
      const bool has4 = c4 > Net::SD_X0EPS, has3 = c3 > Net::SD_X0EPS;
      if (!has4 && !has3) return 0.0;  // both tiny (:2547)
      if (has4 && has3) fin = sd_monod(sd_div(c4, c3), 1.0 / Net::SD_INHIB);
      else fin = has4 ? 1.0 : 0.0;
    }
    sd_factors<r, true>(e, x, c4, c3, f, df, f4, d4, f3, d3);
    drate = drate * f + rate * df;
    rate = rate * f;
    if constexpr (nh4 >= 0) {
      sd_smooth(c4, h, dh);
      d4 = d4 * h + f4 * dh;
      f4 = f4 * h;
    }
    if constexpr (no3 >= 0) {
      sd_smooth(c3, h, dh);
      d3 = d3 * h + f3 * dh;
      f3 = f3 * h;
    }
    // N-rate cap (:2829-2858)
    const double cap = -rate * ns * e.tdt / 0.45;
    if constexpr (nh4 >= 0) {
      const double c = c4 * e.vol, w = cap * fin;
      if (w > c) {
        const double g = sd_monod(c, w - c), dg = sd_dmonod(c, w - c);
        d4 = d4 * g + f4 * dg;
        f4 = f4 * g;
      }
    }
    if constexpr (no3 >= 0) {
      const double c = c3 * e.vol, w = cap * (1.0 - fin);
      if (w > c) {
        const double g = sd_monod(c, w - c), dg = sd_dmonod(c, w - c);
        d3 = d3 * g + f3 * dg;
        f3 = f3 * g;
      }
    }
    const double r4 = rate * f4 * fin, r3 = rate * f3 * (1.0 - fin);
    const double cr = r4 + r3;
    sd_R<ruc>(s, cr);
    sd_R<co2>(s, -cs * cr);
    sd_R<uhr>(s, -cs * cr);
    sd_R<hr>(s, -cs * cr);
    pools_R(cr);
    sd_R<run>(s, unc * cr);
    double nimm = 0.0;
    if constexpr (nh4 >= 0) {
      sd_R<nh4>(s, -ns * r4);
      nimm += ns * r4;
    }
    if constexpr (no3 >= 0) {
      sd_R<no3>(s, -ns * r3);
      nimm += ns * r3;
    }
    sd_R<unimm>(s, ns * cr);
    sd_R<unimp>(s, ns * rate);
    sd_R<gimm>(s, ns * cr);
    sd_R<gimp>(s, ns * rate);
    double dx = drate * (f4 * fin + f3 - f3 * fin);
    {
      const double dco2 = dx * cs, duc = -1.0 * dx;
      const double dn4 = drate * ns * f4 * fin, dn3 = drate * ns * f3 * (1.0 - fin);
      sd_J<co2, ruc>(s, -dco2);
      sd_J<uhr, ruc>(s, -dco2);
      sd_J<hr, ruc>(s, -dco2);
      sd_J<ruc, ruc>(s, -duc);
      pools_J(IC<ruc>{}, duc);
      if constexpr (nh4 >= 0) {
        sd_J<nh4, ruc>(s, -dn4);
        sd_J<unimm, ruc>(s, dn4);
        sd_J<gimm, ruc>(s, dn4);
      }
      if constexpr (no3 >= 0) {
        sd_J<no3, ruc>(s, -dn3);
        sd_J<unimm, ruc>(s, dn3);
        sd_J<gimm, ruc>(s, dn3);
      }
      sd_J<run, ruc>(s, -unc * duc);
    }
    // columns of NH4+ and NO3- (the factors the reference writes,
    // :3180-3470; the derivative of the split between them is off, :2638);
    // dtotal of a species without complexes is the density factor
    sfor<0, 2>([&](auto Q) {
      constexpr int col = decltype(Q)::value == 0 ? nh4 : no3;
      if constexpr (col >= 0) {
        constexpr bool c4q = decltype(Q)::value == 0;
        const double d = c4q ? d4 * fin * rate : d3 * (1.0 - f4 * fin) * rate;
        const double dco2 = d * cs, duc = -1.0 * d;
        const double dn4 = c4q ? d4 * fin * rate * ns : 0.0;
        const double dn3 = c4q ? 0.0 : d3 * (1.0 - fin) * rate * ns;
        if constexpr (co2 == col) sd_J<co2, col>(s, -dco2 * e.dkl);
        sd_J<uhr, col>(s, -dco2);
        sd_J<hr, col>(s, -dco2);
        sd_J<ruc, col>(s, -duc);
        pools_J(IC<col>{}, duc);
        if constexpr (nh4 >= 0) {
          if constexpr (nh4 == col) sd_J<nh4, col>(s, -dn4 * e.dkl);
          sd_J<unimm, col>(s, dn4);
          sd_J<gimm, col>(s, dn4);
        }
        if constexpr (no3 >= 0) {
          if constexpr (no3 == col) sd_J<no3, col>(s, -dn3 * e.dkl);
          sd_J<unimm, col>(s, dn3);
          sd_J<gimm, col>(s, dn3);
        }
        sd_J<run, col>(s, -unc * duc);
      }
    });
    return nimm;
  }
  return 0.0;
}
// SomDecNemission (:3477-3640)
__device__ __forceinline__ void sd_emission(const SdCell& e,
                                            const double (&x)[Net::NAQ + Net::NIMM], double lnh,
                                            double net, SdSum& s) {
  if constexpr (Net::SD_N2O >= 0) {
    constexpr int nh4 = Net::SD_NH4;
    if (!(net > Net::SD_X0EPS) || !(e.em > 0.0)) return;
    double ph = 6.5;
    if constexpr (Net::SD_PROTON >= 0) ph = -lnh / kLogToLn;
    const double f_ph = 0.56 + atan(3.14159265358979323846 * 0.45 * (-5.0 + ph)) /
                                   3.14159265358979323846;
    if (!(f_ph > Net::SD_X0EPS)) return;
    const double tr = e.em * fmin(f_ph, 1.0);
    const double c4 = x[nh4] * e.dkl * e.theta * 1000.0;
    double h, dh;
    sd_smooth(c4, h, dh);
    const double cap = tr * Net::SD_N2OFRAC * net * e.tdt, c = c4 * e.vol;
    if (cap > c) {
      const double g = sd_monod(c, cap - c), dg = sd_dmonod(c, cap - c);
      dh = dh * g + h * dg;
      h = h * g;
    }
    const double rate = tr * Net::SD_N2OFRAC * net * h;
    sd_R<nh4>(s, rate);
    sd_R<Net::SD_N2O>(s, -0.5 * rate);
    sd_R<sd_row(Net::SD_NGASMIN)>(s, -rate);
    const double d = tr * Net::SD_N2OFRAC * net * dh;
    sd_J<nh4, nh4>(s, d * e.dkl);
    sd_J<sd_row(Net::SD_NGASMIN), nh4>(s, -d);
  }
}
#endif  // PFLANE_SD

__device__ __forceinline__ void hand_over(const Args& A, i64 c) {
  A.status[c] = kEscalate;
  if (A.esc_list) A.esc_list[atomicAdd(A.esc_count, 1ull)] = (int)c;
}

// One reaction step for cells [0, ncell) (or, with rescue, the cells whose
// status is kEscalate).  JT: precision of the factorization.
template <typename JT>
__device__ __forceinline__ void lane_step(const Args& A) {
  constexpr int NAQ = Net::NAQ, NIMM = Net::NIMM, N = NAQ + NIMM, NC = Net::NC, NM = Net::NM;
  constexpr int NA1 = NAQ > 0 ? NAQ : 1, NM1 = NM > 0 ? NM : 1;
  constexpr int NT = NAQ > 1 ? NAQ * (NAQ - 1) / 2 : 1;
  constexpr bool NEWTON_ACT = Net::ACT_FREQ == kFreqNewtonIter && NAQ > 0;
  // per-class inverse activity coefficients of the complexes (activity
  // coefficients fixed during the step)
  constexpr int NG = NEWTON_ACT ? 0 : Net::NGCLS;
  constexpr int NG1 = NG > 0 ? NG : 1;
  constexpr int kLdsFields = 2 * N + NAQ + 3 * NM + NG > 0 ? 2 * N + NAQ + 3 * NM + NG : 1;
  constexpr bool F32 = sizeof(JT) == 4;
  // pivot tolerance of the factorization, relative to the diagonal
  constexpr double kPivTol = F32 ? 1.0e-6 : 1.0e-13;
#if PFLANE_SD
  constexpr bool SD = true;
  SdCell sdc;
#else
  constexpr bool SD = false;
#endif
  const i64 ld = A.ld;
  const int lane = (int)__lane_id();
  const int nxcd = A.nxcd;
  const int xcd = (int)(blockIdx.x % (unsigned)nxcd);
  // cells of this pass: all, or a list an earlier kernel wrote (a short
  // list is left to a later pass: the grid returns at once)
  const bool listed = A.list != nullptr;
  const i64 nwork = listed ? (i64)*A.list_count : A.ncell;
  if (listed && nwork <= (i64)A.list_min) return;
  const i64 chunk = (nwork + nxcd - 1) / nxcd;

  // wave-uniform queue of claimed cells [qn, qe); XCD ranges found empty
  i64 qn = 0, qe = 0;
  int steal = 0;
  // lane state.  Per-cell values that the complex loop does not touch live
  // in this lane's own LDS slots (field-major, 256 lanes per field: a wave's
  // accesses are conflict free and no lane reads another's slots).
  __shared__ double lsm[kLdsFields * 256];
  const int tid = (int)threadIdx.x;
#define PF_GUESS(i) lsm[(0 + (i)) * 256 + tid]
#define PF_TINIT(i) lsm[(N + (i)) * 256 + tid]
#define PF_GAM(i) lsm[(2 * N + (i)) * 256 + tid]
#define PF_VF(m) lsm[(2 * N + NAQ + (m)) * 256 + tid]
#define PF_AREA(m) lsm[(2 * N + NAQ + NM + (m)) * 256 + tid]
#define PF_RLAST(m) lsm[(2 * N + NAQ + 2 * NM + (m)) * 256 + tid]
#define PF_GINV(q) lsm[(2 * N + NAQ + 3 * NM + (q)) * 256 + tid]
  bool exhausted = false;
  i64 cell = -1;
  int mode = 0;  // 0: no cell, 1: Newton iteration, 2: write-out evaluation
  double x[N];
  double por = 0.0, sat = 0.0, dkl = 0.0, vol = 0.0, temp = 25.0, ln_aw = 0.0, psv = 0.0;
  double lnT = 0.0, tk = 298.15;
  double target = 0.0, cum = 0.0, tdt = 0.0, r0 = 0.0;
  double sec_I = 0.0, sec_sum = 0.0, I_last = 0.0;
  int nconst = 0, ncuts = 0, nsub = 0, nit_total = 0, nit = 0, status = 0;
  int attempts = 0, last_why = 0;
  bool restore = false;    // outputs of a failed RStep: totals at RReact start
  bool kin = false;        // write-out: the last sub-step's kinetic update is due
  unsigned small = 0u;     // bit i: component i started at or below 1e-40
#pragma unroll
  for (int i = 0; i < N; ++i) x[i] = 1.0;

  for (;;) {
    // lanes without work wait until kServe of them do (or none iterates):
    // writing back and loading touch some 230 rows of the state for however
    // few lanes
    const unsigned long long waiting = __ballot(mode == 2 || (cell < 0 && !exhausted));
    const bool serve = __popcll(waiting) >= kServe || !__ballot(mode == 1);
    if (serve) {
    // ---------------- write finished cells back ----------------
    // totals, secondary molalities, rates and the last sub-step's kinetic
    // update at the final unknowns; apart from the Newton evaluation, which
    // then carries no stores and no write-out tests
    if (mode == 2) {
      const i64 c = cell;
      const i64 lo = opaque(ld);
      const bool ok = status == 0;
      double I = 0.0, sI = 0.0;
      if constexpr (NEWTON_ACT) {  // the last iteration's ionic strength
        I = I_last;
        sI = sqrt(I);
      }
      Acts<NA1> act;
      double tot[NA1];
      sfor<0, NAQ>([&](auto Q) {
        constexpr int i = decltype(Q)::value;
        act_set<i>(act, x[i], PF_GAM(i));
        tot[i] = 0.0;
      });
      double gi[NG1];
      sfor<0, NG>([&](auto Q) {
        constexpr int q = decltype(Q)::value;
        gi[q] = PF_GINV(q);
      });
      double* ps = A.sec_molal + c;
      double* pg = A.sec_act_coef + c;
      sfor<0, NC>([&](auto K) {
        constexpr int k = decltype(K)::value;
        double g = 1.0;
        const double m = cplx_m<k, NEWTON_ACT>(act, lnT, tk, ln_aw, gi, sI, I, g);
        *ps = m;
        ps += lo;
        if constexpr (NEWTON_ACT) {
          *pg = g;
          pg += lo;
        }
        sfor<0, Net::CPLX_N[k]>([&](auto Q) {
          constexpr int a = decltype(Q)::value;
          tot[Net::CPLX_ID[k][a]] += Net::CPLX_NU[k][a] * m;
        });
      });
      double* pp = A.pri_molal + c;
      double* pt = A.total + c;
      double* pa = A.pri_act_coef + c;
      sfor<0, NAQ>([&](auto Q) {
        constexpr int i = decltype(Q)::value;
        *pp = x[i];
        const bool keep = ok && ((small >> i) & 1u);  // original value restored
        if (!keep) *pt = (!ok && restore) ? PF_TINIT(i) : (x[i] + tot[i]) * dkl;
        if constexpr (NEWTON_ACT) *pa = kProd ? PF_GAM(i) : pf_exp(PF_GAM(i));
        pp += lo;
        pt += lo;
        pa += lo;
      });
      sfor<0, NIMM>([&](auto Q) {
        constexpr int i = NAQ + decltype(Q)::value;
        const bool keep = ok && ((small >> i) & 1u);
        if (!keep) A.immobile[(i - NAQ) * lo + c] = (!ok && restore) ? PF_TINIT(i) : x[i];
      });
      sfor<0, NM>([&](auto M) {
        constexpr int m = decltype(M)::value;
        if (kin) {
          // RUpdateKineticState of the last sub-step (reaction_mineral.F90:
          // 1456-1525): rates at the final state, volume fractions of the
          // sub-step's start
          double r = 0.0;
          const double ar = PF_AREA(m);
          if (ar != 0.0) r = mineral_rate<m>(mnrl_q<m>(act, lnT, tk, ln_aw), PF_VF(m), ar, temp).Im;
          double v = PF_VF(m) + r * Net::MNRL_VM[m] * tdt;
          if (v < 0.0) v = 0.0;
          PF_VF(m) = v;
          PF_RLAST(m) = r;
        }
        A.mnrl_volfrac[m * lo + c] = PF_VF(m);
        if (A.mnrl_rate) A.mnrl_rate[m * lo + c] = PF_RLAST(m);
      });
      if constexpr (NEWTON_ACT && Net::ACT_H2O) {
        if (A.ln_act_h2o) A.ln_act_h2o[c] = ln_aw;
      }
      if (A.num_iterations) A.num_iterations[c] = nit_total;
      if (A.num_sub_steps) A.num_sub_steps[c] = nsub;
      if (A.status) A.status[c] = status;
      cell = -1;
      mode = 0;
    }

    // ---------------- work stealing: hand out cells ----------------
    {
      bool needy = cell < 0 && !exhausted;
      unsigned long long mask = __ballot(needy);
      while (mask) {
        if (qn >= qe) {
          if (steal >= nxcd) {  // every range is empty
            if (needy) exhausted = true;
            needy = false;
            break;
          }
          const int xr = xcd + steal < nxcd ? xcd + steal : xcd + steal - nxcd;
          const i64 lo = (i64)xr * chunk;
          const i64 hi = lo + chunk < nwork ? lo + chunk : nwork;
          const int first = __builtin_ctzll(__ballot(1));
          unsigned long long base = 0;
          if (lane == first) base = atomicAdd(A.cursors + 16 * xr, (unsigned long long)kClaim);
          base = __shfl(base, first, 64);
          if (lo + (i64)base >= hi) {
            ++steal;
            continue;
          }
          qn = lo + (i64)base;
          qe = qn + kClaim < hi ? qn + kClaim : hi;
        }
        const int rk = __popcll(mask & ((1ull << lane) - 1ull));
        const i64 avail = qe - qn;
        const int cnt = __popcll(mask);
        if (needy && rk < avail) {
          cell = listed ? (i64)A.list[qn + rk] : qn + rk;
          needy = false;
          // a rescue pass takes only the cells an earlier pass handed over
          if (A.rescue && A.status[cell] != kEscalate) {
            cell = -1;
            needy = true;
          }
        }
        qn += cnt < avail ? cnt : avail;
        mask = __ballot(needy);
      }
    }
    if (__all(cell < 0)) break;  // every lane of the wave is done
    }
    if (cell < 0) continue;
    const i64 c = cell;

    // ---------------- load the cell; RStep set-up ----------------
    if (mode == 2) continue;  // waits to be written back
    if (mode == 0) {
      const i64 lo = opaque(ld);
      // every load of a block is issued before the first value is used: one
      // wavefront per SIMD has nothing else to hide a load's latency with
      por = A.porosity[c];
      sat = A.saturation[c];
      const double den = A.den_kg[c];
      vol = A.volume[c];
      temp = A.temperature ? A.temperature[c] : 25.0;
      ln_aw = (Net::ACT_H2O && A.ln_act_h2o) ? A.ln_act_h2o[c] : 0.0;
      double tin[N], gam[NA1], vf[NM1], ar[NM1];
      {
        const double* pp = A.pri_molal + c;
        const double* pt = A.total + c;
        const double* pg = A.pri_act_coef + c;
        sfor<0, NAQ>([&](auto I) {
          constexpr int i = decltype(I)::value;
          x[i] = *pp;
          tin[i] = *pt;
          gam[i] = *pg;
          pp += lo;
          pt += lo;
          pg += lo;
        });
        sfor<0, NIMM>([&](auto I) {
          constexpr int i = decltype(I)::value;
          x[NAQ + i] = A.immobile[i * lo + c];
          tin[NAQ + i] = x[NAQ + i];
        });
        const double* pv = A.mnrl_volfrac + c;
        const double* pa = A.mnrl_area + c;
        sfor<0, NM>([&](auto M) {
          constexpr int m = decltype(M)::value;
          vf[m] = *pv;
          ar[m] = *pa;
          pv += lo;
          pa += lo;
        });
      }
      issue_loads();
      tk = temp + 273.15;
      lnT = pf_log(tk);
      dkl = den * 1.0e-3;
      psv = por * sat * 1000.0 * vol;
      sfor<0, NAQ>([&](auto I) {
        constexpr int i = decltype(I)::value;
        PF_GAM(i) = act_keep(gam[i]);
      });
      sfor<0, NM>([&](auto M) {
        constexpr int m = decltype(M)::value;
        PF_VF(m) = vf[m];
        PF_AREA(m) = ar[m];
        PF_RLAST(m) = 0.0;
      });
      if constexpr (NEWTON_ACT) {
        sec_I = sec_sum = 0.0;
        sfor<0, NC>([&](auto K) {
          constexpr int k = decltype(K)::value;
          const double mk = A.sec_molal[k * lo + c];
          sec_I += mk * Net::CPLX_Z[k] * Net::CPLX_Z[k];
          sec_sum += mk;
        });
      }
      if constexpr (!NEWTON_ACT) {
        // The Debye-Hueckel law gives complexes of equal charge magnitude
        // and ion size equal coefficients (and neutral ones exactly 1), so
        // each (Z^2, a0) class keeps one inverse coefficient for the whole
        // step.  A cell whose input coefficients break that structure is
        // handed to the team kernel, which reads them per complex.
        bool odd = false;
        double g0[NG1];
        const double* pg = A.sec_act_coef + c;
        constexpr int CH = 16;  // complexes per block of loads
        sfor<0, (NC + CH - 1) / CH>([&](auto B) {
          constexpr int k0 = decltype(B)::value * CH, k1 = k0 + CH < NC ? k0 + CH : NC;
          double g[CH];
          sfor<k0, k1>([&](auto K) {
            g[decltype(K)::value - k0] = *pg;
            pg += lo;
          });
          issue_loads();
          sfor<k0, k1>([&](auto K) {
            constexpr int k = decltype(K)::value;
            constexpr int q = Net::CPLX_GCLS[k];
            if constexpr (q < 0) {
              odd |= !(g[k - k0] == 1.0);
            } else if constexpr (Net::CPLX_GFIRST[k]) {
              g0[q] = g[k - k0];
              PF_GINV(q) = rcp_nr(g[k - k0]);
            } else {
              odd |= !(g[k - k0] == g0[q]);
            }
          });
        });
        if (odd && A.escalate) {
          hand_over(A, c);
          cell = -1;
          continue;
        }
      }
      if constexpr (!Net::FULL_GEOCHEM) {
        // RStep early exit (reaction.F90:3601-3605)
        sfor<0, NAQ>([&](auto I) {
          constexpr int i = decltype(I)::value;
          A.pri_molal[i * lo + c] = tin[i] / den * 1.0e3;
        });
        if (A.num_iterations) A.num_iterations[c] = 0;
        if (A.num_sub_steps) A.num_sub_steps[c] = 0;
        if (A.status) A.status[c] = 0;
        cell = -1;
        continue;
      }
#if PFLANE_SD
      sdc.dkl = dkl;
      sdc.theta = por * sat;
      sdc.vol = vol;
      sdc.sat = sat;
      sd_load(sdc, temp, A.sd_ft != nullptr, A.sd_ft ? A.sd_ft[c] : 1.0, A.sd_fw != nullptr,
              A.sd_fw ? A.sd_fw[c] : 1.0);
#endif
      // clamp small totals (reaction.F90:3617-3631)
      small = 0u;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        if (tin[i] <= 1.0e-40) {
          small |= 1u << i;
          tin[i] = 1.0e-40;
        }
        PF_TINIT(i) = tin[i];
        PF_GUESS(i) = (Net::TOTAL_AS_GUESS && i < NAQ) ? tin[i] : x[i];
      }
      target = A.dt;
      cum = 0.0;
      tdt = A.dt;
      nconst = ncuts = nsub = nit_total = status = attempts = last_why = 0;
      restore = false;
      kin = false;
      nit = -1;
      mode = 1;
    }

    // ---------------- RReact set-up (reaction.F90:3800-3851) ----------------
    if (mode == 1 && nit < 0) {
      if (++attempts > Net::MAX_CALLS) {
        status = last_why ? last_why : kMaxIter;
        mode = 2;
      } else {
#pragma unroll
        for (int i = 0; i < N; ++i) x[i] = PF_GUESS(i);
        nit = 0;
        r0 = 0.0;
      }
    }
    if (mode == 2) continue;  // no call left: written back next time round
    ++nit;

    // ---------------- RTotal + RReaction at x ----------------
    const bool wet = !(sat < kRtMinSat);
    const double itdt = rcp_nr(tdt);
    const double psvd = psv * itdt;
    const double jc = psvd * dkl;
    const double wm = wet ? 1.0 : 0.0;
    // activity coefficients per Newton iteration (LAG at the current pri
    // and last secondary molalities)
    double I = 0.0, sI = 0.0;
    if constexpr (NEWTON_ACT) {
      {
        double Ip = 0.0, sp = 0.0;
        sfor<0, NAQ>([&](auto Q) {
          constexpr int i = decltype(Q)::value;
          Ip += x[i] * Net::ZP[i] * Net::ZP[i];
          if (i != Net::H2O_ID) sp += x[i];
        });
        I = 0.5 * (Ip + sec_I);
        sI = sqrt(I);
        sfor<0, NAQ>([&](auto Q) {
          constexpr int i = decltype(Q)::value;
          if constexpr (Net::ZP[i] > 1.0e-10 || Net::ZP[i] < -1.0e-10)
            PF_GAM(i) = act_keep(dh_gamma(Net::ZP[i], Net::A0P[i], sI, I));
          else
            PF_GAM(i) = act_keep(1.0);
        });
        if constexpr (Net::ACT_H2O) {
          const double a = 1.0 - 0.017 * (sp + sec_sum);
          ln_aw = a > 0.0 ? pf_log(a) : 0.0;
        }
        I_last = I;
      }
    }
    Acts<NA1> act;
    double tot[NA1], D[NA1], sig[NA1];
    JT S[NT];
    sfor<0, NAQ>([&](auto Q) {
      constexpr int i = decltype(Q)::value;
      act_set<i>(act, x[i], PF_GAM(i));
      // FP32 entries are accumulated pre-scaled by sig_i sig_j (any scale
      // works: it is divided out exactly below); FP64 ones are not scaled
      sig[i] = F32 ? __builtin_amdgcn_rsq(x[i]) : 1.0;
      tot[i] = 0.0;
      D[i] = wet ? x[i] : 1.0;
    });
#pragma unroll
    for (int q = 0; q < NT; ++q) S[q] = (JT)0;
    double nsI = 0.0, nss = 0.0;
    double gi[NG1];
    sfor<0, NG>([&](auto Q) {
      constexpr int q = decltype(Q)::value;
      gi[q] = PF_GINV(q);
    });
    // complexes (RTotalAqueous, reaction.F90:4665-4759)
    sfor<0, NC>([&](auto K) {
      constexpr int k = decltype(K)::value;
      constexpr int ns = Net::CPLX_N[k];
      double g;
      const double m = cplx_m<k, NEWTON_ACT>(act, lnT, tk, ln_aw, gi, sI, I, g);
      if constexpr (NEWTON_ACT) {
        nsI += m * (Net::CPLX_Z[k] * Net::CPLX_Z[k]);
        nss += m;
      }
      const double mj = m * wm;
      sfor<0, ns>([&](auto Q) {
        constexpr int a = decltype(Q)::value;
        constexpr int ia = Net::CPLX_ID[k][a];
        constexpr double na = Net::CPLX_NU[k][a];
        tot[ia] += na * m;
        D[ia] += (na * na) * mj;
        const double pa = mj * sig[ia];
        sfor<a + 1, ns>([&](auto Q2) {
          constexpr int b = decltype(Q2)::value;
          constexpr int ib = Net::CPLX_ID[k][b];
          constexpr double nab = na * Net::CPLX_NU[k][b];
          if constexpr (ia == ib) {
            D[ia] += (2.0 * nab) * mj;
          } else {
            S[tri(ia, ib)] += (JT)nab * (JT)(pa * sig[ib]);
          }
        });
      });
    });
    // residual (RTAccumulation, reaction.F90:3899-3916) and its norms
    double res[N], totc[NA1];
    double mx = 0.0, nr2 = 0.0;
    sfor<0, NAQ>([&](auto Q) {
      constexpr int i = decltype(Q)::value;
      totc[i] = (x[i] + tot[i]) * dkl;
      res[i] = wet ? (psv * totc[i] - psv * PF_TINIT(i)) * itdt : 0.0;
    });
    sfor<0, NIMM>([&](auto Q) {
      constexpr int i = NAQ + decltype(Q)::value;
      double r = wet ? (x[i] * vol - PF_TINIT(i) * vol) * itdt : 0.0;
      sfor<0, Net::NDECAY>([&](auto Dq) {
        constexpr int d = decltype(Dq)::value;
        if constexpr (Net::DECAY_ID[d] == i - NAQ) {
          if (wet) r += Net::DECAY_K[d] * vol * x[i];
        }
      });
      res[i] = r;
    });
    // kinetic minerals (RKineticMineral, after the accumulation terms as in
    // RReaction): rates, residual and Jacobian terms
    double rt[NM1];
    const double ijc = wet ? rcp_nr(jc) : 0.0;
    sfor<0, NM>([&](auto Mi) {
      constexpr int mi = decltype(Mi)::value;
      constexpr int ns = Net::MNRL_N[mi];
      rt[mi] = 0.0;
      const double ar = PF_AREA(mi);
      // zero area gives Im = 0.  The plain rate law runs without branches:
      // with a few minerals active per cell some lane of a wavefront has
      // each of them, and the branches kept the complexes' arithmetic from
      // being scheduled across them
      constexpr bool plain = Net::HAS_TEMKIN + Net::HAS_MINSCALE + Net::HAS_AFFPOWER +
                                 Net::HAS_LIMITER + Net::HAS_IRREV + Net::HAS_THRESHOLD +
                                 Net::HAS_EA == 0;
      if (plain || ar != 0.0) {
        const double QK = mnrl_q<mi>(act, lnT, tk, ln_aw);
        MRate r;
        if constexpr (plain) {
          const double aff = 1.0 - QK;
          r.active = ar != 0.0 && (PF_VF(mi) > 0.0 || QK > 1.0);
          r.Im = r.active ? -(ar * aff) * Net::MNRL_K[mi] : 0.0;
          r.dIm = ar * Net::MNRL_K[mi];
        } else {
          r = mineral_rate<mi>(QK, PF_VF(mi), ar, temp);
        }
        if (plain || r.active) {
          rt[mi] = r.Im;
          // dry cells: RReaction adds nothing (reaction.F90:4083)
          const double Rm = r.Im * vol * wm;
          // d res / d ln m_j = nu_i (dIm/dQK QK V rho/1000) nu_j, in units of jc
          // (selected here: an inactive mineral's Q/K may be infinite)
          const double gm = r.active ? r.dIm * vol * QK * dkl * ijc : 0.0;
          sfor<0, ns>([&](auto Q) {
            constexpr int a = decltype(Q)::value;
            constexpr int ia = Net::MNRL_ID[mi][a];
            constexpr double na = Net::MNRL_NU[mi][a];
            res[ia] += na * Rm;
            D[ia] += (na * na) * gm;
            const double pa = gm * sig[ia];
            sfor<a + 1, ns>([&](auto Q2) {
              constexpr int b = decltype(Q2)::value;
              constexpr int ib = Net::MNRL_ID[mi][b];
              constexpr double nab = na * Net::MNRL_NU[mi][b];
              if constexpr (ia == ib) {
                D[ia] += (2.0 * nab) * gm;
              } else {
                S[tri(ia, ib)] += (JT)nab * (JT)(pa * sig[ib]);
              }
            });
          });
        }
      }
    });
#if PFLANE_SD
    SdSum sds;
    bool balanced = false;
#pragma unroll
    for (int i = 0; i < N; ++i) sds.R[i] = 0.0;
#pragma unroll
    for (int q = 0; q < Net::JNNZ; ++q) sds.J[q] = 0.0;
    if (wet) {
      sdc.tdt = tdt;
      sdc.itdt = itdt;
      double nmin = 0.0, nabs = 0.0;
      sfor<0, Net::SDN>([&](auto Q) {
        const double v = sd_reaction<decltype(Q)::value>(sdc, x, sds);
        nmin += v;
        nabs += fabs(v);
      });
      // The N2O emission follows the net N mineralization.  Where that is a
      // small positive difference of mineralization and immobilization, its
      // rounding keeps the relative change of N2O above the tolerance, and
      // whether RReact ends or its step is cut is decided by rounding (every
      // cell of 3.6 million that was cut but one had a net below 1 % of the
      // terms, 99 % of them below 0.5 %; 0.2 % of all cells are that close).
      // Those cells are handed to the team kernel, with them every cell
      // whose step would be cut.
      balanced = Net::SD_N2O >= 0 && nmin > 0.0 && nmin < 0.005 * nabs;
      double lnh = 0.0;
      if constexpr (Net::SD_PROTON >= 0) lnh = act.l[Net::SD_PROTON];
      sd_emission(sdc, x, lnh, nmin, sds);
#pragma unroll
      for (int i = 0; i < N; ++i) res[i] += sds.R[i];
    }
#endif
#pragma unroll
    for (int i = 0; i < N; ++i) {
      mx = fmax(mx, fabs(res[i]));
      nr2 += res[i] * res[i];
    }

    if constexpr (NEWTON_ACT) {
      sec_I = nsI;
      sec_sum = nss;
    }
    sfor<0, NM>([&](auto M) {
      constexpr int m = decltype(M)::value;
      PF_RLAST(m) = rt[m];
    });
    const double nr = sqrt(nr2);
    if (nit == 1) r0 = nr;
    // 0 continue, 1 converged, 2 max iterations, 3 hand over
    int outcome = 0;
    // FP32: when the convergence test first passes on the last sub-step, one
    // more FP32-preconditioned correction of the FP64 residual is applied
    // before the cell exits (the write-out evaluates at the corrected
    // state): the exit test bounds the residual, not the error, and the
    // linear convergence of the FP32-preconditioned iteration would leave
    // up to about 1e-9 of relative error at the exit
    bool polish = false;
    if (nit > Net::MAX_IT) {
      outcome = 2;
    } else if (mx < Net::TOL_ABS || nr / r0 < Net::TOL_REL) {
      if (F32 && !SD && cum + tdt >= target) polish = true;
      else outcome = 1;
    }
    if (outcome == 0) {
      // ---------------- linear solve (RSolve) ----------------
#if PFLANE_SD
      // the sandbox's system is not symmetric, but sparse: a pool's column
      // meets the pools it feeds, NH4+, NO3- and CO2; the other columns are
      // diagonal.  LU in natural order on the pattern closed under fill-in,
      // rows scaled by their accumulation diagonal, columns in the log form
      // (as the team kernel, whose Crout factorization takes the cells a
      // pivot test hands over).
      JT a[Net::JNNZ], b[N], pinv[N];
      bool bad = false;
      double amax[N];
      sfor<0, N>([&](auto Q) {
        constexpr int i = decltype(Q)::value;
        double rs = 1.0, d = 1.0;
        if (wet) rs = i < NAQ ? rcp_nr(jc * x[i]) : rcp_nr(vol * itdt * x[i]);
        sfor<0, Net::NDECAY>([&](auto Dq) {
          constexpr int dd = decltype(Dq)::value;
          if constexpr (Net::DECAY_ID[dd] == i - NAQ && i >= NAQ) {
            if (wet) d += Net::DECAY_K[dd] * vol * x[i] * rs;
          }
        });
        double am = 0.0;
        sfor<0, N>([&](auto Q2) {
          constexpr int j = decltype(Q2)::value;
          constexpr int q = Net::JPOS[i][j];
          if constexpr (q >= 0) {
            double v = sds.J[q] * x[j] * rs;
            if constexpr (i == j) v += d;
            a[q] = (JT)v;
            am = fmax(am, fabs(v));
          }
        });
        amax[i] = am;
        b[i] = (JT)(res[i] * rs);
      });
      constexpr double kLuTol = F32 ? 1.0e-6 : 1.0e-12;
      sfor<0, N>([&](auto P) {
        constexpr int p = decltype(P)::value;
        const JT pv = a[Net::JPOS[p][p]];
        // A pivot small against its row makes the rows below it grow by its
        // multipliers.  A column without entries below the diagonal has
        // none: its unknown (a tracking species, the gases) is read off its
        // own row, whose terms may be any multiple of the pivot, as they are
        // where it starts empty.
        const double av = (double)(pv < (JT)0 ? -pv : pv);
        constexpr bool below = lu_eliminates(p);
        if (!(av > (below ? kLuTol * amax[p] : 0.0) && av < 1.0e300)) bad = true;  // or not finite
        const JT inv = F32 ? (JT)1 / pv : (JT)rcp_nr((double)pv);
        pinv[p] = inv;
        sfor<p + 1, N>([&](auto Q) {
          constexpr int i = decltype(Q)::value;
          if constexpr (Net::JPOS[i][p] >= 0) {
            const JT l = a[Net::JPOS[i][p]] * inv;
            sfor<p + 1, N>([&](auto Q2) {
              constexpr int j = decltype(Q2)::value;
              if constexpr (Net::JPOS[p][j] >= 0) a[Net::JPOS[i][j]] -= l * a[Net::JPOS[p][j]];
            });
            b[i] -= l * b[p];
          }
        });
      });
      double delta[N];
      sfor<0, N>([&](auto Q) {
        constexpr int i = N - 1 - decltype(Q)::value;
        sfor<i + 1, N>([&](auto Q2) {
          constexpr int j = decltype(Q2)::value;
          if constexpr (Net::JPOS[i][j] >= 0) b[i] -= a[Net::JPOS[i][j]] * b[j];
        });
        b[i] *= pinv[i];
        delta[i] = (double)b[i];
        if (!(delta[i] == delta[i])) bad = true;
      });
#else
      // aqueous block M delta = res / jc by L D L^T.  SCALED: symmetric
      // scaling to (about) unit diagonal, A = D^-1/2 M D^-1/2; any positive s
      // gives the same step, so the hardware estimate of 1/sqrt(D_i) is
      // used.  FP64 needs no scaling (the elimination's relative rounding
      // does not depend on it); the pivot test is relative to each diagonal.
      constexpr bool SCALED = F32 || !kProd;
      JT a[NT], dg[NA1], b[NA1], dinv[NA1], piv0[NA1], rr[NA1];
      double s[NA1];
      const double ijs = wet ? ijc : 1.0;
      bool bad = false;
      sfor<0, NAQ>([&](auto Q) {
        constexpr int i = decltype(Q)::value;
        if constexpr (SCALED) {
          s[i] = __builtin_amdgcn_rsq(D[i]);
          rr[i] = F32 ? (JT)(s[i] * rcp_nr(sig[i])) : (JT)s[i];  // ~sqrt(x_i / D_i)
          dg[i] = (JT)(D[i] * s[i] * s[i]);
          b[i] = (JT)(res[i] * s[i] * ijs);
          piv0[i] = (JT)kPivTol;
        } else {
          dg[i] = D[i];
          b[i] = res[i] * ijs;
          piv0[i] = D[i] * kPivTol;
        }
        sfor<0, i>([&](auto Q2) {
          constexpr int j = decltype(Q2)::value;
          if constexpr (SCALED) a[tri(i, j)] = S[tri(i, j)] * rr[i] * rr[j];
          else a[tri(i, j)] = S[tri(i, j)];
        });
      });
      // right-looking
      sfor<0, NAQ>([&](auto P) {
        constexpr int p = decltype(P)::value;
        const JT dp = dg[p];
        if (!((double)dp > (double)piv0[p])) bad = true;  // also for a NaN
        const JT inv = SCALED ? (JT)1 / dp : (JT)rcp_nr((double)dp);
        dinv[p] = inv;
        JT l[NA1];
        sfor<p + 1, NAQ>([&](auto Q) {
          constexpr int i = decltype(Q)::value;
          l[i] = a[tri(i, p)] * inv;
        });
        sfor<p + 1, NAQ>([&](auto Q) {
          constexpr int i = decltype(Q)::value;
          dg[i] -= l[i] * a[tri(i, p)];
          sfor<p + 1, i>([&](auto Q2) {
            constexpr int j = decltype(Q2)::value;
            a[tri(i, j)] -= l[i] * a[tri(j, p)];
          });
        });
        sfor<p + 1, NAQ>([&](auto Q) {
          constexpr int i = decltype(Q)::value;
          a[tri(i, p)] = l[i];
        });
      });
      // forward (L z = b), diagonal, backward (L^T y = z)
      sfor<0, NAQ>([&](auto Q) {
        constexpr int i = decltype(Q)::value;
        sfor<0, i>([&](auto Q2) {
          constexpr int j = decltype(Q2)::value;
          b[i] -= a[tri(i, j)] * b[j];
        });
      });
      sfor<0, NAQ>([&](auto Q) {
        constexpr int i = decltype(Q)::value;
        b[i] *= dinv[i];
      });
      sfor<0, NAQ>([&](auto Q) {
        constexpr int i = NAQ - 1 - decltype(Q)::value;
        sfor<i + 1, NAQ>([&](auto Q2) {
          constexpr int j = decltype(Q2)::value;
          b[i] -= a[tri(j, i)] * b[j];
        });
      });
      double delta[N];
      sfor<0, NAQ>([&](auto Q) {
        constexpr int i = decltype(Q)::value;
        delta[i] = SCALED ? (double)b[i] * s[i] : (double)b[i];
        if (!(delta[i] == delta[i])) bad = true;
      });
      // immobile rows: accumulation + decay on the diagonal
      sfor<0, NIMM>([&](auto Q) {
        constexpr int i = NAQ + decltype(Q)::value;
        double d = vol * itdt * x[i];
        sfor<0, Net::NDECAY>([&](auto Dq) {
          constexpr int dd = decltype(Dq)::value;
          if constexpr (Net::DECAY_ID[dd] == i - NAQ) d += Net::DECAY_K[dd] * vol * x[i];
        });
        if (!wet) d = 1.0;
        delta[i] = res[i] * rcp_nr(d);
        if (!(d > 0.0)) bad = true;
      });
#endif
      if (!Net::LOG_FORM) {
#pragma unroll
        for (int i = 0; i < N; ++i) delta[i] *= x[i];
      }
      if (bad) {
        outcome = 3;
      } else {
        // ---------------- update (reaction.F90:3977-4049) ----------------
        double latest[N], rc = -1.0;
        // The small-step exit holds for the FP32 factorization too: scaled
        // to unit diagonal, M has |M_ij| <= 1 (positive semi-definite
        // terms), so |M| <= n and a step below the tolerance certifies a
        // scaled FP64 residual |b| <= n |y| of the same size.
        if constexpr (Net::LOG_FORM) {
#pragma unroll
          for (int i = 0; i < N; ++i) {
            const double u = copysign(1.0, delta[i]) * fmin(fabs(delta[i]), Net::MAX_DLNC);
            const double f = exp_step(-u);
            latest[i] = x[i] * f;
            // |latest - x| / x
            const double q = kProd || SD ? fabs(f - 1.0) : fabs((latest[i] - x[i]) * rcp_nr(x[i]));
            if (q == q) rc = fmax(rc, q);
          }
        } else {
          double ratio = 1.0e308;
#pragma unroll
          for (int i = 0; i < N; ++i)
            if (x[i] <= delta[i]) ratio = fmin(ratio, fabs(x[i] / delta[i]));
#pragma unroll
          for (int i = 0; i < N; ++i) {
            latest[i] = x[i] - (ratio < 1.0 ? delta[i] * ratio * 0.99 : delta[i]);
            const double q = fabs((latest[i] - x[i]) * rcp_nr(x[i]));
            if (q == q) rc = fmax(rc, q);
          }
        }
        if (polish) {
#pragma unroll
          for (int i = 0; i < N; ++i) x[i] = latest[i];
          outcome = 1;
        } else if (rc >= 0.0 && rc < Net::TOL_CHANGE && (!F32 || !SD || nr <= 1.0e-11 * r0)) {
          // (the certificate above is the symmetric system's: the sandbox's
          // FP32 exit asks the FP64 residual)
          outcome = 1;
        } else {
#pragma unroll
          for (int i = 0; i < N; ++i) x[i] = latest[i];
        }
      }
    }

#if PFLANE_SD
    if (A.escalate && (outcome == 2 || (outcome == 1 && balanced))) outcome = 3;
#endif
    // ---------------- RReact / RStep transitions ----------------
    if (outcome == 1) {
      // RUpdateKineticState (reaction_mineral.F90:1456-1525); the last
      // sub-step's is done by the write-out evaluation at the final state
      const bool last = cum + tdt >= target;
      if (!last) {
        sfor<0, NM>([&](auto M) {
          constexpr int m = decltype(M)::value;
          double v = PF_VF(m) + rt[m] * Net::MNRL_VM[m] * tdt;
          if (v < 0.0) v = 0.0;
          PF_VF(m) = v;
        });
      }
      nit_total += nit;
      cum += tdt;
      ++nsub;
      ++nconst;
      sfor<0, NAQ>([&](auto Q) {
        constexpr int i = decltype(Q)::value;
        PF_TINIT(i) = totc[i];
      });
#pragma unroll
      for (int i = NAQ; i < N; ++i) PF_TINIT(i) = x[i];
#pragma unroll
      for (int i = 0; i < N; ++i) PF_GUESS(i) = x[i];
      nit = -1;
      if (cum >= target) {
        status = 0;
        kin = true;
        mode = 2;  // tdt stays the last sub-step's (the kinetic update uses it)
      } else if (nconst >= 4) {
        --ncuts;
        tdt = fmin(2.0 * tdt, target - cum);
      }
    } else if (outcome == 3 || (outcome == 2 && F32 && A.escalate)) {
      // hand the untouched cell to the next pass
      if (A.escalate) {
        hand_over(A, c);
        cell = -1;
        mode = 0;
        continue;
      }
      // no later pass: a singular system (the reference's zero-row failure)
      nit_total += nit;
      sfor<0, NAQ>([&](auto Q) {
        constexpr int i = decltype(Q)::value;
        PF_TINIT(i) = totc[i];
      });
#pragma unroll
      for (int i = NAQ; i < N; ++i) PF_TINIT(i) = x[i];
      restore = false;
      last_why = kSingular;
      ++ncuts;
      if (ncuts > Net::MAX_CUTS) {
        status = last_why;
        mode = 2;
      } else {
        tdt *= 0.5;
        nconst = 0;
        nit = -1;
      }
    } else if (outcome == 2) {
      // maximum iterations: totals / immobile restored (reaction.F90:3869-3895)
      nit_total += nit;
      restore = true;
      last_why = kMaxIter;
      ++ncuts;
      if (ncuts > Net::MAX_CUTS) {
        status = last_why;
        mode = 2;
      } else {
        tdt *= 0.5;
        nconst = 0;
        nit = -1;
      }
    }
  }
#undef PF_GUESS
#undef PF_TINIT
#undef PF_GAM
#undef PF_VF
#undef PF_AREA
#undef PF_RLAST
#undef PF_GINV
}

}  // namespace pflane

// one module holds the step kernels, or (PFLANE_ADJOINT defined) the adjoint
// kernel, or (PFLANE_GIRT) the GIRT block, so a context compiles what it uses
#if !defined(PFLANE_ADJOINT) && !defined(PFLANE_GIRT)
extern "C" __global__ void __launch_bounds__(256) pfchem_lane_step_f32(pflane::Args a) {
  pflane::lane_step<float>(a);
}
extern "C" __global__ void __launch_bounds__(256) pfchem_lane_step_f64(pflane::Args a) {
  pflane::lane_step<double>(a);
}
#endif

// ---------------------------------------------------------------------------
// Adjoint of one reaction step, one cell per lane, FP64.
//
// The step is RStep's accepted sub-steps s of size h_s, each the converged
// RReact system (reaction.F90:3742-4055)
//   F(m; T0, VF0, p) = psv (T(m; p) - T0) / h + vol sum_q nu_q Im_q(m; p) = 0
// followed by VF = max(0, VF0 + Im V_m h) (reaction_mineral.F90:1456-1525);
// the next sub-step starts from T(m), VF.  Objective per cell:
// f = sum_q wv_q VF_q(end) + sum_k ws_k m_k(end); parameters log10 k_q
// (rate constants) and log10 K_k (complexes).  The forward pass repeats the
// step (the FP64 solve of pfchem_lane_step_f64) and records each accepted
// sub-step (m, VF0, h) in a per-cell log; the reverse pass applies the
// implicit-function theorem at each recorded solution, one solve per
// sub-step.  In the log form J diag(m) = jc M with M symmetric
// (M = diag(m) + S^T diag(m_k) S + sum_q g_q nu_q nu_q^T), so the transposed
// solve J^T lambda = b is M lambda = diag(m) b / jc with the same L D L^T.
// The mineral block of M carries rho/1000 in the Newton iteration (the
// reference's dQK_dmj, reaction_mineral.F90:945) and in the sensitivities
// only when asked (jacobian = 0); otherwise it is the exact derivative.
// Scope: aqueous networks without immobile species, TST rates with optional
// Arrhenius factor, activity coefficients fixed during the step.  A cell the
// pass cannot take (a pivot below tolerance, activity coefficients that do
// not follow the charge/size classes) is left with status kEscalate for the
// general kernel.
namespace pflane {

constexpr int kSensSub = 8;  // sub-steps one cell may record

struct SensArgs {
  i64 ld, ncell;
  const double* pri_molal;
  const double* total;
  const double* pri_act_coef;
  const double* sec_act_coef;
  const double* ln_act_h2o;
  const double* mnrl_volfrac;
  const double* mnrl_area;
  const double* porosity;
  const double* saturation;
  const double* den_kg;
  const double* volume;
  const double* temperature;
  const double* wv;    // [NM] weights of the end-of-step volume fractions
  const double* ws;    // [NC] weights of the end-of-step secondary molalities
  double* grad;        // [(NM + NC) * ldo] per-cell gradient
  i64 ldo;
  double* fcell;       // [ncell] objective per cell, or null
  int* status;         // [ncell]
  double* log;         // [kSensSub * (NAQ + NM + 1) * ldl] sub-step log
  i64 ldl;
  double dt;
  int jacobian;        // 1: exact dF/dm; 0: the reference's mineral block
  int pad;
};
static_assert(sizeof(SensArgs) == 192, "SensArgs layout");

// L D L^T solve of the symmetrically scaled M (diagonal dg, strict lower
// packed a; both overwritten by the factors): M y = b in place; false if a
// pivot is below tolerance
template <int NA>
__device__ __forceinline__ bool sens_ldlt(double (&dg)[NA], double (&a)[NA > 1 ? NA * (NA - 1) / 2 : 1],
                                          double (&b)[NA]) {
  double s[NA], dinv[NA];
  sfor<0, NA>([&](auto Q) {
    constexpr int i = decltype(Q)::value;
    s[i] = __builtin_amdgcn_rsq(dg[i]);
    dg[i] = dg[i] * s[i] * s[i];
    b[i] *= s[i];
  });
  sfor<1, NA>([&](auto Q) {
    constexpr int i = decltype(Q)::value;
    sfor<0, i>([&](auto Q2) {
      constexpr int j = decltype(Q2)::value;
      a[tri(i, j)] *= s[i] * s[j];
    });
  });
  bool bad = false;
  sfor<0, NA>([&](auto P) {
    constexpr int p = decltype(P)::value;
    const double dp = dg[p];
    if (!(dp > 1.0e-13)) bad = true;
    const double inv = 1.0 / dp;
    dinv[p] = inv;
    double l[NA];
    sfor<p + 1, NA>([&](auto Q) {
      constexpr int i = decltype(Q)::value;
      l[i] = a[tri(i, p)] * inv;
    });
    sfor<p + 1, NA>([&](auto Q) {
      constexpr int i = decltype(Q)::value;
      dg[i] -= l[i] * a[tri(i, p)];
      sfor<p + 1, i>([&](auto Q2) {
        constexpr int j = decltype(Q2)::value;
        a[tri(i, j)] -= l[i] * a[tri(j, p)];
      });
    });
    sfor<p + 1, NA>([&](auto Q) {
      constexpr int i = decltype(Q)::value;
      a[tri(i, p)] = l[i];
    });
  });
  sfor<0, NA>([&](auto Q) {
    constexpr int i = decltype(Q)::value;
    sfor<0, i>([&](auto Q2) {
      constexpr int j = decltype(Q2)::value;
      b[i] -= a[tri(i, j)] * b[j];
    });
  });
  sfor<0, NA>([&](auto Q) {
    constexpr int i = decltype(Q)::value;
    b[i] *= dinv[i];
  });
  sfor<0, NA>([&](auto Q) {
    constexpr int i = NA - 1 - decltype(Q)::value;
    sfor<i + 1, NA>([&](auto Q2) {
      constexpr int j = decltype(Q2)::value;
      b[i] -= a[tri(j, i)] * b[j];
    });
  });
  sfor<0, NA>([&](auto Q) {
    constexpr int i = decltype(Q)::value;
    b[i] *= s[i];
    if (!(b[i] == b[i])) bad = true;
  });
  return !bad;
}

__device__ inline void lane_adjoint(const SensArgs& A) {
  constexpr int NAQ = Net::NAQ, NC = Net::NC, NM = Net::NM;
  constexpr int NA1 = NAQ > 0 ? NAQ : 1, NM1 = NM > 0 ? NM : 1;
  constexpr int NT = NA1 > 1 ? NA1 * (NA1 - 1) / 2 : 1;
  constexpr int NG = Net::NGCLS, NG1 = NG > 0 ? NG : 1;
  constexpr int NF = NAQ + NM + 1;  // log fields per sub-step
  const i64 c = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= A.ncell) return;
  const i64 ld = A.ld, ldo = A.ldo, ldl = A.ldl;
  if constexpr (Net::NIMM > 0 || Net::ACT_FREQ == kFreqNewtonIter || !Net::FULL_GEOCHEM) {
    A.status[c] = kEscalate;  // outside this pass's scope
    return;
  } else {
    // ---------------- cell constants ----------------
    const double por = A.porosity[c], sat = A.saturation[c];
    const double den = A.den_kg[c], vol = A.volume[c];
    const double temp = A.temperature ? A.temperature[c] : 25.0;
    const double tk = temp + 273.15, lnT = pf_log(tk);
    const double ln_aw = (Net::ACT_H2O && A.ln_act_h2o) ? A.ln_act_h2o[c] : 0.0;
    const double dkl = den * 1.0e-3, psv = por * sat * 1000.0 * vol;
    auto zero_grad = [&]() {
      sfor<0, NM + NC>([&](auto Q) {
        constexpr int q = decltype(Q)::value;
        A.grad[q * ldo + c] = 0.0;
      });
    };
    if (sat < kRtMinSat) {  // dry: no sensitivity
      zero_grad();
      A.status[c] = 4;  // PFCHEM_CELL_SENS_UNSUPPORTED
      return;
    }
    double gam[NA1], gi[NG1], area[NM1], vf[NM1];
    sfor<0, NAQ>([&](auto Q) {
      constexpr int i = decltype(Q)::value;
      gam[i] = act_keep(A.pri_act_coef[i * ld + c]);
    });
    bool cons = true;
    {
      double g0[NG1];
      const double* pg = A.sec_act_coef + c;
      constexpr int CH = 20;  // loads issued before the first is compared
      sfor<0, (NC + CH - 1) / CH>([&](auto B) {
        constexpr int k0 = decltype(B)::value * CH, k1 = k0 + CH < NC ? k0 + CH : NC;
        double g[CH];
        sfor<k0, k1>([&](auto K) {
          g[decltype(K)::value - k0] = *pg;
          pg += ld;
        });
        issue_loads();
        sfor<k0, k1>([&](auto K) {
          constexpr int k = decltype(K)::value;
          constexpr int q = Net::CPLX_GCLS[k];
          if constexpr (q < 0) {
            cons &= g[k - k0] == 1.0;
          } else if constexpr (Net::CPLX_GFIRST[k]) {
            g0[q] = g[k - k0];
            gi[q] = 1.0 / g[k - k0];
          } else {
            cons &= g[k - k0] == g0[q];
          }
        });
      });
    }
    if (!cons) {
      A.status[c] = kEscalate;
      return;
    }
    sfor<0, NM>([&](auto M) {
      constexpr int m = decltype(M)::value;
      vf[m] = A.mnrl_volfrac[m * ld + c];
      area[m] = A.mnrl_area[m * ld + c];
    });
    // secondary molality of complex K at the activities ac
    auto cplx_m = [&](auto K, const Acts<NA1>& ac) {
      constexpr int k = decltype(K)::value;
      if constexpr (Net::CPLX_GCLS[k] >= 0)
        return cplx_q<k>(ac, lnT, tk, ln_aw, gi[Net::CPLX_GCLS[k]]);
      else
        return cplx_q<k>(ac, lnT, tk, ln_aw, 1.0);
    };
    // rate of mineral M at ac with volume fraction v: Im, dIm/dlnQK
    auto mnrl_r = [&](auto Mq, const Acts<NA1>& ac, double v, double& Im, double& dI) {
      constexpr int mi = decltype(Mq)::value;
      Im = 0.0;
      dI = 0.0;
      if (area[mi] == 0.0) return false;
      const double QK = mnrl_q<mi>(ac, lnT, tk, ln_aw);
      const MRate r = mineral_rate<mi>(QK, v, area[mi], temp);
      if (!r.active) return false;
      Im = r.Im;
      dI = r.dIm * QK;
      return true;
    };
    // the system at molalities x: totals (mol/L), residual, and M's diagonal
    // D / strict lower S (in units of jc) with the mineral block times mf
    auto system = [&](const double(&x)[NA1], const double(&T0)[NA1], const double(&v0)[NM1],
                      double h, double mf, double(&T)[NA1], double(&res)[NA1], double(&D)[NA1],
                      double(&S)[NT]) {
      Acts<NA1> ac;
      double tot[NA1];
      const double jc = psv * dkl / h;
      sfor<0, NAQ>([&](auto Q) {
        constexpr int i = decltype(Q)::value;
        act_set<i>(ac, x[i], gam[i]);
        tot[i] = 0.0;
        D[i] = x[i];
      });
#pragma unroll
      for (int q = 0; q < NT; ++q) S[q] = 0.0;
      sfor<0, NC>([&](auto K) {
        constexpr int k = decltype(K)::value;
        constexpr int ns = Net::CPLX_N[k];
        const double m = cplx_m(K, ac);
        sfor<0, ns>([&](auto Q) {
          constexpr int a = decltype(Q)::value;
          constexpr int ia = Net::CPLX_ID[k][a];
          constexpr double na = Net::CPLX_NU[k][a];
          tot[ia] += na * m;
          D[ia] += (na * na) * m;
          sfor<a + 1, ns>([&](auto Q2) {
            constexpr int b = decltype(Q2)::value;
            constexpr int ib = Net::CPLX_ID[k][b];
            constexpr double nab = na * Net::CPLX_NU[k][b];
            if constexpr (ia == ib) D[ia] += (2.0 * nab) * m;
            else S[tri(ia, ib)] += nab * m;
          });
        });
      });
      sfor<0, NAQ>([&](auto Q) {
        constexpr int i = decltype(Q)::value;
        T[i] = (x[i] + tot[i]) * dkl;
        res[i] = (psv * T[i] - psv * T0[i]) / h;
      });
      sfor<0, NM>([&](auto Mq) {
        constexpr int mi = decltype(Mq)::value;
        constexpr int ns = Net::MNRL_N[mi];
        double Im, dI;
        if (!mnrl_r(Mq, ac, v0[mi], Im, dI)) return;
        const double g = dI * vol * mf / jc;
        sfor<0, ns>([&](auto Q) {
          constexpr int a = decltype(Q)::value;
          constexpr int ia = Net::MNRL_ID[mi][a];
          constexpr double na = Net::MNRL_NU[mi][a];
          res[ia] += na * Im * vol;
          D[ia] += (na * na) * g;
          sfor<a + 1, ns>([&](auto Q2) {
            constexpr int b = decltype(Q2)::value;
            constexpr int ib = Net::MNRL_ID[mi][b];
            constexpr double nab = na * Net::MNRL_NU[mi][b];
            if constexpr (ia == ib) D[ia] += (2.0 * nab) * g;
            else S[tri(ia, ib)] += nab * g;
          });
        });
      });
    };

    // ---------------- forward: RStep with the sub-step log ----------------
    double x[NA1], T0[NA1], guess[NA1], T[NA1];
    sfor<0, NAQ>([&](auto Q) {
      constexpr int i = decltype(Q)::value;
      x[i] = A.pri_molal[i * ld + c];
      T0[i] = A.total[i * ld + c];
      if (T0[i] <= 1.0e-40) T0[i] = 1.0e-40;  // reaction.F90:3617-3631
      guess[i] = Net::TOTAL_AS_GUESS ? T0[i] : x[i];
    });
    int nlog = 0, st = 0, nconst = 0, ncuts = 0, attempts = 0;
    double cum = 0.0, tdt = A.dt;
    bool handover = false;
    while (cum < A.dt) {
      if (++attempts > Net::MAX_CALLS) {
        st = kMaxIter;
        break;
      }
      double r0 = 0.0;
      int why = -1;
#pragma unroll
      for (int i = 0; i < NAQ; ++i) x[i] = guess[i];
      for (int it = 1; why < 0; ++it) {
        double res[NA1], D[NA1], S[NT];
        system(x, T0, vf, tdt, dkl, T, res, D, S);
        double mx = 0.0, nr2 = 0.0;
#pragma unroll
        for (int i = 0; i < NAQ; ++i) {
          mx = fmax(mx, fabs(res[i]));
          nr2 += res[i] * res[i];
        }
        const double nr = sqrt(nr2);
        if (it == 1) r0 = nr;
        if (it > Net::MAX_IT) {
          why = kMaxIter;
          break;
        }
        if (mx < Net::TOL_ABS || nr / r0 < Net::TOL_REL) {
          why = kOk;
          break;
        }
        const double jc = psv * dkl / tdt;
        double delta[NA1];
#pragma unroll
        for (int i = 0; i < NAQ; ++i) delta[i] = res[i] / jc;
        if (!sens_ldlt<NA1>(D, S, delta)) {
          handover = true;
          break;
        }
        if (!Net::LOG_FORM) {
#pragma unroll
          for (int i = 0; i < NAQ; ++i) delta[i] *= x[i];
        }
        double latest[NA1];
        if constexpr (Net::LOG_FORM) {
#pragma unroll
          for (int i = 0; i < NAQ; ++i) {
            const double u = copysign(1.0, delta[i]) * fmin(fabs(delta[i]), Net::MAX_DLNC);
            latest[i] = x[i] * pf_exp(-u);
          }
        } else {
          double ratio = 1.0e308;
#pragma unroll
          for (int i = 0; i < NAQ; ++i)
            if (x[i] <= delta[i]) ratio = fmin(ratio, fabs(x[i] / delta[i]));
#pragma unroll
          for (int i = 0; i < NAQ; ++i)
            latest[i] = x[i] - (ratio < 1.0 ? delta[i] * ratio * 0.99 : delta[i]);
        }
        double rc = -1.0;
#pragma unroll
        for (int i = 0; i < NAQ; ++i) {
          const double q = fabs((latest[i] - x[i]) / x[i]);
          if (q == q) rc = fmax(rc, q);
        }
        if (rc >= 0.0 && rc < Net::TOL_CHANGE) {
          why = kOk;
          break;
        }
#pragma unroll
        for (int i = 0; i < NAQ; ++i) x[i] = latest[i];
      }
      if (handover) break;
      if (why != kOk) {
        // maximum iterations: the totals stay those of the sub-step's start
        if (++ncuts > Net::MAX_CUTS) {
          st = kMaxIter;
          break;
        }
        tdt *= 0.5;
        nconst = 0;
        continue;
      }
      if (nlog == kSensSub) {
        st = 5;  // PFCHEM_CELL_TOO_MANY_SUBSTEPS
        break;
      }
      double* lg = A.log + (i64)nlog * NF * ldl + c;
      sfor<0, NAQ>([&](auto Q) {
        constexpr int i = decltype(Q)::value;
        lg[i * ldl] = x[i];
      });
      // kinetic update with the rates at the sub-step's solution
      {
        Acts<NA1> ac;
        sfor<0, NAQ>([&](auto Q) {
          constexpr int i = decltype(Q)::value;
          act_set<i>(ac, x[i], gam[i]);
        });
        sfor<0, NM>([&](auto Mq) {
          constexpr int mi = decltype(Mq)::value;
          lg[(NAQ + mi) * ldl] = vf[mi];
          double Im, dI;
          mnrl_r(Mq, ac, vf[mi], Im, dI);
          double v = vf[mi] + Im * Net::MNRL_VM[mi] * tdt;
          vf[mi] = v < 0.0 ? 0.0 : v;
        });
      }
      lg[(NAQ + NM) * ldl] = tdt;
      ++nlog;
#pragma unroll
      for (int i = 0; i < NAQ; ++i) {
        T0[i] = T[i];
        guess[i] = x[i];
      }
      cum += tdt;
      if (++nconst >= 4) {
        --ncuts;
        tdt = fmin(2.0 * tdt, A.dt - cum);
      }
    }
    if (handover) {
      A.status[c] = kEscalate;
      return;
    }
    if (st) {
      zero_grad();
      A.status[c] = st;
      return;
    }

    // ---------------- objective and its explicit terms ----------------
    double gm[NA1], gT[NA1], gV[NM1];
    {
      Acts<NA1> ac;
      sfor<0, NAQ>([&](auto Q) {
        constexpr int i = decltype(Q)::value;
        act_set<i>(ac, x[i], gam[i]);
        gm[i] = 0.0;
        gT[i] = 0.0;
      });
      double f = 0.0;
      sfor<0, NM>([&](auto M) {
        constexpr int m = decltype(M)::value;
        gV[m] = A.wv[m];
        f += gV[m] * vf[m];
      });
      sfor<0, NC>([&](auto K) {
        constexpr int k = decltype(K)::value;
        const double wk = A.ws[k];
        if (wk == 0.0) return;
        const double mk = cplx_m(K, ac);
        f += wk * mk;
        sfor<0, Net::CPLX_N[k]>([&](auto Q) {
          constexpr int a = decltype(Q)::value;
          constexpr int ia = Net::CPLX_ID[k][a];
          gm[ia] += wk * mk * Net::CPLX_NU[k][a] / x[ia];
        });
      });
      if (A.fcell) A.fcell[c] = f;
    }

    // ---------------- reverse sweep over the recorded sub-steps ----------------
    const double mf = A.jacobian ? 1.0 : dkl;
    for (int k = nlog - 1; k >= 0; --k) {
      const bool first = k == nlog - 1;
      const double* lg = A.log + (i64)k * NF * ldl + c;
      Acts<NA1> ac;
      double m[NA1], v0[NM1];
      sfor<0, NAQ>([&](auto Q) {
        constexpr int i = decltype(Q)::value;
        m[i] = lg[i * ldl];
        act_set<i>(ac, m[i], gam[i]);
      });
      sfor<0, NM>([&](auto M) {
        constexpr int mi = decltype(M)::value;
        v0[mi] = lg[(NAQ + mi) * ldl];
      });
      const double h = lg[(NAQ + NM) * ldl];
      const double jc = psv * dkl / h;
      // kinetic-state update of this sub-step
      double gkin[NM1], Imq[NM1];
      bool actq[NM1];
      sfor<0, NM>([&](auto Mq) {
        constexpr int mi = decltype(Mq)::value;
        double Im, dI;
        actq[mi] = mnrl_r(Mq, ac, v0[mi], Im, dI);
        Imq[mi] = Im;
        gkin[mi] = 0.0;
        if (v0[mi] + Im * Net::MNRL_VM[mi] * h < 0.0) gV[mi] = 0.0;
        if (gV[mi] == 0.0 || !actq[mi]) return;
        gkin[mi] = gV[mi] * kLogToLn * Im * Net::MNRL_VM[mi] * h;
        sfor<0, Net::MNRL_N[mi]>([&](auto Q) {
          constexpr int a = decltype(Q)::value;
          constexpr int ia = Net::MNRL_ID[mi][a];
          gm[ia] += gV[mi] * Net::MNRL_VM[mi] * h * dI * Net::MNRL_NU[mi][a] / m[ia];
        });
      });
      // the sub-step's end totals feed the next sub-step's accumulation:
      // gm_j += dkl (gT_j + sum_k nu_jk m_k (nu_k . gT) / m_j)
      double D[NA1], S[NT], Tt[NA1], rs[NA1];
      {
        double T0d[NA1];
#pragma unroll
        for (int i = 0; i < NAQ; ++i) T0d[i] = 0.0;
        system(m, T0d, v0, h, mf, Tt, rs, D, S);
      }
      double gt[NA1];
      sfor<0, NAQ>([&](auto Q) {
        constexpr int i = decltype(Q)::value;
        gt[i] = gT[i] * m[i];
      });
      sfor<0, NC>([&](auto K) {
        constexpr int kk = decltype(K)::value;
        constexpr int ns = Net::CPLX_N[kk];
        double dotT = 0.0;
        sfor<0, ns>([&](auto Q) {
          constexpr int a = decltype(Q)::value;
          dotT += Net::CPLX_NU[kk][a] * gT[Net::CPLX_ID[kk][a]];
        });
        if (dotT == 0.0) return;
        const double mk = cplx_m(K, ac);
        sfor<0, ns>([&](auto Q) {
          constexpr int a = decltype(Q)::value;
          gt[Net::CPLX_ID[kk][a]] += Net::CPLX_NU[kk][a] * mk * dotT;
        });
      });
      // J^T lambda = gm  <=>  M lambda = diag(m) gm / jc
      double lam[NA1];
      sfor<0, NAQ>([&](auto Q) {
        constexpr int i = decltype(Q)::value;
        gm[i] += dkl * gt[i] / m[i];
        lam[i] = m[i] * gm[i] / jc;
      });
      if (!sens_ldlt<NA1>(D, S, lam)) {
        A.status[c] = kEscalate;
        return;
      }
      // log K of the complexes: through the sub-step's totals (gT) and
      // through the residual (lambda); at the end of the step also the
      // secondary molality itself
      sfor<0, NC>([&](auto K) {
        constexpr int kk = decltype(K)::value;
        constexpr int ns = Net::CPLX_N[kk];
        double accT = 0.0, accL = 0.0;
        sfor<0, ns>([&](auto Q) {
          constexpr int a = decltype(Q)::value;
          constexpr int ia = Net::CPLX_ID[kk][a];
          accT += gT[ia] * Net::CPLX_NU[kk][a];
          accL += lam[ia] * Net::CPLX_NU[kk][a];
        });
        const double wk = first ? A.ws[kk] : 0.0;
        double* o = A.grad + (i64)(NM + kk) * ldo + c;
        if (accT == 0.0 && accL == 0.0 && wk == 0.0) {
          if (first) *o = 0.0;
          return;
        }
        const double mk = cplx_m(K, ac);
        const double v = (accT - psv / h * accL) * (-kLogToLn * mk * dkl) + wk * (-kLogToLn * mk);
        *o = first ? v : *o + v;
      });
      // rate constants: the rate scales with k
      sfor<0, NM>([&](auto Mq) {
        constexpr int mi = decltype(Mq)::value;
        double v = gkin[mi];
        if (actq[mi]) {
          double acc = 0.0;
          sfor<0, Net::MNRL_N[mi]>([&](auto Q) {
            constexpr int a = decltype(Q)::value;
            acc += lam[Net::MNRL_ID[mi][a]] * Net::MNRL_NU[mi][a];
          });
          v -= acc * vol * kLogToLn * Imq[mi];
        }
        double* o = A.grad + (i64)mi * ldo + c;
        *o = first ? v : *o + v;
      });
      sfor<0, NAQ>([&](auto Q) {
        constexpr int i = decltype(Q)::value;
        gT[i] = lam[i] * psv / h;
        gm[i] = 0.0;
      });
    }
    A.status[c] = 0;
  }
}

}  // namespace pflane

#ifdef PFLANE_ADJOINT
extern "C" __global__ void __launch_bounds__(256) pfchem_lane_adjoint(pflane::SensArgs a) {
  pflane::lane_adjoint(a);
}
#endif

// ---------------------------------------------------------------------------
// GIRT reaction block, one cell per lane, FP64: residual and Jacobian of one
// iterate (RTResidualNonFlux / RTJacobianNonFlux per cell,
// reactive_transport.F90:2393-2430, 2599-2642, 3172-3183, 3270-3300), aqueous
// networks with kinetic minerals and decay.
//   res_i  = (Acc_i(x) - Acc_i(fixed)) / dt + R_i(x)
//   jac_ij = (f S_ij + G_ij) / x_j + delta_ij f,  f = dkl psv / dt,
// S = sum_k nu nu^T m_k and G the minerals' term symmetric: the strict lower
// triangle and the diagonal stay in registers, then every row of the state
// leaves as one contiguous 512-byte store of the wavefront.  The kernel is a
// stream (15 primaries: 3.2 kB a cell): 262,139 cells move 0.84 GB in
// 286 us; the team kernel, whose LDS atomics and dense-tile write-out cost
// more than its traffic, took 1190 us.
namespace pflane {

struct GirtArgs {
  i64 ld, ncell;
  const double* pri_molal;
  double* total;
  const double* immobile;
  double* sec_molal;
  const double* pri_act_coef;
  const double* sec_act_coef;
  const double* ln_act_h2o;
  const double* mnrl_volfrac;
  const double* mnrl_area;
  double* mnrl_rate;
  const double* porosity;
  const double* saturation;
  const double* den_kg;
  const double* volume;
  const double* temperature;
  const double* fixed_total;
  const double* fixed_imm;
  double* res;
  double* jac;  // NULL: residual only
  double dt;
};
static_assert(sizeof(GirtArgs) == 176, "GirtArgs layout");

__device__ inline void lane_girt(const GirtArgs& A) {
  constexpr int NAQ = Net::NAQ, NIMM = Net::NIMM, N = NAQ + NIMM, NC = Net::NC, NM = Net::NM;
  constexpr int NA1 = NAQ > 0 ? NAQ : 1, NI1 = NIMM > 0 ? NIMM : 1, NM1 = NM > 0 ? NM : 1;
  constexpr int NC1 = NC > 0 ? NC : 1, NT = NAQ > 1 ? NAQ * (NAQ - 1) / 2 : 1;
  const i64 c = (i64)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= A.ncell) return;
  const i64 ld = A.ld;
  // every load first
  const double por = A.porosity[c], sat = A.saturation[c], den = A.den_kg[c], vol = A.volume[c];
  const double temp = A.temperature ? A.temperature[c] : 25.0;
  // an input here, whether or not the option to update it is on
  const double ln_aw = A.ln_act_h2o ? A.ln_act_h2o[c] : 0.0;
  double x[N], gam[NA1], fx[N], vf[NM1], ar[NM1], g[NC1];
  {
    const double* pp = A.pri_molal + c;
    const double* pg = A.pri_act_coef + c;
    const double* pf = A.fixed_total + c;
    sfor<0, NAQ>([&](auto I) {
      constexpr int i = decltype(I)::value;
      x[i] = *pp;
      gam[i] = *pg;
      fx[i] = *pf;
      pp += ld;
      pg += ld;
      pf += ld;
    });
    sfor<0, NIMM>([&](auto I) {
      constexpr int i = decltype(I)::value;
      x[NAQ + i] = A.immobile[i * ld + c];
      fx[NAQ + i] = A.fixed_imm[i * ld + c];
    });
    const double* pv = A.mnrl_volfrac + c;
    const double* pa = A.mnrl_area + c;
    sfor<0, NM>([&](auto M) {
      constexpr int m = decltype(M)::value;
      vf[m] = *pv;
      ar[m] = *pa;
      pv += ld;
      pa += ld;
    });
    const double* ps = A.sec_act_coef + c;
    sfor<0, NC>([&](auto K) {
      g[decltype(K)::value] = *ps;
      ps += ld;
    });
  }
  issue_loads();
  const bool wet = !(sat < kRtMinSat);
  const double dkl = den * 1.0e-3, psv = por * sat * 1000.0 * vol;
  const double tk = temp + 273.15, lnT = pf_log(tk);
  const double f = wet ? dkl * (psv / A.dt) : 0.0;
  Acts<NA1> act;
  double tot[NA1], D[NA1], W[NT], xi[NA1], res[N];
  sfor<0, NAQ>([&](auto I) {
    constexpr int i = decltype(I)::value;
    act_set<i>(act, x[i], act_keep(gam[i]));
    xi[i] = 1.0 / x[i];
    tot[i] = 0.0;
    D[i] = 0.0;
  });
#pragma unroll
  for (int q = 0; q < NT; ++q) W[q] = 0.0;
  {
    double* ps = A.sec_molal + c;
    sfor<0, NC>([&](auto K) {
      constexpr int k = decltype(K)::value;
      constexpr int ns = Net::CPLX_N[k];
      const double m = cplx_q<k>(act, lnT, tk, ln_aw, 1.0) * rcp_nr(g[k]);
      *ps = m;
      ps += ld;
      const double mf = m * f;
      sfor<0, ns>([&](auto Q) {
        constexpr int a = decltype(Q)::value;
        constexpr int ia = Net::CPLX_ID[k][a];
        constexpr double na = Net::CPLX_NU[k][a];
        tot[ia] += na * m;
        D[ia] += (na * na) * mf;
        sfor<a + 1, ns>([&](auto Q2) {
          constexpr int b = decltype(Q2)::value;
          constexpr int ib = Net::CPLX_ID[k][b];
          constexpr double nab = na * Net::CPLX_NU[k][b];
          if constexpr (ia == ib) D[ia] += (2.0 * nab) * mf;
          else W[tri(ia, ib)] += nab * mf;
        });
      });
    });
  }
  {
    double* pt = A.total + c;
    sfor<0, NAQ>([&](auto I) {
      constexpr int i = decltype(I)::value;
      const double total = (x[i] + tot[i]) * dkl;
      *pt = total;
      pt += ld;
      res[i] = wet ? (psv * total - psv * fx[i]) / A.dt : 0.0;
    });
  }
  double dimm[NI1];
  sfor<0, NIMM>([&](auto I) {
    constexpr int i = decltype(I)::value;
    double r = (x[NAQ + i] * vol - fx[NAQ + i] * vol) / A.dt, d = vol / A.dt;
    sfor<0, Net::NDECAY>([&](auto Dq) {
      constexpr int q = decltype(Dq)::value;
      if constexpr (Net::DECAY_ID[q] == i) {
        const double kc = Net::DECAY_K[q] * vol;
        r += kc * x[NAQ + i];
        d += kc;
      }
    });
    res[NAQ + i] = wet ? r : 0.0;
    dimm[i] = wet ? d : 1.0;
  });
  sfor<0, NM>([&](auto Mq) {
    constexpr int m = decltype(Mq)::value;
    constexpr int ns = Net::MNRL_N[m];
    double rt = 0.0;
    if (wet && ar[m] != 0.0) {
      const double QK = mnrl_q<m>(act, lnT, tk, ln_aw);
      const MRate r = mineral_rate<m>(QK, vf[m], ar[m], temp);
      if (r.active) {
        rt = r.Im;
        const double Iv = r.Im * vol, gm = r.dIm * vol * QK * dkl;
        sfor<0, ns>([&](auto Q) {
          constexpr int a = decltype(Q)::value;
          constexpr int ia = Net::MNRL_ID[m][a];
          constexpr double na = Net::MNRL_NU[m][a];
          res[ia] += na * Iv;
          D[ia] += (na * na) * gm;
          sfor<a + 1, ns>([&](auto Q2) {
            constexpr int b = decltype(Q2)::value;
            constexpr int ib = Net::MNRL_ID[m][b];
            constexpr double nab = na * Net::MNRL_NU[m][b];
            if constexpr (ia == ib) D[ia] += (2.0 * nab) * gm;
            else W[tri(ia, ib)] += nab * gm;
          });
        });
      }
    }
    if (A.mnrl_rate) A.mnrl_rate[m * ld + c] = rt;
  });
  {
    double* pr = A.res + c;
    sfor<0, N>([&](auto I) {
      *pr = res[decltype(I)::value];
      pr += ld;
    });
  }
  if (A.jac) {
    double* pj = A.jac + c;
    sfor<0, N>([&](auto I) {
      constexpr int i = decltype(I)::value;
      sfor<0, N>([&](auto J) {
        constexpr int j = decltype(J)::value;
        double v = 0.0;
        if constexpr (i < NAQ && j < NAQ) {
          if constexpr (i == j) v = wet ? D[i] * xi[i] + f : 1.0;
          else v = wet ? W[tri(i, j)] * xi[j] : 0.0;
        } else if constexpr (i == j) {
          v = dimm[i - NAQ];
        }
        *pj = v;
        pj += ld;
      });
    });
  }
}

}  // namespace pflane

#ifdef PFLANE_GIRT
extern "C" __global__ void __launch_bounds__(64) pfchem_lane_girt(pflane::GirtArgs a) {
  pflane::lane_girt(a);
}
#endif
