// wadges_device.hpp -- device-side building blocks shared by the WADGES kernels:
// per-node primitive records, the two-point entropy-conservative (Chandrashekar)
// flux in contracted form, and the entropy <-> conservative variable maps.
//
// Math follows the reference (ntan15/scratch_wadge):
//   logmean      okl/Euler3D.okl:55-83, okl/Euler2D.okl:54-66
//   flux         okl/Euler3D.okl:122-162, okl/Euler2D.okl:139-161
//   VU / UV      okl/Euler3D.okl:24-51,85-120, okl/Euler2D.okl:19-33,69-98
// restated for CDNA4 FP64:
//   * per-node quantities (velocity, beta = rho/2p, ln rho, ln beta, |u|^2/2)
//     are computed once per node instead of once per pair;
//   * the log branch of the log mean, (aL-aR)/ln(aL/aR), uses the per-node
//     logs: (aL-aR)/(ln aL - ln aR); the series branch keeps the reference's
//     thresholds (1e-4 with 4 terms in 3D, 1e-3 with 5 terms in 2D);
//   * the divisions of a flux evaluation (two log means, the pressure average
//     and rho_log/beta_log) share two reciprocals, one on smooth states;
//   * the flux is never materialised as a DIM x NFLD matrix: callers contract it
//     with a direction vector n (sum_d n_d F_d) through flux_dot().
// All arithmetic is FP64.
#pragma once

#include <hip/hip_runtime.h>

namespace wadges {

template <int DIM> struct Dims {
  static constexpr int NFLD = DIM + 2;   // conserved fields
  static constexpr int NG = DIM * DIM;   // geometric factors per node
  static constexpr int NFACES = DIM + 1; // faces per simplex
  static constexpr int NFG = DIM + 1;    // face geometric factors per face point
};

// Primitive record of a node: what the flux needs from one side of a pair.
template <int DIM> struct Node {
  double rho;
  double hv[DIM];  // half velocity, u/2
  double beta;     // rho / (2 p)
  double lrho;     // ln rho
  double lbeta;    // ln beta
  double hq;       // |u|^2 / 2
};

// 1/x from v_rcp_f64 (relative error below 2^-24 on gfx950, measured over 4M
// arguments) and one third-order step, r (1 + e + e^2) with e = 1 - x r: the
// omitted e^3 is below 2^-72.  The same results as two Newton steps (at most half
// an ulp off on those arguments) in three multiply-adds instead of four.
// For arguments whose reciprocal is a normal number; 0, infinities and subnormal
// arguments give NaN (IEEE division: infinity and 0).  No admissible state has them.
__device__ __forceinline__ double rcp(double x) {
  const double r = __builtin_amdgcn_rcp(x);
  const double e = __builtin_fma(-x, r, 1.0);
  return __builtin_fma(r, __builtin_fma(e, e, e), r);
}

// a/b given r = rcp(b): one correction of the quotient by its remainder (within
// 0.51 ulp for normal operands and quotients) instead of the scaled IEEE sequence.
// NaN where rcp(b) is, and for an infinite a.
__device__ __forceinline__ double quot(double a, double b, double r) {
  const double q = a * r;
  return __builtin_fma(__builtin_fma(-b, q, a), r, q);
}

// Logarithm, exponential and square root are evaluated once or more per node; the
// math library's take 98, 42 and 22 vector instructions in FP64, and its logarithm
// alone was a fifth of the 2D stage's.  The three below take 50, 27 and 15 and are as
// accurate: against 80-bit arithmetic over 4M arguments each, rms error ln 0.289
// ulp (library 0.289-0.293; arguments in [1/2, 2], [1e-6, 1e6], [1e-300, 1e300]),
// expo 0.302 (0.302; [-8, 8], [-700, 700]), root 0.289 (0.289).  Arguments outside
// their domain give what the library gives (NaN, infinities, zero), but for ln of a
// negative number that rounds to -0 in single precision: -infinity (which quot() turns
// into NaN in the maps to conservative variables).  With them and
// quot() in place of IEEE division: 2D N = 4, K = 32,258, a step 434 -> 397 us; the
// 64-problem ensemble 3.11 -> 2.83 ms for two steps; 3D N = 3, K = 196,608, 8.9 ->
// 8.75 ms.

// A constant in a scalar register at its use.  As plain literals the compiler
// keeps the coefficients of ln in vector registers across the kernel (20-40
// registers, spills in the stage kernels).
__device__ __forceinline__ double sconst(double v) {
  asm volatile("" : "+s"(v));
  return v;
}

constexpr double LN2_HI = 0x1.62e42fefp-1;           // 32 bits: k LN2_HI is exact, |k| < 2^20
constexpr double LN2_LO = 0x1.473de6af278edp-34;     // ln 2 - LN2_HI

// The arrangement of ln is that of fdlibm's log (f and f^2/2 kept out of the rounded
// part, the series in two interleaved chains), with the Taylor coefficients of atanh.
//
// ln x: x = 2^k m with m in [sqrt(1/2), sqrt(2)), f = m - 1 (exact), s = f/(2+f)
// and ln(1+f) = 2 atanh(s) = f - f^2/2 + s (f^2/2 + R(s^2)) with R(z) = 2 (z/3 +
// z^2/5 + ...) (s f = f^2/2 - s f^2/2 ... regroups the first term so that f enters
// exactly); the series to z^10, whose omitted term is below 2e-19.  k ln 2, f and
// f^2/2 are added with their rounding errors.
__device__ __forceinline__ double ln(double x) {
  double m = __builtin_amdgcn_frexp_mant(x);                 // [1/2, 1)
  const int low = m < sconst(0x1.6a09e667f3bcdp-1) ? 1 : 0;
  m = __builtin_amdgcn_ldexp(m, low);
  const double k = (double)(__builtin_amdgcn_frexp_exp(x) - low);
  const double f = m - 1.0;
  const double s = f * rcp(2.0 + f);
  const double z = s * s, w = z * z;
  double r1 = sconst(2.0 / 19.0), r2 = sconst(2.0 / 21.0);
  r1 = __builtin_fma(w, r1, sconst(2.0 / 15.0));
  r2 = __builtin_fma(w, r2, sconst(2.0 / 17.0));
  r1 = __builtin_fma(w, r1, sconst(2.0 / 11.0));
  r2 = __builtin_fma(w, r2, sconst(2.0 / 13.0));
  r1 = __builtin_fma(w, r1, sconst(2.0 / 7.0));
  r2 = __builtin_fma(w, r2, sconst(2.0 / 9.0));
  r1 = __builtin_fma(w, r1, sconst(2.0 / 3.0));
  r2 = __builtin_fma(w, r2, sconst(2.0 / 5.0));
  const double hf = 0.5 * f;
  const double q = hf * f;
  const double q_lo = __builtin_fma(hf, f, -q);
  const double t = s * (q + z * (r1 + z * r2));
  const double a = k * sconst(LN2_HI);
  const double b = a + f;                                    // |a| > |f| or a = 0
  const double b_lo = f - (b - a);
  const double c = b - q;
  const double c_lo = (b - c) - q;
  const double lo = __builtin_fma(k, sconst(LN2_LO), t - q_lo) + (b_lo + c_lo);
  const double v = c + lo;
  // 0, negative, infinite and NaN arguments: as the single-precision instruction
  return __builtin_amdgcn_class(x, 0x180) ? v : (double)__builtin_amdgcn_logf((float)x);
}

// exp x = 2^n exp(r), r = x - n ln 2 in [-ln 2 / 2, ln 2 / 2], Taylor series to
// r^13 (the omitted term is below 5e-18).
__device__ __forceinline__ double expo(double x) {
  const double n = __builtin_rint(x * sconst(1.4426950408889634));
  const double r = __builtin_fma(-n, sconst(LN2_LO), __builtin_fma(-n, sconst(LN2_HI), x));
  double p = sconst(1.0 / 6227020800.0);
  p = __builtin_fma(p, r, sconst(1.0 / 479001600.0));
  p = __builtin_fma(p, r, sconst(1.0 / 39916800.0));
  p = __builtin_fma(p, r, sconst(1.0 / 3628800.0));
  p = __builtin_fma(p, r, sconst(1.0 / 362880.0));
  p = __builtin_fma(p, r, sconst(1.0 / 40320.0));
  p = __builtin_fma(p, r, sconst(1.0 / 5040.0));
  p = __builtin_fma(p, r, sconst(1.0 / 720.0));
  p = __builtin_fma(p, r, sconst(1.0 / 120.0));
  p = __builtin_fma(p, r, sconst(1.0 / 24.0));
  p = __builtin_fma(p, r, sconst(1.0 / 6.0));
  p = __builtin_fma(p, r, 0.5);
  p = __builtin_fma(p, r, 1.0);
  p = __builtin_fma(p, r, 1.0);
  double v = __builtin_amdgcn_ldexp(p, (int)n);
  v = x > sconst(710.0) ? __builtin_huge_val() : v;
  return x < sconst(-746.0) ? 0.0 : v;
}

// 1/sqrt(x) for x > 0: v_rsq_f64 and one third-order step.
__device__ __forceinline__ double rsqrt_pos(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = __builtin_fma(-(x * y), y, 1.0);
  return __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
}

// sqrt(x) from it, corrected by the remainder x - s^2.
__device__ __forceinline__ double root(double x) {
  const double y = rsqrt_pos(x);
  const double s = x * y;
  const double v = __builtin_fma(__builtin_fma(-s, s, x), 0.5 * y, s);
  return __builtin_amdgcn_class(x, 0x260) ? x : v;           // +-0, +inf
}

// Conservative state -> node record.  3D multiplies by 1/rho
// (okl/Euler3D.okl:2252-2256, TESTING); 2D divides (okl/Euler2D.okl:1127-1129).
// LOGS = false leaves ln rho and ln beta out, for a node that serves a single
// pair: pair_flux<DIM, true> then takes the logarithms only where a log-mean
// log branch needs them.
template <int DIM, bool LOGS = true>
__device__ __forceinline__ Node<DIM> make_node(const double (&U)[DIM + 2], double gm1) {
  Node<DIM> n;
  n.rho = U[0];
  double v[DIM];
  if constexpr (DIM == 3) {
    const double inv = rcp(U[0]);
    for (int d = 0; d < DIM; ++d) v[d] = U[1 + d] * inv;
  } else {
    const double inv = rcp(U[0]);
    for (int d = 0; d < DIM; ++d) v[d] = quot(U[1 + d], U[0], inv);
  }
  double uu = v[0] * v[0];
  for (int d = 1; d < DIM; ++d) uu = uu + v[d] * v[d];
  const double p = gm1 * (U[DIM + 1] - 0.5 * U[0] * uu);
  n.beta = quot(0.5 * U[0], p, rcp(p));
  for (int d = 0; d < DIM; ++d) n.hv[d] = 0.5 * v[d];
  n.lrho = LOGS ? ln(n.rho) : 0.0;
  n.lbeta = LOGS ? ln(n.beta) : 0.0;
  n.hq = 0.5 * uu;
  return n;
}

// Pair quantities of the EC flux; F_d = flux_dot with n = e_d.
template <int DIM> struct PairFlux {
  double rholog, pa, f4aux;
  double va[DIM];  // averaged velocity
};

template <int DIM> __device__ __forceinline__ double logmean_series(double u) {
  // 1 + u/3 + u^2/5 + u^3/7 (+ u^4/9 in 2D), Horner form
  if constexpr (DIM == 3)
    return 1.0 + u * (1.0 / 3.0 + u * (1.0 / 5.0 + u * (1.0 / 7.0)));
  else
    return 1.0 + u * (1.0 / 3.0 + u * (1.0 / 5.0 + u * (1.0 / 7.0 + u * (1.0 / 9.0))));
}

// 2 * logmean_series(u), bit for bit: scaling by 2 is exact, so Horner with
// doubled constants rounds every step to twice the value (one multiply fewer).
template <int DIM> __device__ __forceinline__ double logmean_series2(double u) {
  if constexpr (DIM == 3)
    return 2.0 + u * (2.0 / 3.0 + u * (2.0 / 5.0 + u * (2.0 / 7.0)));
  else
    return 2.0 + u * (2.0 / 3.0 + u * (2.0 / 5.0 + u * (2.0 / 7.0 + u * (2.0 / 9.0))));
}

// 1 / (2 F(u)) as the series of 1/F to the order of F itself: 1 - u/3 - 4u^2/45
// - 44u^3/945 (- 428u^4/14175 in 2D) (the coefficients c_n = -sum_k a_k c_{n-k}
// of the reciprocal of a power series).  Below the series thresholds (u < 1e-4
// in 3D, 1e-3 in 2D) the omitted term is below 3e-17 relative, under the
// rounding of the division it replaces.
template <int DIM> __device__ __forceinline__ double logmean_inv_series2(double u) {
  if constexpr (DIM == 3)
    return 0.5 + u * (-1.0 / 6.0 + u * (-2.0 / 45.0 + u * (-22.0 / 945.0)));
  else
    return 0.5 +
           u * (-1.0 / 6.0 + u * (-2.0 / 45.0 + u * (-22.0 / 945.0 + u * (-214.0 / 14175.0))));
}

// True when p holds on every active lane of the wave (a scalar test).
__device__ __forceinline__ bool wave_all(bool p) {
  return __builtin_amdgcn_ballot_w64(p) == __builtin_amdgcn_read_exec();
}

// A flag the caller knows to be the same on every lane, as a value the
// compiler knows to be uniform (a scalar register, tested with a scalar branch
// instead of lane masks).
__device__ __forceinline__ bool uniform_flag(bool p) {
  return __builtin_amdgcn_readfirstlane((int)p) != 0;
}

// Smooth waves.  A node is in band when its rho and beta lie within a relative
// SmoothBand of a reference node's.  When every node of a wave's elements is in
// band, every pair (a, b) of them has |a - b| / (a + b) <= band / (1 - band), so f^2
// < 9.8e-5 (3D) or 9.97e-4 (2D), below the series thresholds: both log means of
// every pair take the series branch.  The records' logarithms are then never
// used and not taken (2D N = 4, K = 32,258, a step 397 -> 376 us; 2D N = 3, K =
// 51,200, 434 -> 405 us), and the pair routines may skip their per-pair wave test
// (the branch they take is the same, so are the bits).
template <int DIM> constexpr double smooth_band() { return DIM == 3 ? 0.0098 : 0.0306; }

template <int DIM>
__device__ __forceinline__ bool in_smooth_band(double rho, double beta, double rho_ref,
                                               double beta_ref) {
  return fabs(rho - rho_ref) <= smooth_band<DIM>() * rho_ref &&
         fabs(beta - beta_ref) <= smooth_band<DIM>() * beta_ref;
}

// inv2gm1 = 1 / (2 (gamma - 1)).  f of both log means and 1/(beta_a + beta_b)
// come from one reciprocal, 1/((rho_a + rho_b)(beta_a + beta_b)).  The series
// branch takes rho_log from the series of 1/(2F) and 1/beta_log = 2F/(beta_a +
// beta_b), so it needs no other; the log branches of both log means share a
// second reciprocal.  Each lane selects the branch of each log mean by itself, so
// a pair's bits do not depend on the pairs its wave holds, and every kernel that
// evaluates a pair gets the same ones.  (Two reciprocals and a selection of both
// quotients' numerators and denominators, four-term reciprocals: 3D N = 4, K =
// 13,182, a step 1.79 -> 1.71 ms; 3D N = 3, K = 196,608, 9.05 -> 8.94 ms.)  In 3D, when every active lane takes the
// series branch of both log means (smooth states: neighbouring nodes differ by far
// less than the 1 % that the series threshold allows), a wave-uniform test skips
// the log branches (same bits).  In the 2D pair loops the test does not pay: the
// kernels aim at four or more waves per SIMD and spilled with it.  LAZY_LOGS: the
// nodes come without logarithms, which are taken only behind that test (the
// surface flux, whose two nodes serve one pair).  Differences of logarithms there
// too, not the logarithm of a quotient: they change sign exactly when the nodes
// change places, so the two elements of a face take the same flux.
// smooth: a wave-uniform flag by which the caller guarantees (3D) that every
// active lane's pair takes the series branch of both log means; the per-pair
// wave test is then skipped (the same branch, so the same bits).
template <int DIM, bool LAZY_LOGS = false>
__device__ __forceinline__ PairFlux<DIM> pair_flux(const Node<DIM> &a, const Node<DIM> &b,
                                                   double inv2gm1, bool smooth = false) {
  constexpr double TH = (DIM == 3) ? 1.0e-4 : 1.0e-3;
  const double sr = a.rho + b.rho, dr = a.rho - b.rho;
  const double sb = a.beta + b.beta, db = a.beta - b.beta;
  const double q1 = rcp(sr * sb);
  const double isr = sb * q1, isb = sr * q1;
  // f = (aL-aR)/(aL+aR) of both log means
  const double fr = dr * isr, fb = db * isb;
  const double ur = fr * fr, ub = fb * fb;
  const bool serR = ur < TH, serB = ub < TH;
  PairFlux<DIM> P;
  P.rholog = sr * logmean_inv_series2<DIM>(ur);
  double ibl = logmean_series2<DIM>(ub) * isb;   // 1 / beta_log
  P.pa = 0.5 * sr * isb;
  const bool all_series = (DIM == 3 || LAZY_LOGS) && (smooth || wave_all(serR && serB));
  if (!all_series) {
    // rho_log = dr / (ln rho_a - ln rho_b), 1/beta_log = (ln beta_a - ln beta_b) / db
    double ldB = LAZY_LOGS ? ln(a.beta) - ln(b.beta) : a.lbeta - b.lbeta;
    // one difference taken before the next pair of logarithms starts (registers)
    if (LAZY_LOGS) asm volatile("" : "+v"(ldB));
    const double ldR = LAZY_LOGS ? ln(a.rho) - ln(b.rho) : a.lrho - b.lrho;
    const double dR = serR ? 1.0 : ldR;
    const double dB = serB ? 1.0 : db;
    const double q2 = rcp(dR * dB);
    P.rholog = serR ? P.rholog : dr * dB * q2;
    ibl = serB ? ibl : ldB * dR * q2;
  }
  const double ratio = P.rholog * ibl;           // rho_log / beta_log
  double vv = 0.0;
  for (int d = 0; d < DIM; ++d) {
    P.va[d] = a.hv[d] + b.hv[d];
    vv = vv + P.va[d] * P.va[d];
  }
  const double vnavg = 2.0 * vv - (a.hq + b.hq);
  P.f4aux = ratio * inv2gm1 + P.pa + 0.5 * P.rholog * vnavg;
  return P;
}

// out[fld] = sum_d n_d F_d[fld] for the EC flux of a pair.
template <int DIM>
__device__ __forceinline__ void flux_dot(const PairFlux<DIM> &P, const double (&n)[DIM],
                                         double (&out)[DIM + 2]) {
  double Un = P.va[0] * n[0];
  for (int d = 1; d < DIM; ++d) Un = Un + P.va[d] * n[d];
  const double rUn = P.rholog * Un;
  out[0] = rUn;
  for (int d = 0; d < DIM; ++d) out[1 + d] = rUn * P.va[d] + P.pa * n[d];
  out[DIM + 1] = P.f4aux * Un;
}

// Wave speed |u| + sqrt(gamma p / rho) of a node (okl/Euler3D.okl:3316-3321):
// 2 hq = |u|^2 and p / rho = 1 / (2 beta).
template <int DIM>
__device__ __forceinline__ double node_speed(const Node<DIM> &n, double gamma) {
  return root(2.0 * n.hq) + root(0.5 * gamma * rcp(n.beta));
}

// Conservative -> entropy variables.  s = ln((gamma-1) rho e) - gamma ln rho
// (the reference evaluates ln((gamma-1) rho e / rho^gamma)).
template <int DIM>
__device__ __forceinline__ void entropy_vars(const double (&U)[DIM + 2], double gamma,
                                             double (&V)[DIM + 2]) {
  const double rho = U[0], E = U[DIM + 1];
  double mm = U[1] * U[1];
  for (int d = 1; d < DIM; ++d) mm = mm + U[1 + d] * U[1 + d];
  const double rhoe = E - quot(0.5 * mm, rho, rcp(rho));
  const double s = ln((gamma - 1.0) * rhoe) - gamma * ln(rho);
  const double invrhoe = rcp(rhoe);
  V[0] = (-E) * invrhoe + ((gamma + 1.0) - s);
  for (int d = 0; d < DIM; ++d) V[1 + d] = U[1 + d] * invrhoe;
  V[DIM + 1] = (-rho) * invrhoe;
}

// Entropy -> conservative variables.
// rho e = ((gamma-1)/(-v_last)^gamma)^(1/(gamma-1)) exp(-s/(gamma-1))
//       = exp((ln(gamma-1) - gamma ln(-v_last) - s) / (gamma-1)).
template <int DIM>
__device__ __forceinline__ void conservative_vars(const double (&V)[DIM + 2], double gamma,
                                                  double lgm1, double (&U)[DIM + 2]) {
  const double vl = V[DIM + 1];
  double vv = V[1] * V[1];
  for (int d = 1; d < DIM; ++d) vv = vv + V[1 + d] * V[1 + d];
  const double h = quot(0.5 * vv, vl, rcp(vl));
  const double s = gamma - V[0] + h;
  const double rhoe = expo(quot(lgm1 - gamma * ln(-vl) - s, gamma - 1.0, rcp(gamma - 1.0)));
  U[0] = rhoe * (-vl);
  for (int d = 0; d < DIM; ++d) U[1 + d] = rhoe * V[1 + d];
  U[DIM + 1] = rhoe * (1.0 - h);
}

// Deterministic accumulation into an LDS accumulator.  The kernels schedule
// pairs so that within one instruction no two lanes of a wave add into the
// same address, and every element's lanes live in one wave; the order of the
// additions is therefore fixed by the program.
__device__ __forceinline__ void lds_add(double *p, double v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// lds_add for a second group of lanes whose addresses coincide with the first
// group's (taken under the complementary lane mask right after it).  Its
// atomic carries another scope, the wave's (the addresses lie in the calling
// wave's own LDS region, which no other wave touches), so the compiler cannot
// merge the two masked adds into one instruction in which two lanes would add
// into one address in an order the program does not fix.
__device__ __forceinline__ void lds_add_second(double *p, double v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

}  // namespace wadges

// ======================================================================
// Reverse mode (discrete adjoint) building blocks.  Hand-written VJPs of the
// forward routines above; derivatives are taken of the mathematical functions
// the forward kernels evaluate (the log mean through whichever branch the
// forward takes, max(lamM, lamP) through its larger argument, M at ties).
// ======================================================================

namespace wadges {

// Cotangent of a node's primitive quantities (rho, velocity u, beta).
template <int DIM> struct PrimBar {
  double rho, u[DIM], beta;
};

template <int DIM> __device__ __forceinline__ void primbar_zero(PrimBar<DIM> &g) {
  g.rho = 0.0;
  for (int d = 0; d < DIM; ++d) g.u[d] = 0.0;
  g.beta = 0.0;
}

// Partial derivatives (dl/da, dl/db) of the log mean l(a, b), in the branch the
// forward evaluation uses: series l = (a+b)/(2F(f^2)), f = (a-b)/(a+b), or
// l = (a-b)/(ln a - ln b).
template <int DIM>
__device__ __forceinline__ void logmean_partials(double a, double b, double la, double lb,
                                                 double &l, double &da, double &db) {
  constexpr double TH = (DIM == 3) ? 1.0e-4 : 1.0e-3;
  const double s = a + b, d = a - b;
  const double is = rcp(s);
  const double f = d * is;
  const double u = f * f;
  if (u < TH) {
    const double F = logmean_series<DIM>(u);
    double Fp;  // F'(u)
    if constexpr (DIM == 3)
      Fp = 1.0 / 3.0 + u * (2.0 / 5.0 + u * (3.0 / 7.0));
    else
      Fp = 1.0 / 3.0 + u * (2.0 / 5.0 + u * (3.0 / 7.0 + u * (4.0 / 9.0)));
    const double iF = rcp(F);
    l = 0.5 * s * iF;
    const double t = 2.0 * f * Fp * is * iF * iF;
    da = 0.5 * iF - t * b;
    db = 0.5 * iF + t * a;
  } else {
    const double iL = rcp(la - lb);
    l = d * iL;
    da = (1.0 - l * rcp(a)) * iL;
    db = (l * rcp(b) - 1.0) * iL;
  }
}

// VJP of L = sum_d sum_fld Gb[d][fld] F_d[fld](a, b) with respect to the
// primitive quantities of both nodes, accumulated into ga, gb, for a cotangent
// of rank NT, Gb[d][fld] = sum_k n_k[d] c_k[fld] (rank one: the contracted
// volume-face and surface couplings; rank two: a volume pair's own row and its
// partner row).  L depends on the flux through A = sum_d Gb[d][0] va_d,
// B = sum_dm Gb[d][1+m] va_d va_m, C = sum_d Gb[d][last] va_d and
// tr = sum_d Gb[d][1+d]; with Un_k = n_k.va and cm_k = sum_m c_k[1+m] va_m these
// are A = sum c_k[0] Un_k, B = sum Un_k cm_k, C = sum c_k[last] Un_k,
// tr = sum_k sum_d n_k[d] c_k[1+d], and the velocity derivative needs, per
// direction, t_d = sum_k n_k[d] (c_k[0] + cm_k) + c_k[1+d] Un_k:
// O(NT (DIM + NFLD)) work instead of the O(DIM^2 NFLD) of a dense Gb.
//
// When every active lane of the wave takes the series branch of both log means
// (smooth states), 1/F comes from the series of 1/F and every reciprocal of the pair
// from one.  LAZY_LOGS: the nodes come without logarithms, which are taken only behind
// that test and kept in them (the surface flux, whose second pair of the same nodes runs
// on some of the first one's lanes and so needs them only if the first did).
template <int DIM, int NT, bool LAZY_LOGS = false, class NA, class NB>
__device__ __forceinline__ void flux_dot_vjp_k(NA &a, NB &b,
                                               const double (&n)[NT][DIM],
                                               const double (&c)[NT][DIM + 2], double inv2gm1,
                                               PrimBar<DIM> &ga, PrimBar<DIM> &gb) {
  constexpr int NF = DIM + 2;
  constexpr double TH = (DIM == 3) ? 1.0e-4 : 1.0e-3;
  const double sr = a.rho + b.rho, sb = a.beta + b.beta;
  const double dr = a.rho - b.rho, db = a.beta - b.beta;
  // f of both log means from one reciprocal
  const double q = rcp(sr * sb);
  const double isr = sb * q, isb = sr * q;
  const double fr = dr * isr, fb = db * isb;
  const double ur = fr * fr, ub = fb * fb;
  double rl, rla, rlb, bla, blb, ibl;   // rho_log, partials of both log means, 1/beta_log
  if (wave_all(ur < TH && ub < TH)) {
    // l = s/(2F(u)); dl/da = 1/(2F) - l' b, dl/db = 1/(2F) + l' a with
    // l' = 2 f F'(u) / (s F^2) = 8 F'(u) (f / s) / (2F)^2  (the partials of the series branch)
    auto partials = [&](double is, double f, double u, double x, double y, double &dx, double &dy) {
      const double h = logmean_inv_series2<DIM>(u);          // 1/(2F)
      double Fp8;                                             // 8 F'(u)
      if constexpr (DIM == 3)
        Fp8 = 8.0 / 3.0 + u * (16.0 / 5.0 + u * (24.0 / 7.0));
      else
        Fp8 = 8.0 / 3.0 + u * (16.0 / 5.0 + u * (24.0 / 7.0 + u * (32.0 / 9.0)));
      const double t = Fp8 * (f * is) * (h * h);
      dx = h - t * y;
      dy = h + t * x;
      return h;
    };
    rl = sr * partials(isr, fr, ur, a.rho, b.rho, rla, rlb);
    partials(isb, fb, ub, a.beta, b.beta, bla, blb);
    ibl = isb * logmean_series2<DIM>(ub);                     // 1/bl = 2F(u_beta)/sb
  } else {
    double bl;
    if constexpr (LAZY_LOGS) {
      a.lrho = ln(a.rho);
      a.lbeta = ln(a.beta);
      b.lrho = ln(b.rho);
      b.lbeta = ln(b.beta);
    }
    logmean_partials<DIM>(a.rho, b.rho, a.lrho, b.lrho, rl, rla, rlb);
    logmean_partials<DIM>(a.beta, b.beta, a.lbeta, b.lbeta, bl, bla, blb);
    ibl = rcp(bl);
  }
  const double pa = 0.5 * sr * isb;
  double va[DIM], vv = 0.0;
  for (int d = 0; d < DIM; ++d) {
    va[d] = a.hv[d] + b.hv[d];
    vv = vv + va[d] * va[d];
  }
  const double hvn = vv - 0.5 * (a.hq + b.hq);                // vnavg / 2
  const double gbl = inv2gm1 * ibl;
  const double rb = rl * gbl;
  const double f4 = rb + pa + rl * hvn;
  double Un[NT], c0m[NT], A = 0.0, C = 0.0, tr = 0.0;
  for (int k = 0; k < NT; ++k) {
    double u = n[k][0] * va[0], cm = c[k][0] + c[k][1] * va[0];
    for (int d = 1; d < DIM; ++d) {
      u = u + n[k][d] * va[d];
      cm = cm + c[k][1 + d] * va[d];
    }
    for (int d = 0; d < DIM; ++d) tr = tr + n[k][d] * c[k][1 + d];
    Un[k] = u;
    c0m[k] = cm;
    A = A + cm * u;                                           // A + B of the comment above
    C = C + c[k][NF - 1] * u;
  }
  const double L_rl = A + C * (gbl + hvn);
  const double L_bl = -C * rb * ibl;
  const double Crl = C * rl;
  const double hrl = 0.5 * rl, hf4 = 0.5 * f4;
  for (int d = 0; d < DIM; ++d) {
    // half the derivative by va_d; the |u|^2 terms of the nodes are -Crl u/2 each
    double t = n[0][d] * c0m[0] + c[0][1 + d] * Un[0];
    double e = n[0][d] * c[0][NF - 1];
    for (int k = 1; k < NT; ++k) {
      t = t + n[k][d] * c0m[k] + c[k][1 + d] * Un[k];
      e = e + n[k][d] * c[k][NF - 1];
    }
    const double g = hrl * t + hf4 * e + Crl * va[d];
    ga.u[d] += g - Crl * a.hv[d];
    gb.u[d] += g - Crl * b.hv[d];
  }
  const double L_pa = (tr + C) * isb;                         // derivative by pa, over sb
  ga.rho += L_rl * rla + 0.5 * L_pa;
  gb.rho += L_rl * rlb + 0.5 * L_pa;
  ga.beta += L_bl * bla - L_pa * pa;
  gb.beta += L_bl * blb - L_pa * pa;
}

template <int DIM, bool LAZY_LOGS = false, class NA, class NB>
__device__ __forceinline__ void flux_dot_vjp(NA &a, NB &b,
                                             const double (&n)[DIM], const double (&c)[DIM + 2],
                                             double inv2gm1, PrimBar<DIM> &ga, PrimBar<DIM> &gb) {
  double nk[1][DIM], ck[1][DIM + 2];
  for (int d = 0; d < DIM; ++d) nk[0][d] = n[d];
  for (int f = 0; f < DIM + 2; ++f) ck[0][f] = c[f];
  flux_dot_vjp_k<DIM, 1, LAZY_LOGS>(a, b, nk, ck, inv2gm1, ga, gb);
}

// Primitive cotangent -> conservative cotangent of one node:
// u = m / rho, beta = rho / (2p), p = (gamma - 1)(E - |m|^2/(2 rho)).
template <int DIM>
__device__ __forceinline__ void primbar_to_cons(const Node<DIM> &n, const PrimBar<DIM> &g,
                                                double gm1, double (&Ub)[DIM + 2]) {
  const double irho = rcp(n.rho);
  const double p = 0.5 * n.rho * rcp(n.beta);      // p = rho / (2 beta)
  const double bp = n.beta * rcp(p);                // beta / p
  double gu_u = 0.0;
  for (int d = 0; d < DIM; ++d) gu_u = gu_u + g.u[d] * (2.0 * n.hv[d]);
  // d beta/d rho = beta/rho - (beta/p)(gamma-1)|u|^2/2
  Ub[0] = g.rho - gu_u * irho + g.beta * (n.beta * irho - bp * gm1 * n.hq);
  for (int d = 0; d < DIM; ++d) Ub[1 + d] = g.u[d] * irho + g.beta * bp * gm1 * (2.0 * n.hv[d]);
  Ub[DIM + 1] = -g.beta * bp * gm1;
}

// Wave speed lambda = |u| + sqrt(gamma p / rho) and its gradient with respect
// to the conservative state.
template <int DIM>
__device__ __forceinline__ double wavespeed(const double (&U)[DIM + 2], double gamma, double gm1,
                                            double (&dl)[DIM + 2]) {
  const double irho = rcp(U[0]);
  double v[DIM], uu = 0.0;
  for (int d = 0; d < DIM; ++d) {
    v[d] = U[1 + d] * irho;
    uu = uu + v[d] * v[d];
  }
  const double p = gm1 * (U[DIM + 1] - 0.5 * U[0] * uu);
  const double su = root(uu);
  const double c = root(gamma * p * irho);
  // d|u|: d(|u|)/du_d = u_d/|u| (0 at rest); u_d = m_d/rho
  const double isu = su > 0.0 ? rcp(su) : 0.0;
  // c^2 = gamma p / rho: d(c)/dq = (gamma/(2c)) d(p/rho)/dq
  const double k = 0.5 * gamma * rcp(c);
  // p/rho = gm1 (E/rho - |m|^2/(2 rho^2))
  const double dpr_rho = gm1 * (-U[DIM + 1] * irho * irho + uu * irho);
  dl[0] = -uu * isu * irho + k * dpr_rho;
  for (int d = 0; d < DIM; ++d) dl[1 + d] = v[d] * isu * irho + k * (-gm1 * v[d] * irho);
  dl[DIM + 1] = k * gm1 * irho;
  return su + c;
}

// VJP of entropy_vars (U -> V) at U.
template <int DIM>
__device__ __forceinline__ void entropy_vars_vjp(const double (&U)[DIM + 2], double gamma,
                                                 const double (&Vb)[DIM + 2], double (&Ub)[DIM + 2]) {
  constexpr int NF = DIM + 2;
  const double rho = U[0], E = U[NF - 1];
  double mm = 0.0;
  for (int d = 0; d < DIM; ++d) mm = mm + U[1 + d] * U[1 + d];
  const double irho = rcp(rho);
  const double rhoe = E - 0.5 * mm * irho;
  const double io = rcp(rhoe);
  // V0 = -E io + (gamma + 1) - s ; V_m = m io ; V_last = -rho io
  double iob = Vb[0] * (-E) + Vb[NF - 1] * (-rho);
  for (int d = 0; d < DIM; ++d) iob = iob + Vb[1 + d] * U[1 + d];
  const double sb = -Vb[0];
  double rhob = -Vb[NF - 1] * io - sb * gamma * irho;     // s = ln((g-1) rho e) - g ln rho
  double Eb = -Vb[0] * io;
  const double rhoeb = -iob * io * io + sb * io;
  Eb = Eb + rhoeb;
  rhob = rhob + rhoeb * 0.5 * mm * irho * irho;
  Ub[0] = rhob;
  for (int d = 0; d < DIM; ++d) Ub[1 + d] = Vb[1 + d] * io - rhoeb * U[1 + d] * irho;
  Ub[NF - 1] = Eb;
}

// VJP of conservative_vars (V -> U) at V.
template <int DIM>
__device__ __forceinline__ void conservative_vars_vjp(const double (&V)[DIM + 2], double gamma,
                                                      double lgm1, const double (&Ub)[DIM + 2],
                                                      double (&Vb)[DIM + 2]) {
  constexpr int NF = DIM + 2;
  const double vl = V[NF - 1];
  double vv = 0.0;
  for (int d = 0; d < DIM; ++d) vv = vv + V[1 + d] * V[1 + d];
  const double ivl = rcp(vl);
  const double h = 0.5 * vv * ivl;
  const double s = gamma - V[0] + h;
  const double igm1 = rcp(gamma - 1.0);
  const double rhoe = expo((lgm1 - gamma * ln(-vl) - s) * igm1);
  double rhoeb = Ub[0] * (-vl) + Ub[NF - 1] * (1.0 - h);
  for (int d = 0; d < DIM; ++d) rhoeb = rhoeb + Ub[1 + d] * V[1 + d];
  double vlb = -Ub[0] * rhoe;
  double hb = -Ub[NF - 1] * rhoe;
  const double Xb = rhoeb * rhoe;
  const double sb = -Xb * igm1;
  vlb = vlb - Xb * gamma * igm1 * ivl;
  Vb[0] = -sb;
  hb = hb + sb;
  const double vvb = 0.5 * hb * ivl;
  vlb = vlb - hb * h * ivl;
  for (int d = 0; d < DIM; ++d) Vb[1 + d] = Ub[1 + d] * rhoe + 2.0 * vvb * V[1 + d];
  Vb[NF - 1] = vlb;
}

}  // namespace wadges
