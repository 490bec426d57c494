// Device-side arithmetic shared by the evaluation and the fused minimization kernels: precision
// traits, DPP row rotation, the Born-radius integral and its radial derivative, the
// work-unit LDS layout and the valence term evaluators.
#pragma once

#include "int95.h"
#include "internal.h"

namespace stormm_amd {

// Generalized Born Taylor-series coefficients (far-field expansion of the HCT integral),
// src/Constants/generalized_born.h:27-36.
constexpr double kGTA = 0.33333333333333333333, kGTB = 0.4, kGTC = 0.42857142857142857143,
                 kGTD = 0.44444444444444444444, kGTDD = 0.45454545454545454545;
constexpr double kGTE = 1.33333333333333333333, kGTF = 2.4, kGTG = 3.42857142857142857143,
                 kGTH = 4.44444444444444444444, kGTHH = 5.45454545454545454545;
constexpr double kGbKscale = 0.73;      // src/Constants/generalized_born.h:120

// ------------------------------------------------------------------------------------------
// Precision traits.  Single precision uses the hardware transcendental units (v_rsq, v_rcp,
// v_log, v_exp); double precision refines the hardware estimates and has its own logarithm and
// hyperbolic tangent for the arguments that occur.
// ------------------------------------------------------------------------------------------
// Nearest integer (ties to even, as rint) of a double as int64.  For |x| < 2^51, adding
// 1.5 * 2^52 rounds x to an integer held in the low bits of the sum's bit pattern; subtracting
// the constant's pattern recovers it in two instructions.  Larger or non-finite values take the
// library conversion.
__device__ __forceinline__ long long round_to_ll(double x) {
  // x must be rounded to double before the addition: never fuse it with the product that made x.
#pragma clang fp contract(off)
  constexpr double kMagic = 6755399441055744.0;  // 1.5 * 2^52
  if (__builtin_expect(fabs(x) < 2251799813685248.0, 1)) {
    return __double_as_longlong(x + kMagic) - __double_as_longlong(kMagic);
  }
  return static_cast<long long>(__builtin_rint(x));
}

template <typename T> struct Prec;

template <> struct Prec<float> {
  using crd_t = int;
  static __device__ __forceinline__ float rsqrt(float x) { return __builtin_amdgcn_rsqf(x); }
  static __device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
  static __device__ __forceinline__ float sqrt(float x) { return __builtin_sqrtf(x); }
  static __device__ __forceinline__ float cbrt(float x) { return ::cbrtf(x); }
  static __device__ __forceinline__ float log(float x) {
    return __builtin_amdgcn_logf(x) * 0.693147180559945309417f;
  }
  static __device__ __forceinline__ float exp(float x) {
    return __builtin_amdgcn_exp2f(x * 1.44269504088896340736f);
  }
  static __device__ __forceinline__ long long fixed(float x) {
    return round_to_ll(static_cast<double>(x));
  }
};

template <> struct Prec<double> {
  using crd_t = double;
  // ln 2 in two parts, the first of 36 bits.
  static constexpr double kLn2High = 0x1.62e42fefap-1, kLn2Low = 0x1.cf79abc9e3b39p-40;
  // The hardware estimates leave residuals e = 1 - x y (reciprocal) and 1 - x y^2 (reciprocal
  // square root) of at most 2^-24 and 2^-22 (measured over a full octave); the binomial series
  // y (1 + e + e^2) and y (1 + e / 2 + 3 e^2 / 8) leave about e^3, below the last bit.  The root's
  // estimate is cut to 26 bits first, so that y^2 and with it the residual are exact: 0.5005 units
  // in the last place at most, where the rounding of x y left 0.99.  Three and six instructions
  // after the estimate, where two Newton-Raphson steps took four and eight.  For positive, finite,
  // normal arguments (distances and radii here).
  static __device__ __forceinline__ double rsqrt(double x) {
    const double y = __longlong_as_double(__double_as_longlong(__builtin_amdgcn_rsq(x)) &
                                          ~0x7ffffffLL);
    const double e = fma(-x, y * y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
  }
  static __device__ __forceinline__ double rcp(double x) {
    const double y = __builtin_amdgcn_rcp(x);
    const double e = fma(-x, y, 1.0);
    return fma(y, fma(e, e, e), y);
  }
  static __device__ __forceinline__ double sqrt(double x) { return ::sqrt(x); }
  static __device__ __forceinline__ double cbrt(double x) { return ::cbrt(x); }
  // Natural logarithm of a positive normal number m 2^e, sqrt(1/2) <= m < sqrt(2): e ln 2 +
  // 2 artanh(f), f = (m - 1) / (m + 1), with (artanh(f) / f - 1) / f^2 interpolated at Chebyshev
  // nodes over f^2 <= 0.0295 (relative error 4e-18 before rounding).  What the quotient (whose
  // denominator m + 1 rounds too) and the sum e ln 2 + 2 f leave is carried along and joined with
  // the smaller terms, and ln 2 is held in two parts, the first of 36 bits so that its multiples
  // are exact: 0.57 units in the last place at most over the ratios of distances that are its
  // arguments, where the library has 0.64 in twice the instructions (98 with its constants).
  static __device__ __forceinline__ double log(double x) {
    double m = __builtin_amdgcn_frexp_mant(x);
    int e = __builtin_amdgcn_frexp_exp(x);
    const bool low = m < 0.70710678118654752440;
    m = low ? m + m : m;
    e -= low ? 1 : 0;
    const double d = m + 1.0;
    const double d_rest = m - (d - 1.0);
    const double inv = rcp(d);
    const double f = (m - 1.0) * inv;
    const double f_rest = fma(-f, d_rest, fma(-f, d, m - 1.0)) * inv;
    const double s = f * f;
    double h = 0.07308292712444311;
    h = fma(h, s, 0.07665855309105386);
    h = fma(h, s, 0.09091444727837474);
    h = fma(h, s, 0.11111105565129939);
    h = fma(h, s, 0.14285714313001635);
    h = fma(h, s, 0.19999999999949722);
    h = fma(h, s, 0.3333333333333335);
    const double k = static_cast<double>(e);
    const double f2 = f + f;
    const double sum = fma(k, kLn2High, f2);
    const double sum_rest = fma(k, kLn2High, -sum) + f2;
    return sum + fma(f2, s * h, fma(2.0, f_rest, fma(k, kLn2Low, sum_rest)));
  }
  // The library's exponential: 42 instructions with its constants.  Shorter ones of this domain
  // were less exact: a reduction by one constant for k ln 2 leaves an error that grows with k (12
  // units in the last place at -40 against 0.87), a two-part one with as long a polynomial 0.93
  // in 39 instructions.
  static __device__ __forceinline__ double exp(double x) { return ::exp(x); }
  // tanh(x) = -E / (2 + E) with E = exp(-2 |x|) - 1, E and the denominator held as a value and
  // what its rounding left.  -2 |x| = k ln 2 + r, |r| <= ln 2 / 2; exp(r) - 1 = r + r^2 g(r) with g
  // interpolated at Chebyshev nodes (relative error 1e-18 of exp); E = (2^k - 1) + 2^k (exp(r) - 1),
  // k >= -58 (below, the result is one).  0.81 units in the last place at most, the library's 0.86,
  // in a third of its 165 instructions.
  static __device__ __forceinline__ double tanh(double x) {
    const double t = -2.0 * fabs(x);
    const double z = (t < -40.0) ? -40.0 : t;
    const double k = __builtin_rint(z * 1.4426950408889634074);
    const double r_high = fma(k, -kLn2High, z);
    const double r = fma(k, -kLn2Low, r_high);
    const double r_rest = fma(k, -kLn2Low, r_high - r);
    double g = 2.0914686968086876e-09;
    g = fma(g, r, 2.5105217004720745e-08);
    g = fma(g, r, 2.75572736431103e-07);
    g = fma(g, r, 2.7557255400206422e-06);
    g = fma(g, r, 2.4801587325547743e-05);
    g = fma(g, r, 0.00019841269874820627);
    g = fma(g, r, 0.0013888888888883748);
    g = fma(g, r, 0.008333333333326136);
    g = fma(g, r, 0.04166666666666667);
    g = fma(g, r, 0.1666666666666667);
    g = fma(g, r, 0.5);
    const double q = fma(r * r, g, r_rest);
    const double p = __builtin_ldexp(1.0, static_cast<int>(k));
    const double p1 = p - 1.0;
    const double a = fma(p, r, p1);
    const double a_rest = fma(p, r, p1 - a) + fma(p, q, p - (p1 + 1.0));
    const double e = a + a_rest;
    const double e_rest = (a - e) + a_rest;
    const double d = 2.0 + e;
    const double d_rest = ((2.0 - d) + e) + e_rest;
    const double inv = rcp(d);
    const double f = e * inv;
    return copysign(fma(fma(-f, d, e) + fma(-f, d_rest, e_rest), inv, f), x);
  }
  // a / b and sqrt(x) from inv_b = rcp(b) and y = rsqrt(x): one residual step leaves them as the
  // IEEE operations round them (the step's own error is 2^-50 units in the last place), in 3 and
  // 4 instructions where those take 12 and 22.  For arguments whose quotient and root are normal.
  static __device__ __forceinline__ double quotient(double a, double b, double inv_b) {
    const double q = a * inv_b;
    return fma(fma(-q, b, a), inv_b, q);
  }
  static __device__ __forceinline__ double root(double x, double y) {
    const double s = x * y;
    return fma(fma(-s, s, x), 0.5 * y, s);
  }
  static __device__ __forceinline__ long long fixed(double x) { return round_to_ll(x); }
};

// ------------------------------------------------------------------------------------------
// Rotation of a value one lane to the right inside each 16-lane DPP row (row_ror:1): after k
// rotations lane L holds what lane (L - k) mod 16 of its row held.
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ int row_rotate(int v) {
  // Every lane of a row has a source under row_ror, so the bound-control and old-value
  // operands never take effect; mov_dpp leaves the old value undefined, which lets the compiler
  // rotate a register in place instead of zero-filling a fresh one each step.
  return __builtin_amdgcn_mov_dpp(v, 0x121, 0xF, 0xF, true);
}
__device__ __forceinline__ float row_rotate(float v) {
  return __int_as_float(row_rotate(__float_as_int(v)));
}
__device__ __forceinline__ double row_rotate(double v) {
  const long long bits = __double_as_longlong(v);
  const int lo = row_rotate(static_cast<int>(bits & 0xffffffffLL));
  const int hi = row_rotate(static_cast<int>(bits >> 32));
  return __longlong_as_double((static_cast<long long>(hi) << 32) |
                              (static_cast<long long>(lo) & 0xffffffffLL));
}

// The value that lane (L - K) mod 16 of the row holds, K = 0..15 (row_ror:K): the j-atom data a
// lane meets at rotation step K while the data stay where they were loaded.  With one use per
// rotated value the compiler folds the move into the arithmetic instruction as its DPP source
// operand, so reading rotated data costs no instruction of its own.
template <int K> __device__ __forceinline__ int row_ror(int v) {
  if constexpr (K == 0) {
    return v;
  }
  else {
    return __builtin_amdgcn_mov_dpp(v, 0x120 + K, 0xF, 0xF, true);
  }
}
template <int K> __device__ __forceinline__ float row_ror(float v) {
  return __int_as_float(row_ror<K>(__float_as_int(v)));
}
template <int K> __device__ __forceinline__ double row_ror(double v) {
  const long long bits = __double_as_longlong(v);
  const int lo = row_ror<K>(static_cast<int>(bits & 0xffffffffLL));
  const int hi = row_ror<K>(static_cast<int>(bits >> 32));
  return __longlong_as_double((static_cast<long long>(hi) << 32) |
                              (static_cast<long long>(lo) & 0xffffffffLL));
}

// Calls f(std::integral_constant<int, K>) for each K of the sequence, in order (rotation steps
// unrolled with compile-time rotation counts).
// A scheduling barrier after each step keeps the steps' live values from overlapping (the
// unrolled steps would otherwise be interleaved past the register budget).
template <typename F, int... K>
__device__ __forceinline__ void unrolled_steps(F &&f, std::integer_sequence<int, K...>) {
  ((f(std::integral_constant<int, K>{}), __builtin_amdgcn_sched_barrier(0)), ...);
}

// Makes x final at this point: an empty statement that reads and rewrites its register, so that
// the arithmetic producing x is not moved below it (into a later block, where the rotated
// operands that arithmetic reads would each need a separate move).
template <typename T> __device__ __forceinline__ void settle(T &x) {
  asm volatile("" : "+v"(x));
}

// Sum of a 64-bit integer over the 16 lanes of a row, on every lane of the row (all 16 lanes must
// be active): rotations, whose moves fold into the additions, where a shuffle goes through the
// LDS crossbar.
template <int K> __device__ __forceinline__ long long row_ror(long long v) {
  const int lo = row_ror<K>(static_cast<int>(v & 0xffffffffLL));
  const int hi = row_ror<K>(static_cast<int>(v >> 32));
  return (static_cast<long long>(hi) << 32) | (static_cast<long long>(lo) & 0xffffffffLL);
}
__device__ __forceinline__ long long row_sum(long long v) {
  v += row_ror<8>(v);
  v += row_ror<4>(v);
  v += row_ror<2>(v);
  v += row_ror<1>(v);
  return v;
}

__device__ __forceinline__ void lds_add(long long *addr, long long v) {
  atomicAdd(reinterpret_cast<unsigned long long *>(addr), static_cast<unsigned long long>(v));
}

// ------------------------------------------------------------------------------------------
// Born-radius integral contribution of a sphere of screened radius sj at distance r onto an
// atom of offset radius ri (HCT pairwise descreening), src/Potential/nonbonded_potential.tpp:
// 578-617, and its radial derivative divided by r (sign convention of :1138-1188).  The
// reference takes a far-field Taylor series in (sj / r)^2 when r > 4 sj and one of three
// analytic branches otherwise:
//   b2  r > ri + sj           : -sj / (2 (r^2 - sj^2))             - ln(|r - sj| / (r + sj)) / (4 r)
//   b3  |ri - sj| < r <= ri+sj: -(1/ri (2 - theta) - 1/(r + sj)) / 4 - ln(ri / (r + sj)) / (4 r)
//   b4  r <= |ri - sj|, ri<sj : -sj / (2 (r^2 - sj^2)) - 1/ri       - ln(|r - sj| / (r + sj)) / (4 r)
// (zero when none applies).  The far and near forms are separate functions so that the tile
// loops can evaluate the cheap series for every lane and hand the rarer near pairs to a
// compacted pass.  The far-field series, -s^3 / r^4 (a + b x + c x^2 + d x^3 + dd x^4) with
// x = (s / r)^2, and its derivative follow :595-598 and :1121-1124.  The near branches share
// one reciprocal and one logarithm: b3 needs 1/(r + sj), b2 and b4 need 1/(r + sj) and
// 1/(r^2 - sj^2), both taken from 1/((r + sj)(r - sj)) since |r - sj| >= ri keeps that product
// away from zero in those branches.
// ------------------------------------------------------------------------------------------
// Squared distance given to an absent pair in the Born-integral and derivative tile loops: far
// beyond 4 screened radii of any atom, with 1 / r^4 below the smallest denormal, so both far-field
// terms round to exactly zero and the pair never enters the near-field queue.
// kCrd is the coordinate (on all three axes, +kCrd for an absent i atom, -kCrd for an absent j
// atom) that puts an absent atom of a tile as far away, with or without a partner present.
template <typename T> struct FarAway;
template <> struct FarAway<float> {
  static constexpr float kR2 = 1.0e30f;
  static constexpr float kCrd = 1.0e15f;
};
template <> struct FarAway<double> {
  static constexpr double kR2 = 1.0e200;
  static constexpr double kCrd = 1.0e100;
};

// Far-field series in x = (s / r)^2: the Born-integral term is -s^3 / r^4 times psi_series(x),
// the derivative term (divided by r) s^3 / r^6 times dpsi_series(x).
template <typename T>
__device__ __forceinline__ T psi_series(T x) {
  return T(kGTA) + x * (T(kGTB) + x * (T(kGTC) + x * (T(kGTD) + x * T(kGTDD))));
}

template <typename T>
__device__ __forceinline__ T dpsi_series(T x) {
  return T(kGTE) + x * (T(kGTF) + x * (T(kGTG) + x * (T(kGTH) + x * T(kGTHH))));
}

// Shared set-up of the near branches: branch flags, 1/(r + sj), 1/(r^2 - sj^2) (b2, b4) and
// the logarithm's argument.
template <typename T> struct NearBranch {
  bool b3, any, b4;
  T uij, t1, lg;
  __device__ __forceinline__ NearBranch(T r, T ri, T sj) {
    using P = Prec<T>;
    const bool b2 = r > ri + sj;
    b3 = (!b2) && (r > fabs(ri - sj));
    b4 = (!b2) && (!b3) && (ri < sj);
    any = b2 || b3 || b4;
    const T rps = r + sj;
    const T rms = r - sj;
    const T inv = P::rcp(b3 ? rps : rps * rms);
    uij = b3 ? inv : rms * inv;
    t1 = inv;
    lg = P::log((b3 ? ri : fabs(rms)) * uij);
  }
};

template <typename T>
__device__ __forceinline__ T psi_near(T r, T r2, T invr, T ri, T iri, T sj) {
  const NearBranch<T> nb(r, ri, sj);
  const T theta = T(0.5) * iri * invr * (r2 + (ri * ri) - (sj * sj));
  const T a3 = -T(0.25) * ((iri * (T(2) - theta)) - nb.uij);
  const T a24 = -(T(0.5) * sj * nb.t1) - (nb.b4 ? iri : T(0));
  const T res = (nb.b3 ? a3 : a24) - (T(0.25) * invr * nb.lg);
  return nb.any ? res : T(0);
}

template <typename T>
__device__ __forceinline__ T dpsi_near(T r, T r2, T invr, T invr2, T ri, T iri, T sj) {
  const NearBranch<T> nb(r, ri, sj);
  const T invr3 = invr2 * invr;
  const T a3 = -T(0.25) * ((-T(0.5) * (r2 - (ri * ri) + (sj * sj)) * invr3 * iri * iri) +
                           (invr * nb.uij * (nb.uij - invr)));
  const T a24 = sj * nb.t1 * (nb.t1 - (T(0.5) * invr2));
  const T res = (nb.b3 ? a3 : a24) + (T(0.25) * invr3 * nb.lg);
  return nb.any ? res : T(0);
}

// Effective Born radius, its inverse, and (OBC) its derivative by the integral psi, from the offset
// radius rho and the intrinsic radius pbr, src/Potential/nonbonded_potential.tpp:731-781, 985-1017.
struct BornRadius {
  double R, inv_R, dr_dpsi;
};
__device__ __forceinline__ BornRadius born_radius(int igb, double al, double be, double ga,
                                                  double rho, double pbr, double psi) {
  using D = Prec<double>;
  BornRadius b;
  b.dr_dpsi = 0.0;
  if (igb == 1) {
    b.R = 1.0 / ((1.0 / rho) + psi);
    b.R = (b.R < 0.0) ? 30.0 : b.R;
    b.inv_R = 1.0 / b.R;
    return b;
  }
  const double fipsi = psi * (-rho);
  const double thi = D::tanh((al - (be * fipsi) + (ga * fipsi * fipsi)) * fipsi);
  const double inv_pbr = D::rcp(pbr);
  b.R = D::rcp(D::rcp(rho) - D::quotient(thi, pbr, inv_pbr));
  b.inv_R = D::rcp(b.R);
  b.dr_dpsi = D::quotient((al - ((2.0 * be) - (3.0 * ga * fipsi)) * fipsi) * (1.0 - thi * thi) *
                              rho, pbr, inv_pbr);
  return b;
}

// Fixed-precision image round(x * 2^bits) of a pair contribution added to an LDS accumulator.
// Single precision converts through 32 bits (rounding at 2^-min(bits, 28), then shifting) when
// the value fits, and through double precision otherwise.
__device__ __forceinline__ long long fixed_contrib(float x, int bits) {
  const int lo = (bits < 28) ? bits : 28;
  const float v = x * __builtin_ldexpf(1.0f, lo);
  if (fabsf(v) < 2147483520.0f) {
    return static_cast<long long>(__float2int_rn(v)) << (bits - lo);
  }
  return round_to_ll(ldexp(static_cast<double>(x), bits));
}
__device__ __forceinline__ long long fixed_contrib(double x, int bits) {
  return round_to_ll(ldexp(x, bits));
}

// Largest block a kernel is compiled for: 16 wavefronts leave 128 registers to a lane, and the
// clash-damped force evaluations in double precision (HEAVY) need 152.
template <typename T, bool HEAVY> struct EvalBlockLimit {
  static constexpr int value = kMaxEvalBlock;
};
template <> struct EvalBlockLimit<double, true> {
  static constexpr int value = kMaxEvalBlockDoubleClash;
};

// ------------------------------------------------------------------------------------------
// Work-unit LDS layout.  Everything the pair loops read or add to of one atom lies in one record,
// so that a lane reaches all of it from one address, with wide reads and constant offsets: with
// one array per quantity the tile set-up and the near-pair passes spent a third of their vector
// instructions on addresses.  The record's 80 bytes (144 in double precision) put the same field
// of 16 consecutive atoms in different LDS banks (20 l mod 64 banks differ for l = 0..15).
// ------------------------------------------------------------------------------------------
template <typename T> struct alignas(16) AtomPos {
  typename Prec<T>::crd_t x, y, z;
  T scr;                    // screened radius
};
template <typename T> struct alignas(16) AtomNb {
  T q, p1, p2;              // charge and Lennard-Jones parameters
  T rad;                    // effective Born radius
};
template <typename T> struct alignas(2 * sizeof(T)) AtomRad {
  T rho, irho;              // offset radius and its inverse
};
template <typename T> struct AtomFields {
  AtomPos<T> pos;
  AtomNb<T> nb;
  AtomRad<T> rr;
  union {
    long long psi;          // Born-radius integral; from the radii stage on dR/dpsi (a double)
    T sd;                   // chain-rule factor, from the chain stage on
  };
  long long fx, fy, fz;     // forces
  long long dedr;           // dE/dR
};
template <typename T> struct AtomRec;
template <> struct AtomRec<float> : AtomFields<float> {};
template <> struct AtomRec<double> : AtomFields<double> {
  double irad;              // inverse Born radius (single precision keeps it in WuLds::irad)
  double pad;
};
static_assert(sizeof(AtomRec<float>) == 80 && sizeof(AtomRec<double>) == 144,
              "atom records keep 16 consecutive atoms' fields in different LDS banks");

template <typename T> struct WuLds {
  using crd_t = typename Prec<T>::crd_t;
  int4 *tasks;              // the unit's tile tasks, placed at their systems' LDS bases
  AtomRec<T> *atom;
  long long *nrg, *org;
  double *move;             // per system: pending line move (coordinate units per direction unit)
  T *irad;                  // inverse Born radius (single precision)
  int *gidx, *slot;
  WuSys *sys;
  int *work;                // per-stage work-item counters (kStageCounters)
  T *clash_d, *clash_r;     // per-system clash distance and sigma ratio of this evaluation
  int *clash_on;            // per-system flag: damped potentials apply
  unsigned *nearq;          // kNearQueueStride entries per wavefront: its near-pair queue

  static constexpr __host__ __device__ size_t bytes(int maxa, int waves) {
    const size_t m = static_cast<size_t>(maxa);
    return (kMaxWuTasks * sizeof(int4)) +
           (m * sizeof(AtomRec<T>)) + (kMaxWuSystems * sizeof(WuSys)) +
           (kMaxWuSystems * 16 * sizeof(long long)) + (3 * kMaxWuSystems * sizeof(long long)) +
           (kMaxWuSystems * sizeof(double)) + (m * sizeof(T)) + (2 * kMaxWuSystems * sizeof(T)) +
           (2 * m * sizeof(int)) + (kStageCounters * sizeof(int)) +
           (kMaxWuSystems * sizeof(int)) +
           (static_cast<size_t>(waves) * kNearQueueStride * sizeof(unsigned));
  }

  // maxa is a multiple of 16 (kTile), so every array below starts on the alignment of its type.
  __device__ WuLds(unsigned char *base, int maxa, int waves) {
    unsigned char *p = base;
    auto take = [&](size_t nbytes) {
      unsigned char *r = p;
      p += nbytes;
      return r;
    };
    const size_t m = static_cast<size_t>(maxa);
    tasks = reinterpret_cast<int4 *>(take(kMaxWuTasks * sizeof(int4)));
    atom = reinterpret_cast<AtomRec<T> *>(take(m * sizeof(AtomRec<T>)));
    sys = reinterpret_cast<WuSys *>(take(kMaxWuSystems * sizeof(WuSys)));
    nrg = reinterpret_cast<long long *>(take(kMaxWuSystems * 16 * sizeof(long long)));
    org = reinterpret_cast<long long *>(take(3 * kMaxWuSystems * sizeof(long long)));
    move = reinterpret_cast<double *>(take(kMaxWuSystems * sizeof(double)));
    irad = reinterpret_cast<T *>(take(m * sizeof(T)));
    clash_d = reinterpret_cast<T *>(take(kMaxWuSystems * sizeof(T)));
    clash_r = reinterpret_cast<T *>(take(kMaxWuSystems * sizeof(T)));
    gidx = reinterpret_cast<int *>(take(m * sizeof(int)));
    slot = reinterpret_cast<int *>(take(m * sizeof(int)));
    work = reinterpret_cast<int *>(take(kStageCounters * sizeof(int)));
    clash_on = reinterpret_cast<int *>(take(kMaxWuSystems * sizeof(int)));
    nearq = reinterpret_cast<unsigned *>(take(static_cast<size_t>(waves) * kNearQueueStride *
                                              sizeof(unsigned)));
  }
};

static_assert(2 * WuLds<double>::bytes(kTwoBlockAtomsDouble, kEvalBlock / 64) <= kLdsPerCu &&
                  2 * WuLds<double>::bytes(kTwoBlockAtomsDouble + kTile, kEvalBlock / 64) >
                      kLdsPerCu,
              "two units of kTwoBlockAtomsDouble atoms, and no larger ones, share a compute unit");

// Threads of an evaluation block.  With no more units than compute units each block has its
// compute unit to itself, and 16 wavefronts hide the latencies that 8 leave open (24 systems of
// 487 atoms 180 -> 144 us); with more units two blocks of 8 share it, whose barriers do not
// coincide (1024 systems 87 us against 100).  In double precision two such blocks need units of
// at most 336 atoms to fit the LDS (600 systems of 20-200 atoms 77 us against 101); beyond that
// one block takes the whole compute unit (1024 systems of 24-256 atoms 158 us against 179 at
// half the size), and a unit alone that is too small for 16 wavefronts takes 8 (200 systems of
// 100 atoms 37 us against 41).  A HEAVY kernel's registers hold 12 wavefronts instead of 16.
// A size that was asked for (the pool takes any) becomes whole wavefronts, no fewer than cover a
// unit's atoms at stage_load's two to a thread.  Results do not depend on the size.
template <typename T, bool HEAVY> inline int eval_block(const MMKit &k, int blocks) {
  constexpr int limit = EvalBlockLimit<T, HEAVY>::value;
  static_assert(limit >= kMinEvalBlock && limit % 64 == 0, "a block is whole wavefronts");
  if (k.block > 0) {
    const int asked = (k.block < limit) ? k.block : limit;
    return (asked < kMinEvalBlock) ? kMinEvalBlock : (asked + 63) / 64 * 64;
  }
  if (sizeof(T) == 4) {
    return (blocks <= k.cus) ? kEvalBlockSparse : kEvalBlock;
  }
  const bool half = (blocks <= k.cus) ? (k.maxa <= kSmallUnitDouble) :
                                        (2 * WuLds<T>::bytes(k.maxa, limit / 128) <= kLdsPerCu);
  return half ? (limit / 2) : limit;
}

// Inverse Born radius of LDS atom a.
__device__ __forceinline__ float &inv_radius(const WuLds<float> &L, int a) { return L.irad[a]; }
__device__ __forceinline__ double &inv_radius(const WuLds<double> &L, int a) {
  return L.atom[a].irad;
}

// The j atoms of a tile in double precision.  A 64-bit value has no DPP operand form, so rotating
// it takes two moves: 16 of the 114 vector instructions of a pair step.  A step reads the j atom
// it meets from the atom records instead, whose byte offset (one 32-bit value) rotates.
struct JRecords {
  AtomRec<double> *atom;
  int off;
  __device__ __forceinline__ JRecords(AtomRec<double> *records, int j0)
      : atom(records), off(j0 * static_cast<int>(sizeof(AtomRec<double>))) {}
  // The record of the atom that the lane meets K steps on.
  template <int K> __device__ __forceinline__ const AtomRec<double> &at() const {
    return *reinterpret_cast<const AtomRec<double> *>(
        reinterpret_cast<const unsigned char *>(atom) + row_ror<K>(off));
  }
  template <int K> __device__ __forceinline__ void rotate() { off = row_ror<K>(off); }
};

// Displacement between two LDS coordinates in Angstroms.
__device__ __forceinline__ float crd_delta(int a, int b, float scale) {
  return static_cast<float>(a - b) * scale;
}
__device__ __forceinline__ double crd_delta(double a, double b, double) { return a - b; }

// exp(-r^2 / (4 Ri Rj)) of the GB pair function as eval(r^2 * (1 / Rj) * (kScale / Ri)): the
// hardware base-2 exponential in single precision (kScale carries log2 e), Prec's in double
// precision.
template <typename T> struct GbExp;
template <> struct GbExp<float> {
  static constexpr float kScale = -0.25f * 1.44269504088896340736f;
  static __device__ __forceinline__ float eval(float x) { return __builtin_amdgcn_exp2f(x); }
};
template <> struct GbExp<double> {
  static constexpr double kScale = -0.25;
  static __device__ __forceinline__ double eval(double x) { return Prec<double>::exp(x); }
};

// Coordinates of a pair tile's atoms in Angstroms in the working precision.  Single precision
// converts the LDS fixed-precision coordinates relative to a point between the tile's two atom
// blocks once per task, as the reference imports tile coordinates relative to the tile's centre
// (src/Potential/nonbonded_potential_tilegroups.cui:395-426), so the rotation steps take plain
// differences.  Double precision holds Angstroms already.
__device__ __forceinline__ int tile_centre(int a, int b) { return (a >> 1) + (b >> 1); }
__device__ __forceinline__ double tile_centre(double, double) { return 0.0; }
__device__ __forceinline__ float tile_crd(int v, int centre, float scale) {
  return static_cast<float>(v - centre) * scale;
}
__device__ __forceinline__ double tile_crd(double v, double, double) { return v; }

// Conversion of a fixed-precision global coordinate to the LDS representation.
template <typename T> struct CrdConv;
template <> struct CrdConv<float> {
  static __device__ __forceinline__ int to_lds(long long v, long long origin, int shift) {
    const long long d = v - origin;
    const long long half = (shift > 0) ? (1LL << (shift - 1)) : 0LL;
    return static_cast<int>((d + half) >> shift);
  }
  static __device__ __forceinline__ bool in_range(long long v, long long origin, int shift) {
    const long long d = (v - origin) >> shift;
    return d > -2147483000LL && d < 2147483000LL;
  }
  // Displacements from a 95-bit value (exact 128-bit difference from the origin).
  static __device__ __forceinline__ int to_lds_wide(__int128 d, int shift) {
    const __int128 half = (shift > 0) ? (static_cast<__int128>(1) << (shift - 1)) : 0;
    return static_cast<int>((d + half) >> shift);
  }
  static __device__ __forceinline__ bool in_range_wide(__int128 d, int shift) {
    const __int128 q = d >> shift;
    return q > -2147483000 && q < 2147483000;
  }
};
template <> struct CrdConv<double> {
  static __device__ __forceinline__ double to_lds(long long v, long long origin, int shift) {
    return static_cast<double>(v - origin) * ldexp(1.0, -shift);
  }
  static __device__ __forceinline__ bool in_range(long long, long long, int) { return true; }
  static __device__ __forceinline__ double to_lds_wide(__int128 d, int shift) {
    return i128_to_double(d) * ldexp(1.0, -shift);
  }
  static __device__ __forceinline__ bool in_range_wide(__int128 d, int shift) {
    const __int128 q = d >> shift;
    return q > -1099511627776LL && q < 1099511627776LL;
  }
};

}  // namespace stormm_amd
