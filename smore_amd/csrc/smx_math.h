// Device math for the distance functors: digamma, trigamma, log-gamma.
//
// Numerical contract: same series as the operator being replaced
// (smore/common/torchext/cuda_math_ext.h:130-211 -- reflection, upward
// recurrence, asymptotic tail), evaluated in the precision of T.
#pragma once
#include <hip/hip_runtime.h>

namespace smx {

template <typename T> struct MathConst;
template <> struct MathConst<float> {
  static constexpr float pi = 3.14159265358979323846f;
};
template <> struct MathConst<double> {
  static constexpr double pi = 3.14159265358979323846;
};

__device__ __forceinline__ float m_acc_log(float x) { return logf(x); }
__device__ __forceinline__ double m_acc_log(double x) { return log(x); }
__device__ __forceinline__ float m_sqrt(float x) { return sqrtf(x); }
__device__ __forceinline__ double m_sqrt(double x) { return sqrt(x); }
__device__ __forceinline__ float m_sin(float x) { return sinf(x); }
__device__ __forceinline__ double m_sin(double x) { return sin(x); }
__device__ __forceinline__ float m_lgamma(float x) { return lgammaf(x); }
__device__ __forceinline__ double m_lgamma(double x) { return lgamma(x); }
__device__ __forceinline__ float m_abs(float x) { return fabsf(x); }
__device__ __forceinline__ double m_abs(double x) { return fabs(x); }
__device__ __forceinline__ float m_min(float a, float b) { return fminf(a, b); }
__device__ __forceinline__ double m_min(double a, double b) { return fmin(a, b); }

// psi(x).  x == 0 -> -/+inf, negative integers -> NaN, x < 0 by reflection.
template <typename T>
__device__ inline T digamma(T x) {
  T shift = 0;
  if (x <= 0) {
    if (x == 0) return copysign((T)INFINITY, -x);
    if (x == trunc(x)) return (T)NAN;
    // the cotangent term is evaluated in double: rounding of pi*x matters near poles
    shift = (T)(-3.14159265358979323846 / tan(3.14159265358979323846 * (double)x));
    x = 1 - x;
  }
  while (x < 10) {
    shift -= 1 / x;
    x += 1;
  }
  if (x == 10) return shift + (T)2.25175258906672110764;
  T tail = 0;
  if (x < (T)1.0e17) {
    const T z = 1 / (x * x);
    T p = (T)8.33333333333333333333E-2;
    p = p * z + (T)-2.10927960927960927961E-2;
    p = p * z + (T)7.57575757575757575758E-3;
    p = p * z + (T)-4.16666666666666666667E-3;
    p = p * z + (T)3.96825396825396825397E-3;
    p = p * z + (T)-8.33333333333333333333E-3;
    p = p * z + (T)8.33333333333333333333E-2;
    tail = z * p;
  }
  return m_acc_log(x) - ((T)0.5 / x) - tail + shift;
}

// psi'(x).  x < 0.5 by reflection, six recurrence steps, asymptotic tail.
template <typename T>
__device__ inline T trigamma(T x) {
  const T pi = MathConst<T>::pi;
  T sign = 1, acc = 0;
  if (x < (T)0.5) {
    sign = -1;
    const T s = m_sin(pi * x);
    acc -= (pi * pi) / (s * s);
    x = 1 - x;
  }
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    acc += 1 / (x * x);
    x += 1;
  }
  const T ixx = 1 / (x * x);
  acc += (1 + 1 / (2 * x) + ixx * ((T)1 / 6 - ixx * ((T)1 / 30 - ixx * ((T)1 / 42)))) / x;
  return sign * acc;
}

// ---- fast fp32 forms for the fused Beta-KL kernels ----------------------------------------------
// For fast_lo <= x <= fast_hi the argument is shifted by a fixed six steps, so there is no
// data-dependent loop and no division:
//   psi(x)    = psi(x+6)  - N(x)/D(x)            D(x) = x(x+1)...(x+5),  N = D'
//   psi'(x)   = psi'(x+6) + P10(x)/D(x)^2        P10 = N^2 - N' D (expanded: all coefficients positive)
//   lgamma(x) = lgamma(x+6) - ln D(x)
// with the asymptotic series at y = x+6 >= 6 (first neglected terms: 2.5e-9, 3.3e-9, 2.1e-9).  The
// polynomials have positive coefficients, so Horner's rule is free of cancellation for x > 0.
// Reciprocals and logarithms use the hardware approximations (1 ulp).  Outside the interval the
// callers fall back to the general routines above.
constexpr float kFastLo = 0.02f;
constexpr float kFastHi = 1000.0f;

__device__ __forceinline__ float f_rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float f_log(float x) {
#pragma clang fp contract(off)
  return __builtin_amdgcn_logf(x) * 0.69314718055994531f;
}

// The multiply-adds of these forms are written out and contraction is off: every kernel gets the same bits for the
// same argument, whatever surrounds the inlined code (the ranking kernels compare scores of one row for equality).
__device__ __forceinline__ float poly_d6(float x) {
#pragma clang fp contract(off)
  float r = __builtin_fmaf(x, x + 15.f, 85.f);
  r = __builtin_fmaf(x, r, 225.f);
  r = __builtin_fmaf(x, r, 274.f);
  r = __builtin_fmaf(x, r, 120.f);
  return x * r;
}
__device__ __forceinline__ float poly_n5(float x) {
  float r = __builtin_fmaf(x, 6.f, 75.f);
  r = __builtin_fmaf(x, r, 340.f);
  r = __builtin_fmaf(x, r, 675.f);
  r = __builtin_fmaf(x, r, 548.f);
  return __builtin_fmaf(x, r, 120.f);
}
__device__ __forceinline__ float poly_p10(float x) {
  float r = __builtin_fmaf(x, 6.f, 150.f);
  r = __builtin_fmaf(x, r, 1635.f);
  r = __builtin_fmaf(x, r, 10200.f);
  r = __builtin_fmaf(x, r, 40208.f);
  r = __builtin_fmaf(x, r, 104370.f);
  r = __builtin_fmaf(x, r, 180455.f);
  r = __builtin_fmaf(x, r, 205800.f);
  r = __builtin_fmaf(x, r, 150152.f);
  r = __builtin_fmaf(x, r, 65760.f);
  return __builtin_fmaf(x, r, 14400.f);
}

struct Shifted {  // what the three functions share for one argument
  float y, ry, z, ln_y, d, rd;
};
__device__ __forceinline__ Shifted shift6(float x, bool want_log) {
#pragma clang fp contract(off)
  Shifted s;
  s.y = x + 6.0f;
  s.ry = f_rcp(s.y);
  s.z = s.ry * s.ry;
  s.ln_y = want_log ? f_log(s.y) : 0.f;
  s.d = poly_d6(x);
  s.rd = f_rcp(s.d);
  return s;
}
__device__ __forceinline__ float digamma_of(float x, const Shifted& s) {
  const float tail = __builtin_fmaf(-s.z, __builtin_fmaf(-s.z, 3.96825397e-3f, 8.33333333e-3f), 8.33333333e-2f);
  const float asym = __builtin_fmaf(-s.z, tail, __builtin_fmaf(-0.5f, s.ry, s.ln_y));
  return __builtin_fmaf(-poly_n5(x), s.rd, asym);
}
__device__ __forceinline__ float trigamma_of(float x, const Shifted& s) {
#pragma clang fp contract(off)
  const float tail = __builtin_fmaf(-s.z, __builtin_fmaf(-s.z, 2.38095238e-2f, 3.33333333e-2f), 1.66666667e-1f);
  const float rz = s.ry * s.z, prd = poly_p10(x) * s.rd;
  const float asym = __builtin_fmaf(rz, tail, __builtin_fmaf(0.5f, s.z, s.ry));
  return __builtin_fmaf(prd, s.rd, asym);
}
// lgamma(x+6) by Stirling's series; lgamma(x) = stirling - ln D(x)
__device__ __forceinline__ float stirling_of(const Shifted& s) {
#pragma clang fp contract(off)
  const float tail = __builtin_fmaf(-s.z, __builtin_fmaf(-s.z, 7.93650794e-4f, 2.77777778e-3f), 8.33333333e-2f);
  const float lead = __builtin_fmaf(s.y - 0.5f, s.ln_y, 0.918938533204672742f - s.y);
  return __builtin_fmaf(s.ry, tail, lead);
}

__device__ __forceinline__ bool fast_ok(float lo, float hi) { return lo >= kFastLo && hi <= kFastHi; }

// (The general routines hand their results back in registers.  By reference they come back through scratch memory, and the
// wait for those loads, where the branches meet, is one for every load in flight.)
typedef float SlowTerms __attribute__((ext_vector_type(4)));

// Entity-side quantities of KL(Beta(a,b) || .): lb = lgamma(a+b) - lgamma(a) - lgamma(b) and the
// three digammas.  One call shares the shifted arguments, logarithms and reciprocals.
static __device__ __noinline__ void beta_terms_slow(float a, float b, float& lb, float& pa, float& pb, float& ps) {
  lb = m_lgamma(a + b) - m_lgamma(a) - m_lgamma(b);
  pa = digamma(a);
  pb = digamma(b);
  ps = digamma(a + b);
}
__device__ __forceinline__ void beta_terms(float a, float b, float& lb, float& pa, float& pb, float& ps) {
#pragma clang fp contract(off)
  const float sum = a + b;
  if (fast_ok(fminf(a, b), sum)) {
    const Shifted sa = shift6(a, true), sb = shift6(b, true), ss = shift6(sum, true);
    pa = digamma_of(a, sa);
    pb = digamma_of(b, sb);
    ps = digamma_of(sum, ss);
    lb = (stirling_of(ss) - stirling_of(sa)) - stirling_of(sb) - f_log(ss.d * sa.rd * sb.rd);
  } else {
    beta_terms_slow(a, b, lb, pa, pb, ps);
  }
}

// ---- the same with the logarithms' sum taken apart -------------------------------------------------
// With w = (x + 3) / 3, y = x + 3 and Stirling's series written out, everything of KL(Beta(a,b) || Beta(qa,qb)) that grows
// with a logarithm has a coefficient of the query alone, because (y - 1/2) ln y of lgamma meets (x - q) ln y of (x - q) psi(x)
// and y - x is 3:
//   KL = k_q + (qs+2.5) ln ws - (qa+2.5) ln wa - (qb+2.5) ln wb + ln(C D(a) D(b) / D(s)) + S(s) - S(a) - S(b)
//        - (a-qa) R(a) - (b-qb) R(b) + (s-qs) R(s)
//   R(x) = ln y - psi(x) = 1/(2y) + V(y) + D'(x)/D(x),  D(x) = x (x + 1) (x + 2),  S, V: what Stirling's series of lgamma and
//   psi leave after the terms written here,  C = e^3 / (3^2.5 sqrt(2 pi)): the constants that are left over,
// and the logarithms are of numbers around 1.  V and S are polynomials of two steps in 1/y^2 fitted for y >= 3 (largest
// error 3.9e-9 and 3.2e-9; the first terms left out of the series at y = x + 6: 2.5e-9 and 2.1e-9), so three steps of
// recurrence do where six are taken above.  BetaE's kernels are bound by the number of their instructions (four cycles each:
// a wavefront that has issued a transcendental one no longer shares its cycles with another), and this is 71 a feature
// instead of 105 in the forward.  One feature's divergence has less than a third of the error (normal rows around 1: 0.5e-6
// instead of 1.7e-6 rms).  512 x 512 pairs of 2 x 400 floats, the forms alone: forward 405 -> 358 us, query gradient 330 -> 299 (437
// and 384 with a branch per feature and the query's values in registers).  Good in the interval of fast_ok.
constexpr float kLn2 = 0.693147180559945f;
constexpr float kBetaConst = 5.14032259e-1f;   // C
constexpr float kLnBetaConst = -6.65469255e-1f;   // ln C
// A constant in a VGPR: an instruction takes one literal, and a scalar register halves the rate of those that have the full one.
__device__ __forceinline__ float vector_const(float c) {
  float v;
  asm("v_mov_b32 %0, %1" : "=v"(v) : "i"(__builtin_bit_cast(int, c)));
  return v;
}
struct BetaArg {
  float w, r;      // (x + 3) / 3 and its reciprocal
  float z;         // r^2
  float d, rd;     // D(x) and its reciprocal; with POLE: (x + 1) (x + 2) and its reciprocal
  float rx;        // POLE: 1/x
  float rest;      // R(x)
  float quot, u;   // not POLE: D'(x)/D(x) and the rest of R(x) without it
};
// POLE: 1/x on its own, D'/D = 1/x + (2x + 3) / ((x + 1) (x + 2)); one special function more, and half the error of psi
// below 5, where the pole is most of it.
template <bool POLE>
__device__ __forceinline__ BetaArg beta_arg(float x) {
#pragma clang fp contract(off)
  BetaArg s;
  s.w = __builtin_fmaf(x, vector_const(3.33333343e-1f), 1.f);
  s.r = f_rcp(s.w);
  s.z = s.r * s.r;
  const float tail = __builtin_fmaf(s.z, __builtin_fmaf(s.z, 4.478603748e-6f, vector_const(-1.023662279e-4f)), 9.259178391e-3f);
  const float u = s.r * __builtin_fmaf(s.r, tail, 1.66666667e-1f);
  if constexpr (POLE) {
    s.d = __builtin_fmaf(x, x + 3.f, 2.f);
    s.rd = f_rcp(s.d);
    s.rx = f_rcp(x);
    s.rest = __builtin_fmaf(__builtin_fmaf(x, 2.f, vector_const(3.f)), s.rd, u) + s.rx;
    s.quot = 0.f;
  } else {
    const float t = __builtin_fmaf(x, x, x + x);
    s.d = t * (x + 1.f);
    s.rd = f_rcp(s.d);
    s.rx = 0.f;
    const float num = __builtin_fmaf(t, vector_const(3.f), 2.f);
    s.rest = __builtin_fmaf(num, s.rd, u);
    s.quot = num * s.rd;
  }
  s.u = u;
  return s;
}
__device__ __forceinline__ float beta_stirling(const BetaArg& s) {   // S(x) / r
#pragma clang fp contract(off)
  return __builtin_fmaf(s.z, __builtin_fmaf(s.z, 2.867135899e-6f, vector_const(-1.026935902e-4f)), 2.777775529e-2f);
}
constexpr float kBetaShift = 2.5f * kLn2;
__device__ __forceinline__ float beta_k(float q) { return __builtin_fmaf(q, kLn2, kBetaShift); }
// lgamma(a+b) - lgamma(a) - lgamma(b) - ln C with ka = (qa+2.5) ln 2 and kb likewise in the place of the row's own.  Query and
// row both go through here: ln C cancels, the sum's coefficient, which is as large as the other two together, is the same rounded
// number on both sides, and a row that equals its query gives the same bits.  (With the coefficient formed from qa + qb for the
// query alone, rows within 1 % of their query were off by 1.1e-4 rms, all of one sign, at 400 features of 1 to 5, and by 1.9e-3 at
// 20 to 60; so they are by 1.6e-5 and 4.2e-4, with the six-step forms above by 5.6e-5 and 6.1e-4.)
__device__ __forceinline__ float beta_logs(const BetaArg& a, const BetaArg& b, const BetaArg& s, float ka, float kb) {
#pragma clang fp contract(off)
  float v = __builtin_amdgcn_logf(a.d * s.rd * b.d) * kLn2;
  v = __builtin_fmaf((ka + kb) - kBetaShift, __builtin_amdgcn_logf(s.w), v);
  v = __builtin_fmaf(-ka, __builtin_amdgcn_logf(a.w), v);
  v = __builtin_fmaf(-kb, __builtin_amdgcn_logf(b.w), v);
  v = __builtin_fmaf(s.r, beta_stirling(s), v);
  v = __builtin_fmaf(-a.r, beta_stirling(a), v);
  return __builtin_fmaf(-b.r, beta_stirling(b), v);
}
// psi'(x) out of the same parts (POLE): 1/x^2 + (2d + 1)/d^2 with d = (x + 1) (x + 2), and psi'(y) = 1/y + 1/(2y^2) plus a
// polynomial fitted as V is (largest error 5.8e-9).  No special function more.  The sum goes from the small terms to 1/y, nearly all
// of it for large x, and 1/x^2, nearly all of it for small x: one rounding each.  (With 1/y first, the gradients of rows at 20 to 60
// had a tenth more error than with the six-step form.)
__device__ __forceinline__ float beta_trigamma(const BetaArg& s) {
#pragma clang fp contract(off)
  const float tail = __builtin_fmaf(s.z, __builtin_fmaf(s.z, 8.307060779e-6f, vector_const(-1.356947031e-4f)), 6.172571429e-3f);
  float v = __builtin_fmaf(s.r * s.z, tail, s.z * 5.55555556e-2f);
  v = __builtin_fmaf(__builtin_fmaf(s.d, 2.f, 1.f), s.rd * s.rd, v);
  return __builtin_fmaf(s.rx, s.rx, __builtin_fmaf(s.r, 3.33333343e-1f, v));
}
// psi(s) - psi(x)
__device__ __forceinline__ float beta_psi_diff(const BetaArg& x, const BetaArg& s) {
#pragma clang fp contract(off)
  return __builtin_fmaf(__builtin_amdgcn_logf(s.w * x.r), kLn2, x.rest - s.rest);
}

static __device__ __noinline__ void digamma3_slow(float a, float b, float& pa, float& pb, float& ps) {
  pa = digamma(a);
  pb = digamma(b);
  ps = digamma(a + b);
}
__device__ __forceinline__ void digamma3(float a, float b, float& pa, float& pb, float& ps) {
  const float sum = a + b;
  if (fast_ok(fminf(a, b), sum)) {
    pa = digamma_of(a, shift6(a, true));
    pb = digamma_of(b, shift6(b, true));
    ps = digamma_of(sum, shift6(sum, true));
  } else {
    digamma3_slow(a, b, pa, pb, ps);
  }
}

// psi(a) - psi(a + b) and psi(b) - psi(a + b), x and y.  In the interval of fast_ok the form of beta_psi_diff, for rows and queries
// alike: a row that equals its query does not pull at it.
__device__ __forceinline__ SlowTerms beta_psi_diffs(float a, float b) {
  const float sum = a + b;
  if (fast_ok(fminf(a, b), sum)) {
    const BetaArg s = beta_arg<true>(sum);
    return SlowTerms{-beta_psi_diff(beta_arg<true>(a), s), -beta_psi_diff(beta_arg<true>(b), s), 0.f, 0.f};
  }
  float pa, pb, ps;
  digamma3_slow(a, b, pa, pb, ps);
  return SlowTerms{pa - ps, pb - ps, 0.f, 0.f};
}
static __device__ __noinline__ SlowTerms beta_psi_diffs_any(float a, float b) { return beta_psi_diffs(a, b); }

static __device__ __noinline__ void trigamma3_slow(float a, float b, float& ta, float& tb, float& ts) {
  ta = trigamma(a);
  tb = trigamma(b);
  ts = trigamma(a + b);
}
__device__ __forceinline__ void trigamma3(float a, float b, float& ta, float& tb, float& ts) {
  const float sum = a + b;
  if (fast_ok(fminf(a, b), sum)) {
    ta = trigamma_of(a, shift6(a, false));
    tb = trigamma_of(b, shift6(b, false));
    ts = trigamma_of(sum, shift6(sum, false));
  } else {
    trigamma3_slow(a, b, ta, tb, ts);
  }
}

// psi' of a, b and their sum: in the interval of fast_ok the form of the entity pass, whatever path the row takes.
static __device__ __noinline__ SlowTerms beta_trigammas_any(float a, float b) {
  const float sum = a + b;
  if (fast_ok(fminf(a, b), sum))
    return SlowTerms{beta_trigamma(beta_arg<true>(a)), beta_trigamma(beta_arg<true>(b)), beta_trigamma(beta_arg<true>(sum)), 0.f};
  float ta, tb, ts;
  trigamma3_slow(a, b, ta, tb, ts);
  return SlowTerms{ta, tb, ts, 0.f};
}

}  // namespace smx
