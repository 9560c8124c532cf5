// Score models of the gather-fused path: logit = gamma - distance, one struct per
// model, built from the per-feature terms in smx_functors.h.
//
//   model      logit                                   reference call site
//   L1         gamma - sum |e-q|                        smore/models/vec.py:85-90
//   L2         gamma - sqrt(sum (e-q)^2)                smore/common/torchext/dist_func/l2_dist.py:59-62
//   BOX        gamma - d_out - cen * d_in               smore/models/box.py:157-164
//   ROTATE     gamma - sum sqrt(dre^2 + dim^2 + 1e-20)  smore/models/rotate.py:137-142
//   BETA_KL    gamma - sum KL(Beta(e) || Beta(q))       smore/models/beta.py:303-308
//   COMPLEX    gamma + sum (e_re q_re + e_im q_im)      smore/models/complex.py:140-148 (a similarity; gamma = 0 there)
//   DISTMULT   gamma + sum e q                          smore/models/distmult.py (distmult_sim; gamma = 0 there)
//
// A model exposes
//   fwd(e1,e2,q,acc0,acc1)      add one feature's term(s) to the lane's accumulators
//   fold(acc0,acc1,p)           the lane's single value to be summed over the wavefront
//   score(sum,p)                logit from that sum
//   coef(g,score,p,c0,c1)       d logit-loss / d accumulator, from the upstream
//                               gradient g of the logit and the saved logit
//   bwd_e / bwd_q               add one feature's gradient w.r.t. entity / query
// Optional entity prologue (BetaE): e' = clamp(e + add, lo, hi)
// (smore/common/modules.py:29-36 applied at smore/models/kg_reasoning.py:352);
// its backward passes gradient where lo <= e + add <= hi.
#pragma once
#include "../../include/smore_amd.h"
#include "smx_functors.h"

namespace smx {

enum Model : int { mL1 = 0, mL2 = 1, mBox = 2, mRotate = 3, mBetaKL = 4, mComplex = 5, mDistmult = 6, mNumModels = 7 };

__host__ __device__ constexpr int model_mul(int m) { return (m == mRotate || m == mBetaKL || m == mComplex) ? 2 : 1; }
__host__ __device__ constexpr int model_nq(int m) { return (m == mL1 || m == mL2 || m == mDistmult) ? 1 : 2; }
// models whose entity derivative can be kept as sign codes (ModelOps<M>::bwd_q_coded / bwd_e_coded)
__host__ __device__ constexpr bool model_coded(int m) { return m == mBox || m == mL1; }

struct ScoreParams {
  float gamma;
  float cen;      // weight of the inside distance (BOX only)
  int reg_on;     // entity prologue on/off
  float reg_add, reg_lo, reg_hi;
  int norm_on;    // COMPLEX, DISTMULT: unit-length halves / rows (the kernels' REG instantiation stands for it there)
};

inline ScoreParams to_params(const smx_score_params* c) {
  return ScoreParams{c->gamma, c->cen, c->reg_on, c->reg_add, c->reg_lo, c->reg_hi, c->norm_on ? 1 : 0};
}
// the entity-side options a model does not have: nullptr, or what to tell the caller
inline const char* params_refused(int model, const smx_score_params* c);

__device__ __forceinline__ float reg_apply(float e, const ScoreParams& p) {
  if (!p.reg_on) return e;
  const float v = e + p.reg_add;
  return fminf(fmaxf(v, p.reg_lo), p.reg_hi);
}
__device__ __forceinline__ float reg_mask(float e_raw, float g, const ScoreParams& p) {
  if (!p.reg_on) return g;
  const float v = e_raw + p.reg_add;
  return (v >= p.reg_lo && v <= p.reg_hi) ? g : 0.0f;
}

inline const char* params_refused(int model, const smx_score_params* c) {
  if (c->reg_on && model != mBetaKL) return "the entity clamp prologue exists for the beta_kl model only";
  if (c->norm_on && model != mComplex && model != mDistmult)
    return "unit-length rows exist for the complex and distmult models only";
  return nullptr;
}

// per-feature query registers kept by a lane for the whole tile
struct QPair {
  float a, b;
};

template <int M> struct ModelOps;

// Hook applied once to a lane's accumulated query gradient before it leaves the registers
// (identity unless a model defers part of its derivative, as BOX does).
template <int M>
__device__ __forceinline__ void finish_query_grad(const typename ModelOps<M>::Q& q, float& g1, float& g2,
                                                  const ScoreParams& p);

// ---- sign codes -----------------------------------------------------------------------------
// Models whose entity derivative is a choice among a few values (L1: +-c0; box: +-c0, +-c1) can keep
// that choice as two bits per feature -- lower bit "outside" (box only), upper bit "negative" -- one
// byte per float4 column; the features of a column are pushed in ascending order, so the last one
// sits in bits 0-1 and feature x of VEC at position VEC-1-x.
// push2: code = 4 * code + 2 * (lane's bit of hi) + (lane's bit of lo): two v_addc with the masks as
// carry-in.  The s_nop covers the wait states a VALU read of an SGPR needs after a VALU compare
// wrote it (the assembler does not look into inline asm).
__device__ __forceinline__ unsigned push2(unsigned code, unsigned long long hi, unsigned long long lo) {
  unsigned long long carry;
  asm("s_nop 1\n\t"
      "v_addc_co_u32_e64 %0, %1, %0, %0, %2\n\t"
      "v_addc_co_u32_e64 %0, %1, %0, %0, %3"
      : "+v"(code), "=&s"(carry)
      : "s"(hi), "s"(lo));
  return code;
}
// the "negative" bit of position x as a sign-bit mask
__device__ __forceinline__ unsigned code_sign(unsigned code, int x) { return (code << (30 - 2 * x)) & 0x80000000u; }

template <> struct ModelOps<mL1> {
  using Q = QPair;
  static __device__ __forceinline__ Q prep(float q1, float) { return {q1, 0.f}; }
  static __device__ __forceinline__ void fwd(float e1, float, const Q& q, float& a0, float&) {
    a0 += Term<kL1, float>::fwd(e1, 0.f, q.a, 0.f);
  }
  static __device__ __forceinline__ float fold(float a0, float, const ScoreParams&) { return a0; }
  static __device__ __forceinline__ float score(float folded, const ScoreParams& p) { return p.gamma - folded; }
  static __device__ __forceinline__ void coef(float g, float, const ScoreParams&, float& c0, float& c1) {
    c0 = -g;
    c1 = 0.f;
  }
  static __device__ __forceinline__ void bwd_e(float c0, float, float e1, float, const Q& q, float& ge1, float&) {
    float s1 = 0, s2 = 0, s3 = 0;
    Term<kL1, float>::bwd(c0, e1, 0.f, q.a, 0.f, ge1, s1, s2, s3);
  }
  static __device__ __forceinline__ void bwd_q(float c0, float, float e1, float, const Q& q, float& gq1, float&) {
    float s1 = 0, s2 = 0, s3 = 0;
    Term<kL1, float>::bwd(c0, e1, 0.f, q.a, 0.f, s1, s2, gq1, s3);
  }
  // sign codes: the derivative is c0 where e - q > 0 and -c0 elsewhere (sign(0) = -1, dist_kernel.h:141)
  static __device__ __forceinline__ float neg_threshold(const Q&) { return 0.f; }
  static __device__ __forceinline__ void fwd_coded(float e1, const Q& q, float, float& a0, float&, unsigned& code) {
    const float d = e1 - q.a;
    a0 += fabsf(d);
    code = push2(code, __ballot(!(d > 0.f)), 0ull);
  }
  static __device__ __forceinline__ void bwd_q_coded(float c0, float, float e1, const Q& q, float, float& gq1, float&,
                                                     unsigned& code) {
    const float d = e1 - q.a;
    const bool pos = d > 0.f;
    gq1 -= pos ? c0 : -c0;
    code = push2(code, __ballot(!pos), 0ull);
  }
  static __device__ __forceinline__ void bwd_q_from_code(float c0, float, unsigned code, int x, float& gq1, float&) {
    gq1 -= __uint_as_float(__float_as_uint(c0) ^ code_sign(code, x));
  }
  static __device__ __forceinline__ void bwd_e_coded(float c0, float, unsigned code, int x, float& ge) {
    ge += __uint_as_float(__float_as_uint(c0) ^ code_sign(code, x));
  }
};

template <> struct ModelOps<mL2> {
  using Q = QPair;
  static __device__ __forceinline__ Q prep(float q1, float) { return {q1, 0.f}; }
  static __device__ __forceinline__ void fwd(float e1, float, const Q& q, float& a0, float&) {
    a0 += Term<kL2, float>::fwd(e1, 0.f, q.a, 0.f);
  }
  static __device__ __forceinline__ float fold(float a0, float, const ScoreParams&) { return a0; }
  // (the root as the hardware instruction, one ulp: the correctly rounded sqrtf is a third of this model's forward)
  static __device__ __forceinline__ float score(float folded, const ScoreParams& p) {
    return p.gamma - __builtin_amdgcn_sqrtf(folded);
  }
  // d(gamma - sqrt(d2)) / d d2 = -1 / (2 sqrt(d2)): the kernels multiply this upstream part by the
  // pair's own 1 / (2 sqrt(d2)), see l2_pair_coef.  At d2 == 0 the coefficient is infinite, as autograd
  // of torch.sqrt makes it in the reference.
  static __device__ __forceinline__ void coef(float g, float, const ScoreParams&, float& c0, float& c1) {
    c0 = -g;
    c1 = 0.f;
  }
  static __device__ __forceinline__ void bwd_e(float c0, float, float e1, float, const Q& q, float& ge1, float&) {
    float s1 = 0, s2 = 0, s3 = 0;
    Term<kL2, float>::bwd(c0, e1, 0.f, q.a, 0.f, ge1, s1, s2, s3);
  }
  static __device__ __forceinline__ void bwd_q(float c0, float, float e1, float, const Q& q, float& gq1, float&) {
    float s1 = 0, s2 = 0, s3 = 0;
    Term<kL2, float>::bwd(c0, e1, 0.f, q.a, 0.f, s1, s2, gq1, s3);
  }
};

// Query2box: acc0 = outside distance, acc1 = inside distance; one row read serves both.
//
// With d = e - c, a = |d|, the terms of smore/common/torchext/dist_kernel.h:58-105 are
//   out = relu(a - o) = a - min(a, o)      (bit-identical: a - o when a > o, else a - a = 0)
//   in  = |min(a, o)|
// and their derivatives, with "outside" := (a - o >= 0), c0 / c1 the coefficients on out / in:
//   outside:  d/de = s_out c0,  d/dc = -s_out c0,  d/do = -c0 + sgn(o) c1   s_out = (d > 0 ? 1 : -1), sgn(o) = (o > 0 ? 1 : -1)
//   inside :  d/de = s_in  c1,  d/dc = -s_in  c1,  d/do = 0                 s_in  = (d >= 0 ? 1 : -1)
// (inside means a < o, so min(a,o) = a, the outer sign of the reference is -1 exactly when a == 0,
// where its inner sign is -1 too: the product is +1 there and sgn(d) elsewhere, i.e. s_in.)
// The offset gradient of a whole query is therefore (sgn(o) cen - 1) * sum over outside pairs of
// c0, so the loop only accumulates that sum and the factor is applied once at the end.
template <> struct ModelOps<mBox> {
  using Q = QPair;  // a = center, b = offset
  static __device__ __forceinline__ Q prep(float q1, float q2) { return {q1, q2}; }
  // min(|d|, o) as the one hardware instruction (fminf semantics for NaN); the compiler's own fminf
  // re-canonicalises the loop-invariant offset for every row
  static __device__ __forceinline__ float min_abs(float d, float o) {
    float mn;
    asm("v_min_f32_e64 %0, |%1|, %2" : "=v"(mn) : "v"(d), "v"(o));
    return mn;
  }
  static __device__ __forceinline__ void fwd(float e1, float, const Q& q, float& a0, float& a1) {
    const float d = e1 - q.a;
    const float a = fabsf(d);
    const float mn = min_abs(d, q.b);
    a0 += a - mn;
    a1 += fabsf(mn);
  }
  static __device__ __forceinline__ float fold(float a0, float a1, const ScoreParams& p) { return a0 + p.cen * a1; }
  static __device__ __forceinline__ float score(float folded, const ScoreParams& p) { return p.gamma - folded; }
  static __device__ __forceinline__ void coef(float g, float, const ScoreParams& p, float& c0, float& c1) {
    c0 = -g;
    c1 = -p.cen * g;
  }
  // gradient of the entity feature; the center's is its negative:
  //   outside (|d| >= o) ? (d > 0 ? c0 : -c0) : (d >= 0 ? c1 : -c1)
  // The two sign rules differ at d == 0 only, and there "outside" means o <= 0: so the sign is  d > t  with
  // t = 0 where o <= 0 and the largest negative float where o > 0 (d > t is then d >= 0), which is -o clamped
  // to [t_min, 0] -- one v_med3 instead of a second compare and a select.
  static __device__ __forceinline__ float de(float c0, float c1, float e1, const Q& q, bool& outside) {
    const float d = e1 - q.a;
    outside = fabsf(d) >= q.b;
    const float mag = outside ? c0 : c1;
    const float t = __builtin_amdgcn_fmed3f(-q.b, __uint_as_float(0x80000001u), 0.f);
    return d > t ? mag : -mag;
  }
  static __device__ __forceinline__ void bwd_e(float c0, float c1, float e1, float, const Q& q, float& ge1, float&) {
    bool outside;
    ge1 += de(c0, c1, e1, q, outside);
  }
  // gc accumulates the center gradient; go accumulates sum(c0 over outside pairs), see finish_q
  static __device__ __forceinline__ void bwd_q(float c0, float c1, float e1, float, const Q& q, float& gc, float& go) {
    bool outside;
    gc -= de(c0, c1, e1, q, outside);
    go += outside ? c0 : 0.f;
  }
  // The same for a kernel that keeps the query in registers: the sign decision of de() is one compare against
  // the feature's neg_threshold (below), which such a kernel computes once per query instead of two compares
  // and a select per pair.  Same decisions for finite operands, same +-c terms, same bits.
  static __device__ __forceinline__ void bwd_q_thr(float c0, float c1, float e1, const Q& q, float neg_thr, float& gc,
                                                   float& go) {
    const float d = e1 - q.a;
    const bool outside = fabsf(d) >= q.b;
    const float mag = outside ? c0 : c1;
    gc -= d < neg_thr ? -mag : mag;
    go += outside ? c0 : 0.f;
  }
  static __device__ __forceinline__ void finish_q(const Q& q, float&, float& go, const ScoreParams& p) {
    go *= (q.b > 0.f ? p.cen : -p.cen) - 1.0f;
  }

  // ---- sign codes ----
  // The derivative of a pair's distance w.r.t. one entity feature is +-c0 or +-c1: two bits say which.
  // The kernels that make these decisions anyway (forward, or the query-gradient kernel) can leave
  // them behind, one byte per four features; the entity pass then sums  +-c  straight from the codes
  // and needs neither the query rows nor the comparisons -- same decisions, same bits.
  // As bwd_q_thr, and pushes this feature's two bits onto `code`.
  static __device__ __forceinline__ void bwd_q_coded(float c0, float c1, float e1, const Q& q, float neg_thr, float& gc,
                                                     float& go, unsigned& code) {
    const float d = e1 - q.a;
    const bool outside = fabsf(d) >= q.b, neg = d < neg_thr;
    const float mag = outside ? c0 : c1;
    gc -= neg ? -mag : mag;
    go += outside ? c0 : 0.f;
    code = push2(code, __ballot(neg), __ballot(outside));
  }
  // As fwd, and pushes this feature's two bits onto `code`: the forward pass
  // can leave the codes too, and then the whole backward works from them without the entity rows.
  // neg_thr (per query feature, loop-invariant): the "negative" decision  outside ? d <= 0 : d < 0  is
  // d < neg_thr with neg_thr = 0 where the offset is positive (d == 0 is then inside the box) and the
  // smallest positive float where it is not (d == 0 is then outside, and d < that means d <= 0): one
  // compare instead of two compares and three mask operations.
  static __device__ __forceinline__ float neg_threshold(const Q& q) { return q.b > 0.f ? 0.f : __uint_as_float(1u); }
  static __device__ __forceinline__ void fwd_coded(float e1, const Q& q, float neg_thr, float& a0, float& a1,
                                                   unsigned& code) {
    const float d = e1 - q.a;
    const float a = fabsf(d);
    const float mn = min_abs(d, q.b);
    a0 += a - mn;
    a1 += fabsf(mn);
    code = push2(code, __ballot(d < neg_thr), __ballot(a >= q.b));
  }
  // (t ? c0 : c1) with its sign flipped when the feature's "negative" bit is set: two three-input bit
  // operations (v_bitop3_b32; table index = src0 << 2 | src1 << 1 | src2).
  static __device__ __forceinline__ float signed_pick(float c0, float c1, unsigned t, unsigned code, int x) {
    const unsigned w = __builtin_amdgcn_bitop3_b32(t, __float_as_uint(c0), __float_as_uint(c1), 0xCA);  // t ? c0 : c1
    const unsigned top = code << (30 - 2 * x);                                    // "negative" bit in bit 31
    return __uint_as_float(__builtin_amdgcn_bitop3_b32(w, top, 0x80000000u, 0x78));  // w ^ (top & sign bit)
  }
  // Query side from a code byte: gc -= derivative of the feature at position x, go += c0 where the pair is outside.
  static __device__ __forceinline__ void bwd_q_from_code(float c0, float c1, unsigned code, int x, float& gc,
                                                         float& go) {
    const unsigned t = (unsigned)__builtin_amdgcn_sbfe((int)code, 2 * x, 1);  // 0 or ~0
    gc -= signed_pick(c0, c1, t, code, x);
    go += __uint_as_float(__float_as_uint(c0) & t);
  }
  // ge += derivative of the feature at position x of the lane's code byte
  static __device__ __forceinline__ void bwd_e_coded(float c0, float c1, unsigned code, int x, float& ge) {
    const unsigned t = (unsigned)__builtin_amdgcn_sbfe((int)code, 2 * x, 1);  // 0 or ~0
    ge += signed_pick(c0, c1, t, code, x);
  }
};

template <> struct ModelOps<mRotate> {
  using Q = QPair;  // a = re, b = im
  static __device__ __forceinline__ Q prep(float q1, float q2) { return {q1, q2}; }
  static __device__ __forceinline__ void fwd(float e1, float e2, const Q& q, float& a0, float&) {
    a0 += Term<kRotate, float>::fwd(e1, e2, q.a, q.b);
  }
  static __device__ __forceinline__ float fold(float a0, float, const ScoreParams&) { return a0; }
  static __device__ __forceinline__ float score(float folded, const ScoreParams& p) { return p.gamma - folded; }
  static __device__ __forceinline__ void coef(float g, float, const ScoreParams&, float& c0, float& c1) {
    c0 = -g;
    c1 = 0.f;
  }
  static __device__ __forceinline__ void bwd_e(float c0, float, float e1, float e2, const Q& q, float& ge1, float& ge2) {
    float s1 = 0, s2 = 0;
    Term<kRotate, float>::bwd(c0, e1, e2, q.a, q.b, ge1, ge2, s1, s2);
  }
  static __device__ __forceinline__ void bwd_q(float c0, float, float e1, float e2, const Q& q, float& g1, float& g2) {
    float s1 = 0, s2 = 0;
    Term<kRotate, float>::bwd(c0, e1, e2, q.a, q.b, s1, s2, g1, g2);
  }
};

// BetaE: KL(Beta(ea,eb) || Beta(qa,qb)) of smore/common/torchext/dist_kernel.h:207-266, regrouped into an
// entity part and a query part so that everything that depends on one side only is evaluated once:
//   KL = [lgG(qa)+lgG(qb)-lgG(sq)] + [lgG(se)-lgG(ea)-lgG(eb)] + (ea-qa)psi(ea) + (eb-qb)psi(eb) + (sq-se)psi(se)
//   dKL/dqa = [psi(qa) - psi(sq)] - psi(ea) + psi(se)                       (same with b)
//   dKL/dea = (ea-qa) psi'(ea) + (sq-se) psi'(se)                            (same with b)
// The bracketed query terms are per (query, feature) constants held in the lane's query registers.
// For the entity gradient the trigammas depend on the entity only, and (ea-qa) + (eb-qb) = se - sq,
// so a segment accumulates S1 = sum c (ea-qa), S2 = sum c (eb-qb) and applies
//   g_a = psi'(ea) S1 - psi'(se) (S1+S2),  g_b = psi'(eb) S2 - psi'(se) (S1+S2)
// once when the segment is finished.
struct QBeta {
  float a, b;  // alpha, beta of the query
  float k;     // forward: lgG(qa)+lgG(qb)-lgG(sq)+ln C, see beta_logs; query backward: psi(qa)-psi(sq)
  float l;     // forward: (qa + 2.5) ln 2, see beta_arg; query backward: psi(qb)-psi(sq)
  float m;     // forward: (qb + 2.5) ln 2
};

// One feature of a row in the interval of fast_ok (see beta_arg).  D'(x)/D(x) meets x - q on its own, after all that is smaller: near
// its pole R(x) is a number of two digits before the point, and the features that a regularizer has clamped are all off by
// the same rounding of it (at 0.05 by 1.2e-6 out of 21.6, D'/D alone by 1.5e-8; normal rows around 1, one feature in 35 clamped:
// error of a score 4.7e-5 -> 3.2e-5 rms for two instructions more, 4.6e-5 with the six-step forms).
static __device__ __forceinline__ float beta_pair_fast(float ea, float eb, const QBeta& q) {
#pragma clang fp contract(off)
  const BetaArg a = beta_arg<false>(ea), b = beta_arg<false>(eb), s = beta_arg<false>(ea + eb);
  float v = q.k + beta_logs(a, b, s, q.l, q.m);
  const float da = ea - q.a, db = eb - q.b;
  v = __builtin_fmaf(-da, a.u, v);
  v = __builtin_fmaf(-db, b.u, v);
  v = __builtin_fmaf(da + db, s.rest, v);
  v = __builtin_fmaf(-da, a.quot, v);
  return __builtin_fmaf(-db, b.quot, v);
}
// ... of any row, the same bits where the feature is in the interval: which form a feature takes is the feature's own affair, as
// it is the query's in prep_fwd.  Not inlined: rows that need it are rare.  (The query's coefficients are formed again: as two
// arguments more they cost the rows of seven floats a lane 17 spilled registers, 584 us instead of 280 for 2 x 400 floats.)
static __device__ __noinline__ float beta_pair_any(float ea, float eb, float qa, float qb, float k) {
  if (fast_ok(fminf(ea, eb), ea + eb)) return beta_pair_fast(ea, eb, {qa, qb, k, beta_k(qa), beta_k(qb)});
  float lb, pa, pb, ps;
  beta_terms_slow(ea, eb, lb, pa, pb, ps);
  return (k + (lb - kLnBetaConst)) + (ea - qa) * pa + (eb - qb) * pb + ((qa + qb) - (ea + eb)) * ps;
}

template <> struct ModelOps<mBetaKL> {
  using Q = QBeta;
  static __device__ __forceinline__ Q prep(float q1, float q2) { return {q1, q2, 0.f, 0.f, 0.f}; }
  static __device__ __forceinline__ Q prep_fwd(float q1, float q2) {
    const float ka = beta_k(q1), kb = beta_k(q2), sum = q1 + q2;
    float lb, pa, pb, ps;
    if (fast_ok(fminf(q1, q2), sum)) lb = beta_logs(beta_arg<false>(q1), beta_arg<false>(q2), beta_arg<false>(sum), ka, kb);
    else {
      beta_terms_slow(q1, q2, lb, pa, pb, ps);
      lb -= kLnBetaConst;
    }
    return {q1, q2, -lb, ka, kb};
  }
  static __device__ __forceinline__ Q prep_bwd_q(float q1, float q2) {
    const SlowTerms t = beta_psi_diffs(q1, q2);
    return {q1, q2, t.x, t.y, 0.f};
  }
  static __device__ __forceinline__ void bwd_q_fast(float c0, float e1, float e2, const Q& q, float& g1, float& g2) {
#pragma clang fp contract(off)
    const BetaArg a = beta_arg<true>(e1), b = beta_arg<true>(e2), s = beta_arg<true>(e1 + e2);
    g1 = __builtin_fmaf(c0, q.k + beta_psi_diff(a, s), g1);
    g2 = __builtin_fmaf(c0, q.l + beta_psi_diff(b, s), g2);
  }
  static __device__ __forceinline__ float fold(float a0, float, const ScoreParams&) { return a0; }
  static __device__ __forceinline__ float score(float folded, const ScoreParams& p) { return p.gamma - folded; }
  static __device__ __forceinline__ void coef(float g, float, const ScoreParams&, float& c0, float& c1) {
    c0 = -g;
    c1 = 0.f;
  }
  // accumulates S1, S2 (see above); finish_e turns them into the gradient
  static __device__ __forceinline__ void bwd_e(float c0, float, float e1, float e2, const Q& q, float& s1, float& s2) {
    s1 += c0 * (e1 - q.a);
    s2 += c0 * (e2 - q.b);
  }
  static __device__ __forceinline__ void finish_e(float e1, float e2, float& g1, float& g2) {
#pragma clang fp contract(off)
    const float sum = e1 + e2;
    float ta, tb, ts;
    if (fast_ok(fminf(e1, e2), sum)) {
      ta = beta_trigamma(beta_arg<true>(e1));
      tb = beta_trigamma(beta_arg<true>(e2));
      ts = beta_trigamma(beta_arg<true>(sum));
    } else {
      const SlowTerms t = beta_trigammas_any(e1, e2);
      ta = t.x;
      tb = t.y;
      ts = t.z;
    }
    const float common = ts * (g1 + g2);
    g1 = __builtin_fmaf(ta, g1, -common);
    g2 = __builtin_fmaf(tb, g2, -common);
  }
  static __device__ __forceinline__ void bwd_q(float c0, float, float e1, float e2, const Q& q, float& g1, float& g2) {
    const SlowTerms t = beta_psi_diffs_any(e1, e2);
    g1 = __builtin_fmaf(c0, q.k - t.x, g1);
    g2 = __builtin_fmaf(c0, q.l - t.y, g2);
  }
};

// BetaE's entity prologue in the kernels built for it: one v_med3 (a NaN gives the lower bound, as fminf(fmaxf()) does).
struct BetaClamp {
  float add, lo, hi;
  bool low_ok;   // the lower bound already is in the interval of fast_ok
  __device__ __forceinline__ BetaClamp(const ScoreParams& p) : add(p.reg_add), lo(fminf(p.reg_lo, p.reg_hi)), hi(p.reg_hi) {
    low_ok = lo >= kFastLo;
  }
  __device__ __forceinline__ float operator()(float e) const { return __builtin_amdgcn_fmed3f(e + add, lo, hi); }
};

// The features of one row, clamped, and whether all of them, in all lanes, lie in the interval of fast_ok: one decision per
// row instead of two compares, an exec mask and a branch per feature.  The largest sum of a pair bounds both, as none is
// negative.  (A sum over all of a lane's features, which was here first, sent rows of 512 floats a half with a mean of 63 to the
// general path, and rows of 2,048 with one of 16.)
template <int VEC, int NIT> struct BetaRow {
  float a[NIT][VEC], b[NIT][VEC];
  template <bool REG, class GetA, class GetB>
  __device__ __forceinline__ bool load(const BetaClamp& clamp, GetA&& ga, GetB&& gb) {
    float high = 0.f;   // (a NaN changes neither bound: the fast forms of one are NaN, as the general ones)
#pragma unroll
    for (int it = 0; it < NIT; ++it)
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        a[it][v] = REG ? clamp(ga(it, v)) : ga(it, v);
        b[it][v] = REG ? clamp(gb(it, v)) : gb(it, v);
        high = fmaxf(high, a[it][v] + b[it][v]);
      }
    bool ok = high <= kFastHi;
    if (!(REG && clamp.low_ok)) {
      float low = __builtin_inff();
#pragma unroll
      for (int it = 0; it < NIT; ++it)
#pragma unroll
        for (int v = 0; v < VEC; ++v) low = fminf(low, fminf(a[it][v], b[it][v]));
      ok = ok && low >= kFastLo;
    }
    return __ballot(!ok) == 0ull;
  }
};

// A lane's part of a row's divergence, and the row's part of the query gradient, from the row's values as they are stored.
// get_q(it, q) fetches the query's values of a column group: the kernels that stream rows keep them in LDS, evaluated once per
// workgroup, which leaves their registers to four wavefronts a SIMD (measured below with beta_arg).
template <int VEC, int NIT, bool REG, class GetA, class GetB, class GetQ>
__device__ __forceinline__ float beta_row_sum(const BetaClamp& clamp, GetA&& ga, GetB&& gb, GetQ&& get_q, int ncol, int lane) {
  BetaRow<VEC, NIT> row;
  const bool fast = row.template load<REG>(clamp, ga, gb);
  float mine = 0.f;
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    QBeta q[VEC];
    get_q(it, q);
    float a0;
    if (fast) {
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        const float x = beta_pair_fast(row.a[it][v], row.b[it][v], q[v]);
        a0 = v == 0 ? x : a0 + x;
      }
    } else {
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        const float x = beta_pair_any(row.a[it][v], row.b[it][v], q[v].a, q[v].b, q[v].k);
        a0 = v == 0 ? x : a0 + x;
      }
    }
    mine += lane + 64 * it < ncol ? a0 : 0.f;
  }
  return mine;
}
template <int VEC, int NIT, bool REG, class GetA, class GetB, class GetQ>
__device__ __forceinline__ void beta_row_query_grad(const BetaClamp& clamp, GetA&& ga, GetB&& gb, float c0, GetQ&& get_q,
                                                    float (&g1)[NIT][VEC], float (&g2)[NIT][VEC]) {
  BetaRow<VEC, NIT> row;
  const bool fast = row.template load<REG>(clamp, ga, gb);
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    QBeta q[VEC];
    get_q(it, q);
    if (fast) {
#pragma unroll
      for (int v = 0; v < VEC; ++v) ModelOps<mBetaKL>::bwd_q_fast(c0, row.a[it][v], row.b[it][v], q[v], g1[it][v], g2[it][v]);
    } else {
#pragma unroll
      for (int v = 0; v < VEC; ++v) ModelOps<mBetaKL>::bwd_q(c0, 0.f, row.a[it][v], row.b[it][v], q[v], g1[it][v], g2[it][v]);
    }
  }
}

// ... and, for the row of a one-pair segment, its gradient with respect to the stored values as well (g = c0 (e - q) through
// the trigammas and the clamp's mask): psi and psi' share every special function.
template <int VEC, int NIT, bool REG, class GetA, class GetB, class GetQ>
__device__ __forceinline__ void beta_row_both_grads(const BetaClamp& clamp, const ScoreParams& p, GetA&& ga, GetB&& gb, float c0,
                                                    GetQ&& get_q, float (&g1)[NIT][VEC], float (&g2)[NIT][VEC],
                                                    float (&ge1)[NIT][VEC], float (&ge2)[NIT][VEC]) {
#pragma clang fp contract(off)
  using O = ModelOps<mBetaKL>;
  BetaRow<VEC, NIT> row;
  const bool fast = row.template load<REG>(clamp, ga, gb);
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    QBeta q[VEC];
    get_q(it, q);
    if (fast) {
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        const float ea = row.a[it][v], eb = row.b[it][v];
        const BetaArg a = beta_arg<true>(ea), b = beta_arg<true>(eb), s = beta_arg<true>(ea + eb);
        g1[it][v] = __builtin_fmaf(c0, q[v].k + beta_psi_diff(a, s), g1[it][v]);
        g2[it][v] = __builtin_fmaf(c0, q[v].l + beta_psi_diff(b, s), g2[it][v]);
        const float s1 = c0 * (ea - q[v].a), s2 = c0 * (eb - q[v].b), common = beta_trigamma(s) * (s1 + s2);
        ge1[it][v] = __builtin_fmaf(beta_trigamma(a), s1, -common);
        ge2[it][v] = __builtin_fmaf(beta_trigamma(b), s2, -common);
      }
    } else {
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        const float ea = row.a[it][v], eb = row.b[it][v];
        O::bwd_q(c0, 0.f, ea, eb, q[v], g1[it][v], g2[it][v]);
        const SlowTerms t = beta_trigammas_any(ea, eb);
        const float s1 = c0 * (ea - q[v].a), s2 = c0 * (eb - q[v].b), common = t.z * (s1 + s2);
        ge1[it][v] = __builtin_fmaf(t.x, s1, -common);
        ge2[it][v] = __builtin_fmaf(t.y, s2, -common);
      }
    }
    if (REG) {
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        ge1[it][v] = reg_mask(ga(it, v), ge1[it][v], p);
        ge2[it][v] = reg_mask(gb(it, v), ge2[it][v], p);
      }
    }
  }
}

// ComplEx and DistMult score by similarity, not distance (dist_kernel.h:187-204, 324-349): the logit grows
// with the inner product, so the upstream coefficient keeps its sign.
template <> struct ModelOps<mComplex> {
  using Q = QPair;  // a = re, b = im
  static __device__ __forceinline__ Q prep(float q1, float q2) { return {q1, q2}; }
  static __device__ __forceinline__ void fwd(float e1, float e2, const Q& q, float& a0, float&) {
    a0 += Term<kComplex, float>::fwd(e1, e2, q.a, q.b);
  }
  static __device__ __forceinline__ float fold(float a0, float, const ScoreParams&) { return a0; }
  static __device__ __forceinline__ float score(float folded, const ScoreParams& p) { return p.gamma + folded; }
  static __device__ __forceinline__ void coef(float g, float, const ScoreParams&, float& c0, float& c1) {
    c0 = g;
    c1 = 0.f;
  }
  static __device__ __forceinline__ void bwd_e(float c0, float, float e1, float e2, const Q& q, float& ge1, float& ge2) {
    float s1 = 0, s2 = 0;
    Term<kComplex, float>::bwd(c0, e1, e2, q.a, q.b, ge1, ge2, s1, s2);
  }
  static __device__ __forceinline__ void bwd_q(float c0, float, float e1, float e2, const Q& q, float& g1, float& g2) {
    float s1 = 0, s2 = 0;
    Term<kComplex, float>::bwd(c0, e1, e2, q.a, q.b, s1, s2, g1, g2);
  }
};

// ComplEx with unit-length halves (complex.py:142-146 when the model's mode names 'norm', complex.py:87-89;
// embed_norm = F.normalize(p = 2, dim = -1), modules.py:38-40):
//   logit = gamma + (re . q_re) / max(|re|, eps) + (im . q_im) / max(|im|, eps),   eps = 1e-12
//   d logit / d q_re = re / max(|re|, eps)
//   d logit / d re   = (q_re - re_n (re_n . q_re)) / |re|   with re_n = re / |re|    (q_re / eps below eps)
// The scaling belongs to the entity, not to the pair: summed over an entity's pairs the gradient is the plain ComplEx
// gradient G = sum c q pushed through the scaling once, g_re = (G_re - re_n (re_n . G_re)) / |re|.  The entity
// kernels therefore accumulate G as they do for plain ComplEx, and the function that finishes a row applies the
// projection.  In the kernels the REG instantiation of the ComplEx model stands for this form.
// DistMult's 'norm' mode (distmult.py:85-87,129-130) is the same with the whole row as its only half:
//   logit = gamma + (e . q) / max(|e|, eps).
constexpr float kNormEps = 1e-12f;
__host__ __device__ constexpr bool model_norm(int m, bool reg) { return (m == mComplex || m == mDistmult) && reg; }
__device__ __forceinline__ float inv_norm(float sumsq) { return 1.f / fmaxf(__builtin_sqrtf(sumsq), kNormEps); }

template <> struct ModelOps<mDistmult> {
  using Q = QPair;
  static __device__ __forceinline__ Q prep(float q1, float) { return {q1, 0.f}; }
  static __device__ __forceinline__ void fwd(float e1, float, const Q& q, float& a0, float&) {
    a0 += Term<kDistmult, float>::fwd(e1, 0.f, q.a, 0.f);
  }
  static __device__ __forceinline__ float fold(float a0, float, const ScoreParams&) { return a0; }
  static __device__ __forceinline__ float score(float folded, const ScoreParams& p) { return p.gamma + folded; }
  static __device__ __forceinline__ void coef(float g, float, const ScoreParams&, float& c0, float& c1) {
    c0 = g;
    c1 = 0.f;
  }
  static __device__ __forceinline__ void bwd_e(float c0, float, float e1, float, const Q& q, float& ge1, float&) {
    float s1 = 0, s2 = 0, s3 = 0;
    Term<kDistmult, float>::bwd(c0, e1, 0.f, q.a, 0.f, ge1, s1, s2, s3);
  }
  static __device__ __forceinline__ void bwd_q(float c0, float, float e1, float, const Q& q, float& gq1, float&) {
    float s1 = 0, s2 = 0, s3 = 0;
    Term<kDistmult, float>::bwd(c0, e1, 0.f, q.a, 0.f, s1, s2, gq1, s3);
  }
};

// Query registers for the forward / the query-backward kernel (models without side constants use prep).
template <int M>
__device__ __forceinline__ typename ModelOps<M>::Q prep_forward(float q1, float q2) {
  if constexpr (M == mBetaKL) return ModelOps<M>::prep_fwd(q1, q2);
  else return ModelOps<M>::prep(q1, q2);
}
template <int M>
__device__ __forceinline__ typename ModelOps<M>::Q prep_backward_query(float q1, float q2) {
  if constexpr (M == mBetaKL) return ModelOps<M>::prep_bwd_q(q1, q2);
  else return ModelOps<M>::prep(q1, q2);
}

// Hook applied once per finished entity row to the summed accumulators (identity unless a model
// defers part of its derivative, as BETA_KL does).  e1 / e2 are the (regularised) entity values.
template <int M>
__device__ __forceinline__ void finish_entity_grad(float e1, float e2, float& g1, float& g2) {
  if constexpr (M == mBetaKL) ModelOps<mBetaKL>::finish_e(e1, e2, g1, g2);
}

template <int M>
__device__ __forceinline__ void finish_query_grad(const typename ModelOps<M>::Q& q, float& g1, float& g2,
                                                  const ScoreParams& p) {
  if constexpr (M == mBox) ModelOps<mBox>::finish_q(q, g1, g2, p);
}

}  // namespace smx
