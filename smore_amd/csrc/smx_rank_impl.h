// Evaluation against all entities: filtered ranks of a query's answers without materialising or
// sorting the [1,N] logit row.
//
// Replaces, for the test_all case of smore/training/train_process.py:112-160,
//   negative_logit = model(None, all_entity_idx, ...)      score of every entity (kg_reasoning.py:349-355)
//   argsort(descending) -> ranking -> ranking[answers] -> sort -> minus arange -> +1   (filtered setting)
// The filtered rank of an answer is 1 + the number of NON-answer entities ranked before it.  So the
// table is streamed once for up to sixteen queries: every lane scores whole rows of its own (rank_scan_kernel), and a
// row that reaches the lowest of a query's answers finds its place among them by a binary search and is counted in
// that place's bin (integer atomics: exact, order-free).  A prefix sum over the bins gives every answer its count.
// Order of equal scores: the lower entity id ranks first (one of the orders an unstable argsort may produce).
// "Beats" is one unsigned compare of (sortable(score) << 32 | ~id) keys; an answer is recognised in the stream by its id.
// The answers' keys come from the same arithmetic, operation by operation, so that equal rows tie.
#pragma once
#include "smx_common.h"
#include "smx_models.h"
#include "smx_wave.h"

#include <type_traits>

namespace smx {

constexpr int kRankQueries = 4;  // query rows a wavefront of the scan keeps sums for; most branches of a union query

struct RankArgs {
  const float* table;
  const float* q1;
  const float* q2;
  int B;
  int U;                // union queries: q1 / q2 hold U branch rows per query, a logit is the maximum over them
                        // (the last line of every custom_cal_logit, smore/models/box.py:163); 1 otherwise
  int ncol, dim;
  unsigned long long n_rows;
  ScoreParams p;
  // answers, per query A slots (the first ans_count[b] are valid), sorted by key descending for the scan
  const long long* ans_id;           // [B, A]
  const unsigned long long* ans_key; // [B, A]   (scan)
  unsigned long long* key_out;       // [B, A]   (answer-key kernel)
  float* score_out;                  // [B, A]   (answer-key kernel)
  const int* ans_count;              // [B]
  int A;
  unsigned* bins;                    // [B, A + 1]
  int lds_bins;                      // the scan counts in LDS first (the bins of its queries fit)
  int lds_keys;                      // and keeps their keys there
  unsigned groups;                   // the scan's groups of kScanRows rows
  int first_list;                    // query of the launch's first list of answers
  long long* rank_out;               // [B, A]
  const int* slot;                   // [B, A] slot of the j-th key in the order the answers were given in, or null
  // ranking among sampled candidates (cand_score_kernel, cand_rank_kernel)
  const long long* cand;             // [B, C], -1 = padding
  int C, H;
  const int* n_hard;                 // [B]: the first n_hard[b] candidates of query b are its hard answers
  float* cand_logit;                 // [B, C] or null
  long long* cand_rank;              // [B, C]
  long long* hard_rank;              // [B, H]
  int* err;
};

enum RankMode : int { kRankScan = 0, kRankKeys = 1, kRankCandidates = 2 };

__device__ __forceinline__ unsigned sortable_bits(float s) {
  const unsigned u = __float_as_uint(s);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);  // ascending in the float order (-0 < +0)
}
__device__ __forceinline__ unsigned long long rank_key(float score, unsigned long long id) {
  return ((unsigned long long)sortable_bits(score) << 32) | (unsigned)(~(unsigned)id);
}

// Whether branch logit s replaces the best so far: torch.max over the branch axis (a NaN wins, the first of equals stays).
__device__ __forceinline__ bool union_takes(float s, float best) { return s > best || (s != s && best == best); }

// Score of one row against one staged query; the value is valid in lane 63.
template <int M, int VEC, int NIT, bool REG>
__device__ __forceinline__ float row_score(const float (&e1)[NIT][VEC], const float (&e2)[NIT][VEC],
                                           const typename ModelOps<M>::Q (&q)[NIT][VEC], int ncol, int lane,
                                           const ScoreParams& p) {
  constexpr int MUL = model_mul(M);
  float mine = 0.f;
  if constexpr (M == mBetaKL) {
    mine = beta_row_sum<VEC, NIT, REG>(BetaClamp(p), [&](int it, int v) { return e1[it][v]; },
                                       [&](int it, int v) { return e2[it][v]; },
                                       [&](int it, QBeta (&to)[VEC]) {
#pragma unroll
                                         for (int v = 0; v < VEC; ++v) to[v] = q[it][v];
                                       }, ncol, lane);
  } else
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    float a0 = 0.f, a1 = 0.f;
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      const float x1 = REG ? reg_apply(e1[it][v], p) : e1[it][v];
      const float x2 = MUL == 2 ? (REG ? reg_apply(e2[it][v], p) : e2[it][v]) : 0.f;
      ModelOps<M>::fwd(x1, x2, q[it][v], a0, a1);
    }
    const float f = ModelOps<M>::fold(a0, a1, p);
    mine += lane + 64 * it < ncol ? f : 0.f;
  }
  return ModelOps<M>::score(wave_sum_last_f32(mine), p);
}

// ComplEx with unit-length halves (REG stands for it there): the row's halves scaled in the lanes' registers, once
// per row however many queries score it.
template <int M, int VEC, int NIT, bool REG>
__device__ __forceinline__ void unit_row(float (&e1)[NIT][VEC], float (&e2)[NIT][VEC], int ncol, int lane) {
  if constexpr (model_norm(M, REG)) {
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      float a = 0.f, b = 0.f;
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        a = __builtin_fmaf(e1[it][v], e1[it][v], a);
        if constexpr (model_mul(M) == 2) b = __builtin_fmaf(e2[it][v], e2[it][v], b);
      }
      const bool in = lane + 64 * it < ncol;
      s1 += in ? a : 0.f;
      s2 += in ? b : 0.f;
    }
    const float i1 = inv_norm(wave_sum_f32(s1));
    const float i2 = model_mul(M) == 2 ? inv_norm(wave_sum_f32(s2)) : 0.f;
#pragma unroll
    for (int it = 0; it < NIT; ++it)
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        e1[it][v] *= i1;
        if constexpr (model_mul(M) == 2) e2[it][v] *= i2;
      }
  }
}

// STREAM: the row is read once (non-temporal)
template <int VEC, int NIT, int MUL, bool STREAM = false>
__device__ __forceinline__ void load_entity(const float* __restrict__ row, int dim, int ncol, int lane,
                                            float (&e1)[NIT][VEC], float (&e2)[NIT][VEC]) {
  typedef float vec4f __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int c = min(lane + 64 * it, ncol - 1);
    if constexpr (VEC == 4) {
      const vec4f* pa = reinterpret_cast<const vec4f*>(row) + c;
      const vec4f a = STREAM ? __builtin_nontemporal_load(pa) : *pa;
      e1[it][0] = a.x; e1[it][1] = a.y; e1[it][2] = a.z; e1[it][3] = a.w;
      if (MUL == 2) {
        const vec4f* pb = reinterpret_cast<const vec4f*>(row + dim) + c;
        const vec4f b = STREAM ? __builtin_nontemporal_load(pb) : *pb;
        e2[it][0] = b.x; e2[it][1] = b.y; e2[it][2] = b.z; e2[it][3] = b.w;
      }
    } else {
      e1[it][0] = STREAM ? __builtin_nontemporal_load(row + c) : row[c];
      if (MUL == 2) e2[it][0] = STREAM ? __builtin_nontemporal_load(row + dim + c) : row[dim + c];
    }
  }
}

template <int M, int VEC, int NIT>
__device__ __forceinline__ void load_rank_query(const float* __restrict__ q1, const float* __restrict__ q2, int b,
                                                int dim, int ncol, int lane,
                                                typename ModelOps<M>::Q (&q)[NIT][VEC]) {
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int c = min(lane + 64 * it, ncol - 1);
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      const float a = q1[(size_t)b * dim + c * VEC + v];
      const float bb = model_nq(M) == 2 ? q2[(size_t)b * dim + c * VEC + v] : 0.f;
      q[it][v] = prep_forward<M>(a, bb);
    }
  }
}

// ---- the scan over all entities ----------------------------------------------------------------
// A workgroup (four wavefronts) holds kScanRows rows of the table at a time, 32 floats of each per step, in LDS; a lane
// owns two of the rows and sums their scores feature by feature, a wavefront does so for NB query rows of its own whose
// values are scalars.  Every lane then works on every feature (a row spread over the lanes leaves 22 % of them without
// a column at 400 floats), nothing is summed across lanes, and the table crosses the fabric once per sixteen queries.
// What bounds it: instruction issue.  Box, per (row, query, feature): subtract, minimum, subtract, multiply-add, add.  An
// addition or multiply-add issues at up to twice the rate of a minimum, and of any instruction with a scalar operand, so
// cen sits in a VGPR: 1 M x 400 rows, 16 queries 0.69 -> 0.65 ms for 32 G operations (a row per wavefront, a pass per four
// queries: 1.57 ms).  (The subtracted query values out of LDS as well, a broadcast read per four features and query row:
// no faster, and RotatE 2 to 5 % slower, LDS then being what bounds it.)
// (Four operations would do: out + cen * in over cen is max(|d|, |d| / cen - o (1 - cen) / cen) for 0 < cen <= 1, 0.65 ms.
// But that rounds values up to 1 / cen times larger than the result: 84 times the error where distances are near the
// offsets, D = 400, cen = 0.02, twice the error elsewhere.)
// The sums of a step (32 features, 16 of two-halves models, 8 of BetaE) are added to the row's total with the rounding
// error carried along, and within a step four features at a time are summed, two such blocks added, and up to four of
// these pairs one after another: no longer a chain than the tree over lanes of the scoring kernels.  (32 features in one
// chain: 1.2 to 2.3 times its error at 33 to 100 floats.)
constexpr int kScanRows = 128;
constexpr int kScanStride = 36;    // floats between two rows' stretches in LDS: 16-byte reads of 8 rows hit 32 banks
constexpr int kScanThreads = 256;

typedef const __attribute__((address_space(4))) float* ScalarRow;  // uniform index: scalar loads
__device__ __forceinline__ ScalarRow scalar_row(const float* p) {
  return reinterpret_cast<ScalarRow>(reinterpret_cast<unsigned long long>(p));
}

// Per-feature arithmetic of the scan and of the answers' keys: every multiply-add is written out and contraction is
// off, so both kernels round alike.
//   kGroup  groups of values a feature has in LDS: 1 (e), 2 (first, second half), 4 (BetaE: ea, eb, psi(ea) - psi(se),
//           psi(eb) - psi(se), evaluated once per row for all queries)
//   kSums   sums per (row, query);  kRowSums  sums per row
// BetaE's log-Beta terms depend on the row or on the query alone; a divergence is what is left when they and the sum over
// psi cancel, digits that its fp32 sums would round away.  They are summed, and the three parts added, in 64 bits: once
// per row, once per query, three additions per pair.  log_beta: with what the rounding of ea + eb changes in lgamma(ea + eb)
// (the pair's sum is over ea and eb themselves, not over that rounded value).
// da, db: psi(a) - psi(a + b), psi(b) - psi(a + b).  The forms are those of the scoring kernels (beta_arg), with the poles of psi(a) and
// psi(b) on their own: at 1/31 to 1/17 these are off by 0.85 of an ulp rms, without by 1.16, in the six-step form by 1.07.  (4 queries
// among 400,000 rows of 2 x 400 floats: 717, 697 and 730 us.)  The logarithms of ratios, which are psi's as well, meet the row's own
// a + 2.5 and b + 2.5 in 64 bits.
__device__ __forceinline__ double log_beta(float a, float b, float& da, float& db) {
#pragma clang fp contract(off)
  const float sum = a + b, from_b = sum - a;
  const float rest = (a - (sum - from_b)) + (b - from_b);   // a + b = sum + rest
  if (fast_ok(fminf(a, b), sum)) {
    const BetaArg xa = beta_arg<true>(a), xb = beta_arg<true>(b), xs = beta_arg<false>(sum);   // (D(x) is x d for the first two)
    const float ga = __builtin_amdgcn_logf(xs.w * xa.r), gb = __builtin_amdgcn_logf(xs.w * xb.r);
    const float gs = __builtin_amdgcn_logf(xs.w);
    const float gd = __builtin_amdgcn_logf(((xa.d * kBetaConst) * xs.rd * xb.d) * (a * b));
    da = -__builtin_fmaf(ga, kLn2, xa.rest - xs.rest);
    db = -__builtin_fmaf(gb, kLn2, xb.rest - xs.rest);
    const float tail = __builtin_fmaf(-xb.r, beta_stirling(xb), __builtin_fmaf(-xa.r, beta_stirling(xa), xs.r * beta_stirling(xs)));
    const double logs = ((double)a + 2.5) * (double)ga + ((double)b + 2.5) * (double)gb + ((double)gd - 2.5 * (double)gs);
    return __builtin_fma(logs, 0.69314718055994531, (double)(tail + rest * (1.f - xs.rest)));
  }
  float lb, pa, pb, ps;
  beta_terms(a, b, lb, pa, pb, ps);
  da = pa - ps;
  db = pb - ps;
  return (double)lb + (double)(rest * ps);
}
// The sum with its error.  Past fp32 the error is a difference of infinities: the total alone then is what a plain sum
// would be (a diverged row scores -inf and ranks last, it does not turn into a NaN above every logit).
__device__ __forceinline__ float with_error(float total, float err) {
#pragma clang fp contract(off)
  return __builtin_isfinite(total) ? total + err : total;
}

template <int M, bool NORM> struct ScanOps {
  static constexpr int kGroup = M == mBetaKL ? 4 : model_mul(M);
  static constexpr int kFeat = 32 / kGroup;   // features per step
  static constexpr int kSums = NORM ? model_mul(M) : 1;
  static constexpr int kRowSums = NORM ? model_mul(M) : 0;
  static constexpr int kKeyStride = kFeat == 8 ? 8 : kFeat + 4;   // floats between two steps of a row in the answers' kernel

  // Sum over N (4 or 1) features; terms that are not products are added as a tree.  SCALAR: a and b are wavefront-uniform.
  template <int N, bool SCALAR>
  static __device__ __forceinline__ void block(const float (&e)[N][kGroup], const float (&a)[N], const float (&b)[N], float cen,
                                               float (&s)[kSums]) {
#pragma clang fp contract(off)
    if constexpr (M == mL1 || M == mBox || M == mRotate) {
      float t[N];
#pragma unroll
      for (int v = 0; v < N; ++v) {
        const float d = e[v][0] - a[v];
        if constexpr (M == mL1) {
          t[v] = fabsf(d);
        } else if constexpr (M == mBox) {
          float mn;
          if constexpr (SCALAR) asm("v_min_f32_e64 %0, |%1|, %2" : "=v"(mn) : "v"(d), "s"(b[v]));   // (no move of the offset)
          else mn = ModelOps<mBox>::min_abs(d, b[v]);
          t[v] = __builtin_fmaf(fabsf(mn), cen, fabsf(d) - mn);
        } else {
          const float y = e[v][1] - b[v];
          t[v] = __builtin_amdgcn_sqrtf(__builtin_fmaf(y, y, __builtin_fmaf(d, d, 1e-20f)));
        }
      }
      s[0] = N == 4 ? (t[0] + t[1]) + (t[N - 2] + t[N - 1]) : t[0];
    } else {
#pragma unroll
      for (int v = 0; v < N; ++v) {
        auto add = [&](int i, bool first, float x, float y) { s[i] = first ? x * y : __builtin_fmaf(x, y, s[i]); };
        if constexpr (M == mL2) {
          const float d = e[v][0] - a[v];
          add(0, v == 0, d, d);
        } else if constexpr (M == mBetaKL) {
          add(0, v == 0, e[v][0] - a[v], e[v][2]);
          add(0, false, e[v][1] - b[v], e[v][3]);
        } else {
          add(0, v == 0, e[v][0], a[v]);
          if constexpr (M == mComplex) add(kSums - 1, kSums == 2 && v == 0, e[v][1], b[v]);
        }
      }
    }
  }
  template <int N>
  static __device__ __forceinline__ void block_row(const float (&e)[N][kGroup], float (&s)[kRowSums > 0 ? kRowSums : 1]) {
#pragma clang fp contract(off)
    if constexpr (NORM) {
#pragma unroll
      for (int i = 0; i < kRowSums; ++i)
#pragma unroll
        for (int v = 0; v < N; ++v) s[i] = v == 0 ? e[v][i] * e[v][i] : __builtin_fmaf(e[v][i], e[v][i], s[i]);
    } else {
      s[0] = 0.f;
    }
  }
  // Product of a query with a half row of squared length r scaled to unit length.  Where r leaves fp32, scaling first (as
  // for candidates) gives zeros, and a NaN for an infinite feature; the product here may be infinite for either.
  static __device__ __forceinline__ float unit_product(float s, float r, const float* half, int dim) {
    if (r != __builtin_inff()) return s * inv_norm(r);
    float zero = 0.f;
    for (int d = 0; d < dim; ++d) zero += half[d] * 0.f;
    return zero;
  }
  // logit from the sums and their errors; row_const: BetaE's sum over the row of lgamma(se) - lgamma(ea) - lgamma(eb),
  // query_const: the same of the query with the other sign
  static __device__ __forceinline__ float score(const float (&total)[kSums], const float (&err)[kSums],
                                                const float (&r)[kRowSums > 0 ? kRowSums : 1], double row_const,
                                                double query_const, const ScoreParams& p, const float* row, int dim) {
#pragma clang fp contract(off)
    if constexpr (M == mBetaKL) {
      const double sum = __builtin_isfinite(total[0]) ? (double)total[0] + (double)err[0] : (double)total[0];
      return p.gamma - (float)(sum + (row_const + query_const));
    }
    float s[kSums];
#pragma unroll
    for (int i = 0; i < kSums; ++i) s[i] = with_error(total[i], err[i]);
    if constexpr (M == mL2) return p.gamma - __builtin_amdgcn_sqrtf(s[0]);
    else if constexpr (M == mComplex || M == mDistmult) {
      float dot = NORM ? unit_product(s[0], r[0], row, dim) : s[0];
      if constexpr (NORM && kSums == 2) dot += unit_product(s[1], r[1], row + dim, dim);
      return p.gamma + dot;
    } else {
      return p.gamma - s[0];
    }
  }
  // a feature's values in LDS from the row's (regularized) values; returns BetaE's log-Beta term
  static __device__ __forceinline__ double expand(float x1, float x2, const ScoreParams& p, float (&e)[kGroup]) {
#pragma clang fp contract(off)
    if constexpr (M == mBetaKL) {
      e[0] = reg_apply(x1, p);
      e[1] = reg_apply(x2, p);
      return log_beta(e[0], e[1], e[2], e[3]);
    } else {
      e[0] = x1;
      if constexpr (kGroup == 2) e[1] = x2;
      return 0.0;
    }
  }
};

// total += step, the rounding error collected in err
__device__ __forceinline__ void add_step(float& total, float& err, float step) {
#pragma clang fp contract(off)
  const float t = total + step;
  err += step - (t - total);
  total = t;
}
__device__ __forceinline__ double beta_eighths(const double (&x)[8]) {
  return ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
}
// BetaE: minus the log-Beta terms of query row bq, summed by a whole wavefront
template <int M>
__device__ __forceinline__ double query_const(const RankArgs& A, int bq, int dim, int lane) {
  if constexpr (M != mBetaKL) return 0.0;
  double mine = 0.0;
  for (int d = lane; d < dim; d += 64) {
    float da, db;
    mine -= log_beta(A.q1[(size_t)bq * dim + d], A.q2[(size_t)bq * dim + d], da, db);
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) mine += __shfl_xor(mine, d);   // (either order of a pair: the same sum in every lane)
  return __longlong_as_double(uniform64(__double_as_longlong(mine)));
}

// Keys (and scores) of the answers.  What bounds it: latency, most calls have a few dozen answers.  2^group_bits lanes share
// an answer and take a step of its features each, out of rows staged in LDS; the steps' sums meet there and are added in
// the scan's order.  (A lane per answer, step after step: 13 us instead of 9 for box at D = 400, 110 for BetaE with its chain
// of special functions.  Lanes that fetch their steps themselves, 64 bytes apart: 59 us instead of 30 for 32,000 answers of
// 2 x 250 floats.)
template <int M, bool NORM, int VEC>
__global__ __launch_bounds__(64) void rank_answer_keys_kernel(RankArgs A, int group_bits, int tiles) {
#pragma clang fp contract(off)
  using O = ScanOps<M, NORM>;
  constexpr int NS = O::kRowSums > 0 ? O::kRowSums : 1, F = O::kFeat, MUL = model_mul(M), kVals = O::kSums + O::kRowSums;
  constexpr bool kBeta = M == mBetaKL;
  // per answer: BetaE's log-Beta terms [steps][8] | (all answers') sums [steps][kVals] | rows [MUL][steps][kKeyStride]
  // | the query's row
  extern __shared__ __attribute__((aligned(16))) double keys_lds[];
  const int lane = threadIdx.x, group = 1 << group_bits, slots = 64 >> group_bits;
  const int mine = lane >> group_bits, s0 = lane & (group - 1);
  const int b = blockIdx.x / tiles, j = (blockIdx.x - b * tiles) * slots + mine;
  const int dim = A.dim, steps = (dim + F - 1) / F;
  const bool valid = j < min(A.ans_count[b], A.A);
  unsigned long long id = valid ? (unsigned long long)A.ans_id[(size_t)b * A.A + j] : 0ull;
  if (id >= A.n_rows) id = 0;  // the host wrapper has already refused such ids
  double* lb = keys_lds + mine * steps * 8;
  float* const parts = reinterpret_cast<float*>(keys_lds + (kBeta ? slots * steps * 8 : 0));
  float* part = parts + mine * steps * kVals;
  float* const rows = parts + ((slots * steps * kVals + 3) & ~3);
  float* const query = rows + slots * MUL * steps * O::kKeyStride;
  {
    typedef std::conditional_t<VEC == 4, float4, float> Piece;
    const int halves = slots * MUL;
    for (int d0 = 0; d0 < dim; d0 += 64 * VEC) {
      const int d = d0 + lane * VEC;
      for (int q0 = 0; q0 < halves; q0 += 8) {   // eight half rows at a time are on their way
        Piece w[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int q = min(q0 + i, halves - 1), from = q / MUL * group;   // (uniform)
          const unsigned long long at = ((unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(id >> 32), from) << 32) |
                                        (unsigned)__builtin_amdgcn_readlane((int)id, from);
          w[i] = *reinterpret_cast<const Piece*>(A.table + (at * MUL + q % MUL) * (size_t)dim + min(d, dim - VEC));
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (q0 + i < halves && d < dim) *reinterpret_cast<Piece*>(rows + ((q0 + i) * steps + d / F) * O::kKeyStride + d % F) = w[i];
      }
    }
  }
  auto fetch = [&](float (&to)[F], const float* from) {   // (what lies past the row's end is not used)
#pragma unroll
    for (int f = 0; f < F; f += 4) {
      const float4 w = reinterpret_cast<const float4*>(from)[f / 4];
      to[f] = w.x;
      to[f + 1] = w.y;
      to[f + 2] = w.z;
      to[f + 3] = w.w;
    }
  };
  float best = 0.f;
  for (int u = 0; u < A.U; ++u) {  // uniform
    const int bq = b * A.U + u;
#pragma unroll
    for (int h = 0; h < model_nq(M); ++h) {
      const float* from = (h == 0 ? A.q1 : A.q2) + (size_t)bq * dim;
      for (int d = lane * VEC; d < dim; d += 64 * VEC) {
        float* to = query + (h * steps + d / F) * O::kKeyStride + d % F;
        if constexpr (VEC == 4) *reinterpret_cast<float4*>(to) = *reinterpret_cast<const float4*>(from + d);
        else *to = from[d];
      }
    }
    __syncthreads();
    for (int c = s0; c < steps; c += group) {
      const int d0 = c * F, n = min(F, dim - d0);
      float x[MUL][F], q1[F], q2[F], s[O::kSums], r[NS];
#pragma unroll
      for (int h = 0; h < MUL; ++h) fetch(x[h], rows + ((mine * MUL + h) * steps + c) * O::kKeyStride);
      fetch(q1, query + c * O::kKeyStride);
      if constexpr (model_nq(M) == 2) fetch(q2, query + (steps + c) * O::kKeyStride);
#pragma unroll
      for (int i = 0; i < O::kSums; ++i) s[i] = 0.f;
#pragma unroll
      for (int i = 0; i < NS; ++i) r[i] = 0.f;
      // N features from f on; the order is the scan's (its `consume`)
      auto block = [&](auto n_tag, int f, float (&ps)[O::kSums], float (&pr)[NS]) {
        constexpr int N = decltype(n_tag)::value;
        float e[N][O::kGroup], qa[N], qb[N];
#pragma unroll
        for (int v = 0; v < N; ++v) {
          const double l = O::expand(x[0][f + v], x[MUL - 1][f + v], A.p, e[v]);
          if constexpr (kBeta) lb[c * 8 + f + v] = l;
          qa[v] = q1[f + v];
          qb[v] = model_nq(M) == 2 ? q2[f + v] : 0.f;
        }
        O::template block<N, false>(e, qa, qb, A.p.cen, ps);
        O::template block_row<N>(e, pr);
      };
      auto take = [&](const float (&ps)[O::kSums], const float (&pr)[NS]) {
#pragma unroll
        for (int i = 0; i < O::kSums; ++i) s[i] += ps[i];
#pragma unroll
        for (int i = 0; i < NS; ++i) r[i] += pr[i];
      };
      float ps[O::kSums], pr[NS], ps2[O::kSums], pr2[NS];
#pragma unroll
      for (int f = 0; f < F; f += 8) {
        if (f + 8 <= n) {
          block(std::integral_constant<int, 4>{}, f, ps, pr);
          block(std::integral_constant<int, 4>{}, f + 4, ps2, pr2);
#pragma unroll
          for (int i = 0; i < O::kSums; ++i) ps[i] += ps2[i];
#pragma unroll
          for (int i = 0; i < NS; ++i) pr[i] += pr2[i];
          take(ps, pr);
        } else if (f < n) {
          const bool four = f + 4 <= n;
          if (four) {
            block(std::integral_constant<int, 4>{}, f, ps, pr);
            take(ps, pr);
          }
#pragma unroll
          for (int v = 0; v < 8; ++v) {
            if (v >= (four ? 4 : 0) && f + v < n) {
              block(std::integral_constant<int, 1>{}, f + v, ps, pr);
              take(ps, pr);
            } else if (kBeta && f + v >= n) {
              lb[c * 8 + f + v] = 0.0;
            }
          }
        }
      }
#pragma unroll
      for (int i = 0; i < O::kSums; ++i) part[c * kVals + i] = s[i];
#pragma unroll
      for (int i = 0; i < O::kRowSums; ++i) part[c * kVals + O::kSums + i] = r[i];
    }
    __syncthreads();
    float tot[O::kSums], err[O::kSums], rtot[NS], rerr[NS];
#pragma unroll
    for (int i = 0; i < O::kSums; ++i) tot[i] = err[i] = 0.f;
#pragma unroll
    for (int i = 0; i < NS; ++i) rtot[i] = rerr[i] = 0.f;
#pragma unroll 4
    for (int c = 0; c < steps; ++c) {
#pragma unroll
      for (int i = 0; i < O::kSums; ++i) add_step(tot[i], err[i], part[c * kVals + i]);
#pragma unroll
      for (int i = 0; i < O::kRowSums; ++i) add_step(rtot[i], rerr[i], part[c * kVals + O::kSums + i]);
    }
    double row_const = 0.0;
    if constexpr (kBeta) {   // (the group has at least eight lanes)
      double sum = 0.0, eighths[8];
      for (int c = 0; c < steps; ++c) sum += lb[c * 8 + (s0 & 7)];
#pragma unroll
      for (int i = 0; i < 8; ++i) eighths[i] = __shfl(sum, mine * group + i);
      row_const = beta_eighths(eighths);
    }
    __syncthreads();  // the next branch writes there
#pragma unroll
    for (int i = 0; i < NS; ++i) rtot[i] = with_error(rtot[i], rerr[i]);
    const float su = O::score(tot, err, rtot, row_const, query_const<M>(A, bq, dim, lane), A.p,
                              A.table + id * (size_t)dim * MUL, dim);
    if (u == 0 || union_takes(su, best)) best = su;
  }
  if (s0 == 0 && j < A.A) {
    if (A.score_out) A.score_out[(size_t)b * A.A + j] = valid ? best : 0.f;
    A.key_out[(size_t)b * A.A + j] = valid ? rank_key(best, id) : 0ull;  // key 0 sorts last and is never counted
  }
}

// NB: query rows per wavefront (four wavefronts share the staged rows).  UP: consecutive query rows that belong to one
// list of answers -- 1, or the branches of a union query padded to 2 or 4 (a row past the last branch repeats it): an
// entity's logit is then the maximum over them.  VEC: floats per table load.
template <int M, bool NORM, int VEC, int NB, int UP>
__global__ __launch_bounds__(kScanThreads) void rank_scan_kernel(RankArgs A) {
#pragma clang fp contract(off)
  using O = ScanOps<M, NORM>;
  constexpr int NS = O::kRowSums > 0 ? O::kRowSums : 1;
  constexpr int R = kScanRows / 64, G = O::kGroup, F = O::kFeat, NL = NB / UP;
  constexpr bool kBeta = M == mBetaKL;
  __shared__ __attribute__((aligned(16))) float stage[2][kScanRows * kScanStride];
  // keys [lists][A], when A.lds_keys | bins [lists][A + 1], when A.lds_bins; the lists of this workgroup
  extern __shared__ unsigned long long lds_keys[];
  const int t = threadIdx.x, lane = t & 63, wave = uniform(t >> 6);
  const int dim = A.dim;
  const size_t row_len = (size_t)dim * model_mul(M);
  const int A1 = A.A + 1;
  const int block_list = A.first_list + (int)blockIdx.y * 4 * NL;
  const int first_list = block_list + wave * NL;   // this wavefront's lists of answers
  const bool active = first_list < A.B;
  const int lists = min(4 * NL, A.B - block_list);
  unsigned* const lds_bins = reinterpret_cast<unsigned*>(lds_keys + (A.lds_keys ? min(4 * NL, A.B) * A.A : 0));
  if (A.lds_bins)
    for (int i = t; i < lists * A1; i += kScanThreads) lds_bins[i] = 0u;
  if (A.lds_keys)
    for (int i = t; i < lists * A.A; i += kScanThreads) lds_keys[i] = A.ans_key[(size_t)block_list * A.A + i];
  __syncthreads();
  int count[NL];                    // answers of the wavefront's lists, and the lowest key of each (uniform)
  unsigned long long lowest[NL];
#pragma unroll
  for (int l = 0; l < NL; ++l) {
    const int b = first_list + l;
    count[l] = b < A.B ? uniform(min(max(A.ans_count[b], 0), A.A)) : 0;
    lowest[l] = count[l] > 0 ? (unsigned long long)uniform64((long long)A.ans_key[(size_t)b * A.A + count[l] - 1]) : ~0ull;
  }
  ScalarRow q1[NB], q2[NB];
  double qc[NB];
#pragma unroll
  for (int x = 0; x < NB; ++x) {
    const int b = min(first_list + x / UP, A.B - 1);   // a list past the last query repeats it and is not counted
    const int bq = b * A.U + min(x % UP, A.U - 1);
    q1[x] = scalar_row(A.q1 + (size_t)bq * dim);
    q2[x] = scalar_row(model_nq(M) == 2 ? A.q2 + (size_t)bq * dim : A.q1);
    qc[x] = active ? query_const<M>(A, bq, dim, lane) : 0.0;
  }

  // Staging.  Rows of 16-byte columns: thread t brings column t % 8 of rows t / 8 + 32 i (two halves: columns 0-3 from
  // the first half, 4-7 from the second).  Others: float t % 32 of rows t / 32 + 8 i.  BetaE: both values of feature
  // t % 8 of rows t / 8 + 32 i, evaluated on the way into LDS.
  constexpr int kItems = kBeta ? 4 : (VEC == 4 ? 4 : 16);
  constexpr int kRowShift = kBeta || VEC == 4 ? 3 : 5, kRowStep = kBeta || VEC == 4 ? 32 : 8;
  typedef float vec4f __attribute__((ext_vector_type(4)));
  // Two halves and few queries, where memory is what bounds: two steps at a time, so that whole 128-byte lines of either half
  // are asked for at once (thread: the same column of both halves; half of the threads then have the first step's).  Four
  // queries, 300 k rows, RotatE 2 x 250 floats 177 -> 167 us, ComplEx 2 x 200 119 -> 117.
  constexpr bool kPairs = G == 2 && NB <= 2;
  typedef std::conditional_t<VEC == 4, vec4f, float> Piece;
  Piece in[kBeta ? 1 : kItems], in_b[kPairs ? kItems : 1];
  float in1[kBeta ? kItems : 1], in2[kBeta ? kItems : 1];
  const int sub = t & ((1 << kRowShift) - 1);
  const int half = G == 2 && !kPairs ? (VEC == 4 ? sub >> 2 : sub >> 4) : 0;
  const int feat = kBeta ? sub : VEC * sub - half * 16;   // first feature within the step (or pair of steps)
  auto request = [&](unsigned g, int d0) {
    if (kPairs && (d0 / F & 1)) return;   // (uniform: on its way since the step before)
    const int d = min(d0 + feat, dim - (kBeta ? 1 : VEC)) + half * dim;
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      const unsigned long long row = min((unsigned long long)g * kScanRows + (t >> kRowShift) + kRowStep * i, A.n_rows - 1);
      const float* p = A.table + row * row_len + d;
      if constexpr (kBeta) {
        in1[i] = p[0];
        in2[i] = p[dim];
      } else {
        in[i] = *reinterpret_cast<const Piece*>(p);
        if constexpr (kPairs) in_b[i] = *reinterpret_cast<const Piece*>(p + dim);
      }
    }
  };
  float cen;   // in a VGPR, see above
  asm("v_mov_b32 %0, %1" : "=v"(cen) : "s"(A.p.cen));
  double lb[kBeta ? kItems : 1];
  auto put = [&](float* to, int d0) {
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      float* at = to + ((t >> kRowShift) + kRowStep * i) * kScanStride;
      if constexpr (kBeta) {
        float e[G];
        const double l = O::expand(in1[i], in2[i], A.p, e);
        lb[i] += d0 + feat < dim ? l : 0.0;
#pragma unroll
        for (int x = 0; x < G; ++x) at[x * F + sub] = e[x];
      } else if constexpr (kPairs) {
        const int f = feat - 16 * (d0 / F & 1);
        if (f >= 0 && f < 16) {
          *reinterpret_cast<Piece*>(at + f) = in[i];
          *reinterpret_cast<Piece*>(at + 16 + f) = in_b[i];
        }
      } else {
        *reinterpret_cast<Piece*>(at + VEC * sub) = in[i];
      }
    }
  };

  float tot[NB][R][O::kSums], err[NB][R][O::kSums], rtot[R][NS], rerr[R][NS];
  // sums over N features (4 or 1) of the staged step, from feature f on
  typedef float Sums[NB][R][O::kSums];
  typedef float RowSums[R][NS];
  auto features = [&](auto n_tag, const float* from, int d0, int f, Sums& s, RowSums& rs) {
    constexpr int N = decltype(n_tag)::value;
    float a[NB][N], b[NB][N], e[R][N][G];
#pragma unroll
    for (int x = 0; x < NB; ++x)
#pragma unroll
      for (int v = 0; v < N; ++v) {
        a[x][v] = q1[x][d0 + f + v];
        b[x][v] = model_nq(M) == 2 ? (float)q2[x][d0 + f + v] : 0.f;
      }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int x = 0; x < G; ++x) {
        const float* at = from + (lane + 64 * r) * kScanStride + x * F + f;
        if constexpr (N == 4) {
          const vec4f w = *reinterpret_cast<const vec4f*>(at);
          e[r][0][x] = w.x; e[r][1][x] = w.y; e[r][2][x] = w.z; e[r][3][x] = w.w;
        } else {
          e[r][0][x] = at[0];
        }
      }
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int x = 0; x < NB; ++x) O::template block<N, true>(e[r], a[x], b[x], cen, s[x][r]);
      O::template block_row<N>(e[r], rs[r]);
    }
  };
  auto consume = [&](const float* from, int d0) {
    Sums s, ps;
    RowSums rs, pr;
    auto add = [&](Sums& to, const Sums& v, RowSums& to_r, const RowSums& v_r) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int x = 0; x < NB; ++x)
#pragma unroll
          for (int i = 0; i < O::kSums; ++i) to[x][r][i] += v[x][r][i];
#pragma unroll
        for (int i = 0; i < NS; ++i) to_r[r][i] += v_r[r][i];
      }
    };
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int x = 0; x < NB; ++x)
#pragma unroll
        for (int i = 0; i < O::kSums; ++i) s[x][r][i] = 0.f;
#pragma unroll
      for (int i = 0; i < NS; ++i) rs[r][i] = 0.f;
    }
    const int n = min(F, dim - d0);
    int f = 0;
    for (; f + 8 <= n; f += 8) {
      Sums ps2;
      RowSums pr2;
      features(std::integral_constant<int, 4>{}, from, d0, f, ps, pr);
      features(std::integral_constant<int, 4>{}, from, d0, f + 4, ps2, pr2);
      add(ps, ps2, pr, pr2);
      add(s, ps, rs, pr);
    }
    if (f + 4 <= n) {
      features(std::integral_constant<int, 4>{}, from, d0, f, ps, pr);
      add(s, ps, rs, pr);
      f += 4;
    }
    for (; f < n; ++f) {
      features(std::integral_constant<int, 1>{}, from, d0, f, ps, pr);
      add(s, ps, rs, pr);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int x = 0; x < NB; ++x)
#pragma unroll
        for (int i = 0; i < O::kSums; ++i) add_step(tot[x][r][i], err[x][r][i], s[x][r][i]);
#pragma unroll
      for (int i = 0; i < NS; ++i) add_step(rtot[r][i], rerr[r][i], rs[r][i]);
    }
  };

  const int steps = (dim + F - 1) / F;
  unsigned g = blockIdx.x;
  request(g, 0);
  int parity = 0;
  for (; g < A.groups; g += gridDim.x) {   // (the same groups for every wavefront of the workgroup)
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int x = 0; x < NB; ++x)
#pragma unroll
        for (int i = 0; i < O::kSums; ++i) tot[x][r][i] = err[x][r][i] = 0.f;
#pragma unroll
      for (int i = 0; i < NS; ++i) rtot[r][i] = rerr[r][i] = 0.f;
    }
    if constexpr (kBeta) {
#pragma unroll
      for (int i = 0; i < kItems; ++i) lb[i] = 0.0;
    }
    for (int c = 0; c < steps; ++c) {
      // the other buffer's readers are behind the barrier of the step before
      put(stage[parity], c * F);
      if (c + 1 < steps) request(g, (c + 1) * F);
      else if (g + gridDim.x < A.groups) request(g + gridDim.x, 0);
      __syncthreads();
      if (active) consume(stage[parity], c * F);
      parity ^= 1;
    }
    double row_const[R];
    if constexpr (kBeta) {   // eight partial sums per row, added in a fixed order
      double* part = reinterpret_cast<double*>(stage[parity]);
#pragma unroll
      for (int i = 0; i < kItems; ++i) part[((t >> kRowShift) + kRowStep * i) * (kScanStride / 2) + sub] = lb[i];
      __syncthreads();
#pragma unroll
      for (int r = 0; r < R; ++r) {
        double x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = part[(lane + 64 * r) * (kScanStride / 2) + i];
        row_const[r] = beta_eighths(x);
      }
      parity ^= 1;
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r) row_const[r] = 0.0;
    }
    if (!active) continue;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const unsigned long long id = (unsigned long long)g * kScanRows + lane + 64 * r;
      float rsum[NS];
#pragma unroll
      for (int i = 0; i < NS; ++i) rsum[i] = with_error(rtot[r][i], rerr[r][i]);
#pragma unroll
      for (int l = 0; l < NL; ++l) {
        float s = 0.f;
#pragma unroll
        for (int u = 0; u < UP; ++u) {
          const float su = O::score(tot[l * UP + u][r], err[l * UP + u][r], rsum, row_const[r], qc[l * UP + u], A.p,
                                    A.table + min(id, A.n_rows - 1) * row_len, dim);
          if (u == 0 || union_takes(su, s)) s = su;
        }
        const unsigned long long key = rank_key(s, id);
        const bool reaches = count[l] > 0 && id < A.n_rows && key >= lowest[l];
        if (__ballot(reaches) == 0ull) continue;   // uniform: no row of these beats any answer of the query
        auto place = [&](const unsigned long long* keys) {
          // answers that the row does not beat: the keys are sorted descending
          int lo = 0, hi = count[l];
          while (__ballot(lo < hi) != 0ull) {
            const int mid = (lo + hi) >> 1;
            if (lo < hi) {
              if (key > keys[mid]) hi = mid;
              else lo = mid + 1;
            }
          }
          // rows that are answers themselves, by the ids in the keys: their own scores may come from elsewhere
          bool is_answer = false;
          for (int j0 = 0; j0 < count[l]; j0 += 64) {
            const unsigned in_group = j0 + lane < count[l] ? ~(unsigned)keys[j0 + lane] - (g * kScanRows + 64 * r) : 64u;
            for (unsigned long long hits = __ballot(in_group < 64u); hits != 0ull; hits &= hits - 1)
              is_answer |= (unsigned)lane == (unsigned)__builtin_amdgcn_readlane((int)in_group, __builtin_ctzll(hits));
          }
          if (reaches && lo < count[l] && !is_answer) {
            if (A.lds_bins) atomicAdd(&lds_bins[(wave * NL + l) * A1 + lo], 1u);
            else atomicAdd(&A.bins[(size_t)(first_list + l) * A1 + lo], 1u);
          }
        };
        if (A.lds_keys) place(lds_keys + (wave * NL + l) * A.A);
        else place(A.ans_key + (size_t)(first_list + l) * A.A);
      }
    }
  }
  if (A.lds_bins) {
    __syncthreads();
    for (int i = t; i < lists * A1; i += kScanThreads) {
      const unsigned v = lds_bins[i];
      if (v) atomicAdd(&A.bins[(size_t)block_list * A1 + i], v);
    }
  }
}

// Evaluation against sampled candidates (the branch of smore/training/train_process.py:118-128 taken when the
// evaluation set brings its own negatives): a query's C candidates are scored -- padding (-1) is scored as entity 0
// with a bias of -1e6 added to the logit, exactly as the reference does -- and ranked among themselves: ranking[j] =
// number of candidates ordered before candidate j by descending biased logit, i.e. the position `argsort(descending)`
// gives it (equal logits: the lower position first, one of the orders an unstable argsort may produce).  The first
// n_hard candidates are the hard answers; their filtered ranks (rank - number of hard answers ranked before it + 1,
// :141-145) come out as well.
// Two launches, so that both halves fill the chip whatever the number of queries: one workgroup per query left 156 of
// 256 compute units idle at 100 queries of 1,001 candidates (RotatE, 2 x 250 floats: one launch 123 us; scores 34 us, the
// fabric's rate for random rows, and ranks 12 us).
// (FUSED, one launch of a workgroup of sixteen wavefronts per query: the second launch costs 3 us, more than it saves up to
// 64 candidates, 5 us instead of 8.)
// Scores: a wavefront takes `per_wave` consecutive candidates of one query, the next row on its way while one is summed.
constexpr int kCandFused = 64;
// ONCE: rows past the caches (candidates_read_once)
template <int M, int VEC, int NIT, bool REG, bool UNION, bool FUSED, bool ONCE = false>
__global__ __launch_bounds__(FUSED ? 1024 : 256) void cand_score_kernel(RankArgs A, int tiles, int per_wave) {
  constexpr int MUL = model_mul(M);
  const int b = blockIdx.x / tiles;
  const int lane = threadIdx.x & 63;
  const int wave = uniform(threadIdx.x >> 6);
  const int dim = A.ncol * VEC;
  const int j0 = ((blockIdx.x - b * tiles) * 4 + wave) * per_wave;
  const int n = min(per_wave, A.C - j0);   // (per_wave <= 64: candidate j0 + i lives in lane i)
  __shared__ unsigned fused_keys[FUSED ? kCandFused : 1];
  if (!FUSED && n <= 0) return;
  if (n > 0) {
    const long long raw = A.cand[(size_t)b * A.C + j0 + min(lane, n - 1)];
    const bool pad = raw == -1;
    unsigned long long id = pad ? 0ull : (unsigned long long)raw;
    const bool bad = id >= A.n_rows;
    if (bad) id = 0;
    if (__ballot(bad) != 0ull && A.err && lane == 0) *A.err = 1;
    const unsigned long long off = id * (size_t)dim * MUL;
    typename ModelOps<M>::Q q[NIT][VEC];
    // The first branch of a union query, or the only row, stays in registers; the others are fetched again per candidate.
    // (BetaE: all of them, in one set of registers.  100 x 500 candidates, two branches: 228 us, 339 with the first kept.)
    constexpr bool kKeep = !UNION || M != mBetaKL;
    if constexpr (kKeep) load_rank_query<M, VEC, NIT>(A.q1, A.q2, b * A.U, dim, A.ncol, lane, q);
    float e1[NIT][VEC], e2[NIT][VEC], next1[NIT][VEC], next2[NIT][VEC];
    auto request = [&](int i) {
      const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)off, i);
      const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(off >> 32), i);
      load_entity<VEC, NIT, MUL, ONCE>(A.table + (((unsigned long long)hi << 32) | lo), dim, A.ncol, lane, next1, next2);
    };
    request(0);
    for (int i = 0; i < n; ++i) {
#pragma unroll
      for (int it = 0; it < NIT; ++it)
#pragma unroll
        for (int v = 0; v < VEC; ++v) {
          e1[it][v] = next1[it][v];
          e2[it][v] = MUL == 2 ? next2[it][v] : 0.f;
        }
      request(min(i + 1, n - 1));
      unit_row<M, VEC, NIT, REG>(e1, e2, A.ncol, lane);
      float s = 0.f;
      if constexpr (kKeep) s = row_score<M, VEC, NIT, REG>(e1, e2, q, A.ncol, lane, A.p);
      if constexpr (UNION) {
        for (int u = kKeep ? 1 : 0; u < A.U; ++u) {  // uniform
          typename ModelOps<M>::Q qu[NIT][VEC];
          load_rank_query<M, VEC, NIT>(A.q1, A.q2, b * A.U + u, dim, A.ncol, lane, qu);
          const float su = row_score<M, VEC, NIT, REG>(e1, e2, qu, A.ncol, lane, A.p);
          if (u == 0 || union_takes(su, s)) s = su;
        }
      }
      s += __builtin_amdgcn_readlane((int)pad, i) ? -1e6f : 0.f;
      if (lane == 63) {
        const size_t at = (size_t)b * A.C + j0 + i;
        if (A.cand_logit) A.cand_logit[at] = s;
        else if (!FUSED) A.cand_rank[at] = (long long)(unsigned long long)__float_as_uint(s);   // the ranking's own slot until it is ranked
        if constexpr (FUSED) fused_keys[j0 + i] = sortable_bits(s);
      }
    }
  }
  if constexpr (FUSED) {   // the ranks, a candidate per lane of the first wavefront
    __syncthreads();
    if (wave != 0 || lane >= A.C) return;
    const unsigned mine = fused_keys[lane];
    const int n_hard = min(A.n_hard[b], min(A.H, A.C));
    int before = 0, ahead = 0;
#pragma unroll 8
    for (int i = 0; i < A.C; ++i) {
      const unsigned k = fused_keys[i];
      const int counts = k > mine || (k == mine && i < lane);
      before += counts;
      ahead += i < n_hard ? counts : 0;
    }
    A.cand_rank[(size_t)b * A.C + lane] = before;
    if (lane < A.H) A.hard_rank[(size_t)b * A.H + lane] = lane < n_hard ? (long long)(before - ahead + 1) : 0ll;
  }
}

// Ranks by counting, 64 candidates per workgroup: each of its wavefronts compares them with its share of the
// query's candidates (four LDS keys per broadcast read) and the counts are added through LDS.  Before position j an
// equal logit counts, behind it only a larger one does, so one 32-bit compare decides and only the stretch that holds
// the workgroup's own positions looks at both.  tiles == 1: the workgroup walks all positions of its query (it then may
// overwrite the scores that stand in the ranking's slots); it has sixteen wavefronts for that if they
// have something to do, four otherwise.
constexpr int cand_padded(int C, int waves) { return (C + 4 * waves - 1) & ~(4 * waves - 1); }
template <int WAVES>
static __global__ __launch_bounds__(64 * WAVES) void cand_rank_kernel(RankArgs A, int tiles) {
  extern __shared__ __attribute__((aligned(16))) unsigned cand_keys[];  // [cand_padded(C, WAVES)] | int [WAVES][64][2]
  const int b = blockIdx.x / tiles, tile = blockIdx.x - b * tiles;
  const int padded = cand_padded(A.C, WAVES);
  int* part = reinterpret_cast<int*>(cand_keys + padded);
  for (int i = threadIdx.x; i < padded; i += 64 * WAVES) {
    unsigned key = 0u;   // (the lowest key, and behind every candidate: never counted)
    if (i < A.C) {
      const size_t at = (size_t)b * A.C + i;
      key = sortable_bits(A.cand_logit ? A.cand_logit[at] : __uint_as_float((unsigned)A.cand_rank[at]));
    }
    cand_keys[i] = key;
  }
  const uint4* keys4 = reinterpret_cast<const uint4*>(cand_keys);
  const int n_hard = min(A.n_hard[b], min(A.H, A.C));
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6);
  const int from = wave * (padded / WAVES), to = from + padded / WAVES;   // (multiples of 4)
  for (int own = tile * 64; own < A.C; own += 64 * tiles) {
    __syncthreads();
    const int j = own + lane;
    const unsigned mine = cand_keys[min(j, A.C - 1)];
    int before = 0, ahead = 0;
    const int lo = min(max(own, from), to), hi = min(max(own + 64, from), to);
#pragma unroll 8
    for (int i = from; i < lo; i += 4) {
      const uint4 k = keys4[i >> 2];
      before += (k.x >= mine) + (k.y >= mine) + (k.z >= mine) + (k.w >= mine);
    }
#pragma unroll 8
    for (int i = lo; i < hi; ++i) {
      const unsigned k = cand_keys[i];
      before += k > mine || (k == mine && i < j);
    }
#pragma unroll 8
    for (int i = hi; i < to; i += 4) {
      const uint4 k = keys4[i >> 2];
      before += (k.x > mine) + (k.y > mine) + (k.z > mine) + (k.w > mine);
    }
    if (own < n_hard) {   // uniform: the hard answers ordered before one of them
      for (int i = from; i < min(to, n_hard); ++i) {
        const unsigned k = cand_keys[i];
        ahead += k > mine || (k == mine && i < j);
      }
    }
    part[(wave * 64 + lane) * 2] = before;
    part[(wave * 64 + lane) * 2 + 1] = ahead;
    __syncthreads();
    if (wave == 0 && j < A.C) {
      before = ahead = 0;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
        before += part[(w * 64 + lane) * 2];
        ahead += part[(w * 64 + lane) * 2 + 1];
      }
      A.cand_rank[(size_t)b * A.C + j] = before;
      if (j < A.H) A.hard_rank[(size_t)b * A.H + j] = j < n_hard ? (long long)(before - ahead + 1) : 0ll;
    }
  }
}

static __global__ __launch_bounds__(256) void rank_clear_kernel(unsigned* bins, size_t n) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) bins[i] = 0u;
}

// filtered rank of answer j (in key order) = 1 + sum of the bins 0..j; one wavefront per query
static __global__ __launch_bounds__(64) void rank_finish_kernel(RankArgs A) {
  const int b = blockIdx.x, lane = threadIdx.x;
  const int n = A.ans_count[b];
  unsigned long long before = 0;
  for (int j0 = 0; j0 < A.A; j0 += 64) {
    const int j = j0 + lane;
    unsigned long long run = j < A.A ? A.bins[(size_t)b * (A.A + 1) + j] : 0u;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
      const unsigned long long left = __shfl_up(run, d);
      if (lane >= d) run += left;
    }
    if (j < A.A)
      A.rank_out[(size_t)b * A.A + (A.slot ? A.slot[(size_t)b * A.A + j] : j)] = j < n ? (long long)(before + run + 1ull) : 0ll;
    before += __shfl(run, 63);
  }
}

// Everything the scan needs beside the keys: the keys in descending order with the slot each came from (unused slots have
// key 0 and go last), the query's bins cleared.  A workgroup places 64 keys, each of its wavefronts by a quarter of the
// query's (one workgroup for all of them: 0.48 ms for a list of 2,000, 6 us now).
static __global__ __launch_bounds__(256) void rank_prepare_kernel(RankArgs A, int tiles, unsigned long long* sorted, int* slot) {
  extern __shared__ unsigned long long sort_keys[];
  __shared__ int before[4][64];
  const int n = A.A, b = blockIdx.x / tiles, tile = blockIdx.x - b * tiles;
  const size_t base = (size_t)b * n;
  for (int i = threadIdx.x; i < n; i += 256) sort_keys[i] = A.key_out[base + i];
  for (int i = tile * 256 + threadIdx.x; i <= n; i += 256 * tiles) A.bins[(size_t)b * (n + 1) + i] = 0u;
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6);
  const int j = tile * 64 + lane, per = (n + 3) / 4;
  const unsigned long long mine = sort_keys[min(j, n - 1)];
  int at = 0;
#pragma unroll 8
  for (int i = wave * per; i < min(n, (wave + 1) * per); ++i) at += sort_keys[i] > mine || (sort_keys[i] == mine && i < j);
  before[wave][lane] = at;
  __syncthreads();
  if (wave == 0 && j < n) {
    at = (before[0][lane] + before[1][lane]) + (before[2][lane] + before[3][lane]);
    sorted[base + at] = mine;
    slot[base + at] = j;
  }
}

// Rows of long lists out of a table that the last-level cache (256 MB) does not hold are loaded past it: no list comes back to
// them, and random rows come at 6.0 TB/s instead of 5.65.  256 lists of 1,500: RotatE 2 x 400 floats, 3.2 GB, 258 -> 243 us, box
// 400 floats, 1.6 GB, 158 -> 152; 256 x 700 x 260 62 -> 58.  The halves' features from 1 GiB on (RotatE
// 2 x 500 floats of 0.7 GB a half 293 / 295, box 128 floats of 0.15 GB 54 / 59, L1 300 floats of 1.1 GB 42.5 / 42.1), lists from 96 MiB on (64 x 400 of 400 floats 38.6 / 39.2), halves from 512 bytes on (440 bytes
// 115 / 114: as good); not BetaE, which is bound by its arithmetic.
inline bool candidates_read_once(const RankArgs& A, int mul) {
  const size_t half = (size_t)A.ncol * 4 * sizeof(float), row = mul * half;
  return half >= 512 && A.n_rows * half >= ((size_t)1 << 30) && (size_t)A.B * A.C * row >= ((size_t)96 << 20);
}

template <int M, int VEC, int NIT, bool REG>
int launch_candidates(hipStream_t st, const RankArgs& A) {
  constexpr bool kOnce = VEC == 4 && M != mBetaKL;
  int per_wave = 16;   // candidates of a wavefront: fewer when the grid would not fill the chip
  while (per_wave > 1 && (size_t)A.B * ((A.C + 4 * per_wave - 1) / (4 * per_wave)) < 2048) per_wave /= 2;
  const int tiles = (A.C + 4 * per_wave - 1) / (4 * per_wave);
  if (A.U == 1 && A.C <= kCandFused) {
    hipLaunchKernelGGL((cand_score_kernel<M, VEC, NIT, REG, false, true>), dim3((unsigned)A.B), dim3(1024), 0, st, A, 1, (A.C + 15) / 16);
    return check_launch("candidate scores and ranks");
  }
  if (A.U > 1)
    hipLaunchKernelGGL((cand_score_kernel<M, VEC, NIT, REG, true, false>), dim3((unsigned)A.B * tiles), dim3(256), 0, st, A, tiles, per_wave);
  else if (kOnce && candidates_read_once(A, model_mul(M)))
    hipLaunchKernelGGL((cand_score_kernel<M, VEC, NIT, REG, false, false, kOnce>), dim3((unsigned)A.B * tiles), dim3(256), 0, st, A, tiles, per_wave);
  else
    hipLaunchKernelGGL((cand_score_kernel<M, VEC, NIT, REG, false, false>), dim3((unsigned)A.B * tiles), dim3(256), 0, st, A, tiles, per_wave);
  if (int rc = check_launch("candidate scores")) return rc;
  auto lds = [&](int waves) { return (size_t)cand_padded(A.C, waves) * sizeof(unsigned) + waves * 64 * 2 * sizeof(int); };
  if (!A.cand_logit && A.C > 256) {   // (2,048 x 128 candidates: 34 us with sixteen wavefronts, 28 with four)
    hipLaunchKernelGGL(cand_rank_kernel<16>, dim3((unsigned)A.B), dim3(1024), lds(16), st, A, 1);
  } else {
    const int rank_tiles = A.cand_logit ? (A.C + 63) / 64 : 1;
    hipLaunchKernelGGL(cand_rank_kernel<4>, dim3((unsigned)A.B * rank_tiles), dim3(256), lds(4), st, A, rank_tiles);
  }
  return check_launch("candidate ranks");
}

template <class K>
unsigned long long resident_workgroups(K kernel, int threads, size_t lds) {
  int dev = 0, cus = 256, per_cu = 2;
  if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, lds) != hipSuccess || per_cu < 1) per_cu = 2;
  return (unsigned long long)cus * per_cu;
}

inline int clear_bins(hipStream_t st, const RankArgs& A) {
  if (A.slot) return SMX_OK;   // (smx_filtered_ranks has cleared them: rank_prepare_kernel)
  const size_t n_bins = (size_t)A.B * (A.A + 1);
  hipLaunchKernelGGL(rank_clear_kernel, dim3((unsigned)((n_bins + 255) / 256)), dim3(256), 0, st, A.bins, n_bins);
  return check_launch("rank scan (bins)");
}
inline int finish_ranks(hipStream_t st, const RankArgs& A) {
  hipLaunchKernelGGL(rank_finish_kernel, dim3((unsigned)A.B), dim3(64), 0, st, A);
  return check_launch("rank scan");
}

template <int M, bool NORM, int VEC, int NB, int UP>
int launch_scan(hipStream_t st, RankArgs A) {
  constexpr int kLists = 4 * (NB / UP);   // lists of answers a workgroup serves
  // Keys and bins in LDS beside 36 KB of staged rows while four workgroups still fit a compute unit; then bins alone up to
  // 24 KB; longer lists count in memory directly.
  const size_t lists = A.B < kLists ? A.B : kLists, bins = lists * (A.A + 1) * sizeof(unsigned);
  const size_t keys = lists * A.A * sizeof(unsigned long long);
  A.lds_bins = bins <= (size_t)24 << 10;
  A.lds_keys = keys + bins <= (size_t)4 << 10;
  const size_t lds = (A.lds_bins ? bins : 0) + (A.lds_keys ? keys : 0);
  // several workgroups per slot: the last ones then spread evenly (BetaE's evaluate their queries first: one per slot)
  const unsigned long long most =
      resident_workgroups(rank_scan_kernel<M, NORM, VEC, NB, UP>, kScanThreads, lds) * (M == mBetaKL ? 1 : 4);
  const unsigned blocks = (unsigned)(A.groups < most ? A.groups : most);
  const unsigned passes = (unsigned)((A.B + kLists - 1) / kLists);
  for (unsigned done = 0; done < passes; done += 65535u) {   // (the second grid extent's limit)
    const unsigned now = passes - done < 65535u ? passes - done : 65535u;
    A.first_list = (int)done * kLists;
    hipLaunchKernelGGL((rank_scan_kernel<M, NORM, VEC, NB, UP>), dim3(blocks, now), dim3(kScanThreads), lds, st, A);
    if (int rc = check_launch("rank scan")) return rc;
  }
  return SMX_OK;
}

template <int M, bool NORM, int VEC>
int launch_scan_vec(hipStream_t st, const RankArgs& A) {
  // query rows per wavefront: four wavefronts take all queries of a small batch between them; a full batch of sixteen
  // reads the table once
  if (A.U == 1) {
    if (A.B <= 4) return launch_scan<M, NORM, VEC, 1, 1>(st, A);
    if (A.B <= 8) return launch_scan<M, NORM, VEC, 2, 1>(st, A);
    return launch_scan<M, NORM, VEC, 4, 1>(st, A);
  }
  if (A.U == 2) return A.B <= 4 ? launch_scan<M, NORM, VEC, 2, 2>(st, A) : launch_scan<M, NORM, VEC, 4, 2>(st, A);
  return launch_scan<M, NORM, VEC, 4, 4>(st, A);
}

template <int M, bool NORM>
int launch_rank_all(hipStream_t st, RankArgs A, int vec, int mode) {
  if (mode == kRankKeys) {
    using O = ScanOps<M, NORM>;
    const int steps = (A.dim + O::kFeat - 1) / O::kFeat;   // at most 256 (BetaE, 2,048 floats per half)
    int bits = M == mBetaKL ? 3 : 0;
    while (bits < 6 && (1 << bits) < steps) ++bits;
    const int slots = 64 >> bits, tiles = (A.A + slots - 1) / slots;
    // (at most 50 KiB: BetaE's 256 steps of one answer, 16 KiB each of them log-Beta terms, row and query)
    const size_t sums = ((size_t)slots * steps * (O::kSums + O::kRowSums) + 3) & ~(size_t)3;
    const size_t lds = (M == mBetaKL ? (size_t)slots * steps * 8 * sizeof(double) : 0) +
                       (sums + ((size_t)slots * model_mul(M) + model_nq(M)) * steps * O::kKeyStride) * sizeof(float);
    if (vec == 4) hipLaunchKernelGGL((rank_answer_keys_kernel<M, NORM, 4>), dim3((unsigned)A.B * tiles), dim3(64), lds, st, A, bits, tiles);
    else hipLaunchKernelGGL((rank_answer_keys_kernel<M, NORM, 1>), dim3((unsigned)A.B * tiles), dim3(64), lds, st, A, bits, tiles);
    return check_launch("rank answer keys");
  }
  if (int rc = clear_bins(st, A)) return rc;
  A.groups = (unsigned)((A.n_rows + kScanRows - 1) / kScanRows);
  int rc;
  if constexpr (M == mBetaKL) rc = launch_scan_vec<M, NORM, 1>(st, A);   // (fetches single floats at any alignment)
  else rc = vec == 4 ? launch_scan_vec<M, NORM, 4>(st, A) : launch_scan_vec<M, NORM, 1>(st, A);
  return rc ? rc : finish_ranks(st, A);
}

// f(VEC, NIT, REG as integral constants) for a call's row shape
template <int M, class F>
int with_row_shape(const RankArgs& A, int vec, int nit, F f) {
  using std::integral_constant;
  auto with_reg = [&](auto vec_tag, auto nit_tag) {
    if constexpr (M == mBetaKL || M == mComplex || M == mDistmult) {
      if (M == mBetaKL ? A.p.reg_on : A.p.norm_on) return f(vec_tag, nit_tag, std::true_type{});
    }
    return f(vec_tag, nit_tag, std::false_type{});
  };
  if (vec == 4) {
    switch (nit) {
      case 1: return with_reg(integral_constant<int, 4>{}, integral_constant<int, 1>{});
      case 2: return with_reg(integral_constant<int, 4>{}, integral_constant<int, 2>{});
      case 4: return with_reg(integral_constant<int, 4>{}, integral_constant<int, 4>{});
      default: return with_reg(integral_constant<int, 4>{}, integral_constant<int, 8>{});
    }
  }
  switch (nit) {
    case 1: return with_reg(integral_constant<int, 1>{}, integral_constant<int, 1>{});
    case 2: return with_reg(integral_constant<int, 1>{}, integral_constant<int, 2>{});
    default: return with_reg(integral_constant<int, 1>{}, integral_constant<int, 4>{});
  }
}

// Instantiated once per model in its own translation unit (smx_rank_inst_*.hip).
template <int M>
int rank_dispatch(hipStream_t st, const RankArgs& A, int vec, int nit, int mode) {
  if (mode == kRankCandidates)
    return with_row_shape<M>(A, vec, nit, [&](auto vec_tag, auto nit_tag, auto reg_tag) {
      return launch_candidates<M, decltype(vec_tag)::value, decltype(nit_tag)::value, decltype(reg_tag)::value>(st, A);
    });
  if constexpr (M == mComplex || M == mDistmult) {
    if (A.p.norm_on) return launch_rank_all<M, true>(st, A, vec, mode);
  }
  return launch_rank_all<M, false>(st, A, vec, mode);   // (BetaE's clamp is a run-time switch of the scan)
}

}  // namespace smx
