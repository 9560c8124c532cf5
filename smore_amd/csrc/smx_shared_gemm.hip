// Negatives shared by the batch as matrix products: BetaE, ComplEx and DistMult.
//
// With --share_negative (smore/cpp_sampler/online_sampler.py:155-157) the same K rows meet all B queries.  For the
// models whose pair score is, or can be regrouped into, an inner product of something per row with something per
// query, the B x K pairs are then a matrix product with an operand shared along each axis -- the one shape on this
// path that the matrix cores fit (v_mfma_f32_32x32x2_f32: fp32 operands, fp32 accumulation in a fixed order).
//
// ComplEx, DistMult (smore/common/torchext/dist_kernel.h:187-204, 324-349): score = gamma + sum_j e[k,j] q[b,j], j over the
// row ([re | im] against [q1 | q2], or the D features of DistMult):
//   forward         [B, J] x [J, K]      (rows of the table gathered by the list's ids as the second operand)
//   query backward  gq = g [B, K] x E [K, J]
//   entity side     R = g^T [K, B] x [q1 | q2] [B, J]: the gradient row of list position k, written where the caller
//                   wants it, or (plan, optimizer, unit-length rows) finished by shared_entity_kernel of smx_shared_impl.h
//
// BetaE: KL(Beta(e) || Beta(q)) per feature (dist_kernel.h:207-266) is
//   [lgG(qa)+lgG(qb)-lgG(sq)] + [lgG(se)-lgG(ea)-lgG(eb)] + (ea-qa) psi(ea) + (eb-qb) psi(eb) + (sq-se) psi(se):
// three digammas and a log-beta of the ENTITY per (pair, feature), which is what makes the per-query kernels
// instruction-bound (smore/models/beta.py:303-308 through beta_dist.py).  Regrouped by what each term depends on,
//   KL[b,k] = Qk[b] + Ek[k] + sum_d qa[b,d] T[k,d] + sum_d qb[b,d] T[k,D+d]
//     T[k,d] = psi(se)-psi(ea),  T[k,D+d] = psi(se)-psi(eb)                       (one row of 2D floats per shared row)
//     Ek[k]  = sum_d [lgG(se)-lgG(ea)-lgG(eb)] + ea psi(ea) + eb psi(eb) - se psi(se)
//     Qk[b]  = sum_d lgG(qa)+lgG(qb)-lgG(sq)
// the special functions are evaluated K x D + B x D times instead of B x K x D, and what is left per pair is the
// product [B, 2D] x [2D, K] with T in the place of the rows.  The query backward is the other product with T,
//   gqa[b,d] = (psi(qa)-psi(sq)) sum_k c[b,k] + sum_k c[b,k] T[k,d]            (c = -upstream gradient; same with b),
// and the entity side (ModelOps<mBetaKL>::bwd_e sums c (ea - qa) and c (eb - qb) over the queries) is
//   S1[k,d] = ea[k,d] C[k] - R[k,d],  S2[k,d] = eb[k,d] C[k] - R[k,D+d],  C[k] = sum_b c[b,k],  R = c^T x [q1 | q2],
// turned into the gradient row (trigamma hook, clamp mask, optimizer) by shared_entity_kernel.  The sums are those of
// ModelOps<mBetaKL>::fwd / bwd_q / bwd_e taken in another order: the groups of terms are summed separately, which
// costs some of the tolerance's headroom (measured in the tests), not the bar.
#include "smx_common.h"
#include "smx_models.h"
#include "smx_wave.h"

namespace smx {

typedef float facc16 __attribute__((ext_vector_type(16)));

// ---- the terms of the shared rows: T [K][2D], then (forward) Ek [K]; one wavefront per row ------------------
template <bool FWD>
__global__ __launch_bounds__(256) void beta_row_terms_kernel(const float* __restrict__ table,
                                                             const long long* __restrict__ ids, int K, int dim,
                                                             unsigned long long n_rows, ScoreParams p,
                                                             float* __restrict__ T, float* __restrict__ Ek, int* err) {
  const int lane = threadIdx.x & 63;
  const int k = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (k >= K) return;
  long long row = ids[k];
  if ((unsigned long long)row >= n_rows) {  // remember it, read row 0 instead (as every scorer of the library does)
    if (err && lane == 0) *err = 1;
    row = 0;
  }
  const float* e = table + (size_t)row * 2 * dim;
  float* out = T + (size_t)k * 2 * dim;
  float mine = 0.f;
  for (int d = lane; d < dim; d += 64) {
    const float ea = reg_apply(e[d], p), eb = reg_apply(e[dim + d], p);
    float lb, pa, pb, ps;
    if constexpr (FWD) {
      beta_terms(ea, eb, lb, pa, pb, ps);
      mine += (lb + ea * pa) + (eb * pb - (ea + eb) * ps);
    } else {
      digamma3(ea, eb, pa, pb, ps);
    }
    out[d] = ps - pa;
    out[dim + d] = ps - pb;
  }
  if constexpr (FWD) {
    const float total = wave_sum_last_f32(mine);
    if (lane == 63) Ek[k] = total;
  }
}

// Qk [B]: one wavefront per query, in the form of the rows' constants: what the two are off by in the same way cancels
__global__ __launch_bounds__(256) void beta_query_terms_kernel(const float* __restrict__ q1, const float* __restrict__ q2,
                                                               int B, int dim, float* __restrict__ Qk) {
  const int lane = threadIdx.x & 63;
  const int b = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (b >= B) return;
  float mine = 0.f;
  for (int d = lane; d < dim; d += 64) {
    float lb, pa, pb, ps;
    beta_terms(q1[(size_t)b * dim + d], q2[(size_t)b * dim + d], lb, pa, pb, ps);
    mine -= lb;
  }
  const float total = wave_sum_last_f32(mine);
  if (lane == 63) Qk[b] = total;
}

// ---- the matrix products ------------------------------------------------------------------------------------
// A 32 x 32 tile of the result is formed by walking the inner dimension two at a time with
// v_mfma_f32_32x32x2_f32.  Operand layout of the instruction: lane l supplies A[l % 32][l / 32] and B[l / 32][l % 32];
// of the 16 accumulators of lane l, number r is the element (8 (r / 4) + 4 (l / 32) + r % 4, l % 32).
__device__ __forceinline__ int acc_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

// What the three products need to know about a call.  BETA: the second operand's rows are rows of T, else rows of
// the table found through the list's ids; nq = query tensors (the inner dimension is nq * dim features).
struct GemmArgs {
  const float* rows;       // T [K][2 dim] (BETA) or the table
  const long long* ids;    // [K] (not BETA); null: `rows` holds the K rows themselves, in list order
  unsigned long long n_rows;
  const float* q1;
  const float* q2;
  const float* gscore;     // [B, K]
  const float* Ek;         // BETA forward
  const float* Qk;
  float* out1;             // score; gq1; R
  float* out2;             // gq2; C
  int B, K, dim, nq;
  float gamma;
  int* err;
};

template <bool BETA>
__device__ __forceinline__ const float* shared_row(const GemmArgs& A, int k, int& bad) {
  if constexpr (BETA) {
    return A.rows + (size_t)k * 2 * A.dim;
  } else {
    if (!A.ids) return A.rows + (size_t)k * A.nq * A.dim;  // uniform
    long long row = A.ids[k];
    if ((unsigned long long)row >= A.n_rows) {  // remember it, read row 0 instead (as every scorer of the library does)
      bad = 1;
      row = 0;
    }
    return A.rows + (size_t)row * A.nq * A.dim;
  }
}

// The three products, M x N results over an inner dimension of length L:
//   forward  M = B, N = K, L = J       score[b,k] = gamma -/+ (... + sum_j q[b,j] row_k[j]), j over the J = nq dim features
//   query    M = B, N = J, L = K       gq[b,n]    = sum_k c[b,k] row_k[n]  (+ kq[b,n] sum_k c[b,k] for BETA)
//   entity   M = K, N = J, L = B       R[k,n]     = sum_b c[b,k] q[b,n],  C[k] = sum_b c[b,k] (BETA)
// with c = -gscore (BETA) or gscore.
//
// A workgroup owns a tile of 32 x 64 (or 32) results.  64 steps of the inner dimension are staged in LDS at a time, in
// 16-byte pieces of whole 128-byte lines, the next two stages already on their way into registers; four wavefronts share each 32 x 32
// part and take a quarter of every stage each, with two accumulators in turn (eight partial sums per element, added in
// a fixed order).  An operand whose memory runs along the inner dimension is read from LDS four values per lane (lanes
// 0-31: inner 8 u .. 8 u + 3, lanes 32-63: the next four), one that runs along the result one value per lane and
// instruction; the strides keep both free of bank conflicts.
// What bounds it: latency and the matrix cores.  B = 512, K = 1024, D = 400, ComplEx (J = 800: 0.84 GFLOP per product,
// 5.3 us at the fp32 matrix rate): 13.4 / 18.6 / 14 us (forward / query / entity); with operands fetched by every
// wavefront straight from memory in the 16-byte pieces the instruction's layout wants, four trips of each line through
// the L1, 20.8 / 24 / 20.6.
enum GemmMode : int { kGemmForward = 0, kGemmQuery = 1, kGemmEntity = 2 };
constexpr int kTileM = 32, kStageL = 64;

// Which tile a workgroup takes.  Workgroups go to the eight XCDs in turn; each XCD gets a block of tiles a quarter of
// the rows high and half the columns wide, so that what its workgroups read fits its L2 and is fetched by two to four
// of the eight instead of all.
__host__ __device__ inline int gemm_blocks_m(int M) { return ((M + kTileM - 1) / kTileM + 3) / 4; }
__host__ __device__ inline int gemm_blocks_n(int N, int tile_n) { return ((N + tile_n - 1) / tile_n + 1) / 2; }

template <int MODE, bool BETA, int kTileN>
__global__ __launch_bounds__(8 * kTileN) void shared_gemm_kernel(GemmArgs A) {
  constexpr int kGemmThreads = 8 * kTileN;                       // four wavefronts per 32 columns
  constexpr int kPiecesA = kTileM * kStageL / 4 / kGemmThreads;  // 16-byte pieces of a stage per thread
  constexpr int kPiecesB = kTileN * kStageL / 4 / kGemmThreads;
  constexpr bool kAInner = MODE != kGemmEntity;    // the operand's memory runs along the inner dimension
  constexpr bool kBInner = MODE == kGemmForward;
  constexpr int SA = kAInner ? kStageL + 4 : kTileM + 8, SB = kBInner ? kStageL + 4 : kTileN + 8;
  constexpr int kA = (kAInner ? kTileM : kStageL) * SA, kB = (kBInner ? kTileN : kStageL) * SB;
  __shared__ __attribute__((aligned(16))) float lds[2 * (kA + kB)];
  typedef float f4 __attribute__((ext_vector_type(4)));
  const f4 zero4 = {0.f, 0.f, 0.f, 0.f};
  const int t = threadIdx.x, lane = t & 63, wave = uniform(t >> 6);
  const int half = lane >> 5, col = lane & 31;
  const int dim = A.dim, J = A.nq * dim;
  const int M = MODE == kGemmEntity ? A.K : A.B, N = MODE == kGemmForward ? A.K : J;
  const int L = MODE == kGemmForward ? J : (MODE == kGemmQuery ? A.K : A.B);
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int bm = gemm_blocks_m(M), bn = gemm_blocks_n(N, kTileN);
  const int m0 = ((xcd >> 1) * bm + local / bn) * kTileM, n0 = ((xcd & 1) * bn + local % bn) * kTileN;
  if (m0 >= M || n0 >= N) return;   // (uniform: the blocks of tiles are rounded up)
  int bad = 0;

  f4 ra[2][kPiecesA], rb[2][kPiecesB];   // [stages on their way][pieces]
  const bool wide = (A.K & 3) == 0 && (reinterpret_cast<unsigned long long>(A.gscore) & 15ull) == 0ull;
  const float* b_row[kPiecesB];   // forward: the table (or T) rows of the pieces
  if constexpr (MODE == kGemmForward) {
#pragma unroll
    for (int i = 0; i < kPiecesB; ++i) b_row[i] = shared_row<BETA>(A, min(n0 + t / 16 + kGemmThreads / 16 * i, N - 1), bad);
    if (bad && A.err) *A.err = 1;
  }
  // four upstream gradients g[b][k .. k + 3]; past the list's end zeros
  auto load_g = [&](int b, int k) -> f4 {
    const float* p = A.gscore + (size_t)min(b, A.B - 1) * A.K;
    if (b >= A.B || k >= A.K) return zero4;
    if (wide) return *reinterpret_cast<const f4*>(p + k);
    f4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = k + e < A.K ? p[min(k + e, A.K - 1)] : 0.f;
    return v;
  };
  // four features of [q1 | q2] of query b from feature j on (j and dim are multiples of four)
  auto load_q = [&](int b, int j) -> f4 {
    return *reinterpret_cast<const f4*>(j < dim ? A.q1 + (size_t)b * dim + j : A.q2 + (size_t)b * dim + (j - dim));
  };
  // query: the rows of a stage are found through ids that were fetched a stage earlier
  long long id_next[kPiecesB] = {};
  auto fetch_ids = [&](int l0) {
    if constexpr (MODE == kGemmQuery && !BETA) {
      if (A.ids) {   // uniform
#pragma unroll
        for (int i = 0; i < kPiecesB; ++i) id_next[i] = A.ids[min(l0 + t / (kTileN / 4) + kGemmThreads / (kTileN / 4) * i, L - 1)];
      }
    }
  };
  auto request = [&](f4 (&ga)[kPiecesA], f4 (&gb)[kPiecesB], int l0) {
#pragma unroll
    for (int i = 0; i < kPiecesA; ++i) {
      if constexpr (MODE == kGemmForward) {
        const int j = l0 + 4 * (t & 15);
        ga[i] = j < L ? load_q(min(m0 + t / 16 + kGemmThreads / 16 * i, M - 1), j) : zero4;
      } else if constexpr (MODE == kGemmQuery) {
        ga[i] = load_g(min(m0 + t / 16 + kGemmThreads / 16 * i, M - 1), l0 + 4 * (t & 15));
      } else {
        ga[i] = load_g(l0 + t / 8 + kGemmThreads / 8 * i, m0 + 4 * (t & 7));
      }
    }
#pragma unroll
    for (int i = 0; i < kPiecesB; ++i) {
      // (forward: 16 pieces per row; the others: kTileN / 4 pieces per inner step)
      constexpr int kPer = kBInner ? 16 : kTileN / 4;
      const int r = t / kPer + kGemmThreads / kPer * i, c = 4 * (t % kPer);
      if constexpr (MODE == kGemmForward) {
        gb[i] = l0 + c < L ? *reinterpret_cast<const f4*>(b_row[i] + l0 + c) : zero4;
      } else if constexpr (MODE == kGemmQuery) {   // (rows past the list repeat its last one: their coefficients are zero)
        long long row = min(l0 + r, L - 1);
        if (!BETA && A.ids) row = (unsigned long long)id_next[i] < A.n_rows ? id_next[i] : 0;   // (outside the table: row 0)
        gb[i] = *reinterpret_cast<const f4*>(A.rows + (size_t)row * J + min(n0 + c, N - 4));
      } else {
        gb[i] = load_q(min(l0 + r, L - 1), min(n0 + c, N - 4));
      }
    }
    fetch_ids(l0 + kStageL);
  };
  auto put = [&](const f4 (&ga)[kPiecesA], const f4 (&gb)[kPiecesB], float* to) {
#pragma unroll
    for (int i = 0; i < kPiecesA; ++i) {
      if constexpr (kAInner) *reinterpret_cast<f4*>(to + (t / 16 + kGemmThreads / 16 * i) * SA + 4 * (t & 15)) = ga[i];
      else *reinterpret_cast<f4*>(to + (t / 8 + kGemmThreads / 8 * i) * SA + 4 * (t & 7)) = ga[i];
    }
#pragma unroll
    for (int i = 0; i < kPiecesB; ++i) {
      constexpr int kPer = kBInner ? 16 : kTileN / 4;
      *reinterpret_cast<f4*>(to + kA + (t / kPer + kGemmThreads / kPer * i) * SB + 4 * (t % kPer)) = gb[i];
    }
  };

  const int ns = wave % (kTileN / 32), kh = wave / (kTileN / 32);   // 32 columns of the tile; a quarter of every stage
  facc16 acc[2] = {{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}, {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}};
  float c_sum = 0.f;
  auto consume = [&](const float* from, int l0) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int i0 = 8 * (kh * 2 + u);
      if (l0 + i0 < L) {   // uniform
        f4 a, b;
        if constexpr (kAInner) {
          a = *reinterpret_cast<const f4*>(from + col * SA + i0 + 4 * half);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) a[e] = from[(i0 + 4 * half + e) * SA + col];
        }
        if constexpr (kBInner) {
          b = *reinterpret_cast<const f4*>(from + kA + (ns * 32 + col) * SB + i0 + 4 * half);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) b[e] = from[kA + (i0 + 4 * half + e) * SB + ns * 32 + col];
        }
        if constexpr (BETA && MODE != kGemmForward) c_sum += (a[0] + a[1]) + (a[2] + a[3]);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[u & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], acc[u & 1], 0, 0, 0);
      }
    }
  };
  const int stages = (L + kStageL - 1) / kStageL;
  float* const buf0 = lds;
  float* const buf1 = lds + kA + kB;
  fetch_ids(0);
  request(ra[0], rb[0], 0);
  if (stages > 1) request(ra[1], rb[1], kStageL);
  for (int s = 0; s < stages; s += 2) {   // (stage s + 1's buffer was last read at stage s - 1, behind a barrier)
    put(ra[0], rb[0], buf0);
    if (s + 2 < stages) request(ra[0], rb[0], (s + 2) * kStageL);
    __syncthreads();
    consume(buf0, s * kStageL);
    if (s + 1 >= stages) break;
    put(ra[1], rb[1], buf1);
    if (s + 3 < stages) request(ra[1], rb[1], (s + 3) * kStageL);
    __syncthreads();
    consume(buf1, (s + 1) * kStageL);
  }
  facc16 sum = acc[0] + acc[1];
  c_sum += __shfl_xor(c_sum, 32);   // row m0 + col: both halves of every eight
  __syncthreads();                  // the stages are dead: their LDS takes the second halves' partial tiles
  if (kh > 0) {
    float* part = lds + ((kh - 1) * (kTileN / 32) + ns) * 17 * 64 + lane;
#pragma unroll
    for (int r = 0; r < 16; ++r) part[r * 64] = sum[r];
    part[16 * 64] = c_sum;
  }
  __syncthreads();
  if (kh > 0) return;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float* part = lds + (k * (kTileN / 32) + ns) * 17 * 64 + lane;
#pragma unroll
    for (int r = 0; r < 16; ++r) sum[r] += part[r * 64];
    c_sum += part[16 * 64];
  }
  const int n = n0 + ns * 32 + col;
  if constexpr (MODE == kGemmForward) {
    if (n >= N) return;
    const float ek = BETA ? A.Ek[n] : 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = m0 + acc_row(r, lane);
      if (m < M) A.out1[(size_t)m * N + n] = BETA ? A.gamma - ((A.Qk[m] + ek) + sum[r]) : A.gamma + sum[r];
    }
  } else if constexpr (MODE == kGemmQuery) {
    const int d = n < dim ? n : n - dim;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = acc_row(r, lane);
      const float g = BETA ? __shfl(c_sum, row) : 0.f;
      const int m = m0 + row;
      if (m < M && n < N) {
        float v = sum[r];
        if constexpr (BETA) {
          float pa, pb, ps;   // (the rows' digammas are of this form)
          digamma3(A.q1[(size_t)m * dim + d], A.q2[(size_t)m * dim + d], pa, pb, ps);
          v = -(v + ((n < dim ? pa : pb) - ps) * g);
        }
        (n < dim ? A.out1 : A.out2)[(size_t)m * dim + d] = v;
      }
    }
  } else {
    if (BETA && n0 == 0 && ns == 0 && half == 0 && m0 + col < M) A.out2[m0 + col] = -c_sum;
    if (n >= N) return;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = m0 + acc_row(r, lane);
      if (m < M) A.out1[(size_t)m * N + n] = BETA ? -sum[r] : sum[r];
    }
  }
}

template <int MODE, bool BETA>
static void launch_gemm(hipStream_t st, const GemmArgs& A) {
  const int J = A.nq * A.dim;
  const int M = MODE == kGemmEntity ? A.K : A.B, N = MODE == kGemmForward ? A.K : J;
  // 64 columns per workgroup where that gives every compute unit one, else 32 (B = 512, K = 1024, D = 400: ComplEx
  // forward, 256 workgroups, 13.4 us against 15.1 with 512; query 19.6 with 208, 18.6 with 400; DistMult query 17.4
  // with 112, 13.1 with 208)
  if (((M + kTileM - 1) / kTileM) * ((N + 63) / 64) >= 256)
    hipLaunchKernelGGL((shared_gemm_kernel<MODE, BETA, 64>), dim3(8u * (unsigned)gemm_blocks_m(M) * (unsigned)gemm_blocks_n(N, 64)),
                       dim3(512), 0, st, A);
  else
    hipLaunchKernelGGL((shared_gemm_kernel<MODE, BETA, 32>), dim3(8u * (unsigned)gemm_blocks_m(M) * (unsigned)gemm_blocks_n(N, 32)),
                       dim3(256), 0, st, A);
}

// ---- the K rows of the list side by side, as the products' second operand -------------------------------------
// UNIT (ComplEx with unit-length halves, width = 2 dim): out [K][2 dim], row k = [re / max(|re|, eps) |
// im / max(|im|, eps)] of table row ids[k]; DistMult with unit-length rows, width = dim: e / max(|e|, eps).  One
// wavefront per row.
// Not UNIT: out [K][width], row k = table row ids[k] as it is, for the distance models' query backward.  (The products
// fetch the ids a stage ahead of the rows and do not need the copy: ComplEx query backward at B = 512, K = 1024,
// D = 400 19.6 us through the ids of a table of 3 to 64 GB, 23.8 with the copy.)
template <bool UNIT>
__global__ __launch_bounds__(256) void list_rows_kernel(const float* __restrict__ table, const long long* __restrict__ ids,
                                                        int K, int dim, int width, unsigned long long n_rows,
                                                        float* __restrict__ En, int* err) {
  const int lane = threadIdx.x & 63;
  const int k = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (k >= K) return;
  long long row = ids[k];
  if ((unsigned long long)row >= n_rows) {
    if (err && lane == 0) *err = 1;
    row = 0;
  }
  const float* e = table + (size_t)row * width;
  float* out = En + (size_t)k * width;
  if constexpr (!UNIT) {
    typedef float f4 __attribute__((ext_vector_type(4)));  // (width is a multiple of four, the rows 16-byte aligned)
    for (int c = lane; c < width / 4; c += 64) reinterpret_cast<f4*>(out)[c] = reinterpret_cast<const f4*>(e)[c];
    return;
  }
  const bool two = width == 2 * dim;  // ComplEx; DistMult: the row is its only half
  float s1 = 0.f, s2 = 0.f;
  for (int d = lane; d < dim; d += 64) {
    s1 = __builtin_fmaf(e[d], e[d], s1);
    if (two) s2 = __builtin_fmaf(e[dim + d], e[dim + d], s2);
  }
  const float i1 = inv_norm(wave_sum_f32(s1)), i2 = inv_norm(wave_sum_f32(s2));
  for (int d = lane; d < dim; d += 64) {
    out[d] = e[d] * i1;
    if (two) out[dim + d] = e[dim + d] * i2;
  }
}

// ---- host side ----------------------------------------------------------------------------------------------
// out [K][width] = table rows ids[k], width a multiple of four floats, everything 16-byte aligned
int shared_list_rows(hipStream_t st, const float* table, size_t n_rows, const long long* ids, size_t K, size_t width,
                     float* out) {
  hipLaunchKernelGGL(list_rows_kernel<false>, dim3((unsigned)((K + 3) / 4)), dim3(256), 0, st, table, ids, (int)K, 0,
                     (int)width, (unsigned long long)n_rows, out, nullptr);
  return check_launch("rows of the shared list, side by side");
}

static bool is_inner(int model) { return model == mComplex || model == mDistmult; }

// floats of workspace a call of the model needs: forward / query backward, and the entity side
// (norm: ComplEx with unit-length halves, whose scaled rows stand in the workspace for the first two)
size_t shared_gemm_workspace_floats(int model, size_t B, size_t K, size_t dim, bool entity, bool norm) {
  if (model == mBetaKL) return entity ? K * (2 * dim + 1) : K * (2 * dim + 1) + B;
  if (is_inner(model)) return entity || norm ? K * (size_t)model_nq(model) * dim : 0;
  return 0;
}

// Whether the call can take these kernels: a model with a product form, float4-aligned operands, room in the workspace.
bool shared_gemm_fits(int model, size_t dim, const void* table, const void* q1, const void* q2, const void* workspace,
                      size_t workspace_bytes, size_t B, size_t K, bool entity, bool norm) {
  if (model != mBetaKL && !is_inner(model)) return false;
  if (dim % 4 != 0 || !aligned16(table) || !aligned16(q1) || (model_nq(model) == 2 && !aligned16(q2))) return false;
  const size_t need = shared_gemm_workspace_floats(model, B, K, dim, entity, norm) * sizeof(float);
  if (need == 0) return true;
  return workspace && aligned16(workspace) && workspace_bytes >= need;
}

static GemmArgs gemm_args(int model, const float* table, size_t n_rows, const long long* ids, const float* q1,
                          const float* q2, const float* gscore, size_t B, size_t K, size_t dim, float gamma, int* err) {
  GemmArgs A{};
  A.rows = table;
  A.ids = ids;
  A.n_rows = n_rows;
  A.q1 = q1;
  A.q2 = q2;
  A.gscore = gscore;
  A.B = (int)B;
  A.K = (int)K;
  A.dim = (int)dim;
  A.nq = model_nq(model);
  A.gamma = gamma;
  A.err = err;
  return A;
}

int shared_gemm_forward(int model, hipStream_t st, const float* table, size_t n_rows, const long long* ids,
                        const float* q1, const float* q2, float* score, size_t B, size_t K, size_t dim,
                        const ScoreParams& p, int* err, float* workspace) {
  GemmArgs A = gemm_args(model, table, n_rows, ids, q1, q2, nullptr, B, K, dim, p.gamma, err);
  A.out1 = score;
  if (model == mBetaKL) {
    float* T = workspace;
    float* Ek = T + K * 2 * dim;
    float* Qk = Ek + K;
    hipLaunchKernelGGL(beta_row_terms_kernel<true>, dim3((unsigned)((K + 3) / 4)), dim3(256), 0, st, table, ids, (int)K,
                       (int)dim, (unsigned long long)n_rows, p, T, Ek, err);
    hipLaunchKernelGGL(beta_query_terms_kernel, dim3((unsigned)((B + 3) / 4)), dim3(256), 0, st, q1, q2, (int)B, (int)dim, Qk);
    A.rows = T;
    A.Ek = Ek;
    A.Qk = Qk;
    launch_gemm<kGemmForward, true>(st, A);
  } else {
    if (p.norm_on) {
      hipLaunchKernelGGL(list_rows_kernel<true>, dim3((unsigned)((K + 3) / 4)), dim3(256), 0, st, table, ids, (int)K,
                         (int)dim, model_nq(model) * (int)dim, (unsigned long long)n_rows, workspace, err);
      A.rows = workspace;
      A.ids = nullptr;
    }
    launch_gemm<kGemmForward, false>(st, A);
  }
  return check_launch("score forward (shared negatives, matrix product)");
}

int shared_gemm_backward_query(int model, hipStream_t st, const float* table, size_t n_rows, const long long* ids,
                               const float* q1, const float* q2, const float* gscore, float* gq1, float* gq2, size_t B,
                               size_t K, size_t dim, const ScoreParams& p, float* workspace) {
  GemmArgs A = gemm_args(model, table, n_rows, ids, q1, q2, gscore, B, K, dim, p.gamma, nullptr);
  A.out1 = gq1;
  A.out2 = gq2;
  if (model == mBetaKL) {
    float* T = workspace;
    hipLaunchKernelGGL(beta_row_terms_kernel<false>, dim3((unsigned)((K + 3) / 4)), dim3(256), 0, st, table, ids, (int)K,
                       (int)dim, (unsigned long long)n_rows, p, T, nullptr, nullptr);
    A.rows = T;
    launch_gemm<kGemmQuery, true>(st, A);
  } else {
    if (p.norm_on) {  // (scaled again rather than kept: the entity side of the previous step has used the workspace since)
      hipLaunchKernelGGL(list_rows_kernel<true>, dim3((unsigned)((K + 3) / 4)), dim3(256), 0, st, table, ids, (int)K,
                         (int)dim, model_nq(model) * (int)dim, (unsigned long long)n_rows, workspace, nullptr);
      A.rows = workspace;
      A.ids = nullptr;
    }
    launch_gemm<kGemmQuery, false>(st, A);
  }
  return check_launch("score backward (query, shared negatives, matrix product)");
}

// R [K][nq dim] (and C [K] for beta_kl) for the entity side; workspace: shared_gemm_workspace_floats(.., true)
int shared_gemm_entity_sums(int model, hipStream_t st, const float* q1, const float* q2, const float* gscore, size_t B,
                            size_t K, size_t dim, float* workspace) {
  GemmArgs A = gemm_args(model, nullptr, 0, nullptr, q1, q2, gscore, B, K, dim, 0.f, nullptr);
  const size_t width = (size_t)model_nq(model) * dim;
  A.out1 = workspace;
  A.out2 = workspace + K * width;
  if (model == mBetaKL) launch_gemm<kGemmEntity, true>(st, A);
  else launch_gemm<kGemmEntity, false>(st, A);
  return check_launch("entity backward (shared negatives, sums as a matrix product)");
}

}  // namespace smx
