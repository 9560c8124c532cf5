// Evaluation against all entities, one or two query rows at a time: a wavefront scores a row at a time, its features spread
// over the lanes, and the table streams past at the rate of memory.  The scan of smx_rank_impl.h, which gives a lane whole
// rows, is bound by latency when one or two of its sixteen query rows are used; this one is bound by instructions beyond
// two.  Scan alone, one query, its first 40 entities as answers, us, this kernel / that one: box 1 M x 400 259 / 270, L1
// 1 M x 100 75 / 79 (78 / 108 with answers all over the table), ComplEx 300 k x 2 x 200 77 / 113, RotatE 300 k x 2 x 250
// 97 / 161; two queries 272 / 280, 116 / 79, 80 / 115, 99 / 163.  That one has the lead below 20 MB of table (L2 15 k x 200
// 20 / 13), with more than 64 answers (this one compares every row with all of them: L1, 500 answers, 293 / 164), and for
// BetaE, whose terms of the row this one evaluates once per query (470 / 460).
// Sums are those of the scoring kernels, a tree over the lanes; keys and scan of a call follow the same rule.
#pragma once
#include "smx_rank_impl.h"

namespace smx {

inline bool rank_streams(int model, unsigned long long n_rows, size_t dim, size_t B, size_t U, size_t A) {
  return model != mBetaKL && B * U <= (model_nq(model) == 1 ? 1 : 2) && A <= 64 && n_rows * dim * model_mul(model) * sizeof(float) >= (20ull << 20);
}

// Keys (and scores) of the answers: one wavefront per (query, answer slot).
template <int M, int VEC, int NIT, bool REG>
__global__ __launch_bounds__(256) void rank_stream_keys_kernel(RankArgs A) {
  constexpr int MUL = model_mul(M);
  const int lane = threadIdx.x & 63;
  const int slot = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (slot >= A.B * A.A) return;
  const int b = slot / A.A, j = slot - b * A.A;
  const int dim = A.ncol * VEC;
  const bool valid = j < A.ans_count[b];
  unsigned long long id = valid ? (unsigned long long)A.ans_id[slot] : 0ull;
  if (id >= A.n_rows) id = 0;  // the host wrapper has already refused such ids
  typename ModelOps<M>::Q q[NIT][VEC];
  float e1[NIT][VEC], e2[NIT][VEC];
  load_entity<VEC, NIT, MUL>(A.table + id * (size_t)dim * MUL, dim, A.ncol, lane, e1, e2);
  unit_row<M, VEC, NIT, REG>(e1, e2, A.ncol, lane);
  float s = 0.f;
  for (int u = 0; u < A.U; ++u) {  // uniform
    load_rank_query<M, VEC, NIT>(A.q1, A.q2, b * A.U + u, dim, A.ncol, lane, q);
    const float su = row_score<M, VEC, NIT, REG>(e1, e2, q, A.ncol, lane, A.p);
    if (u == 0 || union_takes(su, s)) s = su;
  }
  if (lane == 63) {
    if (A.score_out) A.score_out[slot] = valid ? s : 0.f;
    A.key_out[slot] = valid ? rank_key(s, id) : 0ull;  // key 0 sorts last and is never counted
  }
}

// The scan for NB (1 or 2) queries -- or, UNION, for one query with two branch rows: an entity's logit is then the
// maximum over them, and there is one list of answers.  LDS: bins [NL][A + 1], keys [NL][A] with NL = the number of
// answer lists (NB, or 1).
template <int M, int VEC, int NIT, bool REG, int NB, bool UNION = false>
__global__ __launch_bounds__(256) void rank_stream_kernel(RankArgs A) {
  constexpr int NL = UNION ? 1 : NB;
  constexpr int MUL = model_mul(M);
  constexpr int RIF = NIT * MUL <= 2 ? 4 : (NIT * MUL <= 4 ? 2 : 1);
  extern __shared__ unsigned lds_bins[];  // bins [NB][A + 1], then (8-byte aligned) the answers' keys [NB][A]
  const int lane = threadIdx.x & 63;
  const int wave = uniform(threadIdx.x >> 6);
  const int dim = A.ncol * VEC;
  const size_t row_len = (size_t)dim * MUL;
  const int A1 = A.A + 1;
  unsigned long long* lds_keys = reinterpret_cast<unsigned long long*>(lds_bins + ((NL * A1 + 1) & ~1));
  for (int i = threadIdx.x; i < NL * A1; i += 256) lds_bins[i] = 0u;
  for (int i = threadIdx.x; i < NL * A.A; i += 256) {
    const int x = i / A.A, j = i - x * A.A;
    const int b = x;
    lds_keys[i] = j < A.ans_count[b] ? A.ans_key[(size_t)b * A.A + j] : 0ull;
  }
  __syncthreads();

  typename ModelOps<M>::Q q[NB][NIT][VEC];
  int count[NL], qb[NL];
#pragma unroll
  for (int x = 0; x < NL; ++x) {
    qb[x] = x;
    count[x] = min(max(A.ans_count[qb[x]], 0), A.A);  // a count beyond the slots would index past the LDS arrays
  }
#pragma unroll
  for (int x = 0; x < NB; ++x)
    load_rank_query<M, VEC, NIT>(A.q1, A.q2, x, dim, A.ncol, lane, q[x]);
  const int chunks = (A.A + 63) / 64;
  // The first 64 answers' keys stay in registers (most queries have no more); further chunks come from LDS.
  // live[x]: lanes that hold one of them.  my_id[x]: that answer's entity id.
  unsigned long long first_keys[NL], live[NL];
  unsigned my_id[NL];
  // tally[x], lane L: rows so far that beat exactly L of query x's answers (the common cases: L = 0 is
  // every entity ranked below all answers).  Rows that beat 64 or more go to the LDS histogram directly.
  unsigned tally[NL];
#pragma unroll
  for (int x = 0; x < NL; ++x) {
    first_keys[x] = lane < count[x] ? lds_keys[x * A.A + lane] : 0ull;
    live[x] = count[x] >= 64 ? ~0ull : ((1ull << count[x]) - 1ull);
    my_id[x] = (unsigned)~(unsigned)first_keys[x];
    tally[x] = 0u;
  }

  // Wavefronts walk the table together: group g of RIF consecutive rows belongs to wavefront g mod n_waves.
  // Group and row numbers are 32-bit scalars (the host refuses tables of 2^32 - 8 rows or more).  Requests
  // are unconditional -- past the end they repeat the last group -- and rows past the end are scored and
  // then dropped, so that no branch separates a request from the use of the rows requested before it:
  // the counters the compiler waits on then leave the newest RIF loads in flight.
  const unsigned n_waves = gridDim.x * 4u;
  const unsigned wid = blockIdx.x * 4u + (unsigned)wave;
  const unsigned n_rows32 = (unsigned)A.n_rows;
  const unsigned groups = (n_rows32 + RIF - 1) / RIF;
  float ea1[RIF][NIT][VEC], ea2[RIF][NIT][VEC], eb1[RIF][NIT][VEC], eb2[RIF][NIT][VEC];
  auto request = [&](float (&x1)[RIF][NIT][VEC], float (&x2)[RIF][NIT][VEC], unsigned g) {
    g = min(g, groups - 1);
#pragma unroll
    for (int r = 0; r < RIF; ++r) {
      const unsigned row = min(g * RIF + r, n_rows32 - 1);
      load_entity<VEC, NIT, MUL, true>(A.table + row * row_len, dim, A.ncol, lane, x1[r], x2[r]);
    }
  };
  auto consume = [&](const float (&x1)[RIF][NIT][VEC], const float (&x2)[RIF][NIT][VEC], unsigned g) {
#pragma unroll
    for (int r = 0; r < RIF; ++r) {
      const unsigned id = g * RIF + r;  // entity id of the row
      float u1[NIT][VEC], u2[NIT][VEC];  // (the row itself unless the model scales it)
#pragma unroll
      for (int it = 0; it < NIT; ++it)
#pragma unroll
        for (int v = 0; v < VEC; ++v) {
          u1[it][v] = x1[r][it][v];
          u2[it][v] = MUL == 2 ? x2[r][it][v] : 0.f;
        }
      unit_row<M, VEC, NIT, REG>(u1, u2, A.ncol, lane);
#pragma unroll
      for (int x = 0; x < NL; ++x) {
        const float s = row_score<M, VEC, NIT, REG>(u1, u2, q[x], A.ncol, lane, A.p);
        float su = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s), 63));
        if constexpr (UNION) {
#pragma unroll
          for (int u = 1; u < NB; ++u) {
            const float t = row_score<M, VEC, NIT, REG>(u1, u2, q[u], A.ncol, lane, A.p);
            const float tu = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(t), 63));
            if (union_takes(tu, su)) su = tu;
          }
        }
        const unsigned long long key = rank_key(su, id);
        int not_beaten = __popcll(__ballot(!(key > first_keys[x])) & live[x]);
        bool skip = id >= n_rows32 || (__ballot(my_id[x] == id) & live[x]) != 0ull;  // past the end, or an answer
        for (int c = 1; c < chunks; ++c) {
          const int j = c * 64 + lane;
          const bool in_list = j < count[x];
          const unsigned long long ak = in_list ? lds_keys[x * A.A + j] : 0ull;
          not_beaten += __popcll(__ballot(in_list && !(key > ak)));
          skip |= __ballot(in_list && ((unsigned)~(unsigned)ak == id)) != 0ull;
        }
        const int beaten = skip ? -1 : count[x] - not_beaten;  // wave-uniform; -1 matches no lane
        tally[x] += lane == beaten ? 1u : 0u;
        if (beaten >= 64 && lane == 0) atomicAdd(&lds_bins[x * A1 + not_beaten], 1u);
      }
    }
  };
  if (wid < groups) {
    unsigned g = wid;
    request(ea1, ea2, g);
    while (true) {
      // (group numbers stay below 2^30 + 2 * n_waves: no wrap-around)
      request(eb1, eb2, g + n_waves);
      consume(ea1, ea2, g);
      if (g + n_waves >= groups) break;
      request(ea1, ea2, g + 2 * n_waves);
      consume(eb1, eb2, g + n_waves);
      if (g + 2 * n_waves >= groups) break;
      g += 2 * n_waves;
    }
  }
#pragma unroll
  for (int x = 0; x < NL; ++x)
    if (lane <= count[x] && tally[x] != 0u) atomicAdd(&lds_bins[x * A1 + (count[x] - lane)], tally[x]);
  __syncthreads();
#pragma unroll
  for (int x = 0; x < NL; ++x) {
    for (int i = threadIdx.x; i < A1; i += 256) {
      const unsigned v = lds_bins[x * A1 + i];
      if (v) atomicAdd(&A.bins[(size_t)x * A1 + i], v);
    }
  }
}

template <int M, int VEC, int NIT, bool REG>
int launch_rank_stream(hipStream_t st, const RankArgs& A, int mode) {
  if (mode == kRankKeys) {
    hipLaunchKernelGGL((rank_stream_keys_kernel<M, VEC, NIT, REG>), dim3((unsigned)(((size_t)A.B * A.A + 3) / 4)), dim3(256), 0, st, A);
    return check_launch("rank answer keys (streaming form)");
  }
  if (int rc = clear_bins(st, A)) return rc;
  auto launch = [&](auto kernel, int lists) {
    const size_t lds = (((size_t)lists * (A.A + 1) + 1) & ~(size_t)1) * sizeof(unsigned) + (size_t)lists * A.A * sizeof(unsigned long long);
    const unsigned long long want = (A.n_rows + 15) / 16, most = resident_workgroups(kernel, 256, lds);
    hipLaunchKernelGGL(kernel, dim3((unsigned)(want < most ? want : most)), dim3(256), lds, st, A);
  };
  if (A.U == 2) launch(rank_stream_kernel<M, VEC, NIT, REG, 2, true>, 1);
  else if (A.B == 2) launch(rank_stream_kernel<M, VEC, NIT, REG, 2>, 2);
  else launch(rank_stream_kernel<M, VEC, NIT, REG, 1>, 1);
  if (int rc = check_launch("rank scan (streaming form)")) return rc;
  return finish_ranks(st, A);
}

template <int M>
int rank_stream_dispatch(hipStream_t st, const RankArgs& A, int vec, int nit, int mode) {
  return with_row_shape<M>(A, vec, nit, [&](auto vec_tag, auto nit_tag, auto reg_tag) {
    return launch_rank_stream<M, decltype(vec_tag)::value, decltype(nit_tag)::value, decltype(reg_tag)::value>(st, A, mode);
  });
}

}  // namespace smx
