// Gather-fused scoring, forward and query-side backward (fp32).
//
// Replaces, in one pass each, the sequence the reference runs per training
// step for the negative samples (smore/models/kg_reasoning.py:301-307,349-355):
//   rows = table[idx]                      smore/common/embedding/embed_rw.py:74-75
//   [optional clamp(rows + 1, .05, 1e9)]   smore/common/modules.py:29-36
//   d = dist(rows, query)                  smore/common/torchext/common_kernel.h:33-56
//   logit = gamma - d                      custom_cal_logit of smore/models/*.py
// and, backward, the query-gradient kernel common_kernel.h:92-123.  The
// [B,K,D] gathered tensor is never materialised: a wavefront reads each entity
// row straight from the table with 16-byte loads (one float4 column per lane).
//
// Work split.  forward: workgroup = (query b, tile of negatives); the query
// row(s) are staged once in LDS, every lane then keeps the features it owns in
// registers for the whole tile; each of the four wavefronts streams its
// quarter of the tile's rows, two batches of rows in flight at a time.  backward: one workgroup per
// query walks all K negatives, wavefront partial sums are combined through LDS
// in wavefront order, so the gradient has a fixed summation order.
#pragma once
#include "smx_common.h"
#include "smx_models.h"
#include "smx_rowupdate.h"
#include "smx_slab.h"
#include "smx_wave.h"

namespace smx {

struct ScoreArgs {
  const float* table;
  const long long* idx;  // null: `table` holds the B*K rows in pair order
  const float* q1;
  const float* q2;
  float* score_out;      // forward
  const float* score;    // backward: the logits the forward wrote
  const float* gscore;
  float* gq1;
  float* gq2;
  int B, K, ncol;
  int ids_shared;        // idx holds K ids that every query scores (--share_negative, online_sampler.py:155-157), not B*K
  // Union queries (kg_reasoning.py:326, box.py:163): q1 / q2 hold U branch rows per query, [B*U, dim]; a kernel's
  // "query" is then one branch row, number bq = b * U + u, which scores the ids of query b.
  int U;                 // branches per query (1: none of this)
  bool stream_rows;      // one-pair segments are finished in the stream of the rows (beta_rows_in_stream)
  const unsigned char* winner;  // query backward, [B, K]: the branch that gave the pair's logit; a branch row sums its own pairs only
  unsigned long long n_rows;
  ScoreParams p;
  int* err;
  const int* pair_seg;   // one-pair segments finished by the query backward (SINGLES kernels)
  const long long* uniq; // plan's id list: row of a one-pair segment when the kernel runs without the id tensor (GQ = false)
  unsigned char* codes;  // [B*K][NIT*64] sign codes written by this kernel (forward or query backward), or null
  const unsigned char* codes_in;  // query backward: codes the forward left; the entity rows are then not read
  RowSink sink;
};

// BetaE with Adam in place: the query-gradient kernel finishes the rows that occur once.  It is bound by the special functions
// (VALU 95 % busy, the rows at 2.8 TB/s) and the entity pass by the rows' w, m and v, one after the other; here the first hides
// behind the second, a row is read once for both, and psi' costs no special function beyond those of psi.  512 x 512 pairs,
// 2 x 400 floats, 1 M entities, 201 k of 230 k rows occur once: query gradient 299 + entity pass 1001 us -> 849 + 186; 300 x 512
// 1.04 ms a step against 1.31 before (its 300 workgroups take two turns of the 256 CUs), 128 x 1024 0.98 / 1.14, D = 200
// 0.73 / 0.98.  Merged rows, v per row and other optimizers take the entity pass as before.
inline bool beta_rows_in_stream(int model, const RowSink& sink, int vec, int nit) {
  return model == mBetaKL && vec == 4 && nit <= 2 && sink.adam_on == kOptAdam && !sink.squeeze && !sink.merged;
}

template <int VEC> struct Pack {
  float v[VEC];
};

template <int VEC>
__device__ __forceinline__ Pack<VEC> load_pack(const float* __restrict__ base, int col) {
  Pack<VEC> r;
  if constexpr (VEC == 4) {
    const float4 t = reinterpret_cast<const float4*>(base)[col];
    r.v[0] = t.x;
    r.v[1] = t.y;
    r.v[2] = t.z;
    r.v[3] = t.w;
  } else {
    r.v[0] = base[col];
  }
  return r;
}

// Loads the features a lane owns of the staged query into registers.
template <int M, int VEC, int NIT, bool FWD>
__device__ __forceinline__ void load_query_regs(const float* lds, int dim, int ncol, int lane,
                                                typename ModelOps<M>::Q (&q)[NIT][VEC]) {
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int c = lane + 64 * it;
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      const int cc = min(c, ncol - 1);  // lanes past the row end hold a copy of the last column
      const float a = lds[cc * VEC + v];
      const float b = model_nq(M) == 2 ? lds[dim + cc * VEC + v] : 0.f;
      q[it][v] = FWD ? prep_forward<M>(a, b) : prep_backward_query<M>(a, b);
    }
  }
}

template <int M>
__device__ __forceinline__ void stage_query(float* lds, const float* __restrict__ q1, const float* __restrict__ q2,
                                            size_t b, int dim) {
  for (int d = threadIdx.x; d < dim; d += blockDim.x) {
    lds[d] = q1[b * dim + d];
    if (model_nq(M) == 2) lds[dim + d] = q2[b * dim + d];
  }
  __syncthreads();
}

// BetaE's per-query values in LDS, one stretch of dim floats per field, evaluated once per workgroup.  FWD: a, b, k of QBeta, and
// l, m where a lane reads columns of four; a lane that takes single floats forms them again, two multiply-adds in the place of two
// reads with their addresses and a wait (2 x 400 floats, 512 x 512 pairs: 291 -> 286 us).  Query backward: k, l and, where rows are
// finished (ROWS), a, b.
__host__ __device__ constexpr int query_fields(int model, int vec, bool fwd, bool rows = false) {
  return model != mBetaKL ? model_nq(model) : (fwd ? (vec == 1 ? 3 : 5) : (rows ? 4 : 2));
}
template <int VEC, bool FWD, bool ROWS = false>
__device__ __forceinline__ void stage_beta_query(float* lds, const float* __restrict__ q1, const float* __restrict__ q2,
                                                 size_t b, int dim) {
  for (int d = threadIdx.x; d < dim; d += blockDim.x) {
    const float x = q1[b * dim + d], y = q2[b * dim + d];
    const QBeta q = FWD ? prep_forward<mBetaKL>(x, y) : prep_backward_query<mBetaKL>(x, y);
    if constexpr (FWD) {
      lds[d] = q.a;
      lds[dim + d] = q.b;
      lds[2 * dim + d] = q.k;
      if constexpr (VEC != 1) {
        lds[3 * dim + d] = q.l;
        lds[4 * dim + d] = q.m;
      }
    } else {
      lds[d] = q.k;
      lds[dim + d] = q.l;
      if constexpr (ROWS) {
        lds[2 * dim + d] = q.a;
        lds[3 * dim + d] = q.b;
      }
    }
  }
  __syncthreads();
}
template <int VEC>
__device__ __forceinline__ void lds_pack(const float* lds, int col, float (&x)[VEC]) {
  if constexpr (VEC == 4) {
    typedef float vec4 __attribute__((ext_vector_type(4)));
    const vec4 t = reinterpret_cast<const vec4*>(lds)[col];
    x[0] = t.x;
    x[1] = t.y;
    x[2] = t.z;
    x[3] = t.w;
  } else {
    x[0] = lds[col];
  }
}
template <int VEC, bool FWD, bool ROWS = false>
__device__ __forceinline__ void beta_query(const float* lds, int dim, int col, QBeta (&q)[VEC]) {
  float f[5][VEC];
#pragma unroll
  for (int i = 0; i < query_fields(mBetaKL, VEC, FWD, ROWS); ++i) lds_pack<VEC>(lds + i * dim, col, f[i]);
  if constexpr (FWD && VEC == 1) {
    f[3][0] = beta_k(f[0][0]);
    f[4][0] = beta_k(f[1][0]);
  }
#pragma unroll
  for (int v = 0; v < VEC; ++v)
    q[v] = FWD ? QBeta{f[0][v], f[1][v], f[2][v], f[3][v], f[4][v]}
               : QBeta{ROWS ? f[2][v] : 0.f, ROWS ? f[3][v] : 0.f, f[0][v], f[1][v], 0.f};
}

// ---- streaming the rows of up to 64 pairs through a wavefront -----------------------------------
// The lanes first fetch, in one coalesced load, the ids of the pairs the wavefront is about to
// process (pair j of the batch lives in lane j), turn them into row addresses and park them, with the
// pair's two gradient coefficients in the backward kernel, in a 64-entry slab of LDS that belongs to
// the wavefront.  The row loop then finds a row with one LDS read at a uniform address (a broadcast,
// no bank conflicts) instead of v_readlane + scalar address arithmetic per row: the loop is bound by
// instruction issue, and every vector or scalar instruction it does not need is time.  Rows are
// requested RIF at a time into two register sets used in turn: while set A is consumed, set B is
// already on its way.  All loads are unconditional so that they issue as one batch and stay in
// flight together: entries past the batch's end repeat its last pair.

struct PairBatch {
  unsigned off_lo, off_hi;  // this lane's pair: offset of its entity row in floats
  unsigned row;             // ... and the row number (low 32 bits)
};

__device__ __forceinline__ PairBatch load_pair_batch(const long long* __restrict__ idx, size_t first_pair, int cnt,
                                                     int lane, size_t row_len, unsigned long long n_rows, int& bad) {
  const size_t pair = first_pair + min(lane, cnt - 1);
  long long row = idx ? idx[pair] : (long long)pair;
  if ((unsigned long long)row >= n_rows) {  // id outside the table: remember it, read row 0 instead
    bad = 1;
    row = 0;
  }
  const unsigned long long off = (unsigned long long)row * row_len;
  return {(unsigned)off, (unsigned)(off >> 32), (unsigned)row};
}

__device__ __forceinline__ unsigned long long batch_off(const PairBatch& pb, int j) {
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)pb.off_lo, j);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)pb.off_hi, j);
  return ((unsigned long long)hi << 32) | lo;
}

constexpr int kSlabDwords = kSlabEntries * 4;  // per wavefront: 64 entries of {address lo, address hi, c0, c1}

// Orders a wavefront's own LDS writes before its later LDS reads (other lanes' entries).
__device__ __forceinline__ void slab_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ void stage_pairs(unsigned* slab, int lane, const float* __restrict__ table,
                                            const PairBatch& pb, float c0, float c1) {
  slab_fence();  // reads of the previous batch are done
  const unsigned long long addr =
      (unsigned long long)(table + (((unsigned long long)pb.off_hi << 32) | pb.off_lo));
  *reinterpret_cast<uint4*>(slab + 4 * lane) =
      make_uint4((unsigned)addr, (unsigned)(addr >> 32), __float_as_uint(c0), __float_as_uint(c1));
  slab_fence();
}

// The address comes back from LDS as an integer; the pointer made from it is declared global so that
// the row loads are global_load (a generic pointer would make them flat_load, which also counts
// against the LDS wait counter).
typedef const __attribute__((address_space(1))) float* GlobalRow;
__device__ __forceinline__ GlobalRow slab_row(const unsigned* slab, int j) {
  const uint2 a = *reinterpret_cast<const uint2*>(slab + 4 * j);
  return reinterpret_cast<GlobalRow>(((unsigned long long)a.y << 32) | a.x);
}
// ONCE: past the caches (read_once)
template <int VEC, bool ONCE = false>
__device__ __forceinline__ Pack<VEC> load_pack(GlobalRow base, int col) {
  Pack<VEC> r;
  if constexpr (VEC == 4) {
    typedef float vec4 __attribute__((ext_vector_type(4)));
    const __attribute__((address_space(1))) vec4* p = reinterpret_cast<const __attribute__((address_space(1))) vec4*>(base) + col;
    const vec4 t = ONCE ? __builtin_nontemporal_load(p) : *p;
    r.v[0] = t.x;
    r.v[1] = t.y;
    r.v[2] = t.z;
    r.v[3] = t.w;
  } else {
    r.v[0] = base[col];
  }
  return r;
}
__device__ __forceinline__ float2 slab_coef(const unsigned* slab, int j) {
  return *reinterpret_cast<const float2*>(slab + 4 * j + 2);
}

template <int MUL, int VEC, int NIT, int RIF> struct RowSet {
  Pack<VEC> e1[RIF][NIT];
  Pack<VEC> e2[RIF][NIT];
};

// Requests rows g0 .. g0+RIF-1 of the batch, g0 a multiple of RIF: the entries exist (last_group).
template <int MUL, int VEC, int NIT, int RIF, bool ONCE = false>
__device__ __forceinline__ void request_rows(RowSet<MUL, VEC, NIT, RIF>& rs, const unsigned* slab, int g0, int dim,
                                             int ncol, int lane) {
  GlobalRow pe[RIF];
#pragma unroll
  for (int r = 0; r < RIF; ++r) pe[r] = slab_row(slab, g0 + r);
#pragma unroll
  for (int r = 0; r < RIF; ++r) {
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int c = min(lane + 64 * it, ncol - 1);
      rs.e1[r][it] = load_pack<VEC, ONCE>(pe[r], c);
      if (MUL == 2) rs.e2[r][it] = load_pack<VEC, ONCE>(pe[r] + dim, c);
    }
    // Rows are used in the order r = 0, 1, ..: their loads must be issued in that order everywhere (the
    // scheduler is otherwise free to reverse them in the loop prologue), or the wait for row 0 at the top
    // of the streaming loop becomes a wait for every load in flight.
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Streams the first cnt (1 .. 64) rows of a staged batch through `consume(j, e1, e2)`, j ascending.  `slab` is the start of the
// wavefront's own: every group has to lie in it (last_group).
template <int MUL, int VEC, int NIT, int RIF, bool ONCE = false, class Consume>
__device__ __forceinline__ void stream_batch(const unsigned* slab, int cnt, int dim, int ncol, int lane,
                                             Consume&& consume) {
  static_assert(kSlabEntries % RIF == 0, "a group of rows must not straddle the end of the slab");
  RowSet<MUL, VEC, NIT, RIF> a, b;
  const int last = last_group(cnt, RIF);
  request_rows<MUL, VEC, NIT, RIF, ONCE>(a, slab, 0, dim, ncol, lane);
  for (int j0 = 0; j0 < cnt; j0 += 2 * RIF) {
    request_rows<MUL, VEC, NIT, RIF, ONCE>(b, slab, min(j0 + RIF, last), dim, ncol, lane);
#pragma unroll
    for (int r = 0; r < RIF; ++r)
      if (j0 + r < cnt) consume(j0 + r, a.e1[r], a.e2[r]);
    request_rows<MUL, VEC, NIT, RIF, ONCE>(a, slab, min(j0 + 2 * RIF, last), dim, ncol, lane);
#pragma unroll
    for (int r = 0; r < RIF; ++r)
      if (j0 + RIF + r < cnt) consume(j0 + RIF + r, b.e1[r], b.e2[r]);
  }
}

// Sign codes on their way to memory: a wavefront parks each pair's NIT x 64 code bytes in its LDS
// stage and, every 16 pairs (and after the last one), writes the stage out with 16-byte stores -- the
// 16 pairs are contiguous in the code array as well.
constexpr int kStagePairs = 16;
template <int NIT>
__device__ __forceinline__ void flush_codes(const unsigned char* stage, unsigned char* codes, size_t first_pair, int j,
                                            int cnt, int lane) {
  if ((j & (kStagePairs - 1)) == kStagePairs - 1 || j == cnt - 1) {
    slab_fence();
    typedef unsigned vec4u __attribute__((ext_vector_type(4)));
    const int rows_here = (j & (kStagePairs - 1)) + 1;
    vec4u* out = reinterpret_cast<vec4u*>(codes + (first_pair + (j & ~(kStagePairs - 1))) * (size_t)(NIT * 64));
#pragma unroll
    for (int i = 0; i < NIT; ++i) {
      const int chunk = lane + 64 * i;
      if (chunk * 16 < rows_here * NIT * 64)
        __builtin_nontemporal_store(reinterpret_cast<const vec4u*>(stage)[chunk], out + chunk);
    }
    slab_fence();
  }
}

// Wavefronts per SIMD the compiler has to leave registers for: four where BetaE is bound by its arithmetic (with three, 2 x 400
// floats: forward 415 instead of 405 us, query gradient 354 instead of 330; seven floats a lane do not fit the query gradient's
// 128 registers: spills, 381 us instead of 299).
constexpr int arithmetic_waves(int model, int floats_per_lane, bool fwd) {
  return model == mBetaKL && floats_per_lane <= 8 && (fwd || floats_per_lane != 7) ? 4 : 1;
}

// DEDUP: a workgroup scores each DISTINCT entity among the (up to 256) pairs of its tile once.  With skewed ids a
// query's negatives repeat the hot entities many times (Zipf 1.1: ~175 distinct among 256 consecutive negatives,
// ~51 among 64), every repeat costs the same instructions as the first occurrence although its row comes from
// the cache, and at such shapes the kernel is bound by instruction issue.  The lanes enter their ids into a small
// hash table in LDS; the first pair of the tile with an id puts its row on the tile's list of representatives; the
// list (in pair order) is dealt out to the four wavefronts in equal parts and streamed; every pair then takes its
// score (and its code bytes, from the tile's LDS stage) from its representative: the same bits as without
// de-duplication, pair by pair.
constexpr int kDedupSlots = 512;   // hash table entries for the 256 ids of a tile
constexpr unsigned kDedupEmpty = 0xffffffffu;  // (no id: the table has at most 2^32 - 1 rows)
// LDS bytes of the de-duplication tables: ids, first pairs and list positions of the slots, row addresses and
// scores of the list, representatives per wavefront
constexpr size_t kDedupLds = kDedupSlots * 12 + 256 * 8 + 256 * 4 + 16;

// ONCE (with DEDUP): tiles of different ids load their rows past the caches (read_once).  A kernel of its own, as the second
// loop costs the first 8 to 28 registers.
template <int M, int VEC, int NIT, int RIF, bool REG, bool CODED = false, bool DEDUP = false, bool ONCE = false>
__global__ __launch_bounds__(256, arithmetic_waves(M, VEC * NIT, true)) void score_forward_kernel(ScoreArgs A, int tiles, int tile_k) {
  const float* __restrict__ table = A.table;
  const long long* __restrict__ idx = A.idx;
  const float* __restrict__ q1 = A.q1;
  const float* __restrict__ q2 = A.q2;
  float* __restrict__ score = A.score_out;
  const int K = A.K, ncol = A.ncol;
  const unsigned long long n_rows = A.n_rows;
  const ScoreParams p = A.p;
  int* err = A.err;
  constexpr int MUL = model_mul(M);
  extern __shared__ float lds[];
  const int b = blockIdx.x / tiles;
  const int tile = blockIdx.x - b * tiles;
  const int lane = threadIdx.x & 63;
  const int wave = uniform(threadIdx.x >> 6);
  const int dim = ncol * VEC;
  const size_t row_len = (size_t)dim * MUL;

  // this wavefront's share of the tile: per_wave (<= 64) consecutive negatives
  const int per_wave = tile_k / 4;
  const int kw0 = tile * tile_k + wave * per_wave;
  const int cnt = min(per_wave, K - kw0);
  int bad = 0;
  PairBatch pb{0u, 0u};
  if (cnt > 0)
    pb = load_pair_batch(idx, (A.ids_shared ? (size_t)0 : (size_t)(b / A.U) * K) + kw0, cnt, lane, row_len, n_rows, bad);

  // LDS: query | per-wavefront pair slabs | code stage (per wavefront; one for the tile with DEDUP) | DEDUP tables
  constexpr int QF = query_fields(M, VEC, true);
  unsigned* slab = reinterpret_cast<unsigned*>(lds + QF * dim) + wave * kSlabDwords;
  constexpr int kStaged = DEDUP ? 256 : kStagePairs;  // pairs whose code bytes a stage holds (DEDUP: tile_k, at most that)
  unsigned char* stage_base = reinterpret_cast<unsigned char*>(lds + QF * dim + 4 * kSlabDwords);
  unsigned char* stage = DEDUP ? stage_base : stage_base + wave * (kStaged * NIT * 64);
  unsigned char* after_stage = stage_base + (CODED ? (size_t)(DEDUP ? tile_k : 4 * kStaged) * NIT * 64 : 0);
  unsigned* slot_id = reinterpret_cast<unsigned*>(after_stage);                   // [kDedupSlots]
  int* slot_pos = reinterpret_cast<int*>(slot_id + kDedupSlots);                   // [kDedupSlots]
  uint2* rep_addr = reinterpret_cast<uint2*>(slot_pos + kDedupSlots);              // [256]
  float* rep_score = reinterpret_cast<float*>(rep_addr + 256);                     // [256]
  int* slot_first = reinterpret_cast<int*>(rep_score + 256);                        // [kDedupSlots]
  int* wave_reps = slot_first + kDedupSlots;                                        // [4]
  if constexpr (DEDUP) {
    for (int i = threadIdx.x; i < kDedupSlots; i += 256) {
      slot_id[i] = kDedupEmpty;
      slot_first[i] = 0x7fffffff;
    }
  }

  // (either ends with a barrier: the tables are cleared)
  [[maybe_unused]] typename ModelOps<M>::Q q[NIT][VEC];
  if constexpr (M == mBetaKL) {
    stage_beta_query<VEC, true>(lds, q1, q2, b, dim);
  } else {
    stage_query<M>(lds, q1, q2, b, dim);
    load_query_regs<M, VEC, NIT, true>(lds, dim, ncol, lane, q);
  }
  if constexpr (!DEDUP) {
    if (cnt <= 0) return;
  }
  int n_stream = cnt;        // rows this wavefront streams
  int first_rep = 0;         // DEDUP: position on the tile's list of the first of them
  int my_pos = lane;         // DEDUP: position on the list of the row my pair's score comes from
  [[maybe_unused]] bool once = false;   // ONCE: the tile's ids are all different
  if constexpr (DEDUP) {
    // The representative of an id is its first pair of the tile, and the list holds the representatives in pair
    // order: which wavefront scores which row is then the same in every run (a row's bits may depend on where it
    // stands in a wavefront's stream, through the contraction of multiply-adds in the unrolled row loop).
    const int pair_in_tile = wave * per_wave + lane;
    unsigned s = 0;
    if (lane < cnt) {
      const unsigned key = pb.row;
      s = (key * 2654435761u) >> 23;  // 9 bits
      while (true) {
        const unsigned old = atomicCAS(&slot_id[s], kDedupEmpty, key);
        if (old == kDedupEmpty || old == key) break;
        s = (s + 1) & (kDedupSlots - 1);
      }
      atomicMin(&slot_first[s], pair_in_tile);
    }
    __syncthreads();
    const bool is_rep = lane < cnt && slot_first[s] == pair_in_tile;
    const unsigned long long reps = __ballot(is_rep);
    if (lane == 0) wave_reps[wave] = __popcll(reps);
    __syncthreads();
    int before = 0, n_reps = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const int c = wave_reps[w];
      before += w < wave ? c : 0;
      n_reps += c;
    }
    if (is_rep) {
      const int pos = before + (int)lanes_below_in(reps);
      slot_pos[s] = pos;
      const unsigned long long addr =
          (unsigned long long)(table + (((unsigned long long)pb.off_hi << 32) | pb.off_lo));
      rep_addr[pos] = make_uint2((unsigned)addr, (unsigned)(addr >> 32));
    }
    __syncthreads();
    if (lane < cnt) my_pos = slot_pos[s];
    if constexpr (ONCE) once = n_reps == min(tile_k, K - tile * tile_k);
    const int share = (n_reps + 3) / 4;  // <= 64
    first_rep = wave * share;
    n_stream = max(0, min(share, n_reps - first_rep));
    // this wavefront's part of the list goes into its slab (entries past its end repeat the last: the row loop's
    // loads are unconditional)
    if (n_stream > 0) {
      *reinterpret_cast<uint2*>(slab + 4 * lane) = rep_addr[first_rep + min(lane, n_stream - 1)];
      slab_fence();
    }
  } else {
    stage_pairs(slab, lane, table, pb, 0.f, 0.f);
  }

  [[maybe_unused]] const BetaClamp clamp(p);
  float neg_thr[NIT][VEC];
  if constexpr (CODED) {
#pragma unroll
    for (int it = 0; it < NIT; ++it)
#pragma unroll
      for (int v = 0; v < VEC; ++v) neg_thr[it][v] = ModelOps<M>::neg_threshold(q[it][v]);
  }
  float* out = score + (size_t)b * K + kw0;
  auto take = [&](int j, const Pack<VEC>(&e1)[NIT], const Pack<VEC>(&e2)[NIT]) __attribute__((always_inline)) {
    // lanes past the row end hold a copy of the last column: they compute along and are dropped here.
    if constexpr (model_norm(M, REG)) {
      // unit-length halves: the two inner products and the two squared lengths are summed separately
      float dot1 = 0.f, dot2 = 0.f, sq1 = 0.f, sq2 = 0.f;
#pragma unroll
      for (int it = 0; it < NIT; ++it) {
        float a = 0.f, b2 = 0.f, c = 0.f, d = 0.f;
#pragma unroll
        for (int v = 0; v < VEC; ++v) {
          a = __builtin_fmaf(e1[it].v[v], q[it][v].a, a);
          c = __builtin_fmaf(e1[it].v[v], e1[it].v[v], c);
          if constexpr (MUL == 2) {
            b2 = __builtin_fmaf(e2[it].v[v], q[it][v].b, b2);
            d = __builtin_fmaf(e2[it].v[v], e2[it].v[v], d);
          }
        }
        const bool in = lane + 64 * it < ncol;
        dot1 += in ? a : 0.f;
        dot2 += in ? b2 : 0.f;
        sq1 += in ? c : 0.f;
        sq2 += in ? d : 0.f;
      }
      dot1 = wave_sum_last_f32(dot1);
      sq1 = wave_sum_last_f32(sq1);
      float s = dot1 * inv_norm(sq1);
      if constexpr (MUL == 2) {
        dot2 = wave_sum_last_f32(dot2);
        sq2 = wave_sum_last_f32(sq2);
        s += dot2 * inv_norm(sq2);
      }
      s += p.gamma;
      if constexpr (DEDUP) {
        if (lane == 63) rep_score[first_rep + j] = s;
      } else {
        if (lane == 63) out[j] = s;
      }
      return;
    }
    // The logit is linear in the accumulators: fold them per lane, reduce once.
    float mine = 0.f;
    if constexpr (M == mBetaKL) {
      asm volatile("" ::: "memory");   // the query's values are read again for every row, see beta_row_sum
      mine = beta_row_sum<VEC, NIT, REG>(
          clamp, [&](int it, int v) { return e1[it].v[v]; }, [&](int it, int v) { return e2[it].v[v]; },
          [&](int it, QBeta (&to)[VEC]) { beta_query<VEC, true>(lds, dim, min(lane + 64 * it, ncol - 1), to); }, ncol, lane);
    } else
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      float a0 = 0.f, a1 = 0.f;
      if constexpr (CODED) {
        unsigned code = 0;
#pragma unroll
        for (int v = 0; v < VEC; ++v) ModelOps<M>::fwd_coded(e1[it].v[v], q[it][v], neg_thr[it][v], a0, a1, code);
        stage[((DEDUP ? first_rep + j : j) & (kStaged - 1)) * (NIT * 64) + 64 * it + lane] = (unsigned char)code;
      } else {
#pragma unroll
        for (int v = 0; v < VEC; ++v) {
          const float x1 = REG ? reg_apply(e1[it].v[v], p) : e1[it].v[v];
          const float x2 = MUL == 2 ? (REG ? reg_apply(e2[it].v[v], p) : e2[it].v[v]) : 0.f;
          ModelOps<M>::fwd(x1, x2, q[it][v], a0, a1);
        }
      }
      const float f = ModelOps<M>::fold(a0, a1, p);
      mine += lane + 64 * it < ncol ? f : 0.f;
    }
    const float folded = wave_sum_last_f32(mine);
    if constexpr (DEDUP) {
      if (lane == 63) rep_score[first_rep + j] = ModelOps<M>::score(folded, p);
    } else {
      if (lane == 63) out[j] = ModelOps<M>::score(folded, p);
      if constexpr (CODED) flush_codes<NIT>(stage, A.codes, (size_t)b * K + kw0, j, cnt, lane);
    }
  };
  if (n_stream > 0) {
    if (ONCE && once)
      stream_batch<MUL, VEC, NIT, RIF, ONCE>(slab, n_stream, dim, ncol, lane, take);
    else
      stream_batch<MUL, VEC, NIT, RIF>(slab, n_stream, dim, ncol, lane, take);
  }
  if constexpr (DEDUP) {
    // every pair takes what its representative produced: the score from the tile's list ...
    __syncthreads();
    if (lane < cnt) out[lane] = rep_score[my_pos];
    if constexpr (CODED) {
      // ... and its NIT x 64 code bytes from the representative's row of the stage, 16 bytes per lane and turn;
      // the wavefront's pairs are contiguous in the code array
      if (cnt > 0) {
        typedef unsigned vec4u __attribute__((ext_vector_type(4)));
        constexpr int kPer = NIT * 4;  // 16-byte pieces per pair
        vec4u* dst = reinterpret_cast<vec4u*>(A.codes + ((size_t)b * K + kw0) * (size_t)(NIT * 64));
        for (int c0 = 0; c0 < cnt * kPer; c0 += 64) {
          const int c = c0 + lane;
          const int pair = min(c / kPer, cnt - 1);
          const int src_row = __shfl(my_pos, pair);
          if (c < cnt * kPer)
            __builtin_nontemporal_store(reinterpret_cast<const vec4u*>(stage + src_row * (NIT * 64))[c % kPer], dst + c);
        }
      }
    }
  }
  if (__ballot(bad != 0) != 0ull && err && lane == 0) *err = 1;
}

// SINGLES: the plan marks pairs whose entity occurs once in the step.  Such a segment needs no
// reduction, and this kernel already holds the pair's query in registers and has just read its entity
// row, so it finishes the row here (merged-gradient row and/or Adam on w, m, v) instead of leaving it
// to the entity pass, which would have to fetch the query rows and the entity row again.
// SINGLES: 0 = leave every segment to the entity pass, 1 = finish one-pair segments here as merged-gradient
// rows, 2 = ... with an optimizer on w, m, v (and the merged row if asked for), 3 = ... with Adam, in the stream of the rows
// (BetaE, rows of up to 512 floats a half).
// CODES (models with sign codes): 1 = also writes every pair's derivative decisions, one byte per lane
// and column group, for the entity pass to use in place of the query rows; 2 = the forward pass left
// the codes: the query gradient is summed from them and the entity rows are not read at all (except
// those of the one-pair segments finished here).
// GQ = false: only the one-pair segments are finished (optimizer on w, m, v); no query gradient, no
// other pair is touched.  The pairs' rows then come from the plan (uniq[segment]), not from the id tensor:
// this is the half of the work that smx_score_backward_entity hands to this kernel when the query
// gradients were taken earlier (autograd's backward) and the update comes later (apply_grad).
template <int M, int VEC, int NIT, int RIF, int NW, bool REG, int SINGLES, int CODES = 0, bool GQ = true>
__global__ __launch_bounds__(NW * 64, SINGLES == 0 ? arithmetic_waves(M, VEC * NIT, false) : 1) void score_backward_query_kernel(ScoreArgs A) {
  static_assert(GQ || (SINGLES == 2 && CODES == 0), "the one-pair-only form exists with an optimizer");
  const float* __restrict__ table = A.table;
  const long long* __restrict__ idx = A.idx;
  const float* __restrict__ q1 = A.q1;
  const float* __restrict__ q2 = A.q2;
  const float* __restrict__ score = A.score;
  const float* __restrict__ gscore = A.gscore;
  float* __restrict__ gq1 = A.gq1;
  float* __restrict__ gq2 = A.gq2;
  const int K = A.K, ncol = A.ncol;
  const unsigned long long n_rows = A.n_rows;
  const ScoreParams p = A.p;
  constexpr int MUL = model_mul(M);
  constexpr int NQ = model_nq(M);
  constexpr int QF = query_fields(M, VEC, false, SINGLES == 3);
  extern __shared__ float lds[];
  // Queries are taken last to first: the forward walks them first to last, and what it touched last -- the sign
  // codes it wrote, the rows it read -- is what the memory-side cache still holds when this kernel starts
  // (86 M x 200 box workload: backward 0.92 -> 0.91 ms; the kernel by itself, with nothing of a forward left in
  // that cache, takes 0.71 ms instead of 0.63).
  const int b = (int)(gridDim.x - 1u - blockIdx.x);
  const int lane = threadIdx.x & 63;
  const int wave = uniform(threadIdx.x >> 6);
  const int dim = ncol * VEC;
  const size_t row_len = (size_t)dim * MUL;

  [[maybe_unused]] typename ModelOps<M>::Q q[NIT][VEC];
  if constexpr (M == mBetaKL) {
    stage_beta_query<VEC, false, SINGLES != 0>(lds, q1, q2, b, dim);
  } else {
    stage_query<M>(lds, q1, q2, b, dim);
    load_query_regs<M, VEC, NIT, false>(lds, dim, ncol, lane, q);
  }

  [[maybe_unused]] const BetaClamp clamp(p);
  float g1[NIT][VEC], g2[NIT][VEC];
  [[maybe_unused]] float neg_thr[NIT][VEC];  // sign-coded models, when this kernel makes the comparisons itself
#pragma unroll
  for (int it = 0; it < NIT; ++it)
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      g1[it][v] = g2[it][v] = 0.f;
      if constexpr (model_coded(M)) neg_thr[it][v] = ModelOps<M>::neg_threshold(q[it][v]);
    }
  // LDS: query | per-wavefront partial sums | per-wavefront pair slabs
  unsigned* slab = reinterpret_cast<unsigned*>(lds + (NW * NQ + QF) * dim) + wave * kSlabDwords;
  unsigned char* stage =
      reinterpret_cast<unsigned char*>(lds + (NW * NQ + QF) * dim + NW * kSlabDwords) + wave * (kStagePairs * NIT * 64);

  // BetaE: the query's features of a column group for the rows finished here.  They stand behind k and l (SINGLES 1 and 2: where the
  // partial sums go once every wavefront is done with them).  Fetched from memory for each row instead: 4096 x 128 pairs of 2 x 400
  // floats 1457 us against 1450 with merged rows, 2341 against 2330 with Adam and v per row.
  [[maybe_unused]] auto query_features = [&](int it, QBeta (&to)[VEC]) {
    float fa[VEC], fb[VEC];
    const int col = min(lane + 64 * it, ncol - 1);
    lds_pack<VEC>(lds + 2 * dim, col, fa);
    lds_pack<VEC>(lds + 3 * dim, col, fb);
#pragma unroll
    for (int v = 0; v < VEC; ++v) to[v] = QBeta{fa[v], fb[v], 0.f, 0.f, 0.f};
  };
  [[maybe_unused]] QBeta qf[VEC];
  // this wavefront's share of the query's negatives: a contiguous range, walked in batches of 64
  const int per_wave = (K + NW - 1) / NW;
  const int kw0 = wave * per_wave;
  const int kw1 = min(K, kw0 + per_wave);
  int bad = 0;
  for (int kb = kw0; kb < kw1; kb += 64) {
    const int cnt = min(64, kw1 - kb);
    const size_t first = (size_t)(b / A.U) * K + kb;  // pairs belong to queries, a union's branch rows share them
    const size_t mine = first + min(lane, cnt - 1);
    int my_ps = 0;
    unsigned long long singles = 0ull;  // pairs of the batch that are a segment of their own
    if constexpr (SINGLES != 0) {
      my_ps = A.pair_seg[mine];
      singles = __ballot(lane < cnt && my_ps < 0);
    }
    PairBatch pb;
    if constexpr (GQ) {
      pb = load_pair_batch(idx, A.ids_shared ? (size_t)kb : first, cnt, lane, row_len, n_rows, bad);
    } else {
      if (singles == 0ull) continue;  // wave-uniform
      const unsigned long long row = my_ps < 0 ? (unsigned long long)A.uniq[my_ps & 0x7fffffff] : 0ull;
      const unsigned long long off = row * row_len;
      pb = PairBatch{(unsigned)off, (unsigned)(off >> 32), (unsigned)row};
    }
    float my_c0, my_c1;
    ModelOps<M>::coef(gscore[mine], score[mine], p, my_c0, my_c1);
    if constexpr (SINGLES == 3) {
      // the rows to finish behind the others, each kind in pair order: each streams without a branch on the other
      const int to = slab_place(lane, cnt, __popcll(singles), (singles >> lane) & 1ull, (int)lanes_below_in(singles));
      auto moved = [&](unsigned x) { return (unsigned)__builtin_amdgcn_ds_permute(to * 4, (int)x); };
      pb = PairBatch{moved(pb.off_lo), moved(pb.off_hi), moved(pb.row)};
      my_c0 = __uint_as_float(moved(__float_as_uint(my_c0)));
      my_c1 = __uint_as_float(moved(__float_as_uint(my_c1)));
    }
    // Without optimizer state to fetch, such a pair's row is finished the moment it streams by: its entity
    // row and query are in registers, the merged-gradient row is one more store.
    constexpr bool kInStream = SINGLES == 1 && CODES != 2;
    // With the forward's codes and no optimizer the merged-gradient row of such a pair is a function of its
    // code bytes and coefficients alone: it is stored as the codes stream by, and the entity row is never read.
    constexpr bool kFromCodes = SINGLES == 1 && CODES == 2;
    if constexpr (!GQ) {
      // nothing streams: only the rows of the one-pair segments below
    } else if constexpr (CODES == 2) {
      // 8 pairs' code bytes requested at a time, two sets used in turn
      constexpr int CB = 8;
      const unsigned char* pc = A.codes_in + first * (size_t)(NIT * 64) + lane;
      unsigned ca[CB][NIT], cb[CB][NIT];
      auto request = [&](unsigned (&c)[CB][NIT], int j0) {
#pragma unroll
        for (int r = 0; r < CB; ++r) {
          const int j = min(j0 + r, cnt - 1);
#pragma unroll
          for (int it = 0; it < NIT; ++it) c[r][it] = pc[(size_t)j * (NIT * 64) + 64 * it];
        }
      };
      auto consume = [&](const unsigned (&c)[CB][NIT], int j0) {
#pragma unroll
        for (int r = 0; r < CB; ++r) {
          if (j0 + r < cnt) {
            const float c0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(my_c0), j0 + r));
            const float c1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(my_c1), j0 + r));
#pragma unroll
            for (int it = 0; it < NIT; ++it)
#pragma unroll
              for (int v = 0; v < VEC; ++v)
                ModelOps<M>::bwd_q_from_code(c0, c1, c[r][it], VEC - 1 - v, g1[it][v], g2[it][v]);
            if constexpr (kFromCodes) {
              if ((singles >> (j0 + r)) & 1ull) {  // wave-uniform
                RowRegs<MUL, VEC, NIT> none;
                float ge1[NIT][VEC], ge2[NIT][VEC];
#pragma unroll
                for (int it = 0; it < NIT; ++it)
#pragma unroll
                  for (int v = 0; v < VEC; ++v) {
                    none.h[0][it].v[v] = 0.f;
                    ge1[it][v] = ge2[it][v] = 0.f;
                    ModelOps<M>::bwd_e_coded(c0, c1, c[r][it], VEC - 1 - v, ge1[it][v]);
                  }
                const int seg = __builtin_amdgcn_readlane(my_ps, j0 + r) & 0x7fffffff;
                finish_row<M, VEC, NIT, REG, false>(A.sink, lane, 0u, seg, ge1, ge2, none, none, none);
              }
            }
          }
        }
      };
      request(ca, 0);
      for (int j0 = 0; j0 < cnt; j0 += 2 * CB) {
        request(cb, j0 + CB);
        consume(ca, j0);
        request(ca, j0 + 2 * CB);
        consume(cb, j0 + CB);
      }
    } else {
    stage_pairs(slab, lane, table, pb, my_c0, my_c1);
    int n_stream = cnt;
    if constexpr (SINGLES == 0 && CODES == 0) {
      if (A.winner) {  // uniform: a branch row of a union query streams the pairs it won, moved to the front of the slab
        const bool keep = lane < cnt && A.winner[mine] == (unsigned char)(b - (b / A.U) * A.U);
        const unsigned long long won = __ballot(keep);
        n_stream = __popcll(won);
        if (keep) {
          const unsigned long long addr =
              (unsigned long long)(table + (((unsigned long long)pb.off_hi << 32) | pb.off_lo));
          *reinterpret_cast<uint4*>(slab + 4 * lanes_below_in(won)) =
              make_uint4((unsigned)addr, (unsigned)(addr >> 32), __float_as_uint(my_c0), __float_as_uint(my_c1));
        }
        slab_fence();
      }
    }
    if constexpr (SINGLES == 3) {
      // Rows that occur once, Adam: the row with its moments, one ahead of the one in work; every turn has the same number
      // of loads and stores, so that no wait is for more than what it needs (after a branch that may have issued some, the
      // wait is for all of them).
      n_stream = cnt - __popcll(singles);   // the rows to finish are n_stream .. cnt - 1
      RowState<MUL, VEC, NIT> sa, sb;
      auto request = [&](RowState<MUL, VEC, NIT>& s, int j) {
        const unsigned long long off = batch_off(pb, min(j, cnt - 1));
        load_row<MUL, VEC, NIT>(s.e, table + off, dim, ncol, lane);
        load_row<MUL, VEC, NIT, true>(s.m, A.sink.m + off, dim, ncol, lane);
        load_row<MUL, VEC, NIT, true>(s.v, A.sink.v + off, dim, ncol, lane);
        __builtin_amdgcn_sched_barrier(0);
      };
      RowSink sink = A.sink;
      sink.merged = nullptr;
      sink.adam_on = kOptAdam;
      sink.squeeze = 0;
      auto finish = [&](const RowState<MUL, VEC, NIT>& s, int j) {
        const float c0 = slab_coef(slab, j).x;
        float ge1[NIT][VEC], ge2[NIT][VEC];
        asm volatile("" ::: "memory");
        beta_row_both_grads<VEC, NIT, REG>(
            clamp, p, [&](int it, int v) { return s.e.h[0][it].v[v]; }, [&](int it, int v) { return s.e.h[MUL - 1][it].v[v]; }, c0,
            [&](int it, QBeta (&to)[VEC]) { beta_query<VEC, false, true>(lds, dim, min(lane + 64 * it, ncol - 1), to); }, g1, g2,
            ge1, ge2);
        finish_row<M, VEC, NIT, REG, true, true>(sink, lane, (unsigned)__builtin_amdgcn_readlane((int)pb.row, j), 0, ge1, ge2, s.e,
                                                 s.m, s.v);
      };
      if (n_stream < cnt) {
        request(sa, n_stream);
        for (int j = n_stream; j < cnt; j += 2) {
          request(sb, j + 1);
          finish(sa, j);
          if (j + 1 >= cnt) break;
          request(sa, j + 2);
          finish(sb, j + 1);
        }
      }
    }
    // lanes past the row end hold a copy of the last column: what they accumulate is never stored
    if (n_stream > 0)
    stream_batch<MUL, VEC, NIT, RIF>(slab, n_stream, dim, ncol, lane,
                                     [&](int j, const Pack<VEC>(&e1)[NIT], const Pack<VEC>(&e2)[NIT]) {
      float2 c = slab_coef(slab, j);
      [[maybe_unused]] const float c_raw = c.x;
      if constexpr (M == mL2)
        c.x = l2_pair_coef<VEC, NIT>(c.x, ncol, lane, [&](int it, int v) { return e1[it].v[v]; },
                                     [&](int it, int v) { return q[it][v].a; });
      if constexpr (model_norm(M, REG))  // d logit / d q = e / |e| per half: the upstream coefficient over the lengths
        c = norm_pair_coef<VEC, NIT, MUL>(c_raw, ncol, lane, [&](int it, int v) { return e1[it].v[v]; },
                                          [&](int it, int v) { return e2[it].v[v]; });
      if constexpr (CODES == 1) {
        // the pair's code bytes go to the wavefront's LDS stage, see flush_codes
        unsigned char* mine_b = stage + (j & (kStagePairs - 1)) * (NIT * 64) + lane;
#pragma unroll
        for (int it = 0; it < NIT; ++it) {
          unsigned code = 0;
#pragma unroll
          for (int v = 0; v < VEC; ++v)
            ModelOps<M>::bwd_q_coded(c.x, c.y, e1[it].v[v], q[it][v], neg_thr[it][v], g1[it][v], g2[it][v], code);
          mine_b[64 * it] = (unsigned char)code;
        }
        flush_codes<NIT>(stage, A.codes, first, j, cnt, lane);
      } else if constexpr (M == mBetaKL) {
        asm volatile("" ::: "memory");   // (as in the forward)
        beta_row_query_grad<VEC, NIT, REG>(
            clamp, [&](int it, int v) { return e1[it].v[v]; }, [&](int it, int v) { return e2[it].v[v]; }, c.x,
            [&](int it, QBeta (&to)[VEC]) { beta_query<VEC, false>(lds, dim, min(lane + 64 * it, ncol - 1), to); }, g1, g2);
      } else {
#pragma unroll
        for (int it = 0; it < NIT; ++it) {
#pragma unroll
          for (int v = 0; v < VEC; ++v) {
            const float x1 = REG ? reg_apply(e1[it].v[v], p) : e1[it].v[v];
            const float x2 = MUL == 2 ? (REG ? reg_apply(e2[it].v[v], p) : e2[it].v[v]) : 0.f;
            if constexpr (M == mBox) {
              ModelOps<M>::bwd_q_thr(c.x, c.y, x1, q[it][v], neg_thr[it][v], g1[it][v], g2[it][v]);
            } else if constexpr (model_norm(M, REG)) {
              g1[it][v] = __builtin_fmaf(c.x, x1, g1[it][v]);
              if constexpr (MUL == 2) g2[it][v] = __builtin_fmaf(c.y, x2, g2[it][v]);
            } else {
              ModelOps<M>::bwd_q(c.x, c.y, x1, x2, q[it][v], g1[it][v], g2[it][v]);
            }
          }
        }
      }
      if constexpr (kInStream) {
        if ((singles >> j) & 1ull) {  // wave-uniform
          RowRegs<MUL, VEC, NIT> w, none;
          float ge1[NIT][VEC], ge2[NIT][VEC];
#pragma unroll
          for (int it = 0; it < NIT; ++it) {
            if constexpr (M == mBetaKL) query_features(it, qf);
#pragma unroll
            for (int v = 0; v < VEC; ++v) {
              w.h[0][it].v[v] = e1[it].v[v];
              if (MUL == 2) w.h[MUL - 1][it].v[v] = e2[it].v[v];
              ge1[it][v] = ge2[it][v] = 0.f;
              const float x1 = REG ? reg_apply(e1[it].v[v], p) : e1[it].v[v];
              const float x2 = MUL == 2 ? (REG ? reg_apply(e2[it].v[v], p) : e2[it].v[v]) : 0.f;
              if constexpr (M == mBetaKL) ModelOps<M>::bwd_e(c.x, c.y, x1, x2, qf[v], ge1[it][v], ge2[it][v]);
              else ModelOps<M>::bwd_e(model_norm(M, REG) ? c_raw : c.x, c.y, x1, x2, q[it][v], ge1[it][v], ge2[it][v]);
            }
          }
          const int seg = __builtin_amdgcn_readlane(my_ps, j) & 0x7fffffff;
          const unsigned row = (unsigned)__builtin_amdgcn_readlane((int)pb.row, j);
          finish_row<M, VEC, NIT, REG, false>(A.sink, lane, row, seg, ge1, ge2, w, none, none);
        }
      }
    });
    }

    if constexpr (SINGLES != 0 && SINGLES != 3 && !kInStream && !kFromCodes) {
      // S rows at a time per wavefront (their w, m, v loads are all requested before the first is
      // used): the row sets of the streaming loop are dead here, so this costs no extra registers, and
      // it divides the memory latency each one-pair row would otherwise expose by S.
      constexpr int S = NIT * MUL == 1 ? 3 : (NIT * MUL == 2 ? 2 : 1);
      unsigned long long todo = singles;
      while (todo != 0ull) {
        int js[S];
        RowRegs<MUL, VEC, NIT> e[S], m0[S], v0[S];
#pragma unroll
        for (int s = 0; s < S; ++s) {
          js[s] = todo != 0ull ? __builtin_ctzll(todo) : -1;
          if (js[s] >= 0) {  // wave-uniform
            todo &= todo - 1;
            const unsigned long long off = batch_off(pb, js[s]);
            load_row<MUL, VEC, NIT>(e[s], table + off, dim, ncol, lane);
            if constexpr (SINGLES == 2) {
              if (A.sink.adam_on == kOptAdam) load_row<MUL, VEC, NIT, true>(m0[s], A.sink.m + off, dim, ncol, lane);
              if (A.sink.adam_on != kOptSgd && !A.sink.squeeze)
                load_row<MUL, VEC, NIT, true>(v0[s], A.sink.v + off, dim, ncol, lane);
            }
          }
        }
#pragma unroll
        for (int s = 0; s < S; ++s) {
          if (js[s] >= 0) {
            const int j = js[s];
            float c0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(my_c0), j));
            const float c1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(my_c1), j));
            if constexpr (M == mL2)
              c0 = l2_pair_coef<VEC, NIT>(c0, ncol, lane, [&](int it, int v) { return e[s].h[0][it].v[v]; },
                                          [&](int it, int v) { return q[it][v].a; });
            const int seg = __builtin_amdgcn_readlane(my_ps, j) & 0x7fffffff;
            const unsigned row = (unsigned)__builtin_amdgcn_readlane((int)pb.row, j);
            float ge1[NIT][VEC], ge2[NIT][VEC];
#pragma unroll
            for (int it = 0; it < NIT; ++it) {
              if constexpr (M == mBetaKL) query_features(it, qf);
#pragma unroll
              for (int v = 0; v < VEC; ++v) {
                ge1[it][v] = ge2[it][v] = 0.f;
                const float x1 = REG ? reg_apply(e[s].h[0][it].v[v], p) : e[s].h[0][it].v[v];
                const float x2 =
                    MUL == 2 ? (REG ? reg_apply(e[s].h[MUL - 1][it].v[v], p) : e[s].h[MUL - 1][it].v[v]) : 0.f;
                if constexpr (M == mBetaKL) ModelOps<M>::bwd_e(c0, c1, x1, x2, qf[v], ge1[it][v], ge2[it][v]);
                else ModelOps<M>::bwd_e(c0, c1, x1, x2, q[it][v], ge1[it][v], ge2[it][v]);
              }
            }
            finish_row<M, VEC, NIT, REG, SINGLES == 2>(A.sink, lane, row, seg, ge1, ge2, e[s], m0[s], v0[s]);
          }
        }
      }
    }
  }

  if constexpr (!GQ) return;
#pragma unroll
  for (int it = 0; it < NIT; ++it)
#pragma unroll
    for (int v = 0; v < VEC; ++v)
      if constexpr (M != mBetaKL) finish_query_grad<M>(q[it][v], g1[it][v], g2[it][v], p);

  // wavefront partials -> LDS -> fixed-order sum over wavefronts
  float* part = lds + QF * dim;  // [NW][NQ][dim]
  if constexpr (M == mBetaKL && (SINGLES == 1 || SINGLES == 2)) __syncthreads();   // (query_features)
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int c = lane + 64 * it;
    if (c < ncol) {
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        part[(wave * NQ + 0) * dim + c * VEC + v] = g1[it][v];
        if (NQ == 2) part[(wave * NQ + 1) * dim + c * VEC + v] = g2[it][v];
      }
    }
  }
  __syncthreads();
  for (int d = threadIdx.x; d < dim; d += NW * 64) {
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      s1 += part[(w * NQ + 0) * dim + d];
      if (NQ == 2) s2 += part[(w * NQ + 1) * dim + d];
    }
    gq1[(size_t)b * dim + d] = s1;
    if (NQ == 2) gq2[(size_t)b * dim + d] = s2;
  }
}

// rows requested per batch; two batches are in flight at a time
constexpr int rows_in_flight(int nit, int mul) {
  const int r = 4 / (nit * mul);
  return r < 1 ? 1 : r;
}

// Pairs of a forward workgroup: 64 per wavefront, fewer where the grid would not fill the chip.
inline int forward_tile(size_t B, size_t K, int least) {
  int tile_k = 256;
  while (tile_k > least && (B * ((K + tile_k - 1) / tile_k) < 8192 || (size_t)tile_k / 2 >= K)) tile_k /= 2;
  return tile_k;
}

// Tile length from which each distinct entity of a tile is scored once.  Not the short tiles of small batches: few of their ids
// repeat, and the tables, the barriers and the LDS they take -- 49 KiB for sign codes of 400 floats, three workgroups per CU -- cost
// more than the repeats.  Uniform / skewed ids, us with and without: box 512 x 128 x 400 46 / 43 -> 23 / 22, 400 x 400 x 400
// 61 / 57 -> 39 / 30, L1 54 / 46 -> 36 / 27 at 1024 x 128 x 400, L2 512 x 128 x 200 12.8 / 11.5 -> 11.6 / 10.3.  Tiles of 64,
// 1024 x 512 x 400: box 116 / 87 -> 113 / 68, but BetaE, whose pairs are arithmetic, 341 / 300 -> 337 / 336 at 200.  Tiles of 128,
// 2000 x 1000 x 200: L2 162 / 77 -> 164 / 93.
// Below it every pair is scored where it stands, and repeats of one id may then differ in their last bits, as those of two tiles may.
constexpr int distinct_from(int model) { return model == mBetaKL ? 64 : 128; }

// Rows that no cache will hold until they are asked for again are loaded past the caches (non-temporal), in the tiles whose ids
// are all different: then the last-level cache (256 MB) keeps what is asked for again -- the sign codes and the logits, or the
// lines that the query gradient starts with -- and the loads themselves are quicker (random rows of 800 bytes 6.0 TB/s against
// 5.65).  Forward of 1024 x 1024 pairs, RotatE, rows of 4 KB of a table of 10 GB: 736 -> 674 us.  The lines, from whole steps
// (forward, query gradient, entity pass), plain / past the caches in us:
// a table from 1.5 GiB on (below, a share of the rows is still in the cache): box, rows of 800 bytes of 0.8 GB 498 / 507, of 1.7 GB
// 546 / 536, of 8 GB 1054 / 1029; 1600 bytes of 2.4 GB 792 / 775; L1, 800 bytes of 0.8 GB 479 / 485, of 1.7 GB 532 / 521;
// without codes the query gradient reads the rows again: a table from 4 GiB on (RotatE 4 KB of 1.6 GB 2156 / 2157, of 3.3 GB
// 2378 / 2340, 1 KB of 1.7 GB 1308 / 1320, of 5 GB 1414 / 1400; L2 1600 bytes of 1.7 GB 1019 / 1033, of 13 GB 2179 / 2133) and a
// pass of 1.5 GiB (L2 800 bytes x 1 M pairs 669 / 676, 1200 bytes 939 / 934; ComplEx 1600 bytes 1101 / 1095);
// halves from 512 bytes on, or the lines that a row shares with its neighbours are most of it (RotatE, 2 x 400 bytes of 4 GB
// 674 / 683, 2 x 512 bytes 739 / 736).  Not in the kernels that follow: the query gradient of RotatE 1468 / 1498.
inline bool read_once(const ScoreArgs& A, int mul) {
  constexpr size_t kGiB = (size_t)1 << 30;
  const size_t half = (size_t)A.ncol * 4 * sizeof(float), row = mul * half;
  if (half < 512) return false;
  if (A.codes) return A.n_rows * row >= 3 * kGiB / 2;
  return A.n_rows * row >= 4 * kGiB && (size_t)A.B * A.K * row >= 3 * kGiB / 2;
}

template <int M, int VEC, int NIT, bool REG>
int launch_forward_reg(hipStream_t st, const ScoreArgs& A) {
  constexpr bool kOnce = VEC == 4 && NIT <= 2 && M != mBetaKL;   // (BetaE is bound by its arithmetic, longer rows lose a wavefront)
  const bool once = kOnce && read_once(A, model_mul(M));
  constexpr int RIF = rows_in_flight(NIT, model_mul(M));
  const size_t B = (size_t)A.B, K = (size_t)A.K;
  const int tile_k = forward_tile(B, K, 4 * RIF);
  const int tiles = (int)((K + tile_k - 1) / tile_k);
  const size_t lds = ((size_t)query_fields(M, VEC, true) * A.ncol * VEC + 4 * kSlabDwords) * sizeof(float);
  // (not the dense layout, whose rows are all different, nor a list of ids shared by the batch: a sampler's K negatives hardly
  // ever repeat)
  const bool dedup = A.idx != nullptr && !A.ids_shared && tile_k >= distinct_from(M);
  if constexpr (model_coded(M) && !REG) {
    if (A.codes) {
      if (dedup && once)
        hipLaunchKernelGGL((score_forward_kernel<M, VEC, NIT, RIF, REG, true, true, kOnce>), dim3((unsigned)(B * tiles)),
                           dim3(256), lds + (size_t)tile_k * NIT * 64 + kDedupLds, st, A, tiles, tile_k);
      else if (dedup)
        hipLaunchKernelGGL((score_forward_kernel<M, VEC, NIT, RIF, REG, true, true>), dim3((unsigned)(B * tiles)),
                           dim3(256), lds + (size_t)tile_k * NIT * 64 + kDedupLds, st, A, tiles, tile_k);
      else
        hipLaunchKernelGGL((score_forward_kernel<M, VEC, NIT, RIF, REG, true>), dim3((unsigned)(B * tiles)), dim3(256),
                           lds + 4 * kStagePairs * NIT * 64, st, A, tiles, tile_k);
      return check_launch("score forward (coded)");
    }
  }
  if (dedup && once)
    hipLaunchKernelGGL((score_forward_kernel<M, VEC, NIT, RIF, REG, false, true, kOnce>), dim3((unsigned)(B * tiles)),
                       dim3(256), lds + kDedupLds, st, A, tiles, tile_k);
  else if (dedup)
    hipLaunchKernelGGL((score_forward_kernel<M, VEC, NIT, RIF, REG, false, true>), dim3((unsigned)(B * tiles)),
                       dim3(256), lds + kDedupLds, st, A, tiles, tile_k);
  else
    hipLaunchKernelGGL((score_forward_kernel<M, VEC, NIT, RIF, REG>), dim3((unsigned)(B * tiles)), dim3(256), lds, st, A,
                       tiles, tile_k);
  return check_launch("score forward");
}

template <int M, int VEC, int NIT, int NW, bool REG>
int launch_backward_query_reg(hipStream_t st, const ScoreArgs& A) {
  constexpr int RIF = rows_in_flight(NIT, model_mul(M));
  const size_t lds = ((size_t)(NW + 1) * model_nq(M) * A.ncol * VEC + NW * kSlabDwords) * sizeof(float);
  if (!A.gq1) {  // one-pair segments only; built for the shapes that have sign codes
    if constexpr (model_coded(M) && !REG && NW == 8 && NIT <= 2) {
      if (A.pair_seg && A.uniq && A.sink.adam_on) {
        hipLaunchKernelGGL((score_backward_query_kernel<M, VEC, NIT, RIF, NW, REG, 2, 0, false>), dim3((unsigned)A.B),
                           dim3(NW * 64), lds, st, A);
        return check_launch("score backward (one-pair segments)");
      }
    }
    return fail(SMX_ERR_ARG, "the one-pair-segment pass is not available for this model and shape");
  }
  if constexpr (model_coded(M) && !REG) {
    if (A.codes_in) {
      if (A.pair_seg && A.sink.adam_on)
        hipLaunchKernelGGL((score_backward_query_kernel<M, VEC, NIT, RIF, NW, REG, 2, 2>), dim3((unsigned)A.B),
                           dim3(NW * 64), lds, st, A);
      else if (A.pair_seg)
        hipLaunchKernelGGL((score_backward_query_kernel<M, VEC, NIT, RIF, NW, REG, 1, 2>), dim3((unsigned)A.B),
                           dim3(NW * 64), lds, st, A);
      else
        hipLaunchKernelGGL((score_backward_query_kernel<M, VEC, NIT, RIF, NW, REG, 0, 2>), dim3((unsigned)A.B),
                           dim3(NW * 64), lds, st, A);
      return check_launch("score backward (query, from codes)");
    }
    if (A.codes && A.pair_seg) {
      const size_t lds_coded = lds + (size_t)NW * kStagePairs * NIT * 64;
      if (A.sink.adam_on)
        hipLaunchKernelGGL((score_backward_query_kernel<M, VEC, NIT, RIF, NW, REG, 2, 1>), dim3((unsigned)A.B),
                           dim3(NW * 64), lds_coded, st, A);
      else
        hipLaunchKernelGGL((score_backward_query_kernel<M, VEC, NIT, RIF, NW, REG, 1, 1>), dim3((unsigned)A.B),
                           dim3(NW * 64), lds_coded, st, A);
      return check_launch("score backward (query, coded)");
    }
  }
  if constexpr (M == mBetaKL && VEC == 4 && NIT <= 2 && NW == 8) {
    if (A.pair_seg && A.stream_rows) {
      const size_t fields = query_fields(M, VEC, false, true) - model_nq(M);
      hipLaunchKernelGGL((score_backward_query_kernel<M, VEC, NIT, RIF, NW, REG, 3>), dim3((unsigned)A.B), dim3(NW * 64),
                         lds + fields * A.ncol * VEC * sizeof(float), st, A);
      return check_launch("score backward (query, rows in the stream)");
    }
  }
  if (A.pair_seg && A.sink.adam_on)
    hipLaunchKernelGGL((score_backward_query_kernel<M, VEC, NIT, RIF, NW, REG, 2>), dim3((unsigned)A.B),
                       dim3(NW * 64), lds, st, A);
  else if (A.pair_seg)
    hipLaunchKernelGGL((score_backward_query_kernel<M, VEC, NIT, RIF, NW, REG, 1>), dim3((unsigned)A.B),
                       dim3(NW * 64), lds, st, A);
  else
    hipLaunchKernelGGL((score_backward_query_kernel<M, VEC, NIT, RIF, NW, REG, 0>), dim3((unsigned)A.B),
                       dim3(NW * 64), lds, st, A);
  return check_launch("score backward (query)");
}

template <int M, int VEC, int NIT>
int launch_score(hipStream_t st, const ScoreArgs& A, bool forward) {
  const bool reg = (M == mBetaKL && A.p.reg_on) || ((M == mComplex || M == mDistmult) && A.p.norm_on);
  if (forward) {
    if constexpr (M == mBetaKL || M == mComplex || M == mDistmult) {
      if (reg) return launch_forward_reg<M, VEC, NIT, true>(st, A);
    }
    return launch_forward_reg<M, VEC, NIT, false>(st, A);
  }
  // wavefronts per query: as many as 64 KiB of LDS allow -- the staged query and one partial-sum row per
  // wavefront, the wavefronts' 1 KiB pair slabs and, where the kernel writes sign codes, their code stages
  const size_t per_wave = (size_t)model_nq(M) * A.ncol * VEC * sizeof(float);
  const size_t extra = kSlabDwords * sizeof(unsigned) + (model_coded(M) ? (size_t)kStagePairs * NIT * 64 : 0);
  auto fits = [&](size_t n) { return (n + 1) * per_wave + n * extra <= 64 * 1024; };
  const int nw = fits(8) ? 8 : (fits(4) ? 4 : 2);
  if constexpr (M == mBetaKL || M == mComplex || M == mDistmult) {
    if (reg) {
      if (nw == 8) return launch_backward_query_reg<M, VEC, NIT, 8, true>(st, A);
      if (nw == 4) return launch_backward_query_reg<M, VEC, NIT, 4, true>(st, A);
      return launch_backward_query_reg<M, VEC, NIT, 2, true>(st, A);
    }
  }
  if (nw == 8) return launch_backward_query_reg<M, VEC, NIT, 8, false>(st, A);
  if (nw == 4) return launch_backward_query_reg<M, VEC, NIT, 4, false>(st, A);
  return launch_backward_query_reg<M, VEC, NIT, 2, false>(st, A);
}

// BetaE's kernels pay for every feature a lane holds, also past the row's end: 512 for a row of 400 in columns of four floats,
// 448 in single ones.  Those rows, and the short ones (128 floats: two a lane instead of four), are taken a float per lane and
// step; the loads are still whole 256-byte stretches.  Forward, 512 x 512 pairs of 2 x 400 floats: 358 -> 311 us.  Not where
// rows are finished as well: that is bound by memory.
inline int beta_singles(int dim, int nit4) {
  const int n = (dim + 63) / 64;
  return n <= 7 && n < 4 * nit4 ? n : 0;   // (never four: rows of 193 to 256 floats fill their columns of four)
}
int beta_singles_dispatch(hipStream_t st, const ScoreArgs& A, int nit, bool forward);   // smx_score_inst_betakl_singles.hip
template <int NIT>
int launch_beta_singles(hipStream_t st, const ScoreArgs& A, bool forward) {
  if (forward) return A.p.reg_on ? launch_forward_reg<mBetaKL, 1, NIT, true>(st, A) : launch_forward_reg<mBetaKL, 1, NIT, false>(st, A);
  // (rows of up to 448 floats: eight wavefronts' partial sums fit)
  const size_t lds = ((size_t)9 * 2 * A.ncol + 8 * kSlabDwords) * sizeof(float);
  if (A.p.reg_on)
    hipLaunchKernelGGL((score_backward_query_kernel<mBetaKL, 1, NIT, 1, 8, true, 0>), dim3((unsigned)A.B), dim3(512), lds, st, A);
  else
    hipLaunchKernelGGL((score_backward_query_kernel<mBetaKL, 1, NIT, 1, 8, false, 0>), dim3((unsigned)A.B), dim3(512), lds, st, A);
  return check_launch("score backward (query)");
}

// Instantiated once per model in its own translation unit (smx_score_inst_*.hip).
template <int M>
int score_dispatch(hipStream_t st, const ScoreArgs& A, int vec, int nit, bool forward) {
  if constexpr (M == mBetaKL) {
    const int n = vec == 4 && (forward || (A.gq1 && !A.pair_seg)) ? beta_singles(A.ncol * 4, nit) : 0;
    if (n) {
      ScoreArgs S = A;
      S.ncol = A.ncol * 4;
      return beta_singles_dispatch(st, S, n, forward);
    }
  }
  if (vec == 4) {
    switch (nit) {
      case 1: return launch_score<M, 4, 1>(st, A, forward);
      case 2: return launch_score<M, 4, 2>(st, A, forward);
      case 4: return launch_score<M, 4, 4>(st, A, forward);
      default: return launch_score<M, 4, 8>(st, A, forward);
    }
  }
  switch (nit) {
    case 1: return launch_score<M, 1, 1>(st, A, forward);
    case 2: return launch_score<M, 1, 2>(st, A, forward);
    default: return launch_score<M, 1, 4>(st, A, forward);
  }
}

}  // namespace smx
