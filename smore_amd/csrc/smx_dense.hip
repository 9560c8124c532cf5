// Dense distance operators for any broadcast layout, fp32 and fp64.
//
// These are the layout-general kernels behind smx_dist_forward_* /
// smx_dist_backward_*: entity [be,ne,dim*mul] against query [bc,nc,dim] with
// the modulo broadcast rule of the replaced launch loops
// (smore/common/torchext/common_kernel.h:41-49, 73-81, 108-115).
//
// General kernels (any layout, fp32 and fp64):
// forward : one wavefront per output element, lanes stride the feature axis,
//           xor-butterfly reduction over 64 lanes.
// backward: one workgroup per row of the side being differentiated; each
//           thread owns features d, d+blockDim, ... and walks that row's jobs
//           in ascending job order, so every sum has a fixed order and no
//           atomics are needed.
//
// Per-query kernels (fp32, entity [B,N,dim*mul] against query [B,1,dim]: the layout of the models'
// negatives [B,K] and positives [B,1], kg_reasoning.py:342-355): the query lives in LDS / registers,
// every entity row is read once, and the backward writes the row gradient and accumulates the query
// gradient in the same pass.  Shared negatives [1,N,.] and the reverse layout (entity [B,1,.] against
// query [B,N,.]) have kernels of the same build.  Rows of up to 1,024 floats in 16-byte columns; the
// backward of the first two layouts also takes rows of up to 512 floats in 8- or 4-byte columns.
// Everything else, and sizes that the kernels' ints or a launch cannot hold, is left to the general
// kernels (smx_dense_rules.h).
#include <type_traits>

#include "../../include/smx_measure.h"
#include "smx_common.h"
#include "smx_dense_rules.h"
#include "smx_functors.h"

namespace smx {

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int m = kWave / 2; m > 0; m >>= 1) v += __shfl_xor(v, m, kWave);
  return v;
}

template <int K, typename T>
__global__ __launch_bounds__(256) void dense_forward_kernel(const T* __restrict__ ent, const T* __restrict__ q1,
                                                            const T* __restrict__ q2, T* __restrict__ dst, Layout L) {
  constexpr int MUL = kind_mul(K);
  const int lane = threadIdx.x & (kWave - 1);
  const size_t waves_per_block = blockDim.x / kWave;
  const size_t total = L.bsize * L.num;
  for (size_t w = blockIdx.x * waves_per_block + threadIdx.x / kWave; w < total; w += (size_t)gridDim.x * waves_per_block) {
    const size_t i = w / L.num, j = w % L.num;
    const T* pe = ent + ((i % L.be) * L.ne + (j % L.ne)) * L.dim * MUL;
    const size_t qrow = ((i % L.bc) * L.nc + (j % L.nc)) * L.dim;
    T s = 0;
    for (size_t d = lane; d < L.dim; d += kWave) {
      const T e1 = pe[d];
      const T e2 = MUL == 2 ? pe[d + L.dim] : (T)0;
      const T a = q1[qrow + d];
      const T b = kind_nq(K) == 2 ? q2[qrow + d] : (T)0;
      s += Term<K, T>::fwd(e1, e2, a, b);
    }
    s = wave_sum(s);
    if (lane == 0) dst[w] = s;
  }
}

// SIDE 0: gradient of the entity rows, SIDE 1: gradient of the query rows.
template <int K, typename T, int SIDE>
__global__ __launch_bounds__(128) void dense_backward_kernel(const T* __restrict__ gout, const T* __restrict__ ent,
                                                             const T* __restrict__ q1, const T* __restrict__ q2,
                                                             T* __restrict__ g_a, T* __restrict__ g_b, Layout L) {
  constexpr int MUL = kind_mul(K);
  constexpr int NQ = kind_nq(K);
  const size_t row = blockIdx.x;
  const size_t own_b = SIDE == 0 ? L.be : L.bc;
  const size_t own_n = SIDE == 0 ? L.ne : L.nc;
  const size_t d0 = row / own_n, d1 = row % own_n;
  const size_t nji = L.bsize / own_b, njj = L.num / own_n;
  for (size_t d = threadIdx.x; d < L.dim; d += blockDim.x) {
    T acc1 = 0, acc2 = 0;
    T own_e1 = 0, own_e2 = 0, own_q1 = 0, own_q2 = 0;
    if (SIDE == 0) {
      own_e1 = ent[row * L.dim * MUL + d];
      if (MUL == 2) own_e2 = ent[row * L.dim * MUL + d + L.dim];
    } else {
      own_q1 = q1[row * L.dim + d];
      if (NQ == 2) own_q2 = q2[row * L.dim + d];
    }
    for (size_t job = 0; job < nji * njj; ++job) {
      const size_t i = (job / njj) * own_b + d0, j = (job % njj) * own_n + d1;
      const T g = gout[i * L.num + j];
      T sink1 = 0, sink2 = 0;
      if (SIDE == 0) {
        const size_t qrow = ((i % L.bc) * L.nc + (j % L.nc)) * L.dim;
        const T a = q1[qrow + d];
        const T b = NQ == 2 ? q2[qrow + d] : (T)0;
        Term<K, T>::bwd(g, own_e1, own_e2, a, b, acc1, acc2, sink1, sink2);
      } else {
        const T* pe = ent + ((i % L.be) * L.ne + (j % L.ne)) * L.dim * MUL;
        const T e1 = pe[d];
        const T e2 = MUL == 2 ? pe[d + L.dim] : (T)0;
        Term<K, T>::bwd(g, e1, e2, own_q1, own_q2, sink1, sink2, acc1, acc2);
      }
    }
    if (SIDE == 0) {
      g_a[row * L.dim * MUL + d] = acc1;
      if (MUL == 2) g_a[row * L.dim * MUL + d + L.dim] = acc2;
    } else {
      g_a[row * L.dim + d] = acc1;
      if (NQ == 2) g_b[row * L.dim + d] = acc2;
    }
  }
}

// ---- per-query layout, fp32 -------------------------------------------------------------------
typedef float dvec4 __attribute__((ext_vector_type(4)));

template <int K>
__device__ __forceinline__ float pq_row_terms(const dvec4* __restrict__ pe, const float* lds, int ncol, int dim, int lane) {
  constexpr int MUL = kind_mul(K), NQ = kind_nq(K);
  float s = 0.f;
  for (int c = lane; c < ncol; c += kWave) {
    const dvec4 e1 = pe[c];
    const dvec4 e2 = MUL == 2 ? pe[c + ncol] : dvec4{0.f, 0.f, 0.f, 0.f};
    const dvec4 a = reinterpret_cast<const dvec4*>(lds)[c];
    const dvec4 b = NQ == 2 ? reinterpret_cast<const dvec4*>(lds + dim)[c] : dvec4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < 4; ++x) s += Term<K, float>::fwd(e1[x], e2[x], a[x], b[x]);
  }
  return s;
}

// One workgroup per (query, tile of rows); its four wavefronts take the tile's rows two at a time.
template <int K, bool SHARED = false>
__global__ __launch_bounds__(256) void dense_pq_forward_kernel(const float* __restrict__ ent, const float* __restrict__ q1,
                                                               const float* __restrict__ q2, float* __restrict__ dst,
                                                               int num, int dim, int tiles, int rows_per_tile) {
  constexpr int MUL = kind_mul(K), NQ = kind_nq(K);
  extern __shared__ float lds[];  // q1[dim] | q2[dim]
  const int b = blockIdx.x / tiles, tile = blockIdx.x - b * tiles;
  for (int d = threadIdx.x; d < dim; d += 256) {
    lds[d] = q1[(size_t)b * dim + d];
    if (NQ == 2) lds[dim + d] = q2[(size_t)b * dim + d];
  }
  __syncthreads();
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int ncol = dim / 4;
  const int k1 = min(num, (tile + 1) * rows_per_tile);
  const size_t row_len = (size_t)dim * MUL;
  for (int k = tile * rows_per_tile + wave; k < k1; k += 8) {
    const size_t r0 = (size_t)b * num + k;
    const bool two = k + 4 < k1;
    const size_t r1 = two ? r0 + 4 : r0;
    const size_t e0 = SHARED ? (size_t)k : r0, e1 = SHARED ? (size_t)(two ? k + 4 : k) : r1;  // entity rows
    float s0 = pq_row_terms<K>(reinterpret_cast<const dvec4*>(ent + e0 * row_len), lds, ncol, dim, lane);
    float s1 = pq_row_terms<K>(reinterpret_cast<const dvec4*>(ent + e1 * row_len), lds, ncol, dim, lane);
    s0 = wave_sum(s0);
    s1 = wave_sum(s1);
    if (lane == 0) {
      dst[r0] = s0;
      if (two) dst[r1] = s1;
    }
  }
}

template <int VEC> using column = float __attribute__((ext_vector_type(VEC)));

// Stores the lane's column (VEC floats) of a half row through a buffer descriptor: a lane past the row's end stores nothing,
// with no branch around the store.  (Loads and stores share one in-order counter, and a wait has to assume the path that issued
// least: behind a branch, the stores of one row would have to land before the next row, long requested, may be used.)
template <int VEC>
__device__ __forceinline__ void store_column(float* half_row, int dim, int c, column<VEC> v) {
  const __amdgpu_buffer_rsrc_t row = __builtin_amdgcn_make_buffer_rsrc(half_row, 0, dim * (int)sizeof(float), 0x00027000);
  constexpr int kNonTemporal = 2;
  if constexpr (VEC == 1) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[0]), row, c * 4, 0, kNonTemporal);
  } else {
    typedef unsigned bits __attribute__((ext_vector_type(VEC)));
    bits t;
#pragma unroll
    for (int x = 0; x < VEC; ++x) t[x] = __float_as_uint(v[x]);
    if constexpr (VEC == 2) __builtin_amdgcn_raw_buffer_store_b64(t, row, c * 8, 0, kNonTemporal);
    else __builtin_amdgcn_raw_buffer_store_b128(t, row, c * 16, 0, kNonTemporal);
  }
}

// One workgroup per query, of NW wavefronts (NW = 0: as many as launched, at most eight).  Lane l owns the columns l, l+64, ... of the row, VEC floats each
// (NIT of them); wavefront w of nw takes rows w, w+nw, ...  For every row it writes the row's gradient and adds
// the row's contribution to its query-gradient registers, with AHEAD the next row on its way; the partial query gradients are
// summed through LDS in wavefront order, so the result does not depend on timing.
// SHARED: the entity rows are the same [1,N,.] for every query (--share_negative, online_sampler.py:155-157);
// this kernel then gives the query gradients only, and dense_shared_entity_backward_kernel the rows'.
// What bounds it: memory, given enough rows in flight, which is what the number of wavefronts and AHEAD are for (rule and figures
// at per_query_form); arithmetic for BetaE and Fisher.  Box 300 x 333 x 400 54 us, 5.9 TB/s.
template <int K, int NIT, bool SHARED, int NW, int VEC, bool AHEAD>
__global__ __launch_bounds__((NW > 0 ? NW : kPqBwdWaves) * kWave) void dense_pq_backward_kernel(
    const float* __restrict__ gout, const float* __restrict__ ent, const float* __restrict__ q1,
    const float* __restrict__ q2, float* __restrict__ gent, float* __restrict__ gq1, float* __restrict__ gq2, int num,
    int dim) {
  constexpr int MUL = kind_mul(K), NQ = kind_nq(K);
  // (a branch that costs one-half rows more than the group's arithmetic: box 200 x 300 x 800, shared, 47.1 / 48.7 us)
  constexpr bool kSkip = kind_heavy(K) || (SHARED && MUL == 2 && NIT * VEC == 16);
  typedef column<VEC> vec;
  extern __shared__ float lds[];  // [waves][NQ][dim]
  const int b = blockIdx.x;
  const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int nw = NW > 0 ? NW : (int)blockDim.x / kWave;
  const int ncol = dim / VEC;
  const size_t row_len = (size_t)dim * MUL;
  const vec zero = (vec)(0.f);
  vec qa[NIT], qb[NIT], acc1[NIT], acc2[NIT];
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int c = min(lane + kWave * it, ncol - 1);
    qa[it] = reinterpret_cast<const vec*>(q1 + (size_t)b * dim)[c];
    qb[it] = NQ == 2 ? reinterpret_cast<const vec*>(q2 + (size_t)b * dim)[c] : zero;
    acc1[it] = acc2[it] = zero;
  }
  struct Row {
    float g;
    vec e1[NIT], e2[NIT];
  };
  auto request = [&](int k, Row& row) {
    const size_t r = (size_t)b * num + k;
    row.g = gout[r];
    const vec* pe = reinterpret_cast<const vec*>(ent + (SHARED ? (size_t)k : r) * row_len);
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int c = min(lane + kWave * it, ncol - 1);
      row.e1[it] = pe[c];
      row.e2[it] = MUL == 2 ? pe[c + ncol] : zero;
    }
  };
  auto use = [&](int k, const Row& row) {
    float* pg = gent + ((size_t)b * num + k) * row_len;
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int c = lane + kWave * it;
      if (kSkip && kWave * it >= ncol) continue;   // uniform: no column of the row in this group
      if (!AHEAD && c >= ncol) continue;   // (AHEAD: such lanes hold a copy of the last column, what they compute is not stored)
      vec ge1 = zero, ge2 = zero;
#pragma unroll
      for (int x = 0; x < VEC; ++x) {
        float a1 = 0.f, a2 = 0.f, b1 = acc1[it][x], b2 = acc2[it][x];
        Term<K, float>::bwd(row.g, row.e1[it][x], row.e2[it][x], qa[it][x], qb[it][x], a1, a2, b1, b2);
        ge1[x] = a1;
        ge2[x] = a2;
        acc1[it][x] = b1;
        acc2[it][x] = b2;
      }
      if (SHARED) continue;
      if constexpr (AHEAD) {
        store_column<VEC>(pg, dim, c, ge1);
        if (MUL == 2) store_column<VEC>(pg + dim, dim, c, ge2);
      } else {
        __builtin_nontemporal_store(ge1, reinterpret_cast<vec*>(pg) + c);
        if (MUL == 2) __builtin_nontemporal_store(ge2, reinterpret_cast<vec*>(pg + dim) + c);
      }
    }
  };
  if constexpr (AHEAD) {
    if (wave < num) {
      Row row_a, row_b;
      auto next = [&](int k) { return min(k + nw, num - 1); };   // (behind a wavefront's last row: one that is read anyway)
      request(wave, row_a);
      for (int k = wave; k < num; k += nw) {
        request(next(k), row_b);
        use(k, row_a);
        k += nw;
        if (k >= num) break;
        request(next(k), row_a);
        use(k, row_b);
      }
    }
  } else {
    for (int k = wave; k < num; k += nw) {
      Row row;
      request(k, row);
      use(k, row);
    }
  }
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int c = lane + kWave * it;
    if (c < ncol) {
      reinterpret_cast<vec*>(lds + (size_t)(wave * NQ + 0) * dim)[c] = acc1[it];
      if (NQ == 2) reinterpret_cast<vec*>(lds + (size_t)(wave * NQ + 1) * dim)[c] = acc2[it];
    }
  }
  __syncthreads();
  for (int d = threadIdx.x; d < dim; d += nw * kWave) {
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int w = 0; w < nw; ++w) {
      s1 += lds[(size_t)(w * NQ + 0) * dim + d];
      if (NQ == 2) s2 += lds[(size_t)(w * NQ + 1) * dim + d];
    }
    gq1[(size_t)b * dim + d] = s1;
    if (NQ == 2) gq2[(size_t)b * dim + d] = s2;
  }
}

// Shared entity rows: gradient of row j = sum over the queries i of gout[i,j] * d term / d e.  One
// workgroup per row, the row in registers; wavefront w takes queries w, w+8, ... in ascending order and
// the eight partial sums are combined through LDS in wavefront order.
template <int K, int NIT, int VEC>
__global__ __launch_bounds__(kPqBwdWaves * kWave) void dense_shared_entity_backward_kernel(
    const float* __restrict__ gout, const float* __restrict__ ent, const float* __restrict__ q1,
    const float* __restrict__ q2, float* __restrict__ gent, int bsize, int num, int dim) {
  constexpr int MUL = kind_mul(K), NQ = kind_nq(K);
  typedef column<VEC> vec;
  extern __shared__ float lds[];  // [waves][MUL][dim]
  const int j = blockIdx.x;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int ncol = dim / VEC;
  const size_t row_len = (size_t)dim * MUL;
  const vec zero = (vec)(0.f);
  vec e1[NIT], e2[NIT], acc1[NIT], acc2[NIT];
  const vec* pe = reinterpret_cast<const vec*>(ent + (size_t)j * row_len);
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int c = min(lane + kWave * it, ncol - 1);
    e1[it] = pe[c];
    e2[it] = MUL == 2 ? pe[c + ncol] : zero;
    acc1[it] = acc2[it] = zero;
  }
  for (int i = wave; i < bsize; i += kPqBwdWaves) {
    const float g = gout[(size_t)i * num + j];
    const vec* pa = reinterpret_cast<const vec*>(q1 + (size_t)i * dim);
    const vec* pb = reinterpret_cast<const vec*>(q2 + (size_t)i * dim);
    vec qa[NIT], qb[NIT];
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int c = min(lane + kWave * it, ncol - 1);
      qa[it] = pa[c];
      qb[it] = NQ == 2 ? pb[c] : zero;
    }
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
#pragma unroll
      for (int x = 0; x < VEC; ++x) {
        float a1 = acc1[it][x], a2 = acc2[it][x], s1 = 0.f, s2 = 0.f;
        Term<K, float>::bwd(g, e1[it][x], e2[it][x], qa[it][x], qb[it][x], a1, a2, s1, s2);
        acc1[it][x] = a1;
        acc2[it][x] = a2;
      }
    }
  }
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int c = lane + kWave * it;
    if (c < ncol) {
      reinterpret_cast<vec*>(lds + (size_t)(wave * MUL + 0) * dim)[c] = acc1[it];
      if (MUL == 2) reinterpret_cast<vec*>(lds + (size_t)(wave * MUL + 1) * dim)[c] = acc2[it];
    }
  }
  __syncthreads();
  for (int d = threadIdx.x; d < dim * MUL; d += kPqBwdWaves * kWave) {
    const int h = d / dim, dd = d - h * dim;
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < kPqBwdWaves; ++w) sum += lds[(size_t)(w * MUL + h) * dim + dd];
    gent[(size_t)j * row_len + d] = sum;
  }
}

template <int K>
static int backward_shared(hipStream_t st, const float* gout, const float* ent, const float* q1, const float* q2,
                           float* gent, float* gq1, float* gq2, const Layout& L, int vec) {
  const dim3 block(kPqBwdWaves * kWave);
  const int num = (int)L.num, dim = (int)L.dim, bsize = (int)L.bsize;
  const size_t lds_q = (size_t)kPqBwdWaves * kind_nq(K) * L.dim * sizeof(float);
  const size_t lds_e = (size_t)kPqBwdWaves * kind_mul(K) * L.dim * sizeof(float);
  auto launch = [&](auto nit, auto v) {
    constexpr int NIT = decltype(nit)::value, VEC = decltype(v)::value;
    // (long rows of the arithmetic-bound kinds would spill, see per_query_form: BetaE 512 x 128 x 600 474 / 432 us)
    constexpr bool AHEAD = !(VEC == 4 && NIT == 4 && kind_heavy(K));
    hipLaunchKernelGGL((dense_pq_backward_kernel<K, NIT, true, kPqBwdWaves, VEC, AHEAD>), dim3((unsigned)L.bsize), block, lds_q, st,
                       gout, ent, q1, q2, gent, gq1, gq2, num, dim);
    hipLaunchKernelGGL((dense_shared_entity_backward_kernel<K, NIT, VEC>), dim3((unsigned)L.num), block, lds_e, st, gout, ent,
                       q1, q2, gent, bsize, num, dim);
  };
  using std::integral_constant;
  constexpr integral_constant<int, 1> one;
  constexpr integral_constant<int, 2> two;
  constexpr integral_constant<int, 4> four;
  constexpr integral_constant<int, 8> eight;
  const size_t ncol = L.dim / vec;
  if (vec == 2) {
    ncol <= 128 ? launch(two, two) : launch(four, two);
  } else if (vec == 1) {
    ncol <= 256 ? launch(four, one) : launch(eight, one);
  } else if (ncol <= 64) {
    launch(one, four);
  } else if (ncol <= 128) {
    launch(two, four);
  } else {
    launch(four, four);
  }
  return check_launch("dist backward (shared entity rows)");
}

// ---- reverse layout, fp32: entity [B,1,.] against query [B,N,.] -------------------------------------
// (inverse queries: the tail entity is projected back through the relations and compared with one query
// row per candidate, kg_reasoning.py:252-263).  The mirror image of the per-query kernels: the entity row
// is the one that stays (LDS / registers), the query rows stream by, the query gradient is per row and the
// entity gradient is the sum over the rows.
template <int K>
__global__ __launch_bounds__(256) void dense_rev_forward_kernel(const float* __restrict__ ent, const float* __restrict__ q1,
                                                                const float* __restrict__ q2, float* __restrict__ dst,
                                                                int num, int dim, int tiles, int rows_per_tile) {
  constexpr int MUL = kind_mul(K), NQ = kind_nq(K);
  extern __shared__ float lds[];  // e1[dim] | e2[dim]
  const int b = blockIdx.x / tiles, tile = blockIdx.x - b * tiles;
  for (int d = threadIdx.x; d < dim * MUL; d += 256) lds[d] = ent[(size_t)b * dim * MUL + d];
  __syncthreads();
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int ncol = dim / 4;
  const int k1 = min(num, (tile + 1) * rows_per_tile);
  const dvec4 zero = {0.f, 0.f, 0.f, 0.f};
  for (int k = tile * rows_per_tile + wave; k < k1; k += 4) {
    const size_t r = (size_t)b * num + k;
    const dvec4* pa = reinterpret_cast<const dvec4*>(q1 + r * dim);
    const dvec4* pb = reinterpret_cast<const dvec4*>(q2 + r * dim);
    float sum = 0.f;
    for (int c = lane; c < ncol; c += kWave) {
      const dvec4 e1 = reinterpret_cast<const dvec4*>(lds)[c];
      const dvec4 e2 = MUL == 2 ? reinterpret_cast<const dvec4*>(lds + dim)[c] : zero;
      const dvec4 a = pa[c];
      const dvec4 bq = NQ == 2 ? pb[c] : zero;
#pragma unroll
      for (int x = 0; x < 4; ++x) sum += Term<K, float>::fwd(e1[x], e2[x], a[x], bq[x]);
    }
    sum = wave_sum(sum);
    if (lane == 0) dst[r] = sum;
  }
}

template <int K, int NIT>
__global__ __launch_bounds__(kPqBwdWaves * kWave) void dense_rev_backward_kernel(
    const float* __restrict__ gout, const float* __restrict__ ent, const float* __restrict__ q1,
    const float* __restrict__ q2, float* __restrict__ gent, float* __restrict__ gq1, float* __restrict__ gq2, int num,
    int dim) {
  constexpr int MUL = kind_mul(K), NQ = kind_nq(K);
  extern __shared__ float lds[];  // [waves][MUL][dim]
  const int b = blockIdx.x;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int ncol = dim / 4;
  const size_t row_len = (size_t)dim * MUL;
  const dvec4 zero = {0.f, 0.f, 0.f, 0.f};
  dvec4 e1[NIT], e2[NIT], acc1[NIT], acc2[NIT];
  const dvec4* pe = reinterpret_cast<const dvec4*>(ent + (size_t)b * row_len);
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int c = min(lane + kWave * it, ncol - 1);
    e1[it] = pe[c];
    e2[it] = MUL == 2 ? pe[c + ncol] : zero;
    acc1[it] = acc2[it] = zero;
  }
  for (int k = wave; k < num; k += kPqBwdWaves) {
    const size_t r = (size_t)b * num + k;
    const float g = gout[r];
    const dvec4* pa = reinterpret_cast<const dvec4*>(q1 + r * dim);
    const dvec4* pb = reinterpret_cast<const dvec4*>(q2 + r * dim);
    dvec4 qa[NIT], qb[NIT];
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int c = min(lane + kWave * it, ncol - 1);
      qa[it] = pa[c];
      qb[it] = NQ == 2 ? pb[c] : zero;
    }
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int c = lane + kWave * it;
      if (c < ncol) {
        dvec4 g1 = zero, g2 = zero;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          float a1 = acc1[it][x], a2 = acc2[it][x], s1 = 0.f, s2 = 0.f;
          Term<K, float>::bwd(g, e1[it][x], e2[it][x], qa[it][x], qb[it][x], a1, a2, s1, s2);
          acc1[it][x] = a1;
          acc2[it][x] = a2;
          g1[x] = s1;
          g2[x] = s2;
        }
        __builtin_nontemporal_store(g1, reinterpret_cast<dvec4*>(gq1 + r * dim) + c);
        if (NQ == 2) __builtin_nontemporal_store(g2, reinterpret_cast<dvec4*>(gq2 + r * dim) + c);
      }
    }
  }
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const int c = lane + kWave * it;
    if (c < ncol) {
      reinterpret_cast<dvec4*>(lds + (size_t)(wave * MUL + 0) * dim)[c] = acc1[it];
      if (MUL == 2) reinterpret_cast<dvec4*>(lds + (size_t)(wave * MUL + 1) * dim)[c] = acc2[it];
    }
  }
  __syncthreads();
  for (int d = threadIdx.x; d < dim * MUL; d += kPqBwdWaves * kWave) {
    const int h = d / dim, dd = d - h * dim;
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < kPqBwdWaves; ++w) sum += lds[(size_t)(w * MUL + h) * dim + dd];
    gent[(size_t)b * row_len + d] = sum;
  }
}

template <int K>
static int forward_rev(hipStream_t st, const float* ent, const float* q1, const float* q2, float* dst, const Layout& L,
                       int rows_per_tile) {
  const int tiles = (int)((L.num + rows_per_tile - 1) / rows_per_tile);
  const size_t lds = (size_t)kind_mul(K) * L.dim * sizeof(float);
  hipLaunchKernelGGL((dense_rev_forward_kernel<K>), dim3((unsigned)(L.bsize * tiles)), dim3(256), lds, st, ent, q1, q2, dst,
                     (int)L.num, (int)L.dim, tiles, rows_per_tile);
  return check_launch("dist forward (reverse layout)");
}

template <int K>
static int backward_rev(hipStream_t st, const float* gout, const float* ent, const float* q1, const float* q2, float* gent,
                        float* gq1, float* gq2, const Layout& L) {
  const size_t lds = (size_t)kPqBwdWaves * kind_mul(K) * L.dim * sizeof(float);
  const dim3 grid((unsigned)L.bsize), block(kPqBwdWaves * kWave);
  const int num = (int)L.num, dim = (int)L.dim;
  const size_t ncol = L.dim / 4;
  if (ncol <= 64)
    hipLaunchKernelGGL((dense_rev_backward_kernel<K, 1>), grid, block, lds, st, gout, ent, q1, q2, gent, gq1, gq2, num, dim);
  else if (ncol <= 128)
    hipLaunchKernelGGL((dense_rev_backward_kernel<K, 2>), grid, block, lds, st, gout, ent, q1, q2, gent, gq1, gq2, num, dim);
  else
    hipLaunchKernelGGL((dense_rev_backward_kernel<K, 4>), grid, block, lds, st, gout, ent, q1, q2, gent, gq1, gq2, num, dim);
  return check_launch("dist backward (reverse layout)");
}

template <int K, bool SHARED = false>
static int forward_pq(hipStream_t st, const float* ent, const float* q1, const float* q2, float* dst, const Layout& L,
                      int rows_per_tile) {
  const int tiles = (int)((L.num + rows_per_tile - 1) / rows_per_tile);
  const size_t lds = (size_t)kind_nq(K) * L.dim * sizeof(float);
  hipLaunchKernelGGL((dense_pq_forward_kernel<K, SHARED>), dim3((unsigned)(L.bsize * tiles)), dim3(256), lds, st, ent, q1, q2, dst,
                     (int)L.num, (int)L.dim, tiles, rows_per_tile);
  return check_launch("dist forward (per-query layout)");
}

template <int K>
static int backward_pq(hipStream_t st, const float* gout, const float* ent, const float* q1, const float* q2, float* gent,
                       float* gq1, float* gq2, const Layout& L, const BackwardForm& form) {
  const int num = (int)L.num, dim = (int)L.dim;
  using std::integral_constant;
  auto launch = [&](auto nit, auto v) {
    constexpr int NIT = decltype(nit)::value, VEC = decltype(v)::value;
    auto go = [&](auto most, auto ahead) {
      constexpr int NW = decltype(most)::value;
      constexpr bool AHEAD = decltype(ahead)::value;
      hipLaunchKernelGGL((dense_pq_backward_kernel<K, NIT, false, NW, VEC, AHEAD>), dim3((unsigned)L.bsize),
                         dim3(form.waves * kWave), (size_t)form.waves * kind_nq(K) * L.dim * sizeof(float), st, gout, ent, q1,
                         q2, gent, gq1, gq2, num, dim);
    };
    constexpr integral_constant<int, 0> as_launched;
    constexpr integral_constant<int, 8> eight;
    constexpr integral_constant<int, 16> sixteen;
    if (form.waves < kPqBwdWaves) return go(as_launched, std::false_type());
    if constexpr (VEC == 4 && (NIT == 1 || (NIT == 2 && kind_mul(K) == 1))) {
      if (form.waves == 16) return go(sixteen, std::true_type());
    }
    if constexpr (VEC == 4 && NIT == (kind_heavy(K) ? 4 : 1)) {
      if (!form.ahead) return go(eight, std::false_type());
    }
    if constexpr (!(VEC == 4 && NIT == 4 && kind_heavy(K))) go(eight, std::true_type());
  };
  constexpr integral_constant<int, 1> one;
  constexpr integral_constant<int, 2> two;
  constexpr integral_constant<int, 4> four;
  constexpr integral_constant<int, 8> eight;
  const size_t ncol = L.dim / form.vec;
  if (form.vec == 2) {
    ncol <= 128 ? launch(two, two) : launch(four, two);
  } else if (form.vec == 1) {
    ncol <= 256 ? launch(four, one) : launch(eight, one);
  } else if (ncol <= 64) {
    launch(one, four);
  } else if (ncol <= 128) {
    launch(two, four);
  } else {
    launch(four, four);
  }
  return check_launch("dist backward (per-query layout)");
}

static int check_layout(const Layout& L) {
  if (L.bsize == 0 || L.num == 0 || L.dim == 0 || L.be == 0 || L.ne == 0 || L.bc == 0 || L.nc == 0)
    return fail(SMX_ERR_SHAPE, "empty dimension in dist layout");
  if (L.bsize % L.be || L.bsize % L.bc || L.num % L.ne || L.num % L.nc)
    return fail(SMX_ERR_SHAPE, "output [%zu,%zu] is not a multiple of entity [%zu,%zu] / query [%zu,%zu]", L.bsize,
                L.num, L.be, L.ne, L.bc, L.nc);
  if (L.be * L.ne > 0x7fffffffull || L.bc * L.nc > 0x7fffffffull)
    return fail(SMX_ERR_SHAPE, "more than 2^31-1 rows on one side");
  return SMX_OK;
}

template <int K, typename T>
static int forward_k(hipStream_t st, const T* ent, const T* q1, const T* q2, T* dst, const Layout& L) {
  const size_t total = L.bsize * L.num;
  size_t blocks = (total + 3) / 4;
  if (blocks > (1u << 20)) blocks = 1u << 20;
  hipLaunchKernelGGL((dense_forward_kernel<K, T>), dim3((unsigned)blocks), dim3(256), 0, st, ent, q1, q2, dst, L);
  return check_launch("dist forward");
}

template <int K, typename T>
static int backward_k(hipStream_t st, const T* gout, const T* ent, const T* q1, const T* q2, T* gent, T* gq1, T* gq2,
                      const Layout& L) {
  hipLaunchKernelGGL((dense_backward_kernel<K, T, 0>), dim3((unsigned)(L.be * L.ne)), dim3(128), 0, st, gout, ent, q1,
                     q2, gent, (T*)nullptr, L);
  hipLaunchKernelGGL((dense_backward_kernel<K, T, 1>), dim3((unsigned)(L.bc * L.nc)), dim3(128), 0, st, gout, ent, q1,
                     q2, gq1, gq2, L);
  return check_launch("dist backward");
}

#define SMX_FOR_EACH_KIND(X) \
  X(kL1) X(kL2) X(kBoxOut) X(kBoxIn) X(kRotate) X(kBetaKL) X(kComplex) X(kDistmult) X(kBetaL2) X(kBetaFisher)

// Addresses or'ed together: what their lowest bits say holds for all of them.
template <typename... P>
static size_t low_bits(const P*... p) {
  return (size_t)(reinterpret_cast<uintptr_t>(p) | ...);
}

template <typename T>
int dense_forward(int kind, void* stream, const T* ent, const T* q1, const T* q2, T* dst, size_t bsize, size_t num,
                  size_t be, size_t ne, size_t bc, size_t nc, size_t dim) {
  if (kind < 0 || kind >= kNumKinds) return fail(SMX_ERR_KIND, "unknown dist kind %d", kind);
  Layout L{bsize, num, be, ne, bc, nc, dim};
  if (int rc = check_layout(L)) return rc;
  if (!ent || !q1 || !dst || (kind_nq(kind) == 2 && !q2)) return fail(SMX_ERR_ARG, "null tensor pointer");
  hipStream_t st = as_stream(stream);
  if constexpr (std::is_same<T, float>::value) {
    const ForwardForm form = dense_forward_form(L, low_bits(ent, q1, q2, dst));
    if (form.path == kPathPerQuery) {
      switch (kind) {
#define X(KK) \
  case KK:    \
    return forward_pq<KK>(st, ent, q1, q2, dst, L, form.rows_per_tile);
        SMX_FOR_EACH_KIND(X)
#undef X
      }
    }
    if (form.path == kPathShared) {
      switch (kind) {
#define X(KK) \
  case KK:    \
    return forward_pq<KK, true>(st, ent, q1, q2, dst, L, form.rows_per_tile);
        SMX_FOR_EACH_KIND(X)
#undef X
      }
    }
    if (form.path == kPathReverse) {
      switch (kind) {
#define X(KK) \
  case KK:    \
    return forward_rev<KK>(st, ent, q1, q2, dst, L, form.rows_per_tile);
        SMX_FOR_EACH_KIND(X)
#undef X
      }
    }
  }
  switch (kind) {
#define X(KK) \
  case KK:    \
    return forward_k<KK, T>(st, ent, q1, q2, dst, L);
    SMX_FOR_EACH_KIND(X)
#undef X
  }
  return fail(SMX_ERR_KIND, "unknown dist kind %d", kind);
}

template <typename T>
int dense_backward(int kind, void* stream, const T* gout, const T* ent, const T* q1, const T* q2, T* gent, T* gq1,
                   T* gq2, size_t bsize, size_t num, size_t be, size_t ne, size_t bc, size_t nc, size_t dim) {
  if (kind < 0 || kind >= kNumKinds) return fail(SMX_ERR_KIND, "unknown dist kind %d", kind);
  Layout L{bsize, num, be, ne, bc, nc, dim};
  if (int rc = check_layout(L)) return rc;
  if (!gout || !ent || !q1 || !gent || !gq1 || (kind_nq(kind) == 2 && (!q2 || !gq2)))
    return fail(SMX_ERR_ARG, "null tensor pointer");
  hipStream_t st = as_stream(stream);
  if constexpr (std::is_same<T, float>::value) {
    const BackwardForm form = dense_backward_form(L, kind, low_bits(gout, ent, q1, q2, gent, gq1, gq2));
    if (form.path == kPathPerQuery) {
      switch (kind) {
#define X(KK) \
  case KK:    \
    return backward_pq<KK>(st, gout, ent, q1, q2, gent, gq1, gq2, L, form);
        SMX_FOR_EACH_KIND(X)
#undef X
      }
    }
    if (form.path == kPathShared) {
      switch (kind) {
#define X(KK) \
  case KK:    \
    return backward_shared<KK>(st, gout, ent, q1, q2, gent, gq1, gq2, L, form.vec);
        SMX_FOR_EACH_KIND(X)
#undef X
      }
    }
    if (form.path == kPathReverse) {
      switch (kind) {
#define X(KK) \
  case KK:    \
    return backward_rev<KK>(st, gout, ent, q1, q2, gent, gq1, gq2, L);
        SMX_FOR_EACH_KIND(X)
#undef X
      }
    }
  }
  switch (kind) {
#define X(KK) \
  case KK:    \
    return backward_k<KK, T>(st, gout, ent, q1, q2, gent, gq1, gq2, L);
    SMX_FOR_EACH_KIND(X)
#undef X
  }
  return fail(SMX_ERR_KIND, "unknown dist kind %d", kind);
}

}  // namespace smx

extern "C" {

int smx_dist_forward_f32(int kind, void* stream, const float* ent, const float* q1, const float* q2, float* dst,
                         size_t bsize, size_t num, size_t be, size_t ne, size_t bc, size_t nc, size_t dim) {
  return smx::dense_forward<float>(kind, stream, ent, q1, q2, dst, bsize, num, be, ne, bc, nc, dim);
}
int smx_dist_forward_f64(int kind, void* stream, const double* ent, const double* q1, const double* q2, double* dst,
                         size_t bsize, size_t num, size_t be, size_t ne, size_t bc, size_t nc, size_t dim) {
  return smx::dense_forward<double>(kind, stream, ent, q1, q2, dst, bsize, num, be, ne, bc, nc, dim);
}
int smx_dist_backward_f32(int kind, void* stream, const float* gout, const float* ent, const float* q1,
                          const float* q2, float* gent, float* gq1, float* gq2, size_t bsize, size_t num, size_t be,
                          size_t ne, size_t bc, size_t nc, size_t dim) {
  return smx::dense_backward<float>(kind, stream, gout, ent, q1, q2, gent, gq1, gq2, bsize, num, be, ne, bc, nc, dim);
}
int smx_dist_backward_f64(int kind, void* stream, const double* gout, const double* ent, const double* q1,
                          const double* q2, double* gent, double* gq1, double* gq2, size_t bsize, size_t num,
                          size_t be, size_t ne, size_t bc, size_t nc, size_t dim) {
  return smx::dense_backward<double>(kind, stream, gout, ent, q1, q2, gent, gq1, gq2, bsize, num, be, ne, bc, nc, dim);
}
int smx_measure_dense_backward_form(int kind, size_t bsize, size_t num, size_t be, size_t ne, size_t bc, size_t nc, size_t dim,
                                    size_t addresses, int* path, int* vec, int* waves, int* ahead) {
  using namespace smx;
  if (kind < 0 || kind >= kNumKinds) return fail(SMX_ERR_KIND, "unknown dist kind %d", kind);
  const Layout L{bsize, num, be, ne, bc, nc, dim};
  if (int rc = check_layout(L)) return rc;
  const BackwardForm form = dense_backward_form(L, kind, addresses);
  *path = form.path;
  *vec = form.vec;
  *waves = form.waves;
  *ahead = form.ahead;
  return SMX_OK;
}
int smx_measure_dense_forward_form(size_t bsize, size_t num, size_t be, size_t ne, size_t bc, size_t nc, size_t dim,
                                   size_t addresses, int* path, int* rows_per_tile) {
  using namespace smx;
  const Layout L{bsize, num, be, ne, bc, nc, dim};
  if (int rc = check_layout(L)) return rc;
  const ForwardForm form = dense_forward_form(L, addresses);
  *path = form.path;
  *rows_per_tile = form.rows_per_tile;
  return SMX_OK;
}

}  // extern "C"
