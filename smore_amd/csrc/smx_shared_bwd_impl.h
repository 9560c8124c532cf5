// Backward of the distance models box, l1 and rotate for negatives that every query of the batch shares
// (--share_negative, smore/cpp_sampler/online_sampler.py:155-157; [1,K,row] against [B,1,D],
// smore/models/kg_reasoning.py:349-355): the query gradients (common_kernel.h:92-123) and the gradient row of every list
// position (common_kernel.h:59-89), one tiling for both.
//
// All B x K pairs meet in every feature, as in a matrix product whose multiply-add is the model's derivative.  A lane
// owns one float4 column of R rows of one side (the side whose gradient is formed) and walks a stretch of the
// other side's rows: what it fetches per step meets R rows, and the (row group, column) items are dealt to the lanes
// without regard to where a row ends, so no lane is idle past a row's last column (100 columns on 128 lanes: 22 %).
// A workgroup is 16 items x 8 stretches, two wavefronts, small enough that the last round of workgroups costs little;
// the stretches' partial sums are added through LDS in order.  Stretches and order are those of the kernels that give a
// workgroup one row (shared_entity_kernel, score_backward_query_kernel), so are the operations per pair: same bits.
#pragma once
#include "smx_common.h"
#include "smx_models.h"
#include "smx_wave.h"

namespace smx {

struct SharedBwdArgs {
  const float* table;
  const long long* ids;  // [K]; null: `table` holds the list's rows themselves
  const float* q1;
  const float* q2;
  const float* gscore;   // [B, K]
  float* out1;           // ENTITY: gradient rows [K, row]; else gq1
  float* out2;           // gq2
  int B, K, ncol;        // ncol float4 columns per half row
  unsigned long long n_rows;
  ScoreParams p;
};

constexpr int kSbItems = 16;
constexpr int kSbStretches = 8;
constexpr int kSbThreads = kSbItems * kSbStretches;
constexpr int kSbChunk = 64;                // row offsets of a stretch in LDS at a time

typedef float sbvec4 __attribute__((ext_vector_type(4)));
typedef float sbvec4u __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ size_t sb_row(const SharedBwdArgs& A, int k) {
  if (!A.ids) return (size_t)k;
  const long long row = A.ids[k];
  return (unsigned long long)row < A.n_rows ? (size_t)row : 0;  // (the forward has flagged it)
}

template <int M, bool ENTITY, int R>
__global__ __launch_bounds__(kSbThreads) void shared_backward_kernel(SharedBwdArgs A) {
  constexpr int MUL = model_mul(M), NQ = model_nq(M);
  constexpr int NK = ENTITY ? MUL : NQ, NS = ENTITY ? NQ : MUL;  // float4 pieces of a kept and of a streamed row
  __shared__ sbvec4 part[kSbStretches * R * NK * kSbItems];
  __shared__ unsigned long long offs[ENTITY ? 1 : kSbStretches * (kSbChunk + 1)];  // (+ 1: stretches in different banks)
  const int t = threadIdx.x, lane = t & 63, wave = uniform(t >> 6);
  const int item = t & (kSbItems - 1), stretch = t / kSbItems;
  const int ncol = A.ncol, dim = ncol * 4;
  const int n_kept = ENTITY ? A.K : A.B, n_str = ENTITY ? A.B : A.K;
  const int n_items = (n_kept + R - 1) / R * ncol;
  const int at = min((int)blockIdx.x * kSbItems + item, n_items - 1);  // an item past the end repeats the last, unstored
  const int group = at / ncol, col = at - group * ncol;
  const int r0 = min(group * R, n_kept - R);  // the last group overlaps its neighbour: same rows, same values

  sbvec4 kept[R][NK];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if constexpr (ENTITY) {
      const sbvec4* row = reinterpret_cast<const sbvec4*>(A.table + sb_row(A, r0 + r) * (size_t)(dim * MUL));
#pragma unroll
      for (int h = 0; h < NK; ++h) kept[r][h] = row[h * ncol + col];
    } else {
      kept[r][0] = reinterpret_cast<const sbvec4*>(A.q1 + (size_t)(r0 + r) * dim)[col];
      if constexpr (NK == 2) kept[r][1] = reinterpret_cast<const sbvec4*>(A.q2 + (size_t)(r0 + r) * dim)[col];
    }
  }
  float acc[R][2][4];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int x = 0; x < 4; ++x) acc[r][0][x] = acc[r][1][x] = 0.f;

  const int per = (n_str + kSbStretches - 1) / kSbStretches;
  const int lo = stretch * per, hi = min(n_str, lo + per);
  auto use = [&](const sbvec4 (&s)[NS], const float (&g)[R]) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float c0, c1;
      ModelOps<M>::coef(g[r], 0.f, A.p, c0, c1);  // (none of these models needs the score)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const sbvec4* e = ENTITY ? kept[r] : s;
        const sbvec4* q = ENTITY ? s : kept[r];
        const float x1 = e[0][x], x2 = MUL == 2 ? e[MUL - 1][x] : 0.f;
        const typename ModelOps<M>::Q qq = ModelOps<M>::prep(q[0][x], NQ == 2 ? q[NQ - 1][x] : 0.f);
        if constexpr (ENTITY) ModelOps<M>::bwd_e(c0, c1, x1, x2, qq, acc[r][0][x], acc[r][1][x]);
        else ModelOps<M>::bwd_q(c0, c1, x1, x2, qq, acc[r][0][x], acc[r][1][x]);
      }
    }
  };

  if constexpr (ENTITY) {
    typedef float gvec __attribute__((ext_vector_type(R), aligned(4)));
    struct Step { sbvec4 s[NS]; gvec g; };
    auto request = [&](int b) {
      Step n;
      b = min(b, n_str - 1);
      n.s[0] = reinterpret_cast<const sbvec4*>(A.q1 + (size_t)b * dim)[col];
      if constexpr (NS == 2) n.s[1] = reinterpret_cast<const sbvec4*>(A.q2 + (size_t)b * dim)[col];
      n.g = *reinterpret_cast<const gvec*>(A.gscore + (size_t)b * A.K + r0);
      return n;
    };
    Step now = request(lo);
#pragma unroll 2
    for (int i = 0; i < per; ++i) {
      const Step next = request(lo + i + 1);
      if (lo + i < hi) {
        float g[R];
#pragma unroll
        for (int r = 0; r < R; ++r) g[r] = now.g[r];
        use(now.s, g);
      }
      now = next;
    }
  } else {
    struct Row { sbvec4 s[NS]; };
    unsigned long long* my_offs = offs + stretch * (kSbChunk + 1);
    for (int c0 = 0; c0 < per; c0 += kSbChunk) {
      const int cnt = min(kSbChunk, per - c0);
      // a wavefront looks up the rows of its own four stretches
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int st = wave * 4 + j;
        offs[st * (kSbChunk + 1) + lane] = sb_row(A, min(st * per + c0 + lane, n_str - 1)) * (unsigned long long)(dim * MUL);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      auto request = [&](int i) {
        Row n;
        const sbvec4* row = reinterpret_cast<const sbvec4*>(A.table + my_offs[min(i, cnt - 1)]);
#pragma unroll
        for (int h = 0; h < NS; ++h) n.s[h] = row[h * ncol + col];
        return n;
      };
      // the coefficients of four steps at a time, [row][step]; at the list's end the last four, moved up
      struct Coef { sbvec4 r[R]; };
      auto request_g = [&](int k) {
        Coef n;
        const int from = min(k, n_str - 4);
#pragma unroll
        for (int r = 0; r < R; ++r) n.r[r] = *reinterpret_cast<const sbvec4u*>(A.gscore + (size_t)(r0 + r) * A.K + from);
        for (int m = min(k - from, 4); m > 0; --m) {
#pragma unroll
          for (int r = 0; r < R; ++r) n.r[r] = sbvec4{n.r[r][1], n.r[r][2], n.r[r][3], 0.f};
        }
        return n;
      };
      Row now = request(0);
      Coef g_now = request_g(lo + c0);
      for (int i0 = 0; i0 < cnt; i0 += 4) {
        const Coef g_next = request_g(lo + c0 + i0 + 4);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const Row next = request(i0 + u + 1);
          if (lo + c0 + i0 + u < hi) {
            float g[R];
#pragma unroll
            for (int r = 0; r < R; ++r) g[r] = g_now.r[r][u];
            use(now.s, g);
          }
          now = next;
        }
        g_now = g_next;
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int x = 0; x < 4; ++x)
        finish_query_grad<M>(ModelOps<M>::prep(kept[r][0][x], NQ == 2 ? kept[r][NQ - 1][x] : 0.f), acc[r][0][x], acc[r][1][x], A.p);
  }

#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int h = 0; h < NK; ++h)
      part[((stretch * R + r) * NK + h) * kSbItems + item] = sbvec4{acc[r][h][0], acc[r][h][1], acc[r][h][2], acc[r][h][3]};
  __syncthreads();
  // thread -> (row, half) of its own item; the items of a workgroup are the same for every stretch
  const int which = t / kSbItems;
  if (which >= R * NK || (int)blockIdx.x * kSbItems + item >= n_items) return;
  sbvec4 sum = part[which * kSbItems + item];
#pragma unroll
  for (int s = 1; s < kSbStretches; ++s) sum += part[(s * R * NK + which) * kSbItems + item];
  const int r = which / NK, h = which - r * NK;
  float* out = ENTITY ? A.out1 + (size_t)(r0 + r) * (dim * MUL) + h * dim
                      : (h == 0 ? A.out1 : A.out2) + (size_t)(r0 + r) * dim;
  reinterpret_cast<sbvec4*>(out)[col] = sum;
}

// Rows per lane for a call, 0 where the kernels of one row per workgroup are the faster ones (or the shape is not this
// kernel's).  What decides is the number of workgroups the chip gets: more rows per lane make a step cheaper, fewer make
// more of them.  Measured, B x K x D, us (one row or two per workgroup / two rows per lane / four):
//   gradient rows  box 512 x 1024 x 400 60 / 54 / 47, 200 x 512 x 400 (800 workgroups of four) 17 / 13 / 12,
//                  512 x 1024 x 100 (400) 34 / 17 / 24, 100 x 128 x 100 (100 of two) 5.5 / 4.8 / 6.1;
//                  rotate, twice the registers, 512 x 1024 x 400 (1600) 82 / 60 / 71, 400 x 1000 x 500 (1953) 67 / 62 / 58
//   query          l1 512 x 1024 x 400 (800) 40 / 33 / 34, 1024 x 2048 x 500 166 / 162 / 109, 333 x 701 x 252 (331)
//                  18 / 16 / 22; rotate 1024 x 2048 x 200 (3200 of two) 167 / 154 / 157, 512 x 1024 x 400 (1600)
//                  78 / 75 / 79, 200 x 512 x 400 (625) 24 / 24 / 40; box, whose eight operations per pair are the time
//                  in either form, 61 / 62 / 63: stays with the kernel of one query per workgroup
inline int shared_backward_rows(int model, int vec, size_t B, size_t K, size_t ncol, bool entity) {
  if ((model != mL1 && model != mRotate && !(model == mBox && entity)) || vec != 4 || B < 4 || K < 4) return 0;
  const size_t kept = entity ? K : B;
  if (kept * ncol >= (1u << 30)) return 0;
  auto workgroups = [&](size_t rows) { return (kept + rows - 1) / rows * ncol / kSbItems; };
  if (entity) return workgroups(4) >= (model == mRotate ? 1900 : 600) ? 4 : (workgroups(2) >= 96 ? 2 : 0);
  if (model == mL1) return workgroups(4) >= 700 ? 4 : 0;
  return workgroups(2) >= 1600 ? 2 : 0;
}

// Instantiated once per model in its own translation unit (smx_shared_inst_*.hip).
template <int M, bool ENTITY, int R>
int launch_shared_backward(hipStream_t st, const SharedBwdArgs& A) {
  const size_t items = (size_t)((ENTITY ? A.K : A.B) + R - 1) / R * A.ncol;
  hipLaunchKernelGGL((shared_backward_kernel<M, ENTITY, R>), dim3((unsigned)((items + kSbItems - 1) / kSbItems)),
                     dim3(kSbThreads), 0, st, A);
  return check_launch(ENTITY ? "entity backward (shared negatives, columns)" : "score backward (shared negatives, columns)");
}
template <int M>
int shared_entity_columns(hipStream_t st, const SharedBwdArgs& A, int rows) {
  return rows == 4 ? launch_shared_backward<M, true, 4>(st, A) : launch_shared_backward<M, true, 2>(st, A);
}
template <int M>
int shared_query_columns(hipStream_t st, const SharedBwdArgs& A) {
  return launch_shared_backward<M, false, M == mL1 ? 4 : 2>(st, A);
}

}  // namespace smx
