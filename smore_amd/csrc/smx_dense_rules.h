// Which kernel a call of the dense operators gets: rules on sizes and alignment alone, so that they can be asked where there
// is no device (smx_measure_dense_backward_form, smx_measure_dense_forward_form).
#pragma once
#include <cstddef>

#include "smx_functors.h"

namespace smx {

struct Layout {
  size_t bsize, num, be, ne, bc, nc, dim;
};

enum BackwardPath { kPathGeneral = 0, kPathPerQuery = 1, kPathShared = 2, kPathReverse = 3 };

// vec: floats per column of a row; waves: wavefronts of the workgroup that a query gets; ahead: a wavefront has its next row
// on the way while it works on one.  (0 where the path has no choice.)
struct BackwardForm {
  int path, vec, waves, ahead;
};

constexpr int kPqBwdWaves = 8;

// Kinds bound by their arithmetic (logarithms, digamma and trigamma functions), not by their rows' way from memory.
constexpr bool kind_heavy(int kind) { return kind == kBetaKL || kind == kBetaFisher; }

// HIP counts the threads of a launch in 32 bits.
constexpr bool launchable(size_t workgroups, size_t waves) { return workgroups < (1ull << 32) / (waves * 64); }

// Row and query counts that the kernels step through by up to 2 x 16 with an int.
constexpr bool steppable(size_t n) { return n <= 0x7fffffffull - 32; }

// The layouts of the kernels below; low: the addresses of all tensors or'ed together.
inline bool rows_of_16_bytes(const Layout& L, size_t low) { return L.dim % 4 == 0 && L.dim <= 1024 && (low & 15) == 0; }
inline bool per_query_layout(const Layout& L) {   // entity [B,N,.] against query [B,1,.]
  return L.be == L.bsize && L.bc == L.bsize && L.ne == L.num && L.nc == 1 && L.bsize * L.num <= 0x7fffffffull;
}
inline bool shared_layout(const Layout& L) {   // entity [1,N,.] shared by the queries [B,1,.]
  return L.be == 1 && L.bc == L.bsize && L.ne == L.num && L.nc == 1 && L.bsize >= 2 && L.bsize * L.num <= 0x7fffffffull;
}
inline bool reverse_layout(const Layout& L) {   // entity [B,1,.] against query [B,N,.]
  return L.be == L.bsize && L.bc == L.bsize && L.ne == 1 && L.nc == L.num && L.num >= 2 && L.bsize * L.num <= 0x7fffffffull;
}

// Rows that are not made of 16-byte columns take 8- or 4-byte ones up to 512 floats.  (The general kernels form each row's and
// each query's gradient by itself: rotate 300 x 333 x 250 571 us against 76 here, box 300 x 333 x 201 487 against 31, L1
// 100 x 400 x 330 666 against 30; rows shared by the queries, L1 512 x 1024 x 330 2,378 against 135, box 300 x 500 x 283 1,132
// against 66.)
inline int column_floats(const Layout& L, size_t low) {
  if (rows_of_16_bytes(L, low)) return 4;
  if (L.dim > 512) return 0;
  return L.dim % 2 == 0 && (low & 7) == 0 ? 2 : 1;
}

// Wavefronts per query and whether they read ahead, us a call:
// Few rows: a wavefront each (two rows for the arithmetic-bound kinds), because one without a row takes registers and LDS from
// other queries.  (Up to eight rows: of their workgroups of five wavefronts and more a CU holds one.)  Eight wavefronts / this,
// box 16384 x 1 x 400 37 / 25, 262144 x 1 x 32 254 / 62, rotate 16384 x 1 x 100 23 / 11, BetaE 16384 x 1 x 400 378 / 64,
// 4096 x 8 x 400 134 / 97.
// Few queries: a CU has one workgroup of the launch, or none, and sixteen wavefronts.  Eight / sixteen, box 64 x 512 x 400
// 33 / 25, 256 x 512 x 100 29 / 22, 512 x 512 x 32 36 / 26, BetaE 256 x 512 x 100 156 / 137.  Not rows of two long halves,
// whose registers do not suffice (BetaE 300 x 333 x 400 408 / 663), nor larger batches (box 1024 x 256 x 100 35 / 41).
// Reading ahead costs registers and, for the last row, a read.  Short rows of many queries do without, their wavefronts being
// many (box 600 x 512 x 100 49 / 44, L1 16384 x 16 x 64 31 / 29, complex 1024 x 512 x 200 347 / 337 us with / without), and so
// do long rows of the arithmetic-bound kinds, which it makes spill (BetaE 512 x 128 x 600 395 / 278).  With / without where it
// stays: box 1024 x 512 x 200 174 / 181, 64 x 512 x 400 33 / 41, rotate 8192 x 32 x 400 307 / 324, BetaE 300 x 333 x 400 408 / 462.
inline BackwardForm per_query_form(const Layout& L, int kind, int vec) {
  const size_t ncol = L.dim / vec;
  const bool one_half = kind_mul(kind) == 1;
  if (kind_heavy(kind) && L.num <= 8) return {kPathPerQuery, vec, (int)(L.num + 1) / 2, 0};
  if (L.num < kPqBwdWaves) return {kPathPerQuery, vec, (int)L.num, 0};
  if (vec == 4) {
    const size_t sixteen = ncol <= 32 ? (one_half ? 512 : 256) : one_half && ncol <= 128 ? 256 : 0;
    if (L.bsize <= sixteen && L.num >= 128) return {kPathPerQuery, vec, 16, 1};
    if (kind_heavy(kind)) return {kPathPerQuery, vec, kPqBwdWaves, ncol <= 128};
    if (ncol <= (one_half ? 32 : 64) && L.bsize > 256) return {kPathPerQuery, vec, kPqBwdWaves, 0};
  }
  return {kPathPerQuery, vec, kPqBwdWaves, 1};
}

// Batches and row counts whose launch HIP would refuse take the general kernels, whose workgroups are of two wavefronts (and
// one per row on either side).
inline BackwardForm dense_backward_form(const Layout& L, int kind, size_t low) {
  if (per_query_layout(L)) {
    const int vec = column_floats(L, low);
    if (vec == 0 || !steppable(L.num)) return {kPathGeneral, 0, 0, 0};
    const BackwardForm form = per_query_form(L, kind, vec);
    return launchable(L.bsize, form.waves) ? form : BackwardForm{kPathGeneral, 0, 0, 0};
  }
  if (shared_layout(L)) {
    const int vec = column_floats(L, low);
    if (vec == 0 || !steppable(L.num) || !steppable(L.bsize) || !launchable(L.bsize, kPqBwdWaves) || !launchable(L.num, kPqBwdWaves))
      return {kPathGeneral, 0, 0, 0};
    return {kPathShared, vec, kPqBwdWaves, !(kind_heavy(kind) && vec == 4 && L.dim > 512)};
  }
  if (reverse_layout(L) && steppable(L.num) && rows_of_16_bytes(L, low)) return {kPathReverse, 4, kPqBwdWaves, 0};
  return {kPathGeneral, 0, 0, 0};
}

// Per-query, shared and reverse forward: rows per workgroup, enough workgroups to fill the chip, at least eight rows each when
// there are that many.  A tile's end, and a row number stepped by eight beyond it, are ints in those kernels.
struct ForwardForm {
  int path, rows_per_tile;
};

inline ForwardForm dense_forward_form(const Layout& L, size_t low) {
  const ForwardForm general = {kPathGeneral, 0};
  if (!rows_of_16_bytes(L, low)) return general;
  const int path = per_query_layout(L) ? kPathPerQuery : shared_layout(L) ? kPathShared : reverse_layout(L) ? kPathReverse : kPathGeneral;
  if (path == kPathGeneral) return general;
  size_t rows = L.num;
  auto tiles = [&] { return (L.num + rows - 1) / rows; };
  while (rows > 8 && L.bsize * tiles() < 8192) rows = (rows + 1) / 2;
  if (!steppable(L.num + rows) || !launchable(L.bsize * tiles(), 4)) return general;
  return {path, (int)rows};
}

}  // namespace smx
