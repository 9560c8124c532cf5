// Which kernel a call of the dense operators' backward gets: rules on sizes and alignment alone, so that they can be asked
// where there is no device (smx_measure_dense_backward_form).
#pragma once
#include <cstddef>

namespace smx {

struct Layout {
  size_t bsize, num, be, ne, bc, nc, dim;
};

enum BackwardPath { kPathGeneral = 0, kPathPerQuery = 1, kPathShared = 2, kPathReverse = 3 };

// vec: floats per column of a row, waves: wavefronts of the workgroup that a query gets (both 0 where the path has no choice)
struct BackwardForm {
  int path, vec, waves;
};

constexpr int kPqBwdWaves = 8;

// HIP counts the threads of a launch in 32 bits.
constexpr bool launchable(size_t workgroups, size_t waves) { return workgroups < (1ull << 32) / (waves * 64); }

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

// halves: of an entity row.  Batches and row counts whose launch HIP would refuse take the general kernels, whose workgroups
// are of two wavefronts (and one per row on either side).
inline BackwardForm dense_backward_form(const Layout& L, int halves, size_t low) {
  if (per_query_layout(L)) {
    const int vec = column_floats(L, low);
    if (vec == 0 || !launchable(L.bsize, kPqBwdWaves)) return {kPathGeneral, 0, 0};
    const size_t ncol = L.dim / vec;
    // Sixteen wavefronts for short rows, and for few queries: a CU has one workgroup, or none.  Eight / sixteen, box
    // 64 x 512 x 400 32 / 25 us, 512 x 512 x 100 42 / 37; two halves of long rows, BetaE 200 x 200 x 400, are slower with
    // sixteen: 134 / 234, the registers do not suffice.
    const bool many = vec == 4 && (ncol <= 32 || (halves == 1 && ncol <= 128 && L.bsize <= 256));
    return {kPathPerQuery, vec, many && launchable(L.bsize, 16) ? 16 : kPqBwdWaves};
  }
  if (shared_layout(L)) {
    const int vec = column_floats(L, low);
    if (vec == 0 || !launchable(L.bsize, kPqBwdWaves) || !launchable(L.num, kPqBwdWaves)) return {kPathGeneral, 0, 0};
    return {kPathShared, vec, kPqBwdWaves};
  }
  if (reverse_layout(L) && rows_of_16_bytes(L, low)) return {kPathReverse, 4, kPqBwdWaves};
  return {kPathGeneral, 0, 0};
}

}  // namespace smx
