// The entries of a wavefront's slab of staged pairs (smx_score_impl.h): where a pair goes and in which order entries are
// asked for.  Index arithmetic alone, for host and device, so that its bounds can be checked where there is no device
// (smx_measure_slab_walk): an entry asked for is read and used as an address, whether its row is used or not.
#pragma once
#include <hip/hip_runtime.h>

namespace smx {

constexpr int kSlabEntries = 64;   // of a wavefront, one per lane

// Entry of the pair in `lane` of a batch of cnt, `n_singles` of which are finished on their own (`singles_below` of them in
// lower lanes): the others first, both kinds in pair order, because the others are streamed in groups from entry 0 on.
// Entries from cnt on keep what their lanes hold, a copy of the batch's last pair.
__host__ __device__ constexpr int slab_place(int lane, int cnt, int n_singles, bool single, int singles_below) {
  return lane >= cnt ? lane : (single ? cnt - n_singles + singles_below : lane - singles_below);
}

// Rows are requested in groups of rif entries, from entry 0 of the slab on; the last group of cnt entries (1 .. 64) starts at
// a multiple of rif as well, so that the entries asked for are of the slab, at most rif - 1 of them past cnt.
__host__ __device__ constexpr int last_group(int cnt, int rif) { return ((cnt - 1) / rif) * rif; }

}  // namespace smx
