// Point sources and coupling terms of a tile: lists of entries, each adding
// one value to one point of the tile, whose order at a point is fixed.
//
// One wavefront handles a tile's list in groups of 64 entries, a lane each,
// so the entries' loads are in flight together.  Entries of a group that
// name the same point are added in list order: each carries its rank among
// the group's earlier entries at its point, and the lanes add rank by rank.
// One thread walking the list instead waits for every entry's dependent loads
// in turn: a coupled 300x200-element step, whose interface tiles hold 40
// entries per medium, took 61.7 us that way and takes 41.7 us.
#pragma once

#include <cstdint>
#include <vector>

namespace smx {

constexpr int ENTRY_GROUP = 64; // entries a wavefront adds together
constexpr int ENTRY_RANK = 16;  // bits of the code below the rank

// Code of every entry of one tile's list li[off .. off + n): the tile-local
// point and the entry's rank in its group (both below 65536).
inline void entry_codes(const std::vector<int32_t> &li, int off, int n,
                        std::vector<int32_t> &code) {
  for (int k = 0; k < n; ++k) {
    int rank = 0;
    for (int j = k / ENTRY_GROUP * ENTRY_GROUP; j < k; ++j)
      rank += li[off + j] == li[off + k];
    code[off + k] = li[off + k] | (rank << ENTRY_RANK);
  }
}

#ifdef __HIPCC__
// Adds a group's entries: code < 0 for a lane without one; add(point).
// Called by a whole wavefront.
template <typename F>
__device__ __forceinline__ void add_entry_group(int code, F add) {
  for (int r = 0; __any((code >> ENTRY_RANK) >= r); ++r) {
    if ((code >> ENTRY_RANK) == r)
      add(code & ((1 << ENTRY_RANK) - 1));
    // rank r's sums before rank r + 1's: the barrier keeps the wavefront's
    // order of execution, the fences the compiler's order of the accesses
    // (another lane's sum; within a wavefront they cost no instruction)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}
#endif

} // namespace smx
