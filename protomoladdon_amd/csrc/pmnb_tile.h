// Column grid and wave helpers of the tile path (the pair kernels are in
// pmnb_cluster.h and pmnb_adjoint.h).
//
// Cell grid: x/y columns at least half a cutoff wide (a neighbour's column
// offset is -2 .. 2) and z cells of about an eighth of the cutoff; atoms are
// sorted column by column and by z (then atom index) inside a column, so a
// column's z-range of cells is one contiguous run of the sorted arrays (two
// when it wraps).  A work item is 16 consecutive sorted atoms of one column:
// with columns of half a cutoff its atoms fill a box of about 4.9 x 4.9 x 6 A
// (96,000-atom water, 9 A cutoff), whose cutoff shell holds 750 candidates
// of which a third are pairs; columns of a whole cutoff hold 980.
#pragma once

#include "pmnb_common.h"
#include "pmnb_pair.h"

namespace pmnb {

constexpr int kTileAtoms = 16;   // atoms per wave

struct TileGrid {
  int nx, ny, nz;       // grid
  float csx, csy, csz;  // cell sizes
  float lox, loy, loz;  // ... and what rounding to FP32 left of them
};

__device__ __forceinline__ void wave_sync_lds() {
  // LDS written by some lanes of this wave is read by other lanes next.
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int lane_prefix(unsigned long long mask) {
  return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
}

}  // namespace pmnb
