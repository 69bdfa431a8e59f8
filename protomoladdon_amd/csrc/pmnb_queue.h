// Pieces the tile path's kernels share: the geometry of one replica (TileRep),
// the per-replica reduction of the items' partial rows in a fixed order
// (finish_rep_block), fixed-point conversion and scalar-register helpers.
//
// Each replica has its own column grid (TileRep): x/y columns at least half
// a pair cutoff wide, so a neighbour's column offset is -2 .. 2.  On an axis
// with fewer than four columns (box shorter than 2 cutoffs; FP64: five, 2.5
// cutoffs) every column is taken once with the minimum image of every pair along it (as z is when
// the cutoff reaches all z cells), so small boxes keep the reference's
// one-image pair set.
#pragma once

#include <type_traits>

#include "pmnb_cells.h"
#include "pmnb_list.h"
#include "pmnb_tile.h"

namespace pmnb {

constexpr int kQLj = 64;      // LJ table entries held in LDS
constexpr int kQTypeShift = 24;  // bits of an atom index beside its type

// Geometry of one replica on the tile path.  Its atoms occupy the sorted
// slots atom_off ..; they are sorted in bins (a bin: fz z cells of one
// column), and its work items (16 consecutive atoms of a bin) occupy the
// item slots item_off .. item_off + item_max - 1.
struct TileRep {
  Box box;            // FP64 box: minimum image of pairs near the cutoff
  Grid grid;          // FP64 column grid (cell assignment)
  TileGrid tg;        // FP32 cell sizes
  float L[3], iL[3];  // box lengths and inverses
  float Llo[3];       // what rounding the lengths to FP32 left of them
  int wrap[2];        // x, y: per-pair minimum image, each column once
  int cell_off;       // first global cell of the replica
  int bin_off, nbin;  // its bins: (column) * ns + z cell / fz
  int ns, fz;         // bins per column, z cells per bin
  int grp_off;        // its sums of kBinGroup bins start here (-1: none)
  int atom_off, natom;  // first sorted slot (= first atom), atoms
  int item_off, item_max;  // its item slots
};

// Bin of the cell (cx, cy, cz) of a replica, global.
__device__ __forceinline__ int tile_bin(const TileRep &R, int cx, int cy,
                                        int cz) {
  return R.bin_off + (cx * R.grid.n[1] + cy) * R.ns + cz / R.fz;
}

// 64-bit fixed point (2^-32) of an FP32 value, saturating beyond +-2^31;
// equal to to_fixed((double)v).
__device__ __forceinline__ long long to_fixed_f32(float v) {
  v = fminf(fmaxf(v, -2147483520.f), 2147483520.f);
  return (long long)rintf(v * 4294967296.f);
}

// The box of a rare path (pairs near the cutoff, molecule centres): the
// pointer passes through an empty asm statement, so the loads of the box
// fields stay in that branch instead of being hoisted into scalar
// registers held across the whole work item.  The pointer must be equal on
// all lanes (one replica per work item); it is read from the first lane, so
// it sits in scalar registers whatever the compiler infers.
__device__ __forceinline__ const Box &rare_box(const Box *b) {
  const unsigned long long v = (unsigned long long)b;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
  b = (const Box *)(((unsigned long long)hi << 32) | lo);
  __asm__ volatile("" : "+s"(b));
  return *b;
}

// Marks a value equal on all lanes as wave-uniform (scalar register), so the
// loops and branches it controls compile to scalar control flow.
__device__ __forceinline__ int uni(int v) {
  return __builtin_amdgcn_readfirstlane(v);
}
__device__ __forceinline__ float uni(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// Per-replica sum of one accumulator of the item partials (accumulator k
// of item b at partial[k * pstride + b]) by one block of 1024 threads with
// a fixed reduction tree, added into out[20 r + ..]:
// [0] LJ, [1] electrostatic, [2..10] virial 3x3, [11..19] molecular virial.
__device__ __forceinline__ void finish_rep_block(
    const double *__restrict__ partial, int pstride,
    const TileRep *__restrict__ reps, const int *__restrict__ rep_items,
    double *__restrict__ out, int r, int k, int fresh = 0) {
  __shared__ double red[16];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int i0 = reps[r].item_off, i1 = i0 + rep_items[r];
  const double *pk = partial + (size_t)k * pstride;
  // four independent sums per thread, so the loads overlap
  double v0 = 0.0, v1 = 0.0, v2 = 0.0, v3 = 0.0;
  int b = i0 + (int)threadIdx.x;
  for (; b + 3072 < i1; b += 4096) {
    v0 += pk[b];
    v1 += pk[b + 1024];
    v2 += pk[b + 2048];
    v3 += pk[b + 3072];
  }
  for (; b < i1; b += 1024) v0 += pk[b];
  double v = (v0 + v1) + (v2 + v3);
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  if (lane == 0) red[wave] = v;
  __syncthreads();
  if (threadIdx.x != 0) return;
  v = 0.0;
  for (int w = 0; w < 16; w++) v += red[w];
  double *o = out + 20 * r;
  // fresh: every one of the 20 slots is written by exactly one accumulator
  auto put = [&](int slot) { o[slot] = fresh ? v : o[slot] + v; };
  if (k < 2) {
    put(k);
  } else {
    const int base = k < ACC_MXX ? 2 : 11;
    const int u = k < ACC_MXX ? k - ACC_VXX : k - ACC_MXX;
    // u: 0 xx, 1 xy, 2 xz, 3 yy, 4 yz, 5 zz
    switch (u) {
      case 0: put(base + 0); break;
      case 1: put(base + 1); put(base + 3); break;
      case 2: put(base + 2); put(base + 6); break;
      case 3: put(base + 4); break;
      case 4: put(base + 5); put(base + 7); break;
      default: put(base + 8); break;
    }
  }
}

}  // namespace pmnb
