// Cell build of the tile path in two launches: atoms into bins (a bin is fz
// z cells of one x/y column, about 256 atoms at most on average), then one
// block per bin sorts its atoms by z and writes the sorted arrays, the
// bounds of its z cells and its work items.
//
// Bins, not z cells, are counted: 400 instead of 3,200 on the 96,000-atom
// water, so that every block finds its first slot and first item by adding
// the counts of its replica's earlier bins itself, with no scan launch
// between the two kernels (a replica of thousands of bins gets sums of groups
// of bins in a launch of its own).  A replica's atoms and item slots start at
// offsets fixed on the host.
#pragma once

#include "pmnb_queue.h"

namespace pmnb {

constexpr int kBinSort = 1024;  // atoms a block sorts in LDS
constexpr int kBinCells = 256;  // most z cells of a bin
constexpr int kBinGroup = kBlock;  // bins of a sum of k_bin_groups
// Replicas of more bins than this get their counts added by groups first (a
// launch of 4 us).  An evaluation without / with the groups: 4,608 bins 1,263 /
// 1,261 us (1,029,000 atoms), 17,000 bins 369 / 331 (32,000 atoms), 35,000 bins
// 251 / 83 (900 atoms), 98,000 bins 2,513 / 1,019 (999,000 atoms).
constexpr int kGroupBins = 4096;

// Bin of every atom.  Bins of a block's atoms are few (consecutive atoms are
// neighbours): the block counts its atoms per bin in an LDS table (open
// addressing), takes one global atomic add per distinct bin, all issued
// together, and gives each atom the bin's base plus its rank in the block:
// its arrival rank in the bin, at which it is written into the bin's row of
// `bucket` (cap entries per bin; an atom ranked beyond cap is found again
// from bin_of by k_sort_bins).  With pos_copy the positions read (from host
// memory mapped into the device, say) are also stored there for the kernels
// after this one.  Requires blockDim.x == kBlock.
__global__ void __launch_bounds__(kBlock)
k_assign_bins(const TileRep *__restrict__ reps, const int *__restrict__ rep_of,
              const double *__restrict__ pos, int n, int *__restrict__ bin_of,
              int *__restrict__ count, int *__restrict__ bucket, int cap,
              double *__restrict__ pos_copy) {
  __shared__ int key[kBlock], lcount[kBlock], base[kBlock];
  const int t = threadIdx.x;
  const int i = blockIdx.x * kBlock + t;
  key[t] = -1;
  lcount[t] = 0;
  __syncthreads();
  int slot = -1, lrank = 0, c = 0;
  if (i < n) {
    const TileRep &R = reps[rep_of ? rep_of[i] : 0];
    int cx, cy, cz;
    double vx, vy, vz;
    const double px = pos[3 * i], py = pos[3 * i + 1], pz = pos[3 * i + 2];
    if (pos_copy) {
      pos_copy[3 * i] = px;
      pos_copy[3 * i + 1] = py;
      pos_copy[3 * i + 2] = pz;
    }
    cell_coords(R.box, R.grid, px, py, pz, cx, cy, cz, vx, vy, vz);
    c = tile_bin(R, cx, cy, cz);
    bin_of[i] = c;
    // at most kBlock distinct bins in kBlock slots: the probe ends
    int h = c & (kBlock - 1);
    while (true) {
      const int old = atomicCAS(&key[h], -1, c);
      if (old == -1 || old == c) break;
      h = (h + 1) & (kBlock - 1);
    }
    slot = h;
    lrank = atomicAdd(&lcount[h], 1);
  }
  __syncthreads();
  if (key[t] >= 0) base[t] = atomicAdd(&count[key[t]], lcount[t]);
  __syncthreads();
  if (i < n) {
    const int r = base[slot] + lrank;
    if (r < cap) bucket[(size_t)c * cap + r] = i;
  }
}

// Atoms and items of each group of kBinGroup bins of replica r, so that a
// block of k_sort_bins adds groups instead of all earlier bins; the item slots
// are emptied here for those replicas.  One block per group.
__global__ void __launch_bounds__(kBinGroup)
k_bin_groups(const TileRep *__restrict__ reps, int r,
             const int *__restrict__ count, int2 *__restrict__ group,
             int4 *__restrict__ items) {
  __shared__ int red[2][kBinGroup / 64];
  const TileRep &R = reps[r];
  const int t = threadIdx.x, k = blockIdx.x * kBinGroup + t;
  const int c = k < R.nbin ? count[R.bin_off + k] : 0;
  int sa = c, si = (c + kTileAtoms - 1) / kTileAtoms;
  for (int o = 32; o > 0; o >>= 1) {
    sa += __shfl_down(sa, o, 64);
    si += __shfl_down(si, o, 64);
  }
  if ((t & 63) == 0) {
    red[0][t >> 6] = sa;
    red[1][t >> 6] = si;
  }
  for (int j = k; j < R.item_max; j += gridDim.x * kBinGroup)
    items[R.item_off + j] = make_int4(0, 0, 0, 0);
  __syncthreads();
  if (t == 0) {
    sa = si = 0;
#pragma unroll
    for (int w = 0; w < kBinGroup / 64; w++) {
      sa += red[0][w];
      si += red[1][w];
    }
    group[R.grp_off + blockIdx.x] = make_int2(sa, si);
  }
}

// A double as an integer of the same order (a total order, NaN included).
__device__ __forceinline__ long long order_key(double v) {
  const long long b = __double_as_longlong(v);
  return b < 0 ? b ^ 0x7fffffffffffffffll : b;
}

// The sorted arrays of the tile path.
struct BinOut {
  int *sorted;              // atom of each slot
  double *sx, *sy, *sz, *sq;
  float4 *sloc;             // FP32 offset from the cell's lower corner
                            // (computed in FP64), charge
  int *stype, *smol, *scell;
  unsigned *srec;           // atom << 8 | type
  int *cstart, *ccount;     // per z cell: first slot, atoms
  int4 *items;              // {first slot, end slot, local column, replica}
  int *rep_items;           // items of each replica
  unsigned long long *npairs;  // pair counter, cleared here
  const int2 *group;        // sums of k_bin_groups
};

// One block per bin.  The atoms (from the bin's bucket row or, beyond its
// capacity, from bin_of) are counted per z cell in LDS, placed cell by cell,
// and ranked inside their cell by (z, atom index): three atoms per cell on
// water, so the rank is a handful of LDS reads, and the result does not
// depend on the arrival order.  Bins of more than kBinSort atoms (a part of
// the box several times denser than the mean, positions that are not finite)
// are sorted by z cell and atom index from global memory, in time linear in
// their atoms and the replica's: 96,000 atoms without a finite position, all of
// them in one z cell, take 3.2 ms an evaluation.
// GROUPS: there are sums of k_bin_groups (their code costs 0.2 us of 7 on 3,000
// atoms).
template <bool GROUPS>
__global__ void __launch_bounds__(kBlock)
k_sort_bins(const TileRep *__restrict__ reps, const int *__restrict__ bin_rep,
            const double *__restrict__ pos, const int *__restrict__ count,
            const int *__restrict__ bucket, int cap,
            const int *__restrict__ bin_of, const int *__restrict__ type,
            const double *__restrict__ q, const int *__restrict__ mol,
            BinOut O) {
  constexpr int NW = kBlock / 64, NU = kBinSort / kBlock;
  __shared__ long long kz[kBinSort];
  __shared__ int ka[kBinSort];
  __shared__ unsigned char kf[kBinSort];
  __shared__ int hist[kBinCells], first[kBinCells];
  __shared__ int red[2][NW], wsum[NW], found;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int b = blockIdx.x;
  const int r = bin_rep ? bin_rep[b] : 0;
  const TileRep &R = reps[r];
  const int lb = b - R.bin_off, m = count[b];
  const int col = lb / R.ns, z0 = (lb - col * R.ns) * R.fz;
  const int nf = max(0, min(R.fz, R.tg.nz - z0));
  if (b == 0 && t == 0) *O.npairs = 0ull;
  hist[t] = 0;
  if (t == 0) found = 0;
  // first slot and first item: the replica's earlier bins
  int sa = 0, si = 0;
  const bool grouped = GROUPS && R.grp_off >= 0;
  const int g0 = grouped ? lb / kBinGroup : 0;
  for (int k = t; k < g0; k += kBlock) {
    const int2 g = O.group[R.grp_off + k];
    sa += g.x;
    si += g.y;
  }
  for (int k = g0 * kBinGroup + t; k < lb; k += kBlock) {
    const int c = count[R.bin_off + k];
    sa += c;
    si += (c + kTileAtoms - 1) / kTileAtoms;
  }
  for (int o = 32; o > 0; o >>= 1) {
    sa += __shfl_down(sa, o, 64);
    si += __shfl_down(si, o, 64);
  }
  if (lane == 0) {
    red[0][w] = sa;
    red[1][w] = si;
  }
  __syncthreads();
  sa = si = 0;
#pragma unroll
  for (int k = 0; k < NW; k++) {
    sa += red[0][k];
    si += red[1][k];
  }
  const int s0 = R.atom_off + sa, i0 = R.item_off + si;
  const int ni = (m + kTileAtoms - 1) / kTileAtoms;
  for (int k = t; k < ni; k += kBlock)
    O.items[i0 + k] = make_int4(s0 + k * kTileAtoms,
                                min(s0 + (k + 1) * kTileAtoms, s0 + m), col, r);
  if (lb == R.nbin - 1) {
    // the replica's unused item slots are empty
    if (t == 0) O.rep_items[r] = si + ni;
    for (int k = si + ni + t; k < R.item_max && !grouped; k += kBlock)
      O.items[R.item_off + k] = make_int4(0, 0, 0, 0);
  }
  // z cell (in the bin) and order key of atom a
  auto place = [&](int a, int &f, long long &key) {
    int cx, cy, cz;
    double vx, vy, vz;
    cell_coords(R.box, R.grid, pos[3 * a], pos[3 * a + 1], pos[3 * a + 2], cx,
                cy, cz, vx, vy, vz);
    f = min(max(cz - z0, 0), nf - 1);
    key = order_key(vz);
  };
  // slot s receives atom a
  auto put = [&](int s, int a) {
    const double x = pos[3 * a], y = pos[3 * a + 1], z = pos[3 * a + 2];
    int cx, cy, cz;
    double vx, vy, vz;
    cell_coords(R.box, R.grid, x, y, z, cx, cy, cz, vx, vy, vz);
    float4 l;
    l.x = (float)(vx - (double)cx * R.grid.cs[0]);
    l.y = (float)(vy - (double)cy * R.grid.cs[1]);
    l.z = (float)(vz - (double)cz * R.grid.cs[2]);
    l.w = (float)q[a];
    O.sorted[s] = a;
    O.sx[s] = x;
    O.sy[s] = y;
    O.sz[s] = z;
    O.sq[s] = q[a];
    O.sloc[s] = l;
    O.stype[s] = type[a];
    O.smol[s] = mol[a];
    O.scell[s] = R.cell_off + col * R.tg.nz + cz;
    O.srec[s] = ((unsigned)a << 8) | (unsigned)type[a];
  };
  // first[] from hist[], and the cells' bounds (block-wide)
  auto cells = [&]() {
    __syncthreads();
    int v = hist[t], x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    int off = 0;
#pragma unroll
    for (int k = 0; k < NW; k++) off += k < w ? wsum[k] : 0;
    first[t] = off + x - v;
    if (t < nf) {
      const int c = R.cell_off + col * R.tg.nz + z0 + t;
      O.cstart[c] = s0 + off + x - v;
      O.ccount[c] = v;
    }
    __syncthreads();
  };
  if (m <= kBinSort) {
    const int *src = bucket + (size_t)b * cap;
    if (m > cap) {
      for (int i = t; i < R.natom; i += kBlock)
        if (bin_of[R.atom_off + i] == b) ka[atomicAdd(&found, 1)] = R.atom_off + i;
      src = ka;
    }
    __syncthreads();
    int a[NU], f[NU], rk[NU];
    long long key[NU];
#pragma unroll
    for (int u = 0; u < NU; u++) {
      const int k = t + u * kBlock;
      if (k < m) {
        a[u] = src[k];
        place(a[u], f[u], key[u]);
        rk[u] = atomicAdd(&hist[f[u]], 1);
      }
    }
    cells();
#pragma unroll
    for (int u = 0; u < NU; u++) {
      if (t + u * kBlock < m) {
        const int s = first[f[u]] + rk[u];
        ka[s] = a[u];
        kz[s] = key[u];
        kf[s] = (unsigned char)f[u];
      }
    }
    __syncthreads();
    for (int k = t; k < m; k += kBlock) {
      const int ak = ka[k], fk = kf[k];
      const long long zk = kz[k];
      const int lo = first[fk], hi = lo + hist[fk];
      int s = s0 + lo;
      for (int j = lo; j < hi; j++)
        s += (kz[j] < zk || (kz[j] == zk && ka[j] < ak)) ? 1 : 0;
      put(s, ak);
    }
  } else {
    // ascending list of the bin's atoms (in scell until the slots are written),
    // then a stable counting sort by z cell (cells in stype)
    int *list = O.scell + s0, *cell = O.stype + s0;
    constexpr int kRun = 16;
    int at = 0;
    __syncthreads();
    for (int i0 = 0; i0 < R.natom; i0 += kBlock * kRun) {
      const int i = i0 + t * kRun;
      unsigned mine = 0u;
#pragma unroll
      for (int u = 0; u < kRun; u++)
        if (i + u < R.natom && bin_of[R.atom_off + i + u] == b) mine |= 1u << u;
      const int v = __builtin_popcount(mine);
      int x = v;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
      }
      if (lane == 63) wsum[w] = x;
      __syncthreads();
      int k = at + x - v;
#pragma unroll
      for (int j = 0; j < NW; j++) {
        k += j < w ? wsum[j] : 0;
        at += wsum[j];
      }
      for (; mine; mine &= mine - 1, k++)
        if (k < m) list[k] = R.atom_off + i + __builtin_ctz(mine);
      __syncthreads();  // wsum is written again
    }
    __threadfence();
    __syncthreads();
    for (int k = t; k < m; k += kBlock) {
      int f;
      long long key;
      place(list[k], f, key);
      cell[k] = f;
      atomicAdd(&hist[f], 1);
    }
    cells();
    for (int k0 = 0; k0 < m; k0 += kBlock) {
      const int k = k0 + t, f = k < m ? cell[k] : -1;
      ka[t] = f;
      __syncthreads();
      int before = 0, all = 0;
      for (int j = 0; j < kBlock; j++) {
        all += ka[j] == f ? 1 : 0;
        before += ka[j] == f && j < t ? 1 : 0;
      }
      if (f >= 0) O.sorted[s0 + first[f] + before] = list[k];
      __syncthreads();
      if (f >= 0 && before == all - 1) first[f] += all;
    }
    __threadfence();
    __syncthreads();
    for (int k = t; k < m; k += kBlock) put(s0 + k, O.sorted[s0 + k]);
  }
}

}  // namespace pmnb
