// pmnb_pme.h -- smooth particle-mesh Ewald: the reciprocal term of
// ProtoMol's NonbondedPMEwaldSystemForce (mdl/interface/force/nonbonded/
// NonbondedPMEwaldSystemForce.h with Grid.h and BSpline.cpp) for an
// orthogonal periodic box.  Its correction, point-self and charged-system
// terms are the direct Ewald sum's (pmnb_ewald.h), computed by the same
// kernels.
//
// One evaluation:
//   k_pme_bin        one thread per atom: grid coordinates x = r n / L
//                    wrapped into [0, n) as Grid::anterpolateCharge does
//                    (Grid.h:107-131), written with the charge into the
//                    bucket of the atom's bin (4^3 grid cells); an atom
//                    beyond the bucket is spread at once, by atomic adds
//                    into an integer grid that is zero otherwise;
//   k_pme_spread     one block per tile of 8^3 grid points: the atoms of the
//                    bins that reach it, the B-spline weights of
//                    BSpline::set (BSpline.cpp:58-95), and q Mx My Mz summed
//                    over them in LDS as 64-bit fixed-point integers (2^-40),
//                    on top of what k_pme_bin spread:
//                    integer sums do not depend on the order of the adds, so
//                    the grid is the same bits on every run;
//   hipFFT D2Z       the unnormalised transform of the real grid (nx, ny,
//                    nz/2 + 1 half spectrum; the reference transforms the
//                    full complex grid, whose other half is the conjugate);
//   k_pme_scalar     one wave per row of the half spectrum,
//                    the loop of Grid::scalarSum (Grid.h:237-341): theta(m)
//                    = B(m) exp(-pi^2 m^2 / alpha^2) / (pi V m^2), energy
//                    and virial terms (doubled where the reference doubles
//                    them), the spectrum multiplied by theta; per-block sums
//                    in a fixed order; clears the bins for the next run;
//   hipFFT Z2D       back to the real, convolved grid;
//   k_pme_gather     two lanes per atom: the force -q grad (the convolved
//                    grid) n / L, interpolateForce's loop (Grid.h:171-199),
//                    plus the atom's correction pairs, with their energy and
//                    virial; no atomics;
//   k_ew_finish      the blocks' energy and virial sums, half of the grid's
//                    into the output (the reference returns energy * 0.5
//                    and adds virial * 0.5, Grid.h:316-326), and the
//                    correction, self and charged-system terms.
#pragma once

#include "pmnb_ewald.h"

namespace pmnb {

constexpr int kPmeBlock = 256;
constexpr int kPmeTile = 8;      // grid points of a spread tile, per axis
constexpr int kPmeBin = 4;       // grid cells of an atom bin, per axis
constexpr int kPmeList = 512;    // atoms of a tile listed in LDS
// From this order on a lane that finds a tile's list full spreads its atom
// alone: its weights are then formed once, not once a plane (96,000 atoms, 32^3,
// order 8: 1,432 us, 1,730 with another turn of the list; order 4: 376 and 318).
constexpr int kPmeLaneOrder = 6;
constexpr int kPmeRow = kPmeTile + 1;  // LDS row and plane strides of a tile:
constexpr int kPmePlane = kPmeTile * kPmeRow;  // an atom's planes on other banks
constexpr int kPmeScalarBlocks = 4096;
constexpr int kPmeLanes = 2;     // lanes per atom of the gather
// Charge grid resolution 2^-40: with order 8 on a 32^3 grid the rounding of
// 2^-32 moves forces by 1e-9 of the largest, 2^-40 by 3e-12.  A grid value
// must stay below 2^23 (8.4e6, about 4.6e5 elementary charges on one grid
// point) in magnitude; each contribution is clamped to 2^22.
constexpr double kPmeFixScale = 1099511627776.0;       // 2^40
constexpr double kPmeFixInv = 1.0 / 1099511627776.0;
constexpr double kPmeFixClamp = 4194304.0;             // 2^22

// Whether all charges are added in memory: grids of few tiles, of more than 64
// atoms each.  A whole evaluation of 96,000 atoms by tiles / in memory, orders
// 2, 4, 6 and 8: 27 tiles 312 / 70, 627 / 295, 1,420 / 951, 3,094 / 2,338 us; 64
// tiles 178 / 61, 318 / 270, 700 / 876, 1,430 / 2,052; 125 tiles 112 / 64, 183 /
// 226; 900 atoms, 27 tiles 42 / 41, 47 / 55, 63 / 93, 105 / 164.
inline bool pme_all_atomic(long long tiles, int order, int n_atoms) {
  const int few = order == 2 ? 200 : (order == 4 ? 100 : 64);
  return tiles < few && n_atoms / tiles > 64;
}

struct PmeDev {
  int n;                   // atoms
  int nx, ny, nz, nzh;     // grid, nz / 2 + 1
  double hr[3];            // n / L per axis
  int off[3];              // -(order - 1) / 2 + n per axis (Grid.h:509-511)
  double Lr[3];            // 1 / L per axis
  double piVr;             // 1 / (pi V)
  double fac;              // pi^2 / alpha^2
  const double *q;         // scaled charges
  int nb[3];               // atom bins per axis
  int *count;              // atoms per bin, then whether any is beyond its
                           // bucket (zero between runs)
  double4 *bucket;         // cap records {grid x, y, z, charge} per bin
  int cap;                 // 0: all atoms are spread by k_pme_bin
  unsigned long long *qfix;  // nx ny nz: charges of the atoms beyond their
                           // buckets, 2^-40 (zero between runs)
  double *qreal;           // nx ny nz real grid
  double2 *qk;             // nx ny nzh half spectrum
  const double *mod[3];    // B(m) per axis index (Grid::dftmod)
  const double *ex[3];     // exp(-fac m^2) per axis index (ex[2]: k <= nz/2)
  double *part;            // kEwSums rows of n_part scalar-sum blocks
  int n_part;              // scalar-sum blocks
  double *cpart;           // kEwSums rows of n_cpart gather blocks: the
                           // correction's energy and virial
  int n_cpart;
};

// BSpline::set(w) (BSpline.cpp:58-95) with compile-time order P >= 2, in
// the reference's operation order.
template <int P>
__device__ __forceinline__ void pme_bspline(double w, double (&th)[P],
                                            double (&dth)[P]) {
  if constexpr (P == 2) {
    th[1] = w;
    th[0] = 1.0 - w;
    dth[1] = 1.0;
    dth[0] = -1.0;
  } else {
    th[P - 1] = 0.0;
    th[1] = w;
    th[0] = 1.0 - w;
#pragma unroll
    for (int k = 2; k < P - 1; k++) {
      const double div = 1.0 / k;
      th[k] = div * w * th[k - 1];
#pragma unroll
      for (int j = 1; j < k; j++)
        th[k - j] = div * ((w + j) * th[k - j - 1] + (k + 1 - j - w) * th[k - j]);
      th[0] = div * (1 - w) * th[0];
    }
    dth[0] = -th[0];
#pragma unroll
    for (int j = 1; j <= P - 1; j++) dth[j] = th[j - 1] - th[j];
    const double div = 1.0 / (P - 1.0);
    th[P - 1] = div * w * th[P - 2];
#pragma unroll
    for (int j = 1; j < P - 1; j++)
      th[P - 1 - j] = div * ((w + j) * th[P - j - 2] + (P - j - w) * th[P - 1 - j]);
    th[0] = div * (1 - w) * th[0];
  }
}

// Grid coordinate of position p on an axis of n points: p n / L, brought
// into [0, n) by adding or subtracting n as the reference's while loops do
// (Grid.h:111-116); positions more than 64 boxes away and non-finite ones
// are folded in one step, so every loop ends.
__device__ __forceinline__ double pme_coord(double p, double hr, int n) {
  double x = p * hr;
  if (!(x == x) || x > 1e15 || x < -1e15) return 0.0;
  const double dn = (double)n;
  for (int it = 0; it < 64 && x < 0.0; it++) x += dn;
  for (int it = 0; it < 64 && x >= dn; it++) x -= dn;
  if (x < 0.0 || x >= dn) {
    x -= dn * floor(x / dn);
    if (!(x >= 0.0 && x < dn)) x = 0.0;
  }
  return x;
}

// Grid index b + u, b in [0, 2 n), u < n, brought below n.
__device__ __forceinline__ int pme_wrap(int g, int n) {
  g -= g >= 2 * n ? 2 * n : 0;
  return g >= n ? g - n : g;
}

// A contribution in units of 2^-40.  small: |value| <= |charge| < 2048, where
// adding 1.5 * 2^12 leaves the value rounded to 2^-40 in the low bits, the
// rounding of rint.
__device__ __forceinline__ unsigned long long pme_fixed(double val, bool small) {
  if (small)
    return (unsigned long long)__double_as_longlong(val + 6144.0) -
           0x40B8000000000000ull;
  val = fmin(fmax(val, -kPmeFixClamp), kPmeFixClamp);
  return (unsigned long long)(long long)__builtin_rint(val * kPmeFixScale);
}

// Spreads one atom into the integer grid in memory.
template <int P>
__device__ __forceinline__ void pme_spread_global(const PmeDev &d,
                                                  const double4 &r) {
  const int ix = (int)r.x, iy = (int)r.y, iz = (int)r.z;
  double tx[P], ty[P], tz[P], dth[P];
  pme_bspline<P>(r.x - ix, tx, dth);
  pme_bspline<P>(r.y - iy, ty, dth);
  pme_bspline<P>(r.z - iz, tz, dth);
  const bool small = fabs(r.w) < 2048.0;
#pragma unroll
  for (int u = 0; u < P; u++) {
    const size_t plane = (size_t)pme_wrap(ix + d.off[0] + u, d.nx) * d.ny;
    const double av = r.w * tx[u];
#pragma unroll
    for (int v = 0; v < P; v++) {
      unsigned long long *row =
          d.qfix + (plane + pme_wrap(iy + d.off[1] + v, d.ny)) * d.nz;
      const double ab = av * ty[v];
#pragma unroll
      for (int w = 0; w < P; w++)
        atomicAdd(row + pme_wrap(iz + d.off[2] + w, d.nz),
                  pme_fixed(ab * tz[w], small));
    }
  }
}

// The order in a bucket varies from run to run, and so does which atoms are
// beyond it; the integer sums do not.  A bucket holds four times the mean and
// at least 32 atoms (three times what a bin of water holds on a grid of 1.2 A),
// so that atoms are beyond it only on coarse grids, where they are much denser
// than on average.  32,000 atoms in a 68 A cube, 256^3 grid, with a list of
// those atoms that every tile reads / with their charges added in memory: box
// of 300 A 783 / 582 us (none beyond its bucket), of 830 A 1,472 / 693.
// A grid of few tiles leaves the chip idle in k_pme_spread, one block a tile;
// there (pme_all_atomic) all atoms are spread here and the tiles only convert.
template <int P>
__global__ __launch_bounds__(kPmeBlock) void k_pme_bin(PmeDev d,
                                                       const double *x) {
  const int i = blockIdx.x * kPmeBlock + threadIdx.x;
  if (i >= d.n) return;
  const double4 r = make_double4(pme_coord(x[3 * i], d.hr[0], d.nx),
                                 pme_coord(x[3 * i + 1], d.hr[1], d.ny),
                                 pme_coord(x[3 * i + 2], d.hr[2], d.nz), d.q[i]);
  const int b = (((int)r.x / kPmeBin) * d.nb[1] + (int)r.y / kPmeBin) * d.nb[2] +
                (int)r.z / kPmeBin;
  const int k = d.cap ? atomicAdd(d.count + b, 1) : 0;
  if (k < d.cap) {
    d.bucket[(size_t)b * d.cap + k] = r;
  } else {
    pme_spread_global<P>(d, r);
    d.count[(size_t)d.nb[0] * d.nb[1] * d.nb[2]] = 1;
  }
}

// Adds the contributions of stencil plane u of one atom that fall into the
// tile at t0 of extent te.
template <int P>
__device__ __forceinline__ void pme_spread_plane(const PmeDev &d,
                                                 const double4 &r, int u,
                                                 const int (&t0)[3],
                                                 const int (&te)[3],
                                                 unsigned long long *tile) {
  const int ix = (int)r.x, iy = (int)r.y, iz = (int)r.z;
  const int lx = pme_wrap(ix + d.off[0] + u, d.nx) - t0[0];
  if ((unsigned)lx >= (unsigned)te[0]) return;
  double tx[P], ty[P], tz[P], dth[P];
  pme_bspline<P>(r.x - ix, tx, dth);
  pme_bspline<P>(r.y - iy, ty, dth);
  pme_bspline<P>(r.z - iz, tz, dth);
  double mx = tx[0];
#pragma unroll
  for (int k = 1; k < P; k++) mx = u == k ? tx[k] : mx;
  const double av = r.w * mx;
  const bool small = fabs(r.w) < 2048.0;
#pragma unroll
  for (int v = 0; v < P; v++) {
    const int ly = pme_wrap(iy + d.off[1] + v, d.ny) - t0[1];
    if ((unsigned)ly >= (unsigned)te[1]) continue;
    const double ab = av * ty[v];
    unsigned long long *row = tile + lx * kPmePlane + ly * kPmeRow;
#pragma unroll
    for (int w = 0; w < P; w++) {
      const int lz = pme_wrap(iz + d.off[2] + w, d.nz) - t0[2];
      if ((unsigned)lz >= (unsigned)te[2]) continue;
      __hip_atomic_fetch_add(row + lz, pme_fixed(ab * tz[w], small),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }
}

// One block per tile of 8^3 grid points (fewer at the upper faces).  Its
// points are written by it alone, so no global atomics: 6.1 million of them
// took 156 us for 96,000 atoms of order 4 on a 96^3 grid, plus 8 us to convert
// and clear the integer grid; this kernel takes 27 us and k_pme_bin 9 (bound by
// its atomics' latency), this one by its LDS atomics (a tile with margins, which
// needs no test per point but adds 1.9 times as many, took 51).  Bins half a
// tile wide: 4 per axis reach a tile, 8 atoms are read for one of the tile's own
// (27 with bins of a tile).  The listed atoms are spread over the lanes by
// stencil plane, which evens out what the tile's edge cuts off.
template <int P>
__global__ __launch_bounds__(kPmeBlock) void k_pme_spread(PmeDev d) {
  __shared__ unsigned long long tile[kPmeTile * kPmePlane];
  __shared__ double4 list[kPmeList];
  __shared__ int nlist;
  const int t = threadIdx.x;
  const int nn[3] = {d.nx, d.ny, d.nz};
  const int nty = (d.ny + kPmeTile - 1) / kPmeTile,
            ntz = (d.nz + kPmeTile - 1) / kPmeTile;
  const int b = blockIdx.x;
  const int tc[3] = {b / (nty * ntz), b / ntz % nty, b % ntz};
  int t0[3], te[3], first[3], cnt[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    t0[a] = tc[a] * kPmeTile;
    te[a] = min(kPmeTile, nn[a] - t0[a]);
    // cells of the atoms that reach the tile: t0 - P / 2 .. end + (P - 1) / 2;
    // when they leave less than a bin of the axis, every bin once
    const int lo = t0[a] - P / 2, hi = t0[a] + te[a] - 1 + (P - 1) / 2;
    if (hi - lo + 1 > nn[a] - kPmeBin) {
      first[a] = 0;
      cnt[a] = d.nb[a];
    } else {
      first[a] = (lo < 0 ? lo + nn[a] : lo) / kPmeBin;
      const int last = (hi >= nn[a] ? hi - nn[a] : hi) / kPmeBin;
      cnt[a] = last - first[a] + (last < first[a] ? d.nb[a] : 0) + 1;
    }
  }
  const bool pre = d.count[(size_t)d.nb[0] * d.nb[1] * d.nb[2]] > 0;
  for (int k = t; k < kPmeTile * kPmeTile * kPmeTile; k += kPmeBlock) {
    const int lx = k / (kPmeTile * kPmeTile), ly = k / kPmeTile % kPmeTile,
              lz = k % kPmeTile;
    unsigned long long v = 0;
    if (pre && lx < te[0] && ly < te[1] && lz < te[2]) {
      unsigned long long *p =
          d.qfix + ((size_t)(t0[0] + lx) * d.ny + t0[1] + ly) * d.nz + t0[2] + lz;
      v = *p;
      *p = 0;
    }
    tile[lx * kPmePlane + ly * kPmeRow + lz] = v;
  }
  const int nbin = cnt[0] * cnt[1] * cnt[2];
  auto reach = [&](double c, int a) -> bool {  // the atom's stencil meets it
    int g = (int)c + d.off[a] - t0[a];  // first point, from the tile's
    g = g < 0 ? g + nn[a] : g;
    g = g >= 2 * nn[a] ? g - 2 * nn[a] : (g >= nn[a] ? g - nn[a] : g);
    return g < te[a] || g + P > nn[a];
  };
  // four lanes per bin, 64 bins a turn, as often as the list fills up
  for (int k0 = 0; k0 < nbin; k0 += 64) {
    const int k = k0 + (t >> 2);
    const double4 *rec = d.bucket;
    int s = t & 3, n = 0;
    if (k < nbin) {
      int bx = first[0] + k / (cnt[1] * cnt[2]),
          by = first[1] + k / cnt[2] % cnt[1], bz = first[2] + k % cnt[2];
      bx -= bx >= d.nb[0] ? d.nb[0] : 0;
      by -= by >= d.nb[1] ? d.nb[1] : 0;
      bz -= bz >= d.nb[2] ? d.nb[2] : 0;
      const int bin = (bx * d.nb[1] + by) * d.nb[2] + bz;
      n = min(d.count[bin], d.cap);
      rec += (size_t)bin * d.cap;
    }
    while (true) {
      if (t == 0) nlist = 0;
      __syncthreads();
      for (; s < n; s += 4) {
        const double4 r = rec[s];
        if (!(reach(r.x, 0) && reach(r.y, 1) && reach(r.z, 2))) continue;
        const int at = __hip_atomic_fetch_add(&nlist, 1, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_WORKGROUP);
        if (at < kPmeList) {
          list[at] = r;
        } else if (P < kPmeLaneOrder) {
          break;  // again when the list is spread
        } else {
          for (int u = 0; u < P; u++)
            pme_spread_plane<P>(d, r, u, t0, te, tile);
        }
      }
      __syncthreads();
      const int listed = nlist;
      const int items = min(listed, kPmeList) * P;
      for (int j = t; j < items; j += kPmeBlock)
        pme_spread_plane<P>(d, list[j / P], j % P, t0, te, tile);
      __syncthreads();
      if (P >= kPmeLaneOrder || listed <= kPmeList) break;
    }
  }
  for (int k = t; k < kPmeTile * kPmeTile * kPmeTile; k += kPmeBlock) {
    const int lx = k / (kPmeTile * kPmeTile), ly = k / kPmeTile % kPmeTile,
              lz = k % kPmeTile;
    if (lx < te[0] && ly < te[1] && lz < te[2])
      d.qreal[((size_t)(t0[0] + lx) * d.ny + t0[1] + ly) * d.nz + t0[2] + lz] =
          (double)(long long)tile[lx * kPmePlane + ly * kPmeRow + lz] * kPmeFixInv;
  }
}

// One wave per (x, y) row of the spectrum, lanes over z: the row's factors
// are wave-uniform.  Bound by the read and write of the spectrum, 14 MB for
// 96^3, and its latency: 8.4 us (11 with one thread per point, 64-bit
// index divisions and a barrier tree per sum).
__global__ __launch_bounds__(kPmeBlock) void k_pme_scalar(PmeDev d,
                                                          int virial) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(
      (int)(blockIdx.x * (kPmeBlock / 64) + (threadIdx.x >> 6)));
  // the spread of this run is done: clear its bins for the next
  const long long nclear = (long long)d.nb[0] * d.nb[1] * d.nb[2] + 1;
  for (long long k = (long long)blockIdx.x * kPmeBlock + threadIdx.x; k < nclear;
       k += (long long)gridDim.x * kPmeBlock)
    d.count[k] = 0;
  double acc[kEwSums];
#pragma unroll
  for (int c = 0; c < kEwSums; c++) acc[c] = 0.0;
  const int rows = d.nx * d.ny, nw = gridDim.x * (kPmeBlock / 64);
  for (int row = wave; row < rows; row += nw) {
    const int i = row / d.ny, j = row - i * d.ny;
    const int i0 = i <= d.nx / 2 ? i : i - d.nx;
    const int j0 = j <= d.ny / 2 ? j : j - d.ny;
    const double mi = i0 * d.Lr[0], mj = j0 * d.Lr[1];
    const double modxy = d.mod[0][i] * d.mod[1][j];
    const double mij = mi * mi + mj * mj;
    const double exy = d.ex[0][i] * d.piVr * d.ex[1][j];
    double2 *qk = d.qk + (size_t)row * d.nzh;
    for (int k = lane; k < d.nzh; k += 64) {
      double2 s = qk[k];
      const double mk = k * d.Lr[2];
      const double m2 = mij + mk * mk;
      const double im2 = 1.0 / m2;
      const bool zero = row == 0 && k == 0;
      const double theta =
          zero ? 0.0 : modxy * d.mod[2][k] * exy * d.ex[2][k] * im2;
      const double qq = s.x * s.x + s.y * s.y;
      double e = qq * theta;
      if (k > 0 && ((k != d.nz / 2) || (d.nz & 1))) e *= 2.0;
      acc[0] += e;
      if (virial && !zero) {
        const double v = 2.0 * (im2 + d.fac);
        acc[1] += e * (1.0 - v * mi * mi);
        acc[2] -= e * (v * mi * mj);
        acc[3] -= e * (v * mi * mk);
        acc[4] += e * (1.0 - v * mj * mj);
        acc[5] -= e * (v * mj * mk);
        acc[6] += e * (1.0 - v * mk * mk);
      }
      s.x = zero ? 0.0 : s.x * theta;
      s.y = zero ? 0.0 : s.y * theta;
      qk[k] = s;
    }
  }
  ew_store_sums<kPmeBlock / 64>(acc, d.part, d.n_part);
}

// Force of the reciprocal term on each atom and the correction of its
// excluded pairs (ew_correction), added to f in a fixed order.  kPmeLanes lanes
// take the stencil planes and the excluded pairs of an atom in turn: one lane
// per atom leaves 1.5 waves a SIMD on 96,000 atoms, with 64 grid values and two
// erf in one chain each: 16 us, and 15 us more for a pass over the excluded
// pairs' energies.  Two lanes take 15 us for both; four take 24, the weights
// and the erf of a wave with idle lanes being computed twice as often.
template <int P>
__global__ __launch_bounds__(kPmeBlock) void k_pme_gather(PmeDev d, EwDev e,
                                                          const double *x,
                                                          double *f) {
  const int at = blockIdx.x * (kPmeBlock / kPmeLanes) + threadIdx.x / kPmeLanes;
  const int sub = threadIdx.x % kPmeLanes;
  const bool in = at < d.n;
  const int i = in ? at : d.n - 1;  // past the end: a real atom, not written
  const int nn[3] = {d.nx, d.ny, d.nz};
  int b[3];
  double th[3][P], dth[3][P];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    const double g = pme_coord(x[3 * i + a], d.hr[a], nn[a]);
    const int ig = (int)g;
    pme_bspline<P>(g - ig, th[a], dth[a]);
    b[a] = ig + d.off[a];
  }
  int zk[P];
#pragma unroll
  for (int w = 0; w < P; w++) zk[w] = pme_wrap(b[2] + w, d.nz);
  double fx = 0.0, fy = 0.0, fz = 0.0;
#pragma unroll
  for (int u0 = 0; u0 < P; u0 += kPmeLanes) {
    const int u = u0 + sub;
    if (u >= P) break;
    double tx = 0.0, dx = 0.0;
#pragma unroll
    for (int k = u0; k < P && k < u0 + kPmeLanes; k++) {
      tx = u == k ? th[0][k] : tx;
      dx = u == k ? dth[0][k] : dx;
    }
    const double *plane = d.qreal + (size_t)pme_wrap(b[0] + u, d.nx) * d.ny * d.nz;
    double sx = 0.0, sy = 0.0, sz = 0.0;
#pragma unroll
    for (int v = 0; v < P; v++) {
      const double *row = plane + (size_t)pme_wrap(b[1] + v, d.ny) * d.nz;
      double s0 = 0.0, s1 = 0.0;
#pragma unroll
      for (int w = 0; w < P; w++) {
        const double term = row[zk[w]];
        s0 = fma(term, th[2][w], s0);
        s1 = fma(term, dth[2][w], s1);
      }
      sx = fma(th[1][v], s0, sx);
      sy = fma(dth[1][v], s0, sy);
      sz = fma(th[1][v], s1, sz);
    }
    fx = fma(-dx, sx, fx);
    fy = fma(-tx, sy, fy);
    fz = fma(-tx, sz, fz);
  }
  const double q = d.q[i];
  double gx = fx * d.hr[0] * q, gy = fy * d.hr[1] * q, gz = fz * d.hr[2] * q;
  double acc[kEwSums];
#pragma unroll
  for (int c = 0; c < kEwSums; c++) acc[c] = 0.0;
  if (in) ew_correction(e, x, i, sub, kPmeLanes, gx, gy, gz, acc);
#pragma unroll
  for (int o = 1; o < kPmeLanes; o <<= 1) {
    gx += __shfl_xor(gx, o);
    gy += __shfl_xor(gy, o);
    gz += __shfl_xor(gz, o);
  }
  if (in && sub == 0) {
    f[3 * i] += gx;
    f[3 * i + 1] += gy;
    f[3 * i + 2] += gz;
  }
  ew_store_sums<kPmeBlock / 64>(acc, d.cpart, d.n_cpart);
}

}  // namespace pmnb
