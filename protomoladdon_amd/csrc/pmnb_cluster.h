// Pair kernel of the tile path (k_pairs), for one system or a batch of
// replicas, and its finish kernel.
//
// A work item is 16 consecutive sorted atoms of one column (pmnb_bins.h),
// four lanes per atom (lane = atom slot + 16 * split).  Every pair is visited
// from both of its atoms; an atom's force is summed by its own item only and
// added once into the caller's array, each visit takes half the pair's energy
// and virial: no atomics, fixed order.
//
// Candidates.  The neighbour columns (5 x 5; on an axis with fewer than four
// columns, FP64 five, each column once; with four one column at two images)
// give one or two runs of sorted slots each, the z range of a column cut to
// what its x/y distance leaves of the cutoff.  Lane l holds the bounds of run l
// (column l / 2, part l % 2); the runs laid end to end are the positions 0 ..
// total - 1, read in rounds of 64.  A candidate within the cutoff of the item's
// bounding box goes into the wave's LDS buffer.
//
// Streams.  Position p belongs to stream (p / 16) % 4; each stream has its own
// buffer contents and its own partial sums, and the four sums are added in
// stream order.  One wave takes the four streams in turn, or, where the items
// are too few to fill the chip, a block takes one item and each of its four
// waves one stream: the same bits either way, so a replica in a batch gives
// the bits it gives alone.
//
// Buffer.  When it is full (or the stream ends) each lane tests every 4th
// record against its atom into a mask and evaluates the set bits one by one,
// the next record being read from LDS before the current pair's arithmetic.
// Coordinates are relative to the centre of the item's column and z range, at
// most about a cutoff and a half from zero, so the test is |xj|^2 - 2 xi.xj
// <= hi - |xi|^2 with |xj|^2 kept in the record: three FMAs.  Its rounding is
// below a tenth of `band`, one `band` more is let through, and every pair
// within `band` of the cutoff or beyond is decided with the reference's FP64
// minimum image, so the pair set is the FP64 one.  The sizes of box, columns
// and cells carry their FP32 remainders: without them every pair across a
// column is strained alike (up to 6e-8) and the error of the energy grows with
// the number of atoms, where the rounding of single positions averages out.  Items whose atoms spread
// too far for that bound, and axes with a per-pair minimum image, use
// coordinate differences.
//
// Exclusions.  Only partners whose atom index is within the largest excluded
// distance can be excluded, the atom itself among them: one subtraction and
// one comparison per pair; the class then comes from a 62-bit code of the
// lane's own atom (or from its masks when a distance is over 15).
//
// The mixed forms are bound by VALU issue (84% of the issue slots with
// energies, 81% forces only; LDS, L2 and HBM idle most of the time): on the
// 96,000-atom water (9 A, LJ + Ewald real space) 1.1e4 wave instructions an
// item, three quarters of them the pairs' arithmetic.  The FP64 forms issue 61%
// of the slots at three waves a SIMD; what fills the rest is not separated (the
// quarter-rate instructions, or the waits for a pair's FP64 record and LJ entry,
// which are read from LDS right before use).
// Columns of half a cutoff and z runs cut per column leave 2.2 candidates a
// pair where columns of one cutoff left 4.4.  Measured against that layout
// with its z-level loop (3 x 3 columns, one z cell of the columns a time):
//   96,000 atoms   160 -> 137 us forces only, 205 -> 157 with energies
//   the same, FP64 540 -> 417 (508 with IEEE quotients, roots and exp)
//   522,000 atoms in 128 boxes  751 -> 603, 1,076 -> 690 (half shell before)
//   3,000 atoms, 10 A Coulomb   104 -> 35 (a block an item)
//   30,000 atoms of 12 types    1,293 (neighbour list) -> 83
//   adjoint, 250,000 atoms      2,004 -> 780 (a queue of pairs and LDS slots
//                               per atom left two waves a SIMD)
#pragma once

#include <type_traits>

#include "pmnb_adjoint.h"
#include "pmnb_bins.h"
#include "pmnb_list.h"

namespace pmnb {

constexpr int kTmSplit = 4;                 // lanes per atom
constexpr int kTmWaves = kBlock / 64;       // waves per block
constexpr int kStreams = 4;
constexpr int kSegs = 64;                   // runs of candidates per item
constexpr int kLjRow = 16;                  // LDS row stride of the LJ table
constexpr int kLjTypes = 8;                 // types held in LDS

// What k_pairs forms beside the forces and the pair count; kAdjoint forms the
// adjoint of the forces instead.
enum PairMode { kForces = 0, kEnergies = 1, kMolVirial = 2, kAdjoint = 3 };

// Index of the lowest set bit, -1 for 0 (v_ffbl_b32).
__device__ __forceinline__ int ctz_or_none(unsigned m) {
  return m ? __builtin_ctz(m) : -1;
}

// Minimum and maximum over the 16 atom slots (all four copies agree).
__device__ __forceinline__ float slot_min(float v) {
#pragma unroll
  for (int m = 8; m > 0; m >>= 1) v = fminf(v, __shfl_xor(v, m, 64));
  return uni(v);
}
__device__ __forceinline__ float slot_max(float v) {
#pragma unroll
  for (int m = 8; m > 0; m >>= 1) v = fmaxf(v, __shfl_xor(v, m, 64));
  return uni(v);
}

// BIGT: more LJ types than the LDS table holds; the table is read from
// memory.  LOG: the pair record of pmnb_force_pairs is compiled in.  split: a
// block takes one item (a wave one stream); otherwise a wave takes an item.
template <bool F64, int ELEC, int ELSW, int MODE, bool BIGT, bool LOG>
__global__ void __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(
    F64 ? (MODE == kAdjoint ? 2 : 3) : (MODE >= kMolVirial ? 3 : 4))))
k_pairs(ForceParams P, Sorted S, const TileRep *__restrict__ reps,
        const int4 *__restrict__ items, int nslots, int split,
        double *__restrict__ forces, double *__restrict__ partial, int pstride,
        unsigned long long *__restrict__ npairs, PairLog plog, AdjArgs adj) {
  using Real = typename std::conditional<F64, double, float>::type;
  constexpr bool kEn = MODE == kEnergies || MODE == kMolVirial;
  constexpr bool kAdj = MODE == kAdjoint;
  // records buffered per wave
  constexpr int BUF = F64 ? (kAdj ? 128 : 176) : (kAdj ? 192 : 256);
  constexpr bool kLjLds = !F64 && !BIGT;
  constexpr bool kLjLds64 = F64 && !BIGT;
  __shared__ float4 recA[kTmWaves][BUF];    // x, y, z, |x|^2
  __shared__ float2 recB[kTmWaves][BUF];    // charge, atom << 8 | type
  __shared__ int recT[kTmWaves][BUF];       // sorted slot
  __shared__ double4 recD[F64 ? kTmWaves : 1][F64 ? BUF : 1];  // FP64 x, y, z, q
  // adjoint: dL/dF of the record's atom, FP32 or FP64 as the pairs are
  __shared__ float4 recG[kAdj && !F64 ? kTmWaves : 1][kAdj && !F64 ? BUF : 1];
  __shared__ double4 recH[kAdj && F64 ? kTmWaves : 1][kAdj && F64 ? BUF : 1];
  // ... and the lanes' LJ gradients of 1-4 pairs (few, so not in registers)
  __shared__ Real ljm[kAdj ? kTmWaves : 1][kAdj ? 2 * kAdjTypes : 1][64];
  __shared__ int segE[kTmWaves][kSegs];     // end position of each run
  __shared__ int4 segI[kTmWaves][kSegs];    // x, y offset, cell and slot bases
  // what FP32 left of the offsets (FP64 pairs take the sorted positions)
  __shared__ float2 segL[F64 ? 1 : kTmWaves][F64 ? 1 : kSegs];
  __shared__ float2 ljA[kLjLds ? kLjTypes * kLjRow : 1];  // A, B
  __shared__ float2 ljM[kLjLds ? kLjTypes * kLjRow : 1];  // A14, B14
  // FP64: A, B (the 1-4 values are read from memory)
  __shared__ double2 ljD[kLjLds64 ? kLjTypes * kLjTypes : 1];
  __shared__ double combE[kEn ? kTmWaves : 1][MODE == kMolVirial ? 16 : 8];
  __shared__ long long combF[kTmWaves][3 * kTileAtoms];
  const int wave = uni((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const F32Params &F = P.f;
  if (kLjLds) {
    const int T = P.n_types;
    for (int k = threadIdx.x; k < T * T; k += kBlock) {
      const float4 v = S.ljf[k];
      const int at = (k / T) * kLjRow + k % T;
      ljA[at] = make_float2(v.x, v.y);
      ljM[at] = make_float2(v.z, v.w);
    }
    __syncthreads();
  }
  if (kLjLds64) {
    const int T = P.n_types;
    for (int k = threadIdx.x; k < T * T; k += kBlock)
      ljD[(k / T) * kLjTypes + k % T] = make_double2(S.lj[4 * k], S.lj[4 * k + 1]);
    __syncthreads();
  }
  const float hi = F.cut2 + F.band, lo = F.cut2 - F.band;
  const unsigned maxd = (unsigned)P.max_excl_delta;
  const bool small_code = maxd <= 15u;
  const int slot = lane & (kTileAtoms - 1), sp = lane >> 4;
  // Blocks go to the 8 XCDs in turn; block b takes position (b % 8) * per + b
  // / 8 (the grid is a multiple of 8), so each XCD works through one contiguous
  // range of items and the candidates neighbouring items share stay in its L2.
  const int per = gridDim.x / 8;
  const int blk = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  const int first = split ? blk : blk * kTmWaves + wave;
  const int stride = split ? gridDim.x : gridDim.x * kTmWaves;
  unsigned cnt = 0;  // visits: twice the pairs
  for (int it = first; it < nslots; it += stride) {
    const int4 item = items[it];
    const int a0 = uni(item.x), a1 = uni(item.y), col = uni(item.z);
    if (a1 <= a0) continue;  // an empty slot (the whole block when split)
    const TileRep &R = reps[uni(item.w)];
    const TileGrid G = R.tg;
    const bool wx = R.wrap[0] != 0, wy = R.wrap[1] != 0;
    const Box *bptr = &R.box;
    const float L0 = R.L[0], L1 = R.L[1], L2 = R.L[2];
    const float iL0 = R.iL[0], iL1 = R.iL[1], iL2 = R.iL[2];
    const int cx = col / G.ny, cy = col - cx * G.ny;
    const int cbase = R.cell_off + col * G.nz;
    // the lane's own atom, relative to the centre of the column and of the
    // middle z cell of the item
    const int i = a0 + slot;
    const bool active = i < a1;
    const int ii = active ? i : a0;
    const int zc0 = (uni(S.cell[a0]) + uni(S.cell[a1 - 1]) - 2 * cbase) >> 1;
    const float4 li = S.loc[ii];
    const float hx = 0.5f * G.csx, hy = 0.5f * G.csy;
    float xi = li.x - hx, yi = li.y - hy;
    const float zn = (float)(S.cell[ii] - cbase - zc0);
    float zi = fmaf(zn, G.csz, fmaf(zn, G.loz, li.z));
    // an atom without a finite position has no pairs
    const bool live = active && fabsf(xi) + fabsf(yi) + fabsf(zi) < 1e30f;
    xi = live ? xi : 0.f;
    yi = live ? yi : 0.f;
    zi = live ? zi : 0.f;
    const unsigned wi = S.rec[ii];
    const int ti = (int)(wi & 255u), ai = (int)(wi >> 8);
    const unsigned wlo = ((unsigned)ai - maxd) << 8;
    const unsigned wrange = (2u * maxd + 1u) << 8;
    const unsigned long long xcode = S.xcode[ai];
    const double qi = F64 ? S.q[ii] : 0.0;
    const double xd = F64 && live ? S.x[ii] : 0.0,
                 yd = F64 && live ? S.y[ii] : 0.0,
                 zd = F64 && live ? S.z[ii] : 0.0;
    // adjoint: the lane's dL/dF, in FP32 with its remainder
    Real gi0 = 0, gi1 = 0, gi2 = 0, gl0 = 0, gl1 = 0, gl2 = 0;
    if constexpr (kAdj) {
      const double *g = adj.grad_f + 3 * (size_t)ai;
      gi0 = (Real)g[0];
      gi1 = (Real)g[1];
      gi2 = (Real)g[2];
      gl0 = (Real)(g[0] - (double)gi0);
      gl1 = (Real)(g[1] - (double)gi1);
      gl2 = (Real)(g[2] - (double)gi2);
    }
    // dL/d{A, B} / 2 by the partner's type
    Real lj[kAdj ? kAdjTypes : 1][2];
    if constexpr (kAdj)
#pragma unroll
      for (int c = 0; c < kAdjTypes; c++) {
        lj[c][0] = lj[c][1] = Real(0);
        ljm[wave][2 * c][lane] = ljm[wave][2 * c + 1][lane] = Real(0);
      }
    double fq64 = 0.0;
    const float2 *ljr = &ljA[kLjLds ? ti * kLjRow : 0];
    const float4 *ljrow = S.ljf + ti * P.n_types;
    const double *ljrow64 = S.lj + 4 * (ti * P.n_types);
    const float bx0 = slot_min(live ? xi : 1e30f),
                bx1 = slot_max(live ? xi : -1e30f);
    const float by0 = slot_min(live ? yi : 1e30f),
                by1 = slot_max(live ? yi : -1e30f);
    const float bz0 = slot_min(live ? zi : 1e30f),
                bz1 = slot_max(live ? zi : -1e30f);
    const float icsz = 1.f / G.csz;
    const float rch = sqrtf(hi) + 1e-3f;
    // z cells within reach, relative to zc0; when they cover the column, every
    // cell once with the per-pair image
    auto zcell = [&](float z) {  // bounded whatever the positions are
      return (int)floorf(fminf(fmaxf(z * icsz, -1e6f), 1e6f));
    };
    const int kA0 = zcell(bz0 - rch), kB0 = zcell(bz1 + rch);
    const bool wz = kB0 - kA0 + 1 > G.nz;
    const bool wrapped = wx || wy || wz;
    // FMA test allowed: |x|^2 rounding below band / 2 (see the file comment)
    const float ex = fmaxf(fabsf(bx0), fabsf(bx1)),
                ey = fmaxf(fabsf(by0), fabsf(by1)),
                ez = fmaxf(fabsf(bz0), fabsf(bz1));
    const float far = rch + sqrtf(fmaf(ex, ex, fmaf(ey, ey, ez * ez)));
    const bool direct = wrapped || far * far > 8e5f * F.band;
    // -------------------------------------------------- runs of candidates
    int total;
    {
      const int k = lane >> 1, part = lane & 1;
      const int kx = k / 5, ky = k - 5 * kx;
      const int ox = wx ? kx - cx : kx - 2, oy = wy ? ky - cy : ky - 2;
      // (no run without a live atom: the box is empty and so are the z ranges)
      bool ok = k < 25 && bz0 <= bz1 && !(wx && kx >= G.nx) &&
                !(wy && ky >= G.ny);
      int tx = cx + ox, ty = cy + oy;
      tx = tx < 0 ? tx + G.nx : (tx >= G.nx ? tx - G.nx : tx);
      ty = ty < 0 ? ty + G.ny : (ty >= G.ny ? ty - G.ny : ty);
      // column's lower corner
      const double fxd = (double)ox * ((double)G.csx + (double)G.lox) - (double)hx;
      const double fyd = (double)oy * ((double)G.csy + (double)G.loy) - (double)hy;
      const float fx = (float)fxd, fy = (float)fyd;
      const float gx = wx ? 0.f : fmaxf(0.f, fmaxf(fx - bx1, bx0 - fx - G.csx));
      const float gy = wy ? 0.f : fmaxf(0.f, fmaxf(fy - by1, by0 - fy - G.csy));
      // less a margin for the rounding of the coordinates, so that the
      // per-record test alone decides
      const float g2 = fmaxf(0.f, fmaf(gx, gx, gy * gy) - 1e-3f);
      ok = ok && g2 <= hi;
      const int tbase = R.cell_off + (tx * G.ny + ty) * G.nz;
      int w0 = 0, w1 = G.nz - 1, zsub = tbase + zc0;
      if (wz) {
        ok = ok && part == 0;
      } else {
        const float rl = sqrtf(fmaxf(hi - g2, 0.f)) + 1e-3f;  // <= rch
        const int kA = zcell(bz0 - rl), kB = zcell(bz1 + rl);
        const int zA = zc0 + kA, len = kB - kA + 1;
        const int wA = ((zA % G.nz) + G.nz) % G.nz;
        if (part == 0) {
          w0 = wA;
          w1 = min(G.nz - 1, wA + len - 1);
          zsub = tbase - (zA - wA) + zc0;
        } else {
          w1 = wA + len - 1 - G.nz;
          zsub = tbase - (zA - wA + G.nz) + zc0;
          ok = ok && w1 >= 0;
        }
      }
      int start = 0, n = 0;
      if (ok) {
        start = S.cstart[tbase + w0];
        n = S.cstart[tbase + w1] + S.ccount[tbase + w1] - start;
      }
      int inc = n;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(inc, o, 64);
        if (lane >= o) inc += y;
      }
      total = __builtin_amdgcn_readlane(inc, 63);
      segE[wave][lane] = inc;
      if (!F64) segL[wave][lane] = make_float2((float)(fxd - (double)fx),
                                     (float)(fyd - (double)fy));
      segI[wave][lane] = make_int4(__float_as_int(fx), __float_as_int(fy), zsub,
                                   start - (inc - n));
    }
    wave_sync_lds();
    const float thr =
        live ? (hi + F.band) - fmaf(xi, xi, fmaf(yi, yi, zi * zi)) : -1e30f;
    const float tax = -2.f * xi, tay = -2.f * yi, taz = -2.f * zi;
    const float hia = live ? hi : -1e30f;
    // sums of the item: mixed forces are integers (any order); FP64 forces
    // (per atom, on the lanes of split 0) and energies stream by stream
    long long Fx = 0, Fy = 0, Fz = 0;
    double fx64 = 0.0, fy64 = 0.0, fz64 = 0.0;
    double etot = 0.0, mtot = 0.0;
    const int nround = (total + 64 * kStreams - 1) / (64 * kStreams);
    const int st0 = split ? wave : 0, st1 = split ? wave + 1 : kStreams;
    for (int st = st0; st < st1; st++) {
      double sx64 = 0.0, sy64 = 0.0, sz64 = 0.0, erow = 0.0, mrow = 0.0;
      int nbuf = 0;
      for (int rnd = 0; rnd <= nround; rnd++) {
        // ------------------------------------------------ one round of 64
        bool ok = false;
        float4 rf;
        float2 rb;
        int t = 0;
        const int p = 64 * kStreams * rnd + 64 * sp + 16 * st + slot;
        if (rnd < nround && p < total) {
          int k = 0;
#pragma unroll
          for (int o = kSegs / 2; o > 0; o >>= 1)
            k += segE[wave][k + o - 1] <= p ? o : 0;
          const int4 sg = segI[wave][k];
          t = p + sg.w;
          const float4 lt = S.loc[t];
          const float2 sl = F64 ? make_float2(0.f, 0.f) : segL[wave][k];
          rf.x = __int_as_float(sg.x) + (lt.x + sl.x);
          rf.y = __int_as_float(sg.y) + (lt.y + sl.y);
          const float zt = (float)(S.cell[t] - sg.z);
          rf.z = fmaf(zt, G.csz, fmaf(zt, G.loz, lt.z));
          rb = make_float2(lt.w, __uint_as_float(S.rec[t]));
          const float gx = wx ? 0.f : fmaxf(0.f, fmaxf(bx0 - rf.x, rf.x - bx1));
          const float gy = wy ? 0.f : fmaxf(0.f, fmaxf(by0 - rf.y, rf.y - by1));
          const float gz = wz ? 0.f : fmaxf(0.f, fmaxf(bz0 - rf.z, rf.z - bz1));
          rf.w = fmaf(rf.x, rf.x, fmaf(rf.y, rf.y, rf.z * rf.z));
          // finite records only: the buffer's sign test reads no NaN
          ok = fmaf(gx, gx, fmaf(gy, gy, gz * gz)) <= hi && rf.w < 1e30f;
        }
        const unsigned long long ball = __ballot(ok);
        const int nb = __popcll(ball);
        if ((rnd == nround && nbuf > 0) || nbuf + nb > BUF) {
          // ---------------------------------------------- the full buffer
          // up to 15 records after the last get far coordinates, which fail
          // the test (NaN with a per-pair image, which would fold them)
          if (lane < 16 && nbuf + lane < BUF) {
            const float c = wrapped ? __builtin_nanf("") : 1e15f;
            recA[wave][nbuf + lane] = make_float4(c, c, c, c * c);
          }
          wave_sync_lds();
          const int J = ((nbuf + 15) >> 4) << 2;  // records per lane, x 4
          const float4 *ra = &recA[wave][sp];
          // bit j of word w: record 4 (32 w + j) + split
          auto word = [&](int j0, int n, auto in) -> unsigned {
            unsigned m = 0u;
            for (int j = n - 4; j >= 0; j -= 4) {
              const float4 *r = ra + kTmSplit * (j0 + j);
              const float4 r3 = r[12], r2 = r[8], r1 = r[4], r0 = r[0];
              m = in(m, r3);
              m = in(m, r2);
              m = in(m, r1);
              m = in(m, r0);
            }
            return m;
          };
          unsigned m0, m1;
          if (!direct) {
            // the sign of |xj|^2 - 2 xi.xj - thr is the bit, shifted in
            auto test = [&](unsigned m, const float4 &r) -> unsigned {
              const float s =
                  fmaf(tax, r.x, fmaf(tay, r.y, fmaf(taz, r.z, r.w))) - thr;
              return __builtin_amdgcn_alignbit(m, __float_as_uint(s), 31);
            };
            m0 = word(0, min(J, 32), test);
            m1 = J > 32 ? word(32, J - 32, test) : 0u;
          } else {
            auto test = [&](unsigned m, const float4 &r) -> unsigned {
              float dx = r.x - xi, dy = r.y - yi, dz = r.z - zi;
              if (wx) dx = fmaf(-L0, rintf(dx * iL0), dx);
              if (wy) dy = fmaf(-L1, rintf(dy * iL1), dy);
              if (wz) dz = fmaf(-L2, rintf(dz * iL2), dz);
              return (m << 1) +
                     (unsigned)(fmaf(dx, dx, fmaf(dy, dy, dz * dz)) <= hia);
            };
            m0 = word(0, min(J, 32), test);
            m1 = J > 32 ? word(32, J - 32, test) : 0u;
          }
          cnt += __builtin_popcount(m0) + __builtin_popcount(m1);
          Real px = 0, py = 0, pz = 0, pq = 0, pelj = 0, peel = 0;
          Real v0 = 0, v1 = 0, v2 = 0, v3 = 0, v4 = 0, v5 = 0;
          double mv[8];
          if (MODE == kMolVirial)
#pragma unroll
            for (int c = 0; c < 8; c++) mv[c] = 0.0;
          // One pair: record k.  Straight-line: an excluded pair (or a lane
          // without one) runs through and its result is replaced by zero, so
          // only the two rare checks branch.
          auto eval = [&](const float4 &A, const float2 &B, int k, bool valid,
                          auto WR, auto SAME) __attribute__((always_inline)) {
            const unsigned w = __float_as_uint(B.y);
            double2 abd = make_double2(0.0, 0.0);
            if constexpr (kLjLds64) {
              abd = ljD[ti * kLjTypes + (w & 255u)];
            } else if constexpr (F64) {
              const double *lp = ljrow64 + 4 * (w & 255u);
              abd = make_double2(lp[0], lp[1]);
            }
            float2 ab = make_float2(0.f, 0.f);
            float4 ab4 = make_float4(0.f, 0.f, 0.f, 0.f);
            if constexpr (kLjLds) ab = ljr[w & 255u];
            else if constexpr (!F64) ab4 = ljrow[w & 255u];
            float dx = A.x - xi, dy = A.y - yi, dz = A.z - zi;
            if (decltype(WR)::value) {
              auto fold = [](float &d, float L, float lo, float iL) {
                const float k = rintf(d * iL);
                d = fmaf(-lo, k, fmaf(-L, k, d));
              };
              if (wx) fold(dx, L0, R.Llo[0], iL0);
              if (wy) fold(dy, L1, R.Llo[1], iL1);
              if (wz) fold(dz, L2, R.Llo[2], iL2);
            }
            const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
            float qj = B.x;
            bool keep = valid;
            int cls = 0;
            if (valid && w - wlo < wrange) {
              const int d = (int)(w >> 8) - ai;
              if (small_code) cls = (int)(xcode >> (2 * d + 30)) & 3;
              else cls = d == 0 ? 2 : excl_own(S.xown + 4 * (size_t)ai, d);
              if (cls == 2) {
                keep = false;
                cnt--;
              }
              if (!F64 && cls == 1) {
                qj *= F.csf;
                if constexpr (kLjLds) ab = ljM[ti * kLjRow + (w & 255u)];
                else ab4 = make_float4(ab4.z, ab4.w, 0.f, 0.f);
              }
            }
            double exd = 0.0, eyd = 0.0, ezd = 0.0, e2d = 1.0;
            if constexpr (F64) {
              const double4 rd = recD[wave][k];
              min_diff_exact(*bptr, xd, yd, zd, rd.x, rd.y, rd.z, exd, eyd, ezd,
                             e2d);
              if (keep && e2d > P.cut2) {
                keep = false;
                cnt--;
              }
            } else if (keep && r2 >= lo) {
              // near the cutoff: decide with the reference's FP64 minimum image
              const int t2 = recT[wave][k];
              min_diff_exact(rare_box(bptr), S.x[ii], S.y[ii], S.z[ii], S.x[t2],
                             S.y[t2], S.z[t2], exd, eyd, ezd, e2d);
              if (e2d > P.cut2) {
                keep = false;
                cnt--;
              }
            }
            if (LOG && keep && i < recT[wave][k])
              log_pair(plog, ai, (int)(w >> 8), cls);
            if constexpr (kAdj) {
              Real ff, ffp, h, dA, dB, q2, ddx, ddy, ddz, w0, w1, w2;
              if constexpr (F64) {
                if (cls == 1) {
                  const double *lp = ljrow64 + 4 * (w & 255u);
                  abd = make_double2(lp[2], lp[3]);
                }
                q2 = recD[wave][k].w * (cls == 1 ? P.csf : 1.0);
                pair_adj<Real, ELEC, decltype(SAME)::value>(
                    adj.c64, e2d, abd.x, abd.y, qi * q2, ff, ffp, h, dA, dB);
                ddx = exd;
                ddy = eyd;
                ddz = ezd;
                const double4 g = recH[wave][k];
                w0 = g.x - gi0;
                w1 = g.y - gi1;
                w2 = g.z - gi2;
              } else {
                q2 = qj;
                pair_adj<Real, ELEC, decltype(SAME)::value>(
                    adj.c32, r2, ab.x, ab.y, li.w * qj, ff, ffp, h, dA, dB);
                ddx = dx;
                ddy = dy;
                ddz = dz;
                const float4 g = recG[wave][k];
                w0 = (g.x - gi0) - gl0;
                w1 = (g.y - gi1) - gl1;
                w2 = (g.z - gi2) - gl2;
              }
              const Real wd = adj_fma(w0, ddx, adj_fma(w1, ddy, w2 * ddz));
              const Real c2 = Real(2) * ffp * wd;
              px -= keep ? adj_fma(ff, w0, c2 * ddx) : Real(0);
              py -= keep ? adj_fma(ff, w1, c2 * ddy) : Real(0);
              pz -= keep ? adj_fma(ff, w2, c2 * ddz) : Real(0);
              pq += keep ? wd * q2 * h : Real(0);
              const Real hA = keep ? Real(0.5) * wd * dA : Real(0);
              const Real hB = keep ? Real(0.5) * wd * dB : Real(0);
              const int tj = (int)(w & 255u);
              if (cls == 1) {
                ljm[wave][2 * tj][lane] += hA;
                ljm[wave][2 * tj + 1][lane] += hB;
              } else {
#pragma unroll
                for (int c = 0; c < kAdjTypes; c++) {
                  lj[c][0] += tj == c ? hA : Real(0);
                  lj[c][1] += tj == c ? hB : Real(0);
                }
              }
              return;
            }
            const float qq = li.w * qj;
            Real ff, e1, e2, ddx, ddy, ddz;
            if constexpr (F64) {
              double q2 = qi * recD[wave][k].w;
              if (cls == 1) {
                const double *lp = ljrow64 + 4 * (w & 255u);
                abd = make_double2(lp[2], lp[3]);
                q2 *= P.csf;
              }
              pair_fma64<ELEC, ELSW, decltype(SAME)::value>(P, e2d, abd.x, abd.y,
                                                            q2, ff, e1, e2);
              ddx = exd;
              ddy = eyd;
              ddz = ezd;
            } else {
              pair_mix<ELEC, decltype(SAME)::value>(
                  F, r2, kLjLds ? ab.x : ab4.x, kLjLds ? ab.y : ab4.y, qq, ff,
                  e1, e2);
              ddx = dx;
              ddy = dy;
              ddz = dz;
            }
            ff = keep ? ff : Real(0);
            if (decltype(WR)::value) {  // a lane without a pair may hold NaN
              ddx = keep ? ddx : Real(0);
              ddy = keep ? ddy : Real(0);
              ddz = keep ? ddz : Real(0);
            }
            if constexpr (MODE == kForces) {
              if constexpr (F64) {
                px -= ddx * ff;
                py -= ddy * ff;
                pz -= ddz * ff;
              } else {
                px = fmaf(-ddx, ff, px);
                py = fmaf(-ddy, ff, py);
                pz = fmaf(-ddz, ff, pz);
              }
            } else {
              pelj += keep ? e1 : Real(0);
              peel += keep ? e2 : Real(0);
              const Real gx = ddx * ff, gy = ddy * ff, gz = ddz * ff;
              px -= gx;
              py -= gy;
              pz -= gz;
              bool at = (P.flags & 1u) != 0;
              if constexpr (MODE == kMolVirial) {
                const int t2 = recT[wave][k];
                const int mi = S.mol[ii], mj = S.mol[t2];
                if (keep && mi != mj) {
                  at = true;
                  double cdx, cdy, cdz, cd2;
                  min_diff_exact(rare_box(bptr), S.com[3 * mi], S.com[3 * mi + 1],
                                 S.com[3 * mi + 2], S.com[3 * mj],
                                 S.com[3 * mj + 1], S.com[3 * mj + 2], cdx, cdy,
                                 cdz, cd2);
                  const double dgx = gx, dgy = gy, dgz = gz;
                  mv[0] += dgx * cdx;
                  mv[1] += dgx * cdy;
                  mv[2] += dgx * cdz;
                  mv[3] += dgy * cdy;
                  mv[4] += dgy * cdz;
                  mv[5] += dgz * cdz;
                }
              }
              if (at) {
                if constexpr (F64) {
                  v0 += gx * ddx;
                  v1 += gx * ddy;
                  v2 += gx * ddz;
                  v3 += gy * ddy;
                  v4 += gy * ddz;
                  v5 += gz * ddz;
                } else {
                  v0 = fmaf(gx, ddx, v0);
                  v1 = fmaf(gx, ddy, v1);
                  v2 = fmaf(gx, ddz, v2);
                  v3 = fmaf(gy, ddy, v3);
                  v4 = fmaf(gy, ddz, v4);
                  v5 = fmaf(gz, ddz, v5);
                }
              }
            }
          };
          // The set bits, lowest first; two record sets in turn (no register
          // moves) until every lane is through.  An empty word is replaced by
          // the next; the pop of an empty mask gives the last record (every
          // record below nbuf is written), which is read and not used.
          int kb = sp;  // record of bit 0 of the current word
          auto pop = [&]() -> int {
            const bool e = m0 == 0u;
            const unsigned m = e ? m1 : m0;
            m1 = e ? 0u : m1;
            kb = e ? kb + 32 * kTmSplit : kb;
            m0 = m & (m - 1u);
            return (int)min((unsigned)(kb + kTmSplit * ctz_or_none(m)),
                            (unsigned)nbuf - 1u);
          };
          auto run = [&](auto WR, auto SAME) __attribute__((always_inline)) {
            bool g0 = (m0 | m1) != 0u;
            if (!__any(g0)) return;
            int k0 = pop();
            float4 A0 = recA[wave][k0];
            float2 B0 = recB[wave][k0];
            while (true) {
              const bool g1 = (m0 | m1) != 0u;
              const int k1 = pop();
              const float4 A1 = recA[wave][k1];
              const float2 B1 = recB[wave][k1];
              eval(A0, B0, k0, g0, WR, SAME);
              if (!__any(g1)) break;
              g0 = (m0 | m1) != 0u;
              k0 = pop();
              A0 = recA[wave][k0];
              B0 = recB[wave][k0];
              eval(A1, B1, k1, g1, WR, SAME);
              if (!__any(g0)) break;
            }
          };
          if (wrapped) run(std::true_type{}, std::false_type{});
          else if (F.same_switch)
            run(std::false_type{}, std::true_type{});
          else run(std::false_type{}, std::false_type{});
          if constexpr (kAdj) {
            fx64 += px;
            fy64 += py;
            fz64 += pz;
            fq64 += pq;
          } else if constexpr (F64) {
            sx64 += px;
            sy64 += py;
            sz64 += pz;
          } else {
            Fx += to_fixed_f32(px);
            Fy += to_fixed_f32(py);
            Fz += to_fixed_f32(pz);
          }
          if constexpr (kEn) {
            const double e[8] = {(double)pelj, (double)peel, (double)v0,
                                 (double)v1,   (double)v2,   (double)v3,
                                 (double)v4,   (double)v5};
            erow += wave_sum8(e, lane);
            if constexpr (MODE == kMolVirial) mrow += wave_sum8(mv, lane);
          }
          wave_sync_lds();  // the buffer is refilled next
          nbuf = 0;
        }
        if (ok) {
          const int pos = nbuf + lane_prefix(ball);
          recA[wave][pos] = rf;
          recB[wave][pos] = rb;
          recT[wave][pos] = t;
          if (F64)
            recD[wave][pos] = make_double4(S.x[t], S.y[t], S.z[t], S.q[t]);
          if constexpr (kAdj) {
            const double *g =
                adj.grad_f + 3 * (size_t)(__float_as_uint(rb.y) >> 8);
            if constexpr (F64)
              recH[wave][pos] = make_double4(g[0], g[1], g[2], 0.0);
            else
              recG[wave][pos] =
                  make_float4((float)g[0], (float)g[1], (float)g[2], 0.f);
          }
        }
        nbuf += nb;
      }
      if constexpr (F64 && !kAdj) {
        // the four lanes of an atom, then the streams in order
        sx64 += __shfl_xor(sx64, 32, 64);
        sy64 += __shfl_xor(sy64, 32, 64);
        sz64 += __shfl_xor(sz64, 32, 64);
        sx64 += __shfl_xor(sx64, 16, 64);
        sy64 += __shfl_xor(sy64, 16, 64);
        sz64 += __shfl_xor(sz64, 16, 64);
        fx64 += sx64;
        fy64 += sy64;
        fz64 += sz64;
      }
      etot += erow;
      mtot += mrow;
    }
    if constexpr (kAdj) {  // never split
      auto quad = [](double v) {
        v += __shfl_xor(v, 32, 64);
        return v + __shfl_xor(v, 16, 64);
      };
      fx64 = quad(fx64);
      fy64 = quad(fy64);
      fz64 = quad(fz64);
      fq64 = quad(fq64);
      if (active && sp == 0) {
        if (adj.grad_x) {
          double *f = adj.grad_x + 3 * (size_t)ai;
          f[0] += fx64;
          f[1] += fy64;
          f[2] += fz64;
        }
        if (adj.grad_q) adj.grad_q[ai] += fq64;
      }
      if (adj.lj) {
#pragma unroll
        for (int c = 0; c < kAdjTypes; c++)
#pragma unroll
          for (int m = 0; m < 4; m++) {
            double v = (double)(m < 2 ? lj[c][m] : ljm[wave][2 * c + m - 2][lane]);
            v = quad(v);
            if (active && sp == m)
              adj.lj[(size_t)(4 * c + m) * P.n_atoms + i] = v;
          }
      }
      continue;
    }
    if (!F64) {
      Fx += __shfl_xor(Fx, 32, 64);
      Fy += __shfl_xor(Fy, 32, 64);
      Fz += __shfl_xor(Fz, 32, 64);
      Fx += __shfl_xor(Fx, 16, 64);
      Fy += __shfl_xor(Fy, 16, 64);
      Fz += __shfl_xor(Fz, 16, 64);
    }
    if (split) {
      // the streams' sums, added by the first wave in stream order
      if (sp == 0) {
        combF[wave][slot] = F64 ? __double_as_longlong(fx64) : Fx;
        combF[wave][slot + kTileAtoms] = F64 ? __double_as_longlong(fy64) : Fy;
        combF[wave][slot + 2 * kTileAtoms] =
            F64 ? __double_as_longlong(fz64) : Fz;
      }
      if constexpr (kEn) {
        if (lane < 8) {
          combE[wave][lane] = etot;
          if constexpr (MODE == kMolVirial) combE[wave][8 + lane] = mtot;
        }
      }
      __syncthreads();
      if (wave == 0) {
        Fx = Fy = Fz = 0;
        fx64 = fy64 = fz64 = 0.0;
#pragma unroll
        for (int k = 0; k < kStreams; k++) {
          const long long a = combF[k][slot], b = combF[k][slot + kTileAtoms],
                          c = combF[k][slot + 2 * kTileAtoms];
          if (F64) {
            fx64 += __longlong_as_double(a);
            fy64 += __longlong_as_double(b);
            fz64 += __longlong_as_double(c);
          } else {
            Fx += a;
            Fy += b;
            Fz += c;
          }
        }
        if constexpr (kEn) {
          etot = mtot = 0.0;
#pragma unroll
          for (int k = 0; k < kStreams; k++) {
            etot += combE[k][lane & 7];
            if constexpr (MODE == kMolVirial) mtot += combE[k][8 + (lane & 7)];
          }
        }
      }
    }
    if (!split || wave == 0) {
      if (active && sp == 0) {
        const double ox = F64 ? fx64 : (double)Fx * kFixedInv,
                     oy = F64 ? fy64 : (double)Fy * kFixedInv,
                     oz = F64 ? fz64 : (double)Fz * kFixedInv;
        double *f = forces + 3 * (size_t)ai;
        if (P.flags & kFlagFresh) {
          f[0] = ox;
          f[1] = oy;
          f[2] = oz;
        } else {
          f[0] += ox;
          f[1] += oy;
          f[2] += oz;
        }
      }
      if constexpr (kEn) {
        // each pair is seen from both atoms: half of its energy and virial
        if (lane < 8) {
          partial[(size_t)lane * pstride + it] = 0.5 * etot;
          if (lane < 6)
            partial[(size_t)(ACC_MXX + lane) * pstride + it] =
                MODE == kMolVirial ? 0.5 * mtot : 0.0;
        }
      }
    }
    if (split) __syncthreads();  // the sums' LDS is rewritten by the next item
  }
  const unsigned long long tot = block_count<kTmWaves>(cnt);
  if (threadIdx.x == 0 && tot) atomicAdd(npairs, tot);
}

// After the pair kernel: the first rep_blocks blocks sum the item partials of
// one (replica, accumulator) each (finish_rep_block), the first of them also
// storing the pair count in np_out when given (the counter holds visits, two
// per pair); the rest clear the bin counts for the next evaluation.
__global__ void __launch_bounds__(1024)
k_pairs_finish(const double *__restrict__ partial, int pstride,
               const TileRep *__restrict__ reps,
               const int *__restrict__ rep_items, double *__restrict__ out,
               int rep_blocks, int *__restrict__ count, int nbin, int fresh,
               const unsigned long long *__restrict__ npairs,
               unsigned long long *__restrict__ np_out) {
  const int b = blockIdx.x;
  if (b >= rep_blocks) {
    const int c = (b - rep_blocks) * 1024 + threadIdx.x;
    if (c < nbin) count[c] = 0;
    return;
  }
  if (np_out && b == 0 && threadIdx.x == 0) *np_out = *npairs / 2;
  finish_rep_block(partial, pstride, reps, rep_items, out, b / ACC_N, b % ACC_N,
                   fresh);
}

}  // namespace pmnb
