// pmnb_ewald.h -- reciprocal-space and correction terms of ProtoMol's
// NonbondedFullEwaldSystemForce for an orthogonal periodic box.
//
// Reference (force/nonbonded/NonbondedFullEwaldSystemForce.h):
//   :597-652   alpha, rc, kc and the k-vector list (h >= 0 half space),
//              built on the host in the same order
//   :680-700   point self energy and charged-system energy (host)
//   :884-1086  reciprocal term: per-atom sin/cos tables by the addition
//              theorem, structure factor, energy, atomic virial, forces
//   :1092-1130 intramolecular correction over the exclusion table
//
// Work is N x K (atoms x k-vectors), as in the reference, but as two matrix
// products on the FP64 matrix cores.  With X, Y, Z the sines and cosines of
// h x (charge folded in), k y and l z of an atom:
//   k_ew_tables  the tables by the addition theorem, an atom's values
//                together: [X | Y | Z], each (cos, sin) per order;
//   k_ew_sk      C = sum over atoms of (X_a Y_b) Z_c for the four products of
//                (cos, sin) h x and |k| y and both of m z: everything the
//                structure factors of (h, +-k, +-m) need, 2 multiply-adds a
//                k-vector and atom;
//   k_ew_coef    the sums over the atom chunks, the structure factors, energy
//                and virial terms, and the force's coefficients P;
//   k_ew_force   for every (h, k), with w = sin(k r) ps - cos(k r) pc summed
//                over l: w = xys U + xyc V with U = sum_c P_c Z_c, the same
//                for the terms weighted by kz: 4 multiply-adds a k-vector and
//                atom;
//   k_ew_final   the splits' forces in order, and the correction of the
//                atom's excluded pairs, each evaluated by both of its atoms;
//   k_ew_finish  the blocks' energy and virial sums in a fixed order.
// No atomics; every sum has a fixed order.
#pragma once

namespace pmnb {

typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int kEwOrders = 40;   // orders of m a pass holds: 80 columns
constexpr int kEwCols = 2 * kEwOrders;
constexpr int kEwTiles = 8;     // row tiles of a k_ew_sk block (two a wave)
constexpr int kEwStage = 8;     // atoms staged at a time
// staged values of an atom: the tiles' X (2 each) and Y (8 each), and Z
constexpr int kEwX = 0, kEwY = 2 * kEwTiles, kEwZ = kEwY + 8 * kEwTiles,
              kEwVals = kEwZ + kEwCols;
// ... at a stride of 16 doubles mod 32, so two atoms fill the 64 banks
constexpr int kEwStride = 176;
constexpr int kEwAtoms = 32;    // atoms of a k_ew_force wave
constexpr int kEwSteps = kEwCols / 4;  // matrix steps of a pass
constexpr int kEwSums = 7;      // energy, xx, xy, xz, yy, yz, zz

struct EwRun {
  int h, k, l_lo, l_hi, start;  // l in [l_lo, l_hi] at list index start + l - l_lo
};
// Row tile of k_ew_sk: |k| = k0 .. k0 + 3 of one h (four products each),
// orders m0 .. m0 + 8 nc - 1; nc = 0: padding.
struct EwTile {
  int h, k0, m0, nc;
};
// Force tile: k = k0 .. k0 + 3 of one h
struct EwFTile {
  int h, k0;
};
// Per h: the k of its force tiles start at kmin, first tile ft0; runs of
// (h, k) at run0 + k - kmin (every k of the interval has a run)
struct EwH {
  int kmin, kmax, ft0, run0;
};

struct EwDev {
  Box box;
  int n, nk, H;               // atoms, k-vectors, table orders
  const double4 *kv;          // kx, ky, kz, b = exp(-k^2/(4 alpha^2))/k^2
  const EwRun *runs;
  const EwH *hs;
  const EwTile *tiles;
  int n_tiles, n_chunks, chunk;  // row tiles; atom chunks and their size
  const EwFTile *ftiles;
  const int2 *fsteps;         // {first matrix step, steps} per pass and tile
  const int *fsplit;          // first tile of each split, and the end
  int n_ft, n_split, n_pass;
  const double *q;            // scaled charges
  double *tab;                // 6 H per atom
  double *C;                  // n_chunks x n_tiles x 16 rows x 80 columns
  double *P;                  // force coefficients, 64 per matrix step
  double *pf;                 // n_split x n x 3 partial forces
  double *part;               // kEwSums rows of n_tiles blocks
  double *cpart;              // kEwSums rows of n_cpart blocks (correction)
  int n_cpart;
  const int *xptr, *xent;     // per atom: exclusion rows (row << 1 | role)
  const int *xrows;           // 3 per row: a1, a2, class
  int n_excl;
  double alpha, alpha2, two_alpha_pi, csf, Vr, fac;
  double kunit[3];            // 2 pi / L
};

// (s, c) <- (s, c) * exp(i z) for (s1, c1) = (sin z, cos z): the
// addition-theorem step of the tables, with fused multiply-adds.
__device__ __forceinline__ void ew_step(double s1, double c1, double &s,
                                        double &c) {
  const double s2 = fma(s1, c, c1 * s);
  const double c2 = fma(c1, c, -(s1 * s));
  s = s2;
  c = c2;
}

// Intramolecular correction of atom i (:1105-1129): the force of every
// lanes-th excluded pair of i from `sub` on, each pair evaluated by both of
// its atoms (no atomics), its energy and virial (acc: energy, xx, xy, xz, yy,
// yz, zz) by the first.
__device__ __forceinline__ void ew_correction(const EwDev &d, const double *x,
                                              int i, int sub, int lanes,
                                              double &gx, double &gy,
                                              double &gz, double (&acc)[7]) {
  const int e1 = d.xptr[i + 1];
  for (int e = d.xptr[i] + sub; e < e1; e += lanes) {
    const int row = d.xent[e] >> 1, role = d.xent[e] & 1;
    const int a1 = d.xrows[3 * row], a2 = d.xrows[3 * row + 1],
              cls = d.xrows[3 * row + 2];
    double rx, ry, rz, r2;
    min_diff_exact(d.box, x[3 * a1], x[3 * a1 + 1], x[3 * a1 + 2], x[3 * a2],
                   x[3 * a2 + 1], x[3 * a2 + 2], rx, ry, rz, r2);
    double qq = d.q[a1] * d.q[a2];
    if (cls == 1) qq *= 1 - d.csf;  // EXCLUSION_MODIFIED
    const double r = sqrt(r2), rr = 1 / r;
    const double er = erf(d.alpha * r) * rr;
    const double g = qq * (d.two_alpha_pi * exp(-d.alpha2 * r2) - er) * rr * rr;
    const double fx = rx * g, fy = ry * g, fz = rz * g;
    if (role == 0) {
      gx -= fx;
      gy -= fy;
      gz -= fz;
      acc[0] -= qq * er;
      acc[1] += fx * rx;
      acc[2] += fx * ry;
      acc[3] += fx * rz;
      acc[4] += fy * ry;
      acc[5] += fy * rz;
      acc[6] += fz * rz;
    } else {
      gx += fx;
      gy += fy;
      gz += fz;
    }
  }
}

// Sums of kEwSums values over a block of NW waves: rows of part, column
// blockIdx.x, in a fixed order (wave_sum8, then the waves in turn).
template <int NW>
__device__ __forceinline__ void ew_store_sums(const double (&acc)[kEwSums],
                                              double *part, int n_part) {
  __shared__ double red[NW][8];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const double v8[8] = {acc[0], acc[1], acc[2], acc[3],
                        acc[4], acc[5], acc[6], 0.0};
  const double s = wave_sum8(v8, lane);
  if (lane < 8) red[wave][lane] = s;
  __syncthreads();
  if (threadIdx.x < kEwSums) {
    double v = 0.0;
#pragma unroll
    for (int w = 0; w < NW; w++) v += red[w][threadIdx.x];
    part[(size_t)threadIdx.x * n_part + blockIdx.x] = v;
  }
}

// One wave per axis, 64 atoms a block.  16 orders at a time go through LDS, so
// that an atom's values are written together (256 bytes).
__global__ __launch_bounds__(192) void k_ew_tables(EwDev d, const double *x) {
  __shared__ double buf[3][32][65];
  const int a = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int a0 = blockIdx.x * 64, i = min(a0 + lane, d.n - 1);
  double r[3];
  min_pos_exact(d.box, x[3 * i], x[3 * i + 1], x[3 * i + 2], r[0], r[1], r[2]);
  const double ra = a == 0 ? r[0] : (a == 1 ? r[1] : r[2]);
  const double xa = ra * 2.0 * M_PI * d.box.er[a];
  const double sn = sin(xa), cs = cos(xa);
  double s = 0.0, c = a == 0 ? d.q[i] : 1.0;
  for (int m0 = 0; m0 < d.H; m0 += 16) {
#pragma unroll
    for (int m = 0; m < 16; m++) {
      buf[a][2 * m][lane] = c;
      buf[a][2 * m + 1][lane] = s;
      ew_step(sn, cs, s, c);
    }
    wave_sync_lds();
    const int comp = lane & 31;
    const bool in = 2 * m0 + comp < 2 * d.H;
    for (int p = lane >> 5; p < 64; p += 2)
      if (in && a0 + p < d.n)
        d.tab[((size_t)(a0 + p) * 3 + a) * 2 * d.H + 2 * m0 + comp] =
            buf[a][comp][p];
    wave_sync_lds();
  }
}

__device__ __forceinline__ double ew_wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// C of eight row tiles over one chunk of atoms: a 16 x 80 block of a matrix
// product per tile, its inner dimension the atoms.  A wave holds two tiles in
// its accumulators, so a Z value read from LDS feeds two matrix instructions;
// the left operand is one product X Y per lane.  Eight atoms at a time are
// staged in two buffers, the next being read from memory meanwhile.
// Bound by the FP64 matrix rate: 96,000 atoms, 83,013 k-vectors 786 us (2,918 a
// lane an atom with the vector unit, bound by reading the tables 6,107 times);
// the matrix instructions alone are 545.  32 chunks of atoms instead of 48: 895
// (last blocks alone on the chip), 16 atoms a stage: 827.
template <int NC>
__device__ __forceinline__ void ew_sk_tiles(const EwDev &d, const EwTile *tiles,
                                            double (&buf)[2][kEwStage][kEwStride]) {
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int H2 = 2 * d.H;
  // what this thread stages: kEwStage x kEwVals values, 5 a thread
  constexpr int kPer = kEwStage * kEwVals / 256;
  static_assert(kPer * 256 == kEwStage * kEwVals, "whole rounds");
  unsigned src[kPer];
  int dst[kPer], sat[kPer];
#pragma unroll
  for (int p = 0; p < kPer; p++) {
    const int e = t + 256 * p, at = e / kEwVals, j = e % kEwVals;
    int off;
    if (j < kEwY) {
      off = 2 * tiles[j / 2].h + j % 2;
    } else if (j < kEwZ) {
      const int ti = (j - kEwY) / 8, kk = (j - kEwY) % 8;
      off = H2 + 2 * min(tiles[ti].k0 + kk / 2, d.H - 1) + kk % 2;
    } else {
      off = 2 * H2 + min(2 * tiles[0].m0 + j - kEwZ, H2 - 1);
    }
    src[p] = (unsigned)(at * 3 * H2 + off);
    sat[p] = at;
    dst[p] = at * kEwStride + j;
  }
  const int i0 = blockIdx.x * d.chunk, i1 = min(i0 + d.chunk, d.n);
  double next[kPer];
  auto fetch = [&](int i) {
    const double *row = d.tab + (size_t)i * 3 * H2;
    if (i + kEwStage <= i1) {
#pragma unroll
      for (int p = 0; p < kPer; p++) next[p] = row[src[p]];
    } else {  // atoms past the end count nothing
#pragma unroll
      for (int p = 0; p < kPer; p++) next[p] = i + sat[p] < i1 ? row[src[p]] : 0.0;
    }
  };
  // operand rows: 4 kq + product; products cos cos, sin sin, sin cos, cos sin
  const int t0 = 2 * wave, row = lane & 15, g = lane >> 4, pr = row & 3;
  const int xo = kEwX + 2 * t0 + (pr == 1 || pr == 2 ? 1 : 0) + g * kEwStride;
  const int yo = kEwY + 8 * t0 + 2 * (row >> 2) + (pr & 1) + g * kEwStride;
  const int zo = kEwZ + row + g * kEwStride;
  constexpr int kAcc = NC > 0 ? NC : 1;
  v4d acc[2][kAcc];
#pragma unroll
  for (int r = 0; r < 2; r++)
#pragma unroll
    for (int c = 0; c < kAcc; c++) acc[r][c] = v4d{0, 0, 0, 0};
  // the stage at i from buffer b, the next one fetched meanwhile
  auto stage = [&](int i, auto B) {
    constexpr int b = decltype(B)::value;
    const bool more = i + kEwStage < i1;
    if (more) fetch(i + kEwStage);
#pragma unroll
    for (int ks = 0; ks < kEwStage / 4; ks++) {
      const double *v = &buf[b][4 * ks][0];
      const double a0 = v[xo] * v[yo], a1 = v[xo + 2] * v[yo + 8];
#pragma unroll
      for (int c = 0; c < NC; c++) {
        const double z = v[zo + 16 * c];
        acc[0][c] =
            __builtin_amdgcn_mfma_f64_16x16x4f64(a0, z, acc[0][c], 0, 0, 0);
        acc[1][c] =
            __builtin_amdgcn_mfma_f64_16x16x4f64(a1, z, acc[1][c], 0, 0, 0);
      }
    }
    if (more) {
#pragma unroll
      for (int p = 0; p < kPer; p++) (&buf[b ^ 1][0][0])[dst[p]] = next[p];
    }
    __syncthreads();
  };
  fetch(i0);
#pragma unroll
  for (int p = 0; p < kPer; p++) (&buf[0][0][0])[dst[p]] = next[p];
  __syncthreads();
  for (int i = i0; i < i1; i += 2 * kEwStage) {
    stage(i, std::integral_constant<int, 0>{});
    if (i + kEwStage < i1)
      stage(i + kEwStage, std::integral_constant<int, 1>{});
  }
  // register v of lane group g is row 4 v + g: |k| = k0 + v, product g
#pragma unroll
  for (int r = 0; r < 2; r++) {
    const int ti = blockIdx.y * kEwTiles + t0 + r;
    double *out = d.C + ((size_t)blockIdx.x * d.n_tiles + ti) * 16 * kEwCols;
#pragma unroll
    for (int c = 0; c < NC; c++)
      if (c < tiles[t0 + r].nc)
#pragma unroll
        for (int v = 0; v < 4; v++)
          out[(4 * v + g) * kEwCols + 16 * c + row] = acc[r][c][v];
  }
}

__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(2))) void k_ew_sk(EwDev d) {
  __shared__ double buf[2][kEwStage][kEwStride];
  const EwTile *tiles = d.tiles + blockIdx.y * kEwTiles;
  // one width for the block (the barriers are inside): the widest, the first
  switch (tiles[0].nc) {
    case 1: ew_sk_tiles<1>(d, tiles, buf); break;
    case 2: ew_sk_tiles<2>(d, tiles, buf); break;
    case 3: ew_sk_tiles<3>(d, tiles, buf); break;
    case 4: ew_sk_tiles<4>(d, tiles, buf); break;
    default: ew_sk_tiles<5>(d, tiles, buf); break;
  }
}

// One block per row tile: the sums of C over the atom chunks in order, then
// one thread per (|k|, m): the structure factors of (h, +-k, +-m), their
// energy and virial, and the force's coefficients.
constexpr int kEwCoefBlock = 16 * kEwOrders;  // a thread per row and m
__global__ __launch_bounds__(kEwCoefBlock) void k_ew_coef(EwDev d) {
  __shared__ double Cs[16][kEwCols];
  const EwTile ti = d.tiles[blockIdx.x];
  const int t = threadIdx.x;
  {
    const int row = t / kEwOrders, mm = t % kEwOrders;
    double a = 0.0, b = 0.0;
    if (mm < 8 * ti.nc) {
      const double2 *p = reinterpret_cast<const double2 *>(
          d.C + ((size_t)blockIdx.x * 16 + row) * kEwCols + 2 * mm);
      const size_t step = (size_t)d.n_tiles * 16 * kEwCols / 2;
#pragma unroll 8
      for (int c = 0; c < d.n_chunks; c++) {
        const double2 v = p[c * step];
        a += v.x;
        b += v.y;
      }
    }
    Cs[row][2 * mm] = a;
    Cs[row][2 * mm + 1] = b;
  }
  __syncthreads();
  double acc[kEwSums] = {0, 0, 0, 0, 0, 0, 0};
  const int kq = t / kEwOrders, mm = t % kEwOrders;
  const int ka = ti.k0 + kq, m = ti.m0 + mm;
  if (kq < 4 && mm < 8 * ti.nc) {
    const EwH hh = d.hs[ti.h];
    const double cc[2] = {Cs[4 * kq][2 * mm], Cs[4 * kq][2 * mm + 1]};
    const double ss[2] = {Cs[4 * kq + 1][2 * mm], Cs[4 * kq + 1][2 * mm + 1]};
    const double sc[2] = {Cs[4 * kq + 2][2 * mm], Cs[4 * kq + 2][2 * mm + 1]};
    const double cs[2] = {Cs[4 * kq + 3][2 * mm], Cs[4 * kq + 3][2 * mm + 1]};
    for (int sk = 0; sk < (ka == 0 ? 1 : 2); sk++) {
      const int k = sk == 0 ? ka : -ka;
      if (k < hh.kmin || k > hh.kmax) continue;
      const double sg = sk == 0 ? 1.0 : -1.0;
      const EwRun r = d.runs[hh.run0 + k - hh.kmin];
      // sums of cos(h x + k y) z and sin(h x + k y) z, z = cos, sin(m z)
      const double xyc[2] = {cc[0] - sg * ss[0], cc[1] - sg * ss[1]};
      const double xys[2] = {sc[0] + sg * cs[0], sc[1] + sg * cs[1]};
      double ps[2] = {0, 0}, pc[2] = {0, 0};  // l = +m, -m
      double kz = 0.0;
      bool any = false;
      for (int sl = 0; sl < (m == 0 ? 1 : 2); sl++) {
        const int l = sl == 0 ? m : -m;
        if (l < r.l_lo || l > r.l_hi) continue;
        const double tg = sl == 0 ? 1.0 : -1.0;
        const double4 kv = d.kv[r.start + (l - r.l_lo)];
        const double S = xys[0] + tg * xyc[1], Cc = xyc[0] - tg * xys[1];
        const double k2 = kv.x * kv.x + kv.y * kv.y + kv.z * kv.z;
        const double e = kv.w * (S * S + Cc * Cc);
        const double f = 2.0 * (1.0 / k2 + d.fac);
        acc[0] += e;
        acc[1] += e * (1.0 - f * kv.x * kv.x);
        acc[2] -= e * f * kv.x * kv.y;
        acc[3] -= e * f * kv.x * kv.z;
        acc[4] += e * (1.0 - f * kv.y * kv.y);
        acc[5] -= e * f * kv.y * kv.z;
        acc[6] += e * (1.0 - f * kv.z * kv.z);
        const double ak = 8.0 * M_PI * d.Vr * kv.w;
        ps[sl] = ak * Cc;
        pc[sl] = ak * S;
        kz = sl == 0 ? kv.z : -kv.z;
        any = true;
      }
      if (!any) continue;
      const int j = (k - hh.kmin) & 3;
      const int2 fs = d.fsteps[(ti.m0 / kEwOrders) * d.n_ft + hh.ft0 +
                               ((k - hh.kmin) >> 2)];
      // column 2 mm (cos) and 2 mm + 1 (sin); row 4 output + j
      double *P = d.P + (size_t)(fs.x + (mm >> 1)) * 64 + (2 * mm & 3) * 16 + j;
      P[0] = ps[0] + ps[1];                  // U, cos
      P[4] = -(pc[0] + pc[1]);               // V, cos
      P[8] = kz * (ps[0] - ps[1]);           // U', cos
      P[12] = -kz * (pc[0] - pc[1]);         // V', cos
      P[16] = pc[0] - pc[1];                 // U, sin
      P[20] = ps[0] - ps[1];                 // V, sin
      P[24] = kz * (pc[0] + pc[1]);          // U', sin
      P[28] = kz * (ps[0] + ps[1]);          // V', sin
    }
  }
  ew_store_sums<kEwCoefBlock / 64>(acc, d.part, d.n_tiles);
}

// Forces of 32 atoms a wave over a split of the (h, k) tiles.  The matrix
// product's rows are the four outputs U, V, U', V' of four k, its columns the
// atoms and its inner dimension the columns of Z, which stay in registers for
// the whole pass; a step's coefficients are 512 contiguous bytes, read four
// steps ahead, the same for all waves.  A lane gets the four outputs
// of one k and one atom; exp(i (h x + k y)) goes from tile to tile of one h by
// a rotation of 4 y.  Bound by the FP64
// matrix rate: 96,000 atoms, 83,013 k-vectors 1,360 us (4,660 with 11 vector
// operations a k-vector and atom); the matrix instructions alone are 938, an
// eighth of them on columns beyond the sphere.
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(3))) void k_ew_force(EwDev d) {
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int a0 = (blockIdx.x * 4 + wave) * kEwAtoms;
  if (a0 >= d.n) return;
  const int H2 = 2 * d.H;
  const int f0 = d.fsplit[blockIdx.y], f1 = d.fsplit[blockIdx.y + 1];
  const double *row[2];
  double c4[2], s4[2], fx[2], fy[2], fz[2];
#pragma unroll
  for (int u = 0; u < 2; u++) {
    row[u] = d.tab + (size_t)min(a0 + 16 * u + col, d.n - 1) * 3 * H2;
    const double c1 = row[u][H2 + 2], s1 = row[u][H2 + 3];
    double s = s1, c = c1;
    ew_step(s1, c1, s, c);
    s4[u] = s;
    c4[u] = c;
    ew_step(s, c, s4[u], c4[u]);
    fx[u] = fy[u] = fz[u] = 0.0;
  }
  for (int pass = 0; pass < d.n_pass; pass++) {
    double z[2][kEwSteps];
#pragma unroll
    for (int s = 0; s < kEwSteps; s++)
#pragma unroll
      for (int u = 0; u < 2; u++)
        z[u][s] = row[u][2 * H2 + min(pass * kEwCols + 4 * s + g, H2 - 1)];
    const int2 *fs = d.fsteps + (size_t)pass * d.n_ft;
    // P is wave-uniform; p0 .. p3 hold the next four steps' coefficients
    const double *P = d.P + (size_t)fs[f0].x * 64;
    double p0 = P[lane], p1 = P[64 + lane], p2 = P[128 + lane],
           p3 = P[192 + lane];
    double xyc[2] = {0, 0}, xys[2] = {0, 0}, W[2] = {0, 0};
    int h = -1;
    EwFTile tl = d.ftiles[f0];
    int nst = fs[f0].y;
    for (int ft = f0; ft < f1; ft++) {
      const int fn = min(ft + 1, f1 - 1);
      const EwFTile tn = d.ftiles[fn];
      const int nn = fs[fn].y;
      if (tl.h != h) {
        const double kx = h * d.kunit[0];
        const int k = tl.k0 + g, ka = min(k < 0 ? -k : k, d.H - 1);
        h = tl.h;
#pragma unroll
        for (int u = 0; u < 2; u++) {
          fx[u] = fma(kx, W[u], fx[u]);
          W[u] = 0.0;
          const double xc = row[u][2 * h], xs = row[u][2 * h + 1];
          const double yc = row[u][H2 + 2 * ka];
          const double y1 = row[u][H2 + 2 * ka + 1], ys = k < 0 ? -y1 : y1;
          xyc[u] = fma(xc, yc, -(xs * ys));
          xys[u] = fma(xs, yc, xc * ys);
        }
      } else {
#pragma unroll
        for (int u = 0; u < 2; u++) ew_step(s4[u], c4[u], xys[u], xyc[u]);
      }
      const int k0 = tl.k0, steps = nst;
      tl = tn;
      nst = nn;
      if (steps == 0) continue;
      v4d o[2] = {v4d{0, 0, 0, 0}, v4d{0, 0, 0, 0}};
      auto two = [&](int s, double &pa, double &pb) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; u++)
          o[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(pa, z[u][s], o[u], 0, 0, 0);
        pa = P[(s + 4) * 64 + lane];
#pragma unroll
        for (int u = 0; u < 2; u++)
          o[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(pb, z[u][s + 1], o[u], 0, 0, 0);
        pb = P[(s + 5) * 64 + lane];
      };
      // an odd number of pairs leaves the registers' turns swapped
      two(0, p0, p1);
#pragma unroll
      for (int s = 2; s < kEwSteps; s += 4) {
        if (s < steps) two(s, p2, p3);
        if (s + 2 < steps && s + 2 < kEwSteps) two(s + 2, p0, p1);
      }
      if (steps & 2) {
        const double q0 = p0, q1 = p1;
        p0 = p2;
        p1 = p3;
        p2 = q0;
        p3 = q1;
      }
      P += steps * 64;
      const double ky = (k0 + g) * d.kunit[1];
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const double w = fma(xys[u], o[u][0], xyc[u] * o[u][1]);
        W[u] += w;
        fy[u] = fma(ky, w, fy[u]);
        fz[u] = fma(xys[u], o[u][2], fma(xyc[u], o[u][3], fz[u]));
      }
    }
    const double kx = h * d.kunit[0];
#pragma unroll
    for (int u = 0; u < 2; u++) fx[u] = fma(kx, W[u], fx[u]);
  }
  // the four k of a tile, then the atom's partial force
#pragma unroll
  for (int u = 0; u < 2; u++) {
    fx[u] += __shfl_xor(fx[u], 16);
    fy[u] += __shfl_xor(fy[u], 16);
    fz[u] += __shfl_xor(fz[u], 16);
    fx[u] += __shfl_xor(fx[u], 32);
    fy[u] += __shfl_xor(fy[u], 32);
    fz[u] += __shfl_xor(fz[u], 32);
    const int i = a0 + 16 * u + col;
    if (i < d.n && g < 3)
      d.pf[((size_t)blockIdx.y * d.n + i) * 3 + g] =
          g == 0 ? fx[u] : (g == 1 ? fy[u] : fz[u]);
  }
}

// The splits' forces in order and the correction, two lanes per atom.
constexpr int kEwFinalLanes = 2;
__global__ __launch_bounds__(256) void k_ew_final(EwDev d, const double *x,
                                                  double *f) {
  const int at = blockIdx.x * (256 / kEwFinalLanes) + threadIdx.x / kEwFinalLanes;
  const int sub = threadIdx.x % kEwFinalLanes;
  double acc[kEwSums] = {0, 0, 0, 0, 0, 0, 0};
  double gx = 0.0, gy = 0.0, gz = 0.0;
  if (at < d.n) {
    if (sub == 0)
      for (int s = 0; s < d.n_split; s++) {
        const double *p = d.pf + ((size_t)s * d.n + at) * 3;
        gx += p[0];
        gy += p[1];
        gz += p[2];
      }
    ew_correction(d, x, at, sub, kEwFinalLanes, gx, gy, gz, acc);
  }
  gx += __shfl_xor(gx, 1);
  gy += __shfl_xor(gy, 1);
  gz += __shfl_xor(gz, 1);
  if (at < d.n && sub == 0) {
    f[3 * at] += gx;
    f[3 * at + 1] += gy;
    f[3 * at + 2] += gz;
  }
  ew_store_sums<4>(acc, d.cpart, d.n_cpart);
}

// Sums of the k-space terms over the blocks: wave w < 14 adds one of them
// (lanes by stride, then by halving: a fixed order; one lane per sum took
// 235 us over 1,764 blocks).  out[1] += scale energy + correction + constant
// energies, and with the virial flag the virial slots XX..ZZ += scale virial +
// the correction's + the charged-system diagonal.
__global__ __launch_bounds__(1024) void k_ew_finish(
    const double *part, int n_part, const double *cpart, int n_cpart,
    double scale, double *out, int virial, double e_const, double e_charged) {
  __shared__ double tot[2 * kEwSums];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (w < 2 * kEwSums) {
    const bool corr = w >= kEwSums;
    const int n = corr ? n_cpart : n_part;
    const double *p =
        (corr ? cpart : part) + (size_t)(corr ? w - kEwSums : w) * n;
    double v0 = 0.0, v1 = 0.0, v2 = 0.0, v3 = 0.0;
    int b = lane;
    for (; b + 192 < n; b += 256) {
      v0 += p[b];
      v1 += p[b + 64];
      v2 += p[b + 128];
      v3 += p[b + 192];
    }
    for (; b < n; b += 64) v0 += p[b];
    const double v = ew_wave_sum((v0 + v1) + (v2 + v3));
    if (lane == 0) tot[w] = v;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const double *c = tot + kEwSums;
    out[1] += tot[0] * scale + c[0] + e_const;
    if (virial) {
      // slots XX XY XZ YX YY YZ ZX ZY ZZ (ScalarStructure::addVirial)
      const double xx = tot[1] * scale + c[1] + e_charged;
      const double xy = tot[2] * scale + c[2], xz = tot[3] * scale + c[3];
      const double yy = tot[4] * scale + c[4] + e_charged;
      const double yz = tot[5] * scale + c[5];
      const double zz = tot[6] * scale + c[6] + e_charged;
      out[2] += xx; out[3] += xy; out[4] += xz;
      out[5] += xy; out[6] += yy; out[7] += yz;
      out[8] += xz; out[9] += yz; out[10] += zz;
    }
  }
}

}  // namespace pmnb
