// Adjoint (reverse-mode derivative) of the cutoff force.
//
// Given an upstream gradient g = dL/dF (3 per atom), returns
//   dL/dx_k = sum_j dL/dF_j . dF_j/dx_k   (a Hessian-vector product, -H g)
//   dL/dq~_k for every scaled charge, and
//   dL/d{A, B, A14, B14} for every unordered LJ type pair,
// recomputing the pairs from the cell list instead of storing them.
//
// The force on atom i from pair (i, j) is F_i = -d ff(a), d = x_j - x_i
// (minimum image), a = |d|^2, ff = F/r of OneAtomPairTwo::doOneAtomPair
// (force/OneAtomPairTwo.h:96-111): ff = F S - E S~ for each of the two terms,
// with S the switch and S~ its derivative divided by r.  Its Jacobian is
// dF_i/dx_i = ff I + 2 ff' d d^T (ff' = dff/da), the negative of the pair
// Hessian block the reference builds in ReducedHessLennardJones
// (force/hessian/ReducedHessLennardJones.cpp:7-42) and ReducedHessCoulomb
// (force/hessian/ReducedHessCoulomb.cpp:6-35) with the C2 switch Hessian
// (switch/C2SwitchingFunction.cpp:43-52).  With w = g_j - g_i:
//   dL/dx_i  += -(ff w + 2 ff' (w . d) d)
//   dL/dq~_i += (w . d) q~_j h        (ff of the electrostatic term = qq h)
//   dL/dA    += (w . d) dff/dA / 2    (each unordered pair seen twice)
// For the Ewald term ff' differentiates the force expression as the
// reference writes it (the erfc of its energy is the A&S approximation,
// its force uses the exact erfc derivative), so the Jacobian is that of the
// forces actually computed.
//
// k_pairs (pmnb_cluster.h) walks the pairs, in its mode kAdjoint: a lane keeps
// its atom's dL/dx and dL/dq~ in registers and, per type of the partner, the
// LJ-parameter gradients; the four lanes of an atom are added in a fixed order
// and the parameter gradients written per atom, which k_adj_lj_part and
// k_adj_lj_finish add by type pair.
#pragma once

#include "pmnb_queue.h"
#include "pmnb_pair.h"

namespace pmnb {

constexpr int kAdjTypes = 4;  // most LJ types of the adjoint

// Constants of the adjoint in the kernel's precision.
template <typename R>
struct AdjC {
  R on2l, cut2l, s1l, s2l, s3l;   // C2 switch of the LJ term
  R on2e, cut2e, s1e, s2e, s3e;   // C2 switch of the electrostatic term
  R alpha, c2ap, csf;             // alpha, 2 alpha / sqrt(pi), 1-4 factor
};

// What k_pairs takes for the adjoint.
struct AdjArgs {
  const double *grad_f;           // dL/dF, 3 per atom
  double *grad_x, *grad_q;        // dL/dx, dL/dq~ (null: not wanted)
  double *lj;                     // (4 tj + c) rows of n sorted atoms (null:
                                  // not wanted): dL/d{A, B, A14, B14} / 2
  AdjC<float> c32;
  AdjC<double> c64;
};

__device__ __forceinline__ float adj_rsq(float x) {
  return __builtin_amdgcn_rsqf(x);
}
__device__ __forceinline__ double adj_rsq(double x) { return rsq64(x); }
__device__ __forceinline__ float adj_rcp(float x) {
  return __builtin_amdgcn_rcpf(x);
}
__device__ __forceinline__ double adj_rcp(double x) { return rcp64(x); }
__device__ __forceinline__ float adj_exp(float x) {
  return __builtin_amdgcn_exp2f(x * 1.4426950408889634f);
}
__device__ __forceinline__ double adj_exp(double x) { return exp64_neg(x); }
__device__ __forceinline__ float adj_fma(float a, float b, float c) {
  return fmaf(a, b, c);
}
__device__ __forceinline__ double adj_fma(double a, double b, double c) {
  return fma(a, b, c);
}

// C2 value S, S~ = (dS/dr) / r = 2 dS/da and S'' = d2S/da2
// (switch/C2SwitchingFunction.h:42-53, .cpp:43-52).
template <typename R>
__device__ __forceinline__ void c2_adj(R a, R on2, R cut2, R s1, R s2, R s3,
                                       R &S, R &Sd, R &S2) {
  const R c2 = cut2 - a;
  const R b = adj_fma(R(2), a, s2);
  const R c4 = c2 * b;
  const bool on = a >= on2, in = a <= cut2;
  S = on ? (in ? s1 * (c2 * c4) : R(0)) : R(1);
  Sd = on && in ? s3 * adj_fma(c2, c2, -c4) : R(0);
  S2 = on && in ? R(2) * s1 * adj_fma(R(-4), c2, b) : R(0);
}

// Per-pair terms of the adjoint: ff, ff' = dff/da, h = (electrostatic ff) /
// qq, and dff/dA, dff/dB.  A, B are the MODIFIED (A14, B14) values for a
// 1-4 pair; qq includes the 1-4 factor.  SAME: one switch for both terms.
// The LJ terms use dE/da = -F / 2.
template <typename R, int ELEC, bool SAME>
__device__ __forceinline__ void pair_adj(const AdjC<R> &C, R a, R A, R B,
                                         R qq, R &ff, R &ffp, R &h, R &dA,
                                         R &dB) {
  const R rr = ELEC != 0 ? adj_rsq(a) : R(0);
  const R ia = ELEC != 0 ? rr * rr : adj_rcp(a);
  const R ia3 = ia * ia * ia, ia6 = ia3 * ia3;
  // LennardJonesForce (force/LennardJonesForce.h:29-61): E = A/r^12 - B/r^6
  const R a6 = A * ia3;
  const R E = ia3 * (a6 - B);
  const R F = adj_fma(ia3, a6, E) * (R(6) * ia);
  const R Fp = R(-12) * (ia * ia) * ia3 * adj_fma(R(7), a6, R(-2) * B);
  R S, Sd, S2;
  c2_adj(a, C.on2l, C.cut2l, C.s1l, C.s2l, C.s3l, S, Sd, S2);
  ff = adj_fma(F, S, -E * Sd);
  ffp = adj_fma(Fp, S, adj_fma(F, Sd, R(-2) * E * S2));
  dA = ia6 * adj_fma(R(12) * ia, S, -Sd);
  dB = -ia3 * adj_fma(R(6) * ia, S, -Sd);
  h = R(0);
  if (ELEC == 0) return;
  R u, up, v, vp;
  if (ELEC == 1) {
    // CoulombForce (force/CoulombForce.h:27-38): E = qq / r, F/r = E / r^2
    u = rr;
    up = R(-0.5) * rr * ia;
    v = u * ia;
    vp = R(-1.5) * v * ia;
  } else {
    // Ewald real space: E = qq erfc(alpha r) / r with the A&S erfc
    // (base/MathUtilities.cpp:39-49), F/r = (E + qq 2 alpha/sqrt(pi)
    // exp(-alpha^2 r^2)) / r^2 (force/nonbonded/NonbondedFullEwaldSystemForce
    // .h:810-821)
    const R r = a * rr;
    const R ar = C.alpha * r, al2 = C.alpha * C.alpha;
    const R t = adj_rcp(adj_fma(R(0.3275911), ar, R(1)));
    const R e1 = R(0.254829592), e2 = R(-0.284496736), e3 = R(1.421413741),
            e4 = R(-1.453152027), e5 = R(1.061405429);
    const R P = t * adj_fma(t, adj_fma(t, adj_fma(t, adj_fma(t, e5, e4), e3), e2), e1);
    const R Pt = adj_fma(
        t,
        adj_fma(t, adj_fma(t, adj_fma(t, R(5) * e5, R(4) * e4), R(3) * e3),
                R(2) * e2),
        e1);
    const R x = adj_exp(-al2 * a);
    const R tp = R(-0.5) * R(0.3275911) * C.alpha * t * t * rr;  // dt/da
    const R xr = x * rr, cx = C.c2ap * x;
    u = P * xr;
    up = adj_fma(xr * Pt, tp, -u * adj_fma(R(0.5), ia, al2));
    v = (u + cx) * ia;
    vp = ia * (adj_fma(-al2, cx, up) - v);
  }
  if (!SAME) c2_adj(a, C.on2e, C.cut2e, C.s1e, C.s2e, C.s3e, S, Sd, S2);
  h = adj_fma(v, S, -u * Sd);
  const R hp = adj_fma(vp, S, adj_fma(R(0.5) * v - up, Sd, R(-2) * u * S2));
  ff = adj_fma(qq, h, ff);
  ffp = adj_fma(qq, hp, ffp);
}

// LJ-parameter gradients from the atoms' rows.  k_adj_lj_part: block (chunk,
// row) adds its slice of sorted atoms by the atom's type (fixed tree);
// k_adj_lj_finish adds the chunks of the ordered type pairs (ti, tj) and (tj,
// ti) in order, and adds them to grad_lj (T x T x 4, {A, B, A14, B14}), half
// of an unordered off-diagonal pair's gradient to each of its two entries.
constexpr int kAdjChunks = 64, kAdjRows = 4 * kAdjTypes;
__global__ void __launch_bounds__(kBlock)
k_adj_lj_part(const double *__restrict__ lj, const int *__restrict__ stype,
              int n, double *__restrict__ part) {
  __shared__ double red[kBlock / 64][kAdjTypes];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int per = (n + kAdjChunks - 1) / kAdjChunks;
  const int i0 = blockIdx.x * per, i1 = min(i0 + per, n);
  const double *row = lj + (size_t)blockIdx.y * n;
  double acc[kAdjTypes] = {0, 0, 0, 0};
  for (int i = i0 + (int)threadIdx.x; i < i1; i += kBlock) {
    const double v = row[i];
    const int ty = stype[i];
#pragma unroll
    for (int c = 0; c < kAdjTypes; c++) acc[c] += ty == c ? v : 0.0;
  }
#pragma unroll
  for (int c = 0; c < kAdjTypes; c++) {
    double v = acc[c];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if (lane == 0) red[wave][c] = v;
  }
  __syncthreads();
  if (threadIdx.x < kAdjTypes) {
    double v = 0.0;
    for (int w = 0; w < kBlock / 64; w++) v += red[w][threadIdx.x];
    part[((size_t)blockIdx.x * kAdjRows + blockIdx.y) * kAdjTypes +
         threadIdx.x] = v;
  }
}

// One block: thread (ti, tj, c) of kAdjTypes x kAdjTypes x 4.
__global__ void __launch_bounds__(64)
k_adj_lj_finish(const double *__restrict__ part, int T,
                double *__restrict__ grad_lj) {
  __shared__ double sum[kAdjTypes][kAdjTypes][4];
  const int t = threadIdx.x;
  const int ti = t / (4 * kAdjTypes), tj = t / 4 % kAdjTypes, c = t % 4;
  double v = 0.0;
  for (int k = 0; k < kAdjChunks; k++)
    v += part[((size_t)k * kAdjRows + 4 * tj + c) * kAdjTypes + ti];
  sum[ti][tj][c] = v;
  __syncthreads();
  if (ti >= T || tj >= T) return;
  const double both = ti == tj ? sum[ti][tj][c]
                               : 0.5 * (sum[min(ti, tj)][max(ti, tj)][c] +
                                        sum[max(ti, tj)][min(ti, tj)][c]);
  grad_lj[4 * (ti * T + tj) + c] += both;
}

}  // namespace pmnb
