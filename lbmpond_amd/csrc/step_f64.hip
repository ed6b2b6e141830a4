// step_f64.hip -- plain FP64 PonD step for gfx950, reference operation order.
//
// Replaces PonDstep -> LBMpull<> (update.cu:11-14, steps.cu:356-588) and PonDstepD3Q125
// (steps.cu:151-250).  Every rounding step of the reference is reproduced: loops run in the
// reference order, expression trees are kept, the build disables FMA contraction.  The only
// changes are ones that cannot alter a bit:
//   * pure sub-expressions are hoisted (the node's sqrt(|T0|)*sign(T0), the per-target
//     constants, the shared left prefixes W*gx, (W*gx)*gy of the left-associated products);
//   * a node's transfer to a given target is computed once and reused where the reference
//     recomputes it (the three overlapping WENO sub-stencils; 1D grids, where all y/z stencil
//     nodes are the same cell);
//   * the transfer's NaN/Inf test is made on its sum (terms27);
//   * the moment sums (structs.cuh:323-327) run over the stored iterate in the same population order.
//
// D3Q27 mapping: nine lanes per cell, one (ey, ez) group of three targets each; WENO5 cells that go on
// iterating, one workgroup each.  D1Q5 lines: 32 lanes per cell; other D1Q5 grids: one lane per
// cell, 64 consecutive cells (x fastest) per wave.  D3Q125 mapping: one 128-lane block per cell, lane =
// target population (as the reference's 125-thread block), the nodes of the fixed 3x3x3 neighbourhood
// through scalar loads.
#include <type_traits>
#include "pond_device.h"

namespace pond {

// ---------------------------------------------------------------------------------------------
// Gauge transfer, D3Q27 (structs.cuh:525-548)

struct Tgt27 {
  double u1x, u1y, u1z, T1;
  double W;           // (wk*wl)*wm
  double Cx, Cy, Cz;  // (e_inew*sqrt(|T1|))*sign(T1)
  bool kx, ky, kz;    // e_inew component != 0
};

// target population with velocity components (ex, ey, ez)
__device__ __forceinline__ Tgt27 make_tgt27e(int ex, int ey, int ez, double u1x, double u1y, double u1z, double T1) {
  Tgt27 t;
  t.u1x = u1x; t.u1y = u1y; t.u1z = u1z; t.T1 = T1;
  double wk = 1. / (2 * T1), wl = wk, wm = wk;
  if (ex == 0) wk = -1. / T1;
  if (ey == 0) wl = -1. / T1;
  if (ez == 0) wm = -1. / T1;
  t.W = wk * wl * wm;
  const double sq1 = sqrt(fabs(T1));
  const double sg1 = (double)isign_d(T1);
  t.Cx = (double)ex * sq1 * sg1;
  t.Cy = (double)ey * sq1 * sg1;
  t.Cz = (double)ez * sq1 * sg1;
  t.kx = ex != 0; t.ky = ey != 0; t.kz = ez != 0;
  return t;
}

// Node data of the load state: plane bases plus a per-node 32-bit byte offset.
struct NodeSrc {
  const double* __restrict__ f;          // population planes, stride g.plane
  const double* __restrict__ m;          // rho, ux, uy, uz, T planes
  const double* __restrict__ P;          // sqrt(|T|)*sign(T) per cell (params.h:110-112)
  Grid g;
};

__device__ __forceinline__ double ldp(const double* base, int64_t k, int64_t plane, uint32_t boff) {
  return *(const double*)((const char*)(base + k * plane) + boff);
}

__device__ __forceinline__ uint32_t node_off(const Grid& g, int x, int y, int z) {
  return ((uint32_t)x + (uint32_t)g.nx * ((uint32_t)y + (uint32_t)g.ny * (uint32_t)z)) * 8u;
}

// The D3Q27 node data as raw buffer resources: pair planes 4j .. 4j+3 in resource j, the plane
// selected by the scalar offset, the per-lane address a single 32-bit offset (a global load needs a
// 64-bit per-lane address: two VGPRs and a 64-bit add per load).  Resource sizes are exact, so the
// hardware range check returns 0 rather than reading past an array.  Word 3 (0x00020000) is the
// raw-buffer configuration of the gfx9 family.  Usable while four pair planes fit in 4 GiB (plane <=
// 67,108,800 cells).
constexpr int kRawBufferWord3 = 0x00020000;

struct NodeBuf {
  __amdgpu_buffer_rsrc_t f[4], P;
  uint32_t qbytes;  // bytes per pair plane
  Grid g;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc64(const void* base, uint64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)(uint32_t)bytes, kRawBufferWord3);
}

__device__ __forceinline__ NodeBuf make_nodebuf(const NodeSrc& s) {
  NodeBuf b;
  const uint64_t pb = (uint64_t)s.g.plane * 8u;
  b.qbytes = (uint32_t)(2 * pb);
  for (int j = 0; j < 4; j++) {
    const int cnt = 14 - 4 * j < 4 ? 14 - 4 * j : 4;
    b.f[j] = rsrc64(s.f + (int64_t)8 * j * s.g.plane, (uint64_t)cnt * 2 * pb);
  }
  b.P = rsrc64(s.P, 4 * pb);
  b.g = s.g;
  return b;
}

// node accessors: population k, moment plane k, P of the node at byte offset boff
__device__ __forceinline__ double node_f(const NodeSrc& s, int k, uint32_t boff) { return ldp(s.f, k, s.g.plane, boff); }
__device__ __forceinline__ double node_m(const NodeSrc& s, int k, uint32_t boff) { return ldp(s.m, k, s.g.plane, boff); }
__device__ __forceinline__ double node_P(const NodeSrc& s, uint32_t boff) { return ldp(s.P, 0, s.g.plane, boff); }

// D3Q27: the node's gauge record (ux, uy, uz, sqrt(|T|)*sign(T)), 32 bytes per cell, written by
// k_node_prep into the P buffer, at byte offset boff of an FP64 plane (boff = 8 * cell)
// (64-bit byte offsets: 4 * boff leaves 32 bits from 2^27 cells on, the grids this path serves)
__device__ __forceinline__ void node_g4(const NodeSrc& s, uint32_t boff, double& ux, double& uy, double& uz,
                                       double& P) {
  const double2 a = *(const double2*)((const char*)s.P + 4ull * boff);
  const double2 b = *(const double2*)((const char*)s.P + 4ull * boff + 16ull);
  ux = a.x; uy = a.y; uz = b.x; P = b.y;
}
__device__ __forceinline__ double dbl_of(uint32_t lo, uint32_t hi) {
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ void node_g4(const NodeBuf& s, uint32_t boff, double& ux, double& uy, double& uz,
                                       double& P) {
  const auto a = __builtin_amdgcn_raw_buffer_load_b128(s.P, (int)(4u * boff), 0, 0);
  const auto b = __builtin_amdgcn_raw_buffer_load_b128(s.P, (int)(4u * boff), 16, 0);
  ux = dbl_of((uint32_t)a[0], (uint32_t)a[1]);
  uy = dbl_of((uint32_t)a[2], (uint32_t)a[3]);
  uz = dbl_of((uint32_t)b[0], (uint32_t)b[1]);
  P = dbl_of((uint32_t)b[2], (uint32_t)b[3]);
}

// the 27 populations of a D3Q27 node (pair-plane layout) at byte offset boff of an FP64 plane
__device__ __forceinline__ void node_f27(const NodeSrc& s, uint32_t boff, double f[27]) {
#pragma unroll
  for (int j = 0; j < 14; j++) {
    const double2 v = *(const double2*)((const char*)(s.f + (int64_t)2 * j * s.g.plane) + 2ull * boff);
    f[2 * j] = v.x;
    if (2 * j + 1 < 27) f[2 * j + 1] = v.y;
  }
}
__device__ __forceinline__ void node_f27(const NodeBuf& s, uint32_t boff, double f[27]) {
#pragma unroll
  for (int j = 0; j < 14; j++) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(s.f[j >> 2], (int)(2u * boff), (int)((uint32_t)(j & 3) * s.qbytes), 0);
    f[2 * j] = __builtin_bit_cast(double, ((uint64_t)(uint32_t)v[1] << 32) | (uint32_t)v[0]);
    if (2 * j + 1 < 27) f[2 * j + 1] = __builtin_bit_cast(double, ((uint64_t)(uint32_t)v[3] << 32) | (uint32_t)v[2]);
  }
}

// basis values of a node with gauge (u0, P) for target t (structs.cuh:530-538).
// e_iold*sqrt(|T0|)*sign(T0) for e_iold = -1, 0, +1 is exactly {-P, 0*P, P}.
__device__ __forceinline__ void basis27(double u0x, double u0y, double u0z, double Pn, const Tgt27& t, double sqTb,
                                        double gx[3], double gy[3], double gz[3]) {
  const double Dx = (t.u1x - u0x) * sqTb;
  const double Dy = (t.u1y - u0y) * sqTb;
  const double Dz = (t.u1z - u0z) * sqTb;
  const double E[3] = {-Pn, 0.0 * Pn, Pn};
#pragma unroll
  for (int j = 0; j < 3; j++) {
    const double ax = Dx - E[j], ay = Dy - E[j], az = Dz - E[j];
    gx[j] = ax * ax - (t.kx ? t.Cx * ax : t.T1);
    gy[j] = ay * ay - (t.ky ? t.Cy * ay : t.T1);
    gz[j] = az * az - (t.kz ? t.Cz * az : t.T1);
  }
}

// The transfer's term loop (structs.cuh:539-548) over the populations f.  The reference drops every
// NaN or infinite term; a sum that comes out finite has dropped none (one such term leaves the plain
// sum NaN or infinite), so the plain sum is formed and only a non-finite one is formed again with
// the test on every term, from the start: kept for that, the 27 products took 54 registers of every
// node (128^3 vortex 63.7 -> 55.8 ms per step without).
__device__ __forceinline__ double terms27(double W, const double (&gx)[3], const double (&gy)[3],
                                          const double (&gz)[3], const double (&f)[27]) {
  double p2[3][3];
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++) p2[a][b] = W * gx[a] * gy[b];
  double fnew = 0;
#pragma unroll
  for (int iold = 0; iold < 27; iold++) {
    const int jx = kE27[iold][0] + 1, jy = kE27[iold][1] + 1, jz = kE27[iold][2] + 1;
    fnew += p2[jx][jy] * gz[jz] * f[iold];
  }
  if (!finite_d(fnew)) {
    fnew = 0;
    double Wa = W;  // (the compiler would keep the products of the plain sum)
    asm volatile("" : "+v"(Wa));
#pragma unroll
    for (int iold = 0; iold < 27; iold++) {
      const int jx = kE27[iold][0] + 1, jy = kE27[iold][1] + 1, jz = kE27[iold][2] + 1;
      const double fadd = Wa * gx[jx] * gy[jy] * gz[jz] * f[iold];
      if (finite_d(fadd)) fnew += fadd;
    }
  }
  return fnew;
}

// exchanges the populations of a D3Q27 record with their mirror images along axis AX in the lanes
// with m set
template <int AX>
__device__ __forceinline__ void mirror27(bool m, double (&f)[27]) {
#pragma unroll
  for (int i = 0; i < 27; i++) {
    if (kE27[i][AX] != 1) continue;
    const int j = kIdx27.v[AX == 0 ? 0 : kE27[i][0] + 1][AX == 1 ? 0 : kE27[i][1] + 1][AX == 2 ? 0 : kE27[i][2] + 1];
    const double a = f[i], b = f[j];
    f[i] = m ? b : a;
    f[j] = m ? a : b;
  }
}

// gauge transfer of the node at byte offset boff to target t (structs.cuh:525-548)
template <class SRC>
__device__ __forceinline__ double transfer27(const SRC& s, uint32_t boff, const Tgt27& t, double sqTb) {
  double u0x, u0y, u0z, Pn;
  node_g4(s, boff, u0x, u0y, u0z, Pn);
  double gx[3], gy[3], gz[3];
  basis27(u0x, u0y, u0z, Pn, t, sqTb, gx, gy, gz);
  double f[27];
  node_f27(s, boff, f);
  return terms27(t.W, gx, gy, gz, f);
}

// transfer27 of the node's mirror image on the axes set in mx, my, mz (Cell::mirrX/Y/Z,
// structs.cuh:552-578): the axis velocity negated and every population exchanged with its mirror
// image (kIdx27 with that component negated), then the same term loop
template <class SRC>
__device__ double transfer27_mirrored(const SRC& s, uint32_t boff, const Tgt27& t, double sqTb, bool mx, bool my,
                                      bool mz) {
  double u0x, u0y, u0z, Pn;
  node_g4(s, boff, u0x, u0y, u0z, Pn);
  if (mx) u0x = -u0x;
  if (my) u0y = -u0y;
  if (mz) u0z = -u0z;
  double gx[3], gy[3], gz[3];
  basis27(u0x, u0y, u0z, Pn, t, sqTb, gx, gy, gz);
  double f[27];
  node_f27(s, boff, f);
  mirror27<0>(mx, f);
  mirror27<1>(my, f);
  mirror27<2>(mz, f);
  return terms27(t.W, gx, gy, gz, f);
}

// ---------------------------------------------------------------------------------------------
// Gauge transfer, D1Q5 (structs.cuh:352-395)

struct Tgt5 {
  double u1x, et, wk, fnew0;
  double e1sq, e2sq, E, etet;
  bool k0;  // inew == 0
};

__device__ __forceinline__ Tgt5 make_tgt5(int inew, double u1x, double T1) {
  Tgt5 t;
  t.u1x = u1x;
  const double s1 = sqrts_d(T1 / 1.0);
  const double e1_to = kA5[1] * s1, e2_to = kA5[3] * s1;
  t.et = kA5[inew] * s1;
  const double ef = kA5[inew];
  // (one division of the selected denominator: the target varies across the lanes of the line step)
  const double den = ef == 0            ? e1_to * e1_to * e2_to * e2_to
                     : fabs(ef) == kEc1 ? 2 * e1_to * e1_to * (e1_to * e1_to - e2_to * e2_to)
                                        : 2 * e2_to * e2_to * (e2_to * e2_to - e1_to * e1_to);
  const double wk = 1. / den;
  t.wk = wk;
  t.fnew0 = wk * 0.0;
  t.e1sq = e1_to * e1_to;
  t.e2sq = e2_to * e2_to;
  t.E = t.e1sq + t.e2sq;
  t.etet = t.et * t.et;
  t.k0 = inew == 0;
  return t;
}

// transfer of a node with axis velocity u0x, s0 = sqrts(T0/1.0) and populations f to target t
__device__ __forceinline__ double transfer5v(double u0x, double s0, const double (&f)[5], const Tgt5& t) {
  const double et = t.et;
  const double difu = t.u1x - u0x;
  double fadd[5];
#pragma unroll
  for (int iold = 0; iold < 5; iold++) {
    const double e = kA5[iold] * s0;
    double K0, K1, K2, K3;
    const double K4 = 1;
    K3 = -4 * e - et;
    if (t.k0) {
      K2 = 6 * e * e - t.E;
      K1 = 2 * e * (t.E - 2 * e * e);
      K0 = (t.e1sq - e * e) * (t.e2sq - e * e);
    } else {
      K2 = 6 * e * e + 3 * e * et - (t.E - t.etet);
      K1 = (2 * e + et) * (t.E - t.etet) - e * e * (4 * e + 3 * et);
      K0 = e * (e * e - t.E + t.etet) * (e + et);
    }
    double dm4 = u0x + e;
    dm4 = dm4 * dm4 * dm4 * dm4;
    dm4 *= 0;
    const double gx = K4 * difu * difu * difu * difu + K3 * difu * difu * difu + K2 * difu * difu + K1 * difu + K0 - dm4;
    fadd[iold] = t.wk * gx * f[iold];
  }
  // non-finite terms are dropped (structs.cuh:390); a finite sum has none (as in terms27)
  double fnew = t.fnew0;
#pragma unroll
  for (int iold = 0; iold < 5; iold++) fnew += fadd[iold];
  if (!finite_d(fnew)) {
    fnew = t.fnew0;
#pragma unroll
    for (int iold = 0; iold < 5; iold++)
      if (finite_d(fadd[iold])) fnew += fadd[iold];
  }
  return fnew;
}

// MIRX: the node's mirror image in x (Cell::mirrX, structs.cuh:552-559): u0x negated and the
// populations +e/-e exchanged
template <bool MIRX = false, class SRC>
__device__ __forceinline__ double transfer5(const SRC& s, uint32_t boff, const Tgt5& t, bool mx = false) {
  double u0x = node_m(s, 1, boff);
  double f[5];
#pragma unroll
  for (int i = 0; i < 5; i++) f[i] = node_f(s, i, boff);
  if (MIRX && mx) {
    u0x = -u0x;
    const double f1 = f[1], f3 = f[3];
    f[1] = f[2]; f[2] = f1;
    f[3] = f[4]; f[4] = f3;
  }
  return transfer5v(u0x, node_P(s, boff), f, t);  // node_P: sqrts(T0/1.0) = sqrt(|T0|)*sign(T0)
}

// ---------------------------------------------------------------------------------------------
// Lattice traits: the transfer to one target (interp_weno5, interp_lagr4), and for D1Q5 what the
// one-lane-per-cell kernel needs besides

template <int LAT>
struct Lat;

template <>
struct Lat<kD3Q27> {
  using Tgt = Tgt27;
  template <class SRC>
  __device__ static double xfer(const SRC& s, uint32_t boff, const Tgt& t, double sqTb) {
    return transfer27(s, boff, t, sqTb);
  }
  template <class SRC>
  __device__ static double xferm(const SRC& s, uint32_t boff, const Tgt& t, double sqTb, bool mx, bool my, bool mz) {
    return transfer27_mirrored(s, boff, t, sqTb, mx, my, mz);
  }
};

template <>
struct Lat<kD1Q5> {
  static constexpr int Q = 5;
  using Tgt = Tgt5;
  __device__ static double efc(int i, int d) { return d == 0 ? kA5[i] : 0.0; }
  __device__ static Tgt tgt(int i, const double* g) { return make_tgt5(i, g[0], g[3]); }
  template <class SRC>
  __device__ static double xfer(const SRC& s, uint32_t boff, const Tgt& t, double) {
    return transfer5(s, boff, t);
  }
  // D1Q5 velocities have no y or z component: a mirror in y or z only negates the unused uy, uz
  template <class SRC>
  __device__ static double xferm(const SRC& s, uint32_t boff, const Tgt& t, double, bool mx, bool, bool) {
    return transfer5<true>(s, boff, t, mx);
  }
};

// ---------------------------------------------------------------------------------------------
// Interpolators

// the two factors (s-p)/(i-p), p != i, p ascending, of the 3-node Lagrange basis (steps.cu:597)
__device__ __forceinline__ void lag3_factors(double s, double F[3][2]) {
  F[0][0] = (s - 1) / (0 - 1); F[0][1] = (s - 2) / (0 - 2);
  F[1][0] = (s - 0) / (1 - 0); F[1][1] = (s - 2) / (1 - 2);
  F[2][0] = (s - 0) / (2 - 0); F[2][1] = (s - 1) / (2 - 1);
}

// its factors of node i alone (i the same in every lane)
__device__ __forceinline__ void lag3_row(double s, int i, double (&f)[2]) {
  if (i == 0) {
    f[0] = (s - 1) / (0 - 1); f[1] = (s - 2) / (0 - 2);
  } else if (i == 1) {
    f[0] = (s - 0) / (1 - 0); f[1] = (s - 2) / (1 - 2);
  } else {
    f[0] = (s - 0) / (2 - 0); f[1] = (s - 1) / (2 - 1);
  }
}

__device__ __forceinline__ void lag4_factors(double s, double F[4][3]) {
#pragma unroll
  for (int i = 0; i < 4; i++) {
    int c = 0;
#pragma unroll
    for (int p = 0; p < 4; p++)
      if (p != i) F[i][c++] = (s - p) / (double)(i - p);
  }
}

// the WENO5 combination of the three sub-stencil sums (S0: left window, S2: right) with the
// smoothness samples ub at the five window positions, in the operation order of form VAR
template <int VAR>
__device__ __forceinline__ double weno5_combine_f64(double cdist, const double (&ub)[5], double S0, double S1,
                                                    double S2) {
  const double u1 = ub[0], u2 = ub[1], u3 = ub[2], u4 = ub[3], u5 = ub[4];
  if (VAR == 2) {
    // S0, S1, S2 of steps.cu:617-619 are this function's right, middle and left sums
    const double d0 = (cdist * cdist + 3 * cdist + 2) / 12.;
    const double d2 = (cdist * cdist - 3 * cdist + 2) / 12.;
    const double d1 = 1. - d0 - d2;
    const double beta0 = (10 * u3 * u3 - 31 * u3 * u4 + 25 * u4 * u4 + 11 * u3 * u5 - 19 * u4 * u5 + 4 * u5 * u5) / 3.0;
    const double beta1 = (4 * u2 * u2 - 13 * u2 * u3 + 13 * u3 * u3 + 5 * u2 * u4 - 13 * u3 * u4 + 4 * u4 * u4) / 3.0;
    const double beta2 = (4 * u1 * u1 - 19 * u1 * u2 + 25 * u2 * u2 + 11 * u1 * u3 - 31 * u2 * u3 + 10 * u3 * u3) / 3.0;
    double w0 = d0 / ((1e-6 + beta0) * (1e-6 + beta0));
    double w1 = d1 / ((1e-6 + beta1) * (1e-6 + beta1));
    double w2 = d2 / ((1e-6 + beta2) * (1e-6 + beta2));
    const double wsum = w0 + w1 + w2;
    w0 /= wsum;
    w1 /= wsum;
    w2 /= wsum;
    return w0 * S2 + w1 * S1 + w2 * S0;
  }
  const double d0 = (cdist * cdist - 3 * cdist + 2) / 12.;
  const double d2 = (cdist * cdist + 3 * cdist + 2) / 12.;
  const double d1 = 1. - d0 - d2;
  const double beta0 = (10 * u3 * u3 + (11 * u1 - 31 * u2) * u3 + 25 * u2 * u2 - 19 * u1 * u2 + 4 * u1 * u1) / 3.0;
  const double beta1 = (4 * u4 * u4 + (5 * u2 - 13 * u3) * u4 + 13 * u3 * u3 - 13 * u2 * u3 + 4 * u2 * u2) / 3.0;
  const double beta2 = (4 * u5 * u5 + (11 * u3 - 19 * u4) * u5 + 25 * u4 * u4 - 31 * u3 * u4 + 10 * u3 * u3) / 3.0;
  double w0 = d0 * 1, w1 = d1 * 1, w2 = d2 * 1;
  const double sc = 1e-6;
  w0 /= (sc + beta0) * (sc + beta0);
  w1 /= (sc + beta1) * (sc + beta1);
  w2 /= (sc + beta2) * (sc + beta2);
  const double wsum = w0 + w1 + w2;
  w0 /= wsum;
  w1 /= wsum;
  w2 /= wsum;
  return w0 * S0 + w1 * S1 + w2 * S2;
}

// WENO5 interpolation, three forms (VAR):
// 0: propagateWENO<3,5> (steps.cu:774-825) with LagrEval<3> (steps.cu:924-937), as written:
//    y/z sub-stencil nodes floor(y+0.5)+0..2 and smoothness samples on the row
//    (r mod Ny, r mod Nz), r = floor(x+0.5) (steps.cu:776-783).  This extrapolates downwind in
//    y and z and is unstable in 3D (grid-scale modes grow every step).
// 1: the corrected variant (not in the reference): y/z nodes floor(y+0.5)-1..+1 and smoothness
//    samples on the departure point's own row, which is the middle node of every slice, so
//    they reuse that slice's transfers.
// 2: the generic propagateWENO<5,M> (steps.cu:610-654) with propagate3 (steps.cu:909-923): the
//    nodes, samples and interpolant of form 0, with the sub-stencils numbered from the right
//    (lshift = 1), the indicators written expanded and each weight formed in one expression;
//    only the rounding differs from form 0.
template <int LAT, int VAR, class SRC>
__device__ double interp_weno5(const SRC& src, double cx, double cy, double cz, const typename Lat<LAT>::Tgt& t,
                               double sqTb) {
  constexpr bool CENTRED = VAR == 1;
  const Grid& g = src.g;
  const int r = floor_int(cx + 0.5);
  const int ry = floor_int(cy + 0.5) - (CENTRED ? 1 : 0), rz = floor_int(cz + 0.5) - (CENTRED ? 1 : 0);
  const double sy = cy - ry, sz = cz - rz;
  double Fy[3][2], Fz[3][2];
  lag3_factors(sy, Fy);
  lag3_factors(sz, Fz);
  // x parts of LagrPol<3> for sub-stencils k = 0,1,2 with left node r-2+k
  double px[3][3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    double Fx[3][2];
    lag3_factors(cx - (r - 2 + k), Fx);
#pragma unroll
    for (int ix = 0; ix < 3; ix++) px[k][ix] = 1 * Fx[ix][0] * Fx[ix][1];
  }
  int yy[3], zz[3];
#pragma unroll
  for (int a = 0; a < 3; a++) { yy[a] = wrapi(ry + a, g.ny); zz[a] = wrapi(rz + a, g.nz); }
  const bool line = (g.ny == 1) && (g.nz == 1);
  const int by = CENTRED ? yy[1] : wrapi(r, g.ny), bz = CENTRED ? zz[1] : wrapi(r, g.nz);
  double S0 = 0, S1 = 0, S2 = 0;
  double ub[5];
  for (int xs = 0; xs < 5; xs++) {
    const int x = wrapi(r - 2 + xs, g.nx);
    double T[9];
    if (line) {
      const double v = Lat<LAT>::xfer(src, (uint32_t)x * 8u, t, sqTb);
#pragma unroll
      for (int q = 0; q < 9; q++) T[q] = v;
      ub[xs] = v;  // smoothness row (r mod 1, r mod 1) = (0,0): same node
    } else {
#pragma unroll
      for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) {
          T[3 * a + b] = Lat<LAT>::xfer(src, node_off(g, x, yy[a], zz[b]), t, sqTb);
        }
      if (CENTRED) {
        ub[xs] = T[4];
      } else {
        ub[xs] = Lat<LAT>::xfer(src, node_off(g, x, by, bz), t, sqTb);
      }
    }
    // accumulate into every sub-stencil that contains this x slice, in (iy, iz) order
    if (xs <= 2) {
      const double p = xs == 0 ? px[0][0] : xs == 1 ? px[0][1] : px[0][2];
#pragma unroll
      for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) S0 += p * Fy[a][0] * Fy[a][1] * Fz[b][0] * Fz[b][1] * T[3 * a + b];
    }
    if (xs >= 1 && xs <= 3) {
      const double p = xs == 1 ? px[1][0] : xs == 2 ? px[1][1] : px[1][2];
#pragma unroll
      for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) S1 += p * Fy[a][0] * Fy[a][1] * Fz[b][0] * Fz[b][1] * T[3 * a + b];
    }
    if (xs >= 2) {
      const double p = xs == 2 ? px[2][0] : xs == 3 ? px[2][1] : px[2][2];
#pragma unroll
      for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) S2 += p * Fy[a][0] * Fy[a][1] * Fz[b][0] * Fz[b][1] * T[3 * a + b];
    }
  }
  return weno5_combine_f64<VAR>(cx - r, ub, S0, S1, S2);
}

// ---------------------------------------------------------------------------------------------
// D3Q27 targets in (ey, ez) groups: the three targets with ex = -1, 0, +1 share their departure
// point's y and z (v_y and v_z depend on ey, ez only), so their stencils share the y/z rows and
// differ in x only.  A node of the union of their windows is loaded once and transferred to each
// target whose window holds it, with exactly transfer27's operations for that target; the y and
// z basis values, which the three share, are evaluated once.  Each target's interpolation sums
// receive their terms in the order of the one-target code (slices in increasing x, rows (a, b)
// in order inside a slice), so every value is bitwise what interp_weno5 / interp_lagr4 give.

// The three targets of a group: the fields of Tgt27 they share (u1, T1 and the y, z target
// components) once, the x ones per target.  An axis' term is C*a for a moving target component and
// T1 for a resting one: with (Cy, Ty) = (C, 0) or (0, T1) it is Cy*a + Ty, the same bits for finite a
// (the terms of a non-finite one are dropped in either form).
struct Tgt27g3 {
  double u1x, u1y, u1z, T1, Cy, Ty, Cz, Tz;
  bool ky, kz;
  double W0, W1, Cx;  // W of ex = 0 and of ex = -1, +1; C of ex = +1 (its negative for ex = -1)
};

// one stencil node's data in registers
struct Node27 {
  double ux, uy, uz, P, f[27];
};

template <class SRC>
__device__ __forceinline__ void load_node27(const SRC& s, uint32_t boff, Node27& n) {
  node_g4(s, boff, n.ux, n.uy, n.uz, n.P);
  node_f27(s, boff, n.f);
}

// transfer27 of one node to the targets k with use[k] (T[k]; the others untouched).  MIR: of its
// mirror image on the axes set in mx, my, mz (transfer27_mirrored)
template <bool MIR = false>
__device__ __forceinline__ void transfer27_g3(Node27& n, const Tgt27g3& t, const bool (&use)[3], double sqTb,
                                              double (&T)[3], bool mx = false, bool my = false, bool mz = false) {
  double u0x = n.ux, u0y = n.uy, u0z = n.uz;
  if (MIR) {
    u0x = mx ? -u0x : u0x;
    u0y = my ? -u0y : u0y;
    u0z = mz ? -u0z : u0z;
  }
  // basis27u, split into the x part (per target) and the shared y and z parts
  const double Dx = (t.u1x - u0x) * sqTb;
  const double Dy = (t.u1y - u0y) * sqTb;
  const double Dz = (t.u1z - u0z) * sqTb;
  const double E[3] = {-n.P, 0.0 * n.P, n.P};
  double ax[3], gy[3], gz[3];
#pragma unroll
  for (int j = 0; j < 3; j++) {
    ax[j] = Dx - E[j];
    const double ay = Dy - E[j], az = Dz - E[j];
    gy[j] = ay * ay - (t.Cy * ay + t.Ty);
    gz[j] = az * az - (t.Cz * az + t.Tz);
  }
  if (MIR) {
    if (__any(mx)) mirror27<0>(mx, n.f);
    if (__any(my)) mirror27<1>(my, n.f);
    if (__any(mz)) mirror27<2>(mz, n.f);
  }
#pragma unroll
  for (int k = 0; k < 3; k++) {
    if (!use[k]) continue;
    double gx[3];
#pragma unroll
    for (int j = 0; j < 3; j++) gx[j] = ax[j] * ax[j] - (k == 0 ? -t.Cx * ax[j] : k == 2 ? t.Cx * ax[j] : t.T1);
    T[k] = terms27(k == 1 ? t.W0 : t.W1, gx, gy, gz, n.f);
  }
}

// x part of LagrPol<3> of window node ix of sub-stencil q for a departure point at cx whose
// window starts at r - 2 (the value interp_weno5 keeps in px[q][ix])
__device__ __forceinline__ double lag3x(double cx, int r, int q, int ix) {
  double Fx[3][2];
  lag3_factors(cx - (r - 2 + q), Fx);
  return ix == 0 ? 1 * Fx[0][0] * Fx[0][1] : ix == 1 ? 1 * Fx[1][0] * Fx[1][1] : 1 * Fx[2][0] * Fx[2][1];
}

__device__ __forceinline__ Tgt27 tgt27_of(const Tgt27g3& t, int k) {
  Tgt27 tk;
  tk.u1x = t.u1x; tk.u1y = t.u1y; tk.u1z = t.u1z; tk.T1 = t.T1;
  tk.W = k == 1 ? t.W0 : t.W1; tk.Cx = k == 0 ? -t.Cx : t.Cx; tk.Cy = t.Cy; tk.Cz = t.Cz;
  tk.kx = k != 1; tk.ky = t.ky; tk.kz = t.kz;
  return tk;
}

// The walk over the stencil nodes of a group: slices d = dlo .. dhi relative to the cell's x, NR rows in
// y from ry and in z from rz.  Calls slice(d) at the start of a slice, row(a) at the start of a row,
// and node(n, d, a, b) with the node's data.  Row offsets are 32-bit (node_off, mod 2^32).
//
// Tried, and no faster (128^3 vortex, this walk 56 ms per step): the loads of a node issued before the
// weighting of the one before (57 ms: the other wave of the SIMD covers the wait already); each
// different node of a wave's cells loaded once, 16 bytes per lane, and handed out through LDS (112
// ms when the walk took 65: the loaders' addresses go to scratch, and a scratch access occupies the
// L1 for as long as a 16-byte load); held to three waves per SIMD (91 ms, scratch in the walk itself).
template <int NR, bool MIR, class SRC, class FS, class FR, class FN>
__device__ __forceinline__ void walk27(const SRC& src, int x, int ry, int rz, int dlo, int dhi, FS&& slice, FR&& row,
                                       FN&& node) {
  const Grid& g = src.g;
  bool rv;
  uint32_t yo[NR], zo[NR];
#pragma unroll
  for (int q = 0; q < NR; q++) {
    yo[q] = (uint32_t)(MIR ? mirror_wrap(ry + q, g.ny, (g.mirror & 2) != 0, rv) : wrapi(ry + q, g.ny)) * (uint32_t)g.nx;
    zo[q] = (uint32_t)(MIR ? mirror_wrap(rz + q, g.nz, (g.mirror & 4) != 0, rv) : wrapi(rz + q, g.nz)) *
            ((uint32_t)g.nx * (uint32_t)g.ny);
  }
#pragma unroll 1
  for (int d = dlo; d <= dhi; d++) {
    slice(d);
    const uint32_t xw = (uint32_t)(MIR ? mirror_wrap(x + d, g.nx, (g.mirror & 1) != 0, rv) : wrapi(x + d, g.nx));
#pragma unroll 1
    for (int a = 0; a < NR; a++) {
      row(a);
      const uint32_t xy = xw + (a == 0 ? yo[0] : a == 1 ? yo[1] : a == 2 ? yo[2] : yo[NR - 1]);
#pragma unroll 1
      for (int b = 0; b < NR; b++) {
        Node27 n;
        load_node27(src, (xy + (b == 0 ? zo[0] : b == 1 ? zo[1] : b == 2 ? zo[2] : zo[NR - 1])) * 8u, n);
        node(n, d, a, b);
      }
    }
  }
}

// The WENO5 step's cell slot of a lane: cells in pairs, a group's two lanes side by side (lane 18 p +
// 2 group + cell of pair p), the seventh cell's groups in lanes 54 .. 62
__device__ __forceinline__ int weno_slot27(int lane) { return lane < 54 ? lane / 18 * 2 + (lane & 1) : lane < 63 ? 6 : 7; }

// interp_weno5<kD3Q27, VAR> for the three targets of a group (cx[k] of target ex = k - 1; cy, cz
// shared), on a grid that is not a line, without mirrors.  Window positions are taken relative
// to the cell's own x, so lanes of a wave whose flow is alike visit the same positions.  Taken
// only for s = sqrt(T1/TLat) <= 1.5 (f64_group): the windows of ex = -1 and +1 are 2s apart, so
// the union spans at most 9 slices.
//
// Registers are what this is short of: the departure points and windows in x are formed again at
// every slice and the y and z Lagrange factors at every row and node instead of being kept.
template <int VAR, class SRC>
__device__ __forceinline__ void interp_weno5_g3(const SRC& src, int x, double s, double cy, double cz,
                                                const Tgt27g3& t, double sqTb, double (&fn)[3]) {
  constexpr bool CENTRED = VAR == 1;
  const Grid& g = src.g;
  const int ry = floor_int(cy + 0.5) - (CENTRED ? 1 : 0), rz = floor_int(cz + 0.5) - (CENTRED ? 1 : 0);
  const double sy = cy - ry, sz = cz - rz;
  auto target_x = [&](int k, double& cx, int& r) {  // departure point and window middle of ex = k - 1
    cx = (double)x - (s * (double)(k - 1) + t.u1x);
    r = floor_int(cx + 0.5);
  };
  int wlo = 0, whi = 0;  // lowest and highest window start relative to x
#pragma unroll
  for (int k = 0; k < 3; k++) {
    double cx;
    int r;
    target_x(k, cx, r);
    const int w = (r - 2) - x;
    wlo = k == 0 ? w : min(wlo, w);
    whi = k == 0 ? w : max(whi, w);
  }
  const int dlo = wlo;
  // (at most dlo + 8 for s <= 1.5; the bound keeps the loop finite whatever the caller passes)
  const int dhi = min(whi + 4, dlo + 8);
  // The smoothness samples of the three targets wait in LDS (one wave per block), which keeps the
  // sub-stencil sums and a node's populations in registers; so do the slice's x weights (the same
  // for a cell's lanes), which a row takes up with its own y factors: the products' left prefixes,
  // shared by the row's nodes.
  __shared__ double s_ub[3][5][64];
  __shared__ double s_pw[3][3][8];
  const int lane = threadIdx.x & 63, slot = weno_slot27(lane);
  double S[3][3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
#pragma unroll
    for (int q = 0; q < 3; q++) S[k][q] = 0;
#pragma unroll
    for (int j = 0; j < 5; j++) s_ub[k][j][lane] = 0;
  }
  const bool finite_w = finite_d(cy) && finite_d(cz);
  int xs[3] = {0, 0, 0};
  bool use[3] = {false, false, false};
  double pf[3][3];  // per target, the left prefix of the row's weights in sub-stencils 0, 1, 2
  auto slice = [&](int d) {
    wave_lds_order();
#pragma unroll
    for (int k = 0; k < 3; k++) {
      double cx;
      int r;
      target_x(k, cx, r);
      const int j = d - ((r - 2) - x);
      xs[k] = j;
      use[k] = j >= 0 && j <= 4;
#pragma unroll
      for (int q = 0; q < 3; q++) s_pw[k][q][slot] = (j - q >= 0 && j - q <= 2) ? lag3x(cx, r, q, j - q) : 0.0;
    }
    wave_lds_order();
  };
  auto row = [&](int a) {
    double fy[2];
    lag3_row(sy, a, fy);
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
      for (int q = 0; q < 3; q++) pf[k][q] = s_pw[k][q][slot] * fy[0] * fy[1];
  };
  auto node = [&](Node27& n, int d, int a, int b) {
    double T[3] = {0, 0, 0};
    transfer27_g3(n, t, use, sqTb, T);
    double fz[2];
    lag3_row(sz, b, fz);
#pragma unroll
    for (int k = 0; k < 3; k++) {
      if (__ballot(use[k]) == 0) continue;
      // a sub-stencil that does not hold the slice has weight zero, and adding a zero changes no sum
      // that started from +0; only with a value or weight that is not finite it is left out
      if (__ballot(!(finite_w && finite_d(T[k]))) == 0) {
#pragma unroll
        for (int q = 0; q < 3; q++) S[k][q] += pf[k][q] * fz[0] * fz[1] * T[k];
      } else {
        const int j = xs[k];
#pragma unroll
        for (int q = 0; q < 3; q++)
          if (use[k] && j - q >= 0 && j - q <= 2) S[k][q] += pf[k][q] * fz[0] * fz[1] * T[k];
      }
      if (CENTRED && a == 1 && b == 1 && use[k]) s_ub[k][xs[k]][lane] = T[k];
    }
    if (!CENTRED && a == 2 && b == 2) {
      // smoothness samples on the row (r mod Ny, r mod Nz) of each target
#pragma unroll
      for (int k = 0; k < 3; k++) {
        if (!use[k]) continue;
        double cx;
        int r;
        target_x(k, cx, r);
        s_ub[k][xs[k]][lane] =
            transfer27(src, node_off(g, wrapi(x + d, g.nx), wrapi(r, g.ny), wrapi(r, g.nz)), tgt27_of(t, k), sqTb);
      }
    }
  };
  walk27<3, false>(src, x, ry, rz, dlo, dhi, slice, row, node);
#pragma unroll
  for (int k = 0; k < 3; k++) {
    double ub[5], cx;
    int r;
    target_x(k, cx, r);
#pragma unroll
    for (int j = 0; j < 5; j++) ub[j] = s_ub[k][j][lane];
    fn[k] = weno5_combine_f64<VAR>(cx - r, ub, S[k][0], S[k][1], S[k][2]);
  }
}

// x part of LagrPol<4> of node ix for a departure point at cx whose window starts at lx (the
// value interp_lagr4 forms as p)
__device__ __forceinline__ double lag4x(double cx, int lx, int ix) {
  double Fx[4][3];
  lag4_factors(cx - lx, Fx);
  return ix == 0   ? 1 * Fx[0][0] * Fx[0][1] * Fx[0][2]
         : ix == 1 ? 1 * Fx[1][0] * Fx[1][1] * Fx[1][2]
         : ix == 2 ? 1 * Fx[2][0] * Fx[2][1] * Fx[2][2]
                   : 1 * Fx[3][0] * Fx[3][1] * Fx[3][2];
}

// interp_lagr4<kD3Q27, MIR> for the three targets of a group, as interp_weno5_g3 does for
// WENO5: each node of the union of their windows (at most 8 slices for s <= 1.5) loaded once,
// each target's sum in its own node order.
template <bool MIR, class SRC>
__device__ __forceinline__ void interp_lagr4_g3(const SRC& src, int x, double s, double cy, double cz,
                                                const Tgt27g3& t, double sqTb, double (&fn)[3]) {
  const Grid& g = src.g;
  const int ly = floor_int(cy) - 4 / 2 + 1;
  const int lz = floor_int(cz) - 4 / 2 + 1;
  // the y and z Lagrange factors wait in LDS
  __shared__ double s_fy[12][64], s_fz[12][64];
  const int lane = threadIdx.x & 63;
  {
    double F[4][3];
    lag4_factors(cy - ly, F);
#pragma unroll
    for (int q = 0; q < 12; q++) s_fy[q][lane] = F[q / 3][q % 3];
    lag4_factors(cz - lz, F);
#pragma unroll
    for (int q = 0; q < 12; q++) s_fz[q][lane] = F[q / 3][q % 3];
  }
  auto target_x = [&](int k, double& cx, int& lx) {  // departure point and window start of ex = k - 1
    cx = (double)x - (s * (double)(k - 1) + t.u1x);
    lx = floor_int(cx) - 4 / 2 + 1;
  };
  int wlo = 0, whi = 0;  // lowest and highest window start relative to x
#pragma unroll
  for (int k = 0; k < 3; k++) {
    double cx;
    int lx;
    target_x(k, cx, lx);
    wlo = k == 0 ? lx - x : min(wlo, lx - x);
    whi = k == 0 ? lx - x : max(whi, lx - x);
    fn[k] = 0;
  }
  const int dlo = wlo;
  // (at most dlo + 7 for s <= 1.5; the bound keeps the loop finite whatever the caller passes)
  const int dhi = min(whi + 3, dlo + 7);
  bool use[3] = {false, false, false};
  double p[3] = {0, 0, 0}, pf[3] = {0, 0, 0};
  auto slice = [&](int d) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      double cx;
      int lx;
      target_x(k, cx, lx);
      const int ix = d - (lx - x);
      use[k] = ix >= 0 && ix <= 3;
      p[k] = use[k] ? lag4x(cx, lx, ix) : 0.0;
    }
  };
  auto row = [&](int a) {
    const double fy0 = s_fy[3 * a][lane], fy1 = s_fy[3 * a + 1][lane], fy2 = s_fy[3 * a + 2][lane];
#pragma unroll
    for (int k = 0; k < 3; k++) pf[k] = p[k] * fy0 * fy1 * fy2;
  };
  auto node = [&](Node27& n, int d, int a, int b) {
    bool mx = false, my = false, mz = false;
    if (MIR) {
      mirror_wrap(x + d, g.nx, (g.mirror & 1) != 0, mx);
      mirror_wrap(ly + a, g.ny, (g.mirror & 2) != 0, my);
      mirror_wrap(lz + b, g.nz, (g.mirror & 4) != 0, mz);
    }
    double T[3] = {0, 0, 0};
    transfer27_g3<MIR>(n, t, use, sqTb, T, mx, my, mz);
    const double fz0 = s_fz[3 * b][lane], fz1 = s_fz[3 * b + 1][lane], fz2 = s_fz[3 * b + 2][lane];
#pragma unroll
    for (int k = 0; k < 3; k++)
      if (use[k]) fn[k] += pf[k] * fz0 * fz1 * fz2 * T[k];
  };
  walk27<4, MIR>(src, x, ly, lz, dlo, dhi, slice, row, node);
}

// propagate<4> (steps.cu:986-1036): tricubic Lagrange on floor(x)-1 .. floor(x)+2.
// MIR: mirror boundaries on the axes of g.mirror (steps.cu:1004-1022): nodes beyond a mirrored
// face are the mirror images of the cells inside.
template <int LAT, bool MIR, class SRC>
__device__ double interp_lagr4(const SRC& src, double cx, double cy, double cz, const typename Lat<LAT>::Tgt& t,
                               double sqTb) {
  const Grid& g = src.g;
  const int lx = floor_int(cx) - 4 / 2 + 1;
  const int ly = floor_int(cy) - 4 / 2 + 1;
  const int lz = floor_int(cz) - 4 / 2 + 1;
  double Fx[4][3], Fy[4][3], Fz[4][3];
  lag4_factors(cx - lx, Fx);
  lag4_factors(cy - ly, Fy);
  lag4_factors(cz - lz, Fz);
  int yy[4], zz[4];
  bool ry[4] = {false, false, false, false}, rz[4] = {false, false, false, false};
#pragma unroll
  for (int a = 0; a < 4; a++) {
    if (MIR) {
      yy[a] = mirror_wrap(ly + a, g.ny, (g.mirror & 2) != 0, ry[a]);
      zz[a] = mirror_wrap(lz + a, g.nz, (g.mirror & 4) != 0, rz[a]);
    } else {
      yy[a] = wrapi(ly + a, g.ny);
      zz[a] = wrapi(lz + a, g.nz);
    }
  }
  const bool line = (g.ny == 1) && (g.nz == 1);
  double fpr = 0;
  for (int ix = 0; ix < 4; ix++) {
    bool rx = false;
    const int x = MIR ? mirror_wrap(lx + ix, g.nx, (g.mirror & 1) != 0, rx) : wrapi(lx + ix, g.nx);
    const double p = 1 * Fx[ix][0] * Fx[ix][1] * Fx[ix][2];
    double v1 = 0;
    if (line && !MIR) v1 = Lat<LAT>::xfer(src, (uint32_t)x * 8u, t, sqTb);
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
      for (int b = 0; b < 4; b++) {
        double T;
        if (MIR) {
          const uint32_t off = node_off(g, x, yy[a], zz[b]);
          T = (rx || ry[a] || rz[b]) ? Lat<LAT>::xferm(src, off, t, sqTb, rx, ry[a], rz[b])
                                     : Lat<LAT>::xfer(src, off, t, sqTb);
        } else if (line) {
          T = v1;
        } else {
          T = Lat<LAT>::xfer(src, node_off(g, x, yy[a], zz[b]), t, sqTb);
        }
        fpr += p * Fy[a][0] * Fy[a][1] * Fy[a][2] * Fz[b][0] * Fz[b][1] * Fz[b][2] * T;
      }
  }
  return fpr;
}

// ---------------------------------------------------------------------------------------------
// One lane per cell: LBMpull (steps.cu:356-365, 421-512, 557-564, 582)

// Iteration state of one cell: gauge c0, density rho0, count niter.  The iterate's
// populations live in fout.
struct F64Iter {
  double c0[4];
  double rho0;
  int niter;
};

// One fixed-point iteration (LBMpull, steps.cu:421-512) of one cell: true when it has converged.
template <int LAT, int INTERP, class SRC>
__device__ __forceinline__ bool f64_once(const SRC& src, const NodeSrc& gsrc, double* __restrict__ fout, int64_t cell,
                                         int x, int y, int z, bool zero, F64Iter& st, const StepArgs& a) {
  constexpr int Q = Lat<LAT>::Q;
  const int64_t P = a.g.plane;
  double* c0 = st.c0;
  {
    st.niter++;
    const int niter = st.niter;
    const double uT[4] = {c0[0], c0[1], c0[2], c0[3]};
    const double s = sqrt(uT[3] / a.tlat);
    double rho = 0, m0 = 0, m1 = 0, m2 = 0, m3 = 0;
    bool conv = true;
    for (int i = 0; i < Q; i++) {
      const double vx = s * Lat<LAT>::efc(i, 0) + uT[0];
      const double vy = s * Lat<LAT>::efc(i, 1) + uT[1];
      const double vz = s * Lat<LAT>::efc(i, 2) + uT[2];
      const typename Lat<LAT>::Tgt t = Lat<LAT>::tgt(i, uT);
      const double cx = (double)x - vx, cy = (double)y - vy, cz = (double)z - vz;
      // INTERP 3: Lagrange-4 with mirror boundaries; 4: the generic WENO5
      const double fn = INTERP == 1   ? interp_lagr4<LAT, false>(src, cx, cy, cz, t, a.sqrt_tbase)
                        : INTERP == 3 ? interp_lagr4<LAT, true>(src, cx, cy, cz, t, a.sqrt_tbase)
                        : INTERP == 2 ? interp_weno5<LAT, 1>(src, cx, cy, cz, t, a.sqrt_tbase)
                        : INTERP == 4 ? interp_weno5<LAT, 2>(src, cx, cy, cz, t, a.sqrt_tbase)
                                      : interp_weno5<LAT, 0>(src, cx, cy, cz, t, a.sqrt_tbase);
      rho += fn;
      m0 += fn * vx;
      m1 += fn * vy;
      m2 += fn * vz;
      m3 += fn * (vx * vx + vy * vy + vz * vz);
      const int64_t o = f64_fidx(LAT, i, cell, P);
      const double fo = niter > 1 ? fout[o] : (zero ? a.w[i] * 1.0 : gsrc.f[o]);
      if (fabs(fn - fo) >= a.tol_abs + a.tol_rel * fabs(fn)) conv = false;
      fout[o] = fn;
    }
    // Cell::calcMoments (structs.cuh:329-330)
    if (rho != 0) { m0 /= rho; m1 /= rho; m2 /= rho; m3 /= rho; }
    m3 = (m3 - m0 * m0 - m1 * m1 - m2 * m2) * a.inv_dim;
    if (m3 < 0) m3 = c0[3];  // steps.cu:475-478
    const double mn[4] = {m0, m1, m2, m3};
#pragma unroll
    for (int k = 0; k < 4; k++)
      if (fabs(mn[k] - c0[k]) >= a.tol_abs + a.tol_rel * fabs(mn[k])) conv = false;
    st.rho0 = rho;
    c0[0] = m0; c0[1] = m1; c0[2] = m2; c0[3] = m3;
    return conv;
  }
}

// Fixed-point iterations from state st until convergence (true) or until the count reaches
// stop_at (false).
template <int LAT, int INTERP, class SRC>
__device__ bool f64_iterate(const SRC& src, const NodeSrc& gsrc, double* __restrict__ fout, int64_t cell, int x, int y,
                            int z, bool zero, F64Iter& st, int stop_at, const StepArgs& a) {
  while (st.niter < stop_at)
    if (f64_once<LAT, INTERP>(src, gsrc, fout, cell, x, y, z, zero, st, a)) return true;
  return false;
}

// starting state of a cell: its previous gauge; an all-zero cell is reset to set_base(1,
// (0,0,0,TLat)) (steps.cu:360-363)
__device__ __forceinline__ bool f64_start(const NodeSrc& gsrc, int64_t cell, const StepArgs& a, F64Iter& st) {
  const int64_t P = a.g.plane;
  st.rho0 = gsrc.m[cell];
  st.c0[0] = gsrc.m[P + cell]; st.c0[1] = gsrc.m[2 * P + cell]; st.c0[2] = gsrc.m[3 * P + cell];
  st.c0[3] = gsrc.m[4 * P + cell];
  const bool zero = st.rho0 == 0 && st.c0[0] == 0 && st.c0[1] == 0 && st.c0[2] == 0 && st.c0[3] == 0;
  if (zero) { st.rho0 = 1; st.c0[3] = a.tlat; }
  st.niter = 0;
  return zero;
}

// BGK towards rho*w_i in the converged gauge (steps.cu:557-564) and the cell's outputs
__device__ __forceinline__ void f64_finish(double* __restrict__ fout, double* __restrict__ mout,
                                           int* __restrict__ niter_out, int64_t cell, const F64Iter& st,
                                           const StepArgs& a) {
  const int64_t P = a.g.plane;
  for (int i = 0; i < 5; i++) {
    const int64_t o = f64_fidx(kD1Q5, i, cell, P);
    double f = fout[o];
    const double feq = st.rho0 * a.w[i];
    f += a.dtau * (feq - f);
    fout[o] = f;
  }
  mout[cell] = st.rho0;
  mout[P + cell] = st.c0[0];
  mout[2 * P + cell] = st.c0[1];
  mout[3 * P + cell] = st.c0[2];
  mout[4 * P + cell] = st.c0[3];
  niter_out[cell] = st.niter;
}

// D1Q5 with one lane per cell (grids that are no line, and long Lagrange-4 lines).  First pass: every cell
// iterates up to a.pass1_iters times; cells still unconverged are appended to the pending list (one
// atomic per wave) and finished by a second pass over that list (k_step_f64_rest).  A wave runs as long
// as its slowest cell, and a thin layer of cells on shocks and contact discontinuities needs several
// times the mean count.  Each cell's arithmetic and operation order are those of a single pass.
template <int LAT, int INTERP>
__global__ __launch_bounds__(64) void k_step_f64(const NodeSrc gsrc, double* __restrict__ fout,
                                                 double* __restrict__ mout, int* __restrict__ niter_out, Pending pend,
                                                 const StepArgs a) {
  const NodeSrc& src = gsrc;
  const Grid& g = a.g;
  int x, y, z;
  bool active = tile_cell(g, xcd_block(blockIdx.x, gridDim.x), threadIdx.x, x, y, z);
  const int64_t cell = active ? cell_index(g, x, y, z) : 0;
  // a switched-off cell is not stepped: its output record and iteration count keep what they
  // held (LBMpull, steps.cu:359)
  if (active && a.cell_set && a.cell_set[cell] == 0) active = false;
  bool pending = false;
  F64Iter st;
  if (active) {
    const bool zero = f64_start(gsrc, cell, a, st);
    const int stop = a.pass1_iters < a.max_iter ? a.pass1_iters : a.max_iter;
    const bool conv = f64_iterate<LAT, INTERP>(src, gsrc, fout, cell, x, y, z, zero, st, stop, a);
    pending = !conv && st.niter < a.max_iter;
    if (!pending) f64_finish(fout, mout, niter_out, cell, st, a);
  }
  bool any;
  const int64_t e = pending_slot(pend, pending, any);
  if (pending) {
    pend.cell[e] = (int)cell;
    for (int k = 0; k < 4; k++) pend.g[k * pend.cap + e] = st.c0[k];
    pend.res[e] = st.rho0;
    pend.meta[e] = st.niter;
  }
}

// ---------------------------------------------------------------------------------------------
// D3Q27 step: nine lanes per cell, lane = (ey, ez) group of three targets, seven cells per wave.
//
// One lane per cell (all 27 targets one after the other) left two thirds of the lanes idle behind
// the slowest cell of their tile (the mean count is 1.3 to 5 iterations, the slowest of 64 cells
// several times that), gave a small grid a fraction of the chip (8316 cells: 130 waves for 1024
// SIMDs, 10 ms per step), sent the populations through global memory between iterations and needed a
// second pass for the slow cells.  Here a cell's groups run side by side, a slot whose cell has
// converged takes the next one, the iterate stays in LDS and the previous one in registers; the
// lanes of a cell mostly want the same nodes, so a load touches a few cache lines.  Each value is the
// same sequence of operations (bit for bit).
// Per step, before and after: 33x18x14 vortex 10.0 -> 0.85 ms; 128^3 vortex 86 -> 56 ms; 256x128x128
// shock-bubble 289 -> 181 ms; Lagrange-4 128^3 255 -> 124 ms, 100x52x46 with walls 109 -> 15.8 ms.
// Bound by FP64 issue where the flow is smooth: 128^3 vortex VALU busy 75 % (texture-address unit 53 %), 332
// instructions per node where no contraction and every rounding of the reference leave about 290.  On the 384^3
// shock-bubble 59 and 62 %, with 53 lanes in use: neither is full, and two waves per SIMD do not hide the loads.
// The kernel spills 113 registers (364 bytes per lane; WENO5 as written 128 and 424, Lagrange-4 69 and 280),
// all of them outside the loop over the nodes: 13 GB written per step at 128^3 against 0.56 GB of output, 192 GB at 384^3.
template <int INTERP, class SRC>
__device__ __forceinline__ void f64_group(const SRC& src, int x, int y, int z, int ey, int ez, const double (&uT)[4],
                                          double s, const StepArgs& a, double (&fn)[3]) {
  constexpr int VAR = INTERP == 2 ? 1 : INTERP == 4 ? 2 : 0;
  const double cy = (double)y - (s * (double)ey + uT[1]), cz = (double)z - (s * (double)ez + uT[2]);
  // the three together off a line, for gauges whose targets' windows lie close (s <= 1.5, not
  // NaN); hotter or non-finite ones, one target at a time
  if ((a.g.ny > 1 || a.g.nz > 1) && s <= 1.5) {
    // (W and C of ex = -1 and +1 are the same up to C's sign)
    const Tgt27 t0 = make_tgt27e(0, ey, ez, uT[0], uT[1], uT[2], uT[3]);
    const Tgt27 t1 = make_tgt27e(1, ey, ez, uT[0], uT[1], uT[2], uT[3]);
    Tgt27g3 t;
    t.u1x = uT[0]; t.u1y = uT[1]; t.u1z = uT[2]; t.T1 = uT[3];
    t.W0 = t0.W; t.W1 = t1.W; t.Cx = t1.Cx;
    t.Cy = t0.ky ? t0.Cy : 0.0; t.Ty = t0.ky ? 0.0 : uT[3];
    t.Cz = t0.kz ? t0.Cz : 0.0; t.Tz = t0.kz ? 0.0 : uT[3];
    t.ky = t0.ky; t.kz = t0.kz;
    if constexpr (INTERP == 1 || INTERP == 3) interp_lagr4_g3<INTERP == 3>(src, x, s, cy, cz, t, a.sqrt_tbase, fn);
    else interp_weno5_g3<VAR>(src, x, s, cy, cz, t, a.sqrt_tbase, fn);
  } else {
#pragma unroll 1
    for (int k = 0; k < 3; k++) {
      const Tgt27 tk = make_tgt27e(k - 1, ey, ez, uT[0], uT[1], uT[2], uT[3]);
      const double c = (double)x - (s * (double)(k - 1) + uT[0]);
      double v;
      if constexpr (INTERP == 1 || INTERP == 3) v = interp_lagr4<kD3Q27, INTERP == 3>(src, c, cy, cz, tk, a.sqrt_tbase);
      else v = interp_weno5<kD3Q27, VAR>(src, c, cy, cz, tk, a.sqrt_tbase);
      fn[0] = k == 0 ? v : fn[0];
      fn[1] = k == 1 ? v : fn[1];
      fn[2] = k == 2 ? v : fn[2];
    }
  }
}

// A WENO5 cell late in its iterations goes to k_step_f64_27_wide where its wave has no cell left to start and
// no more than this many slots (of 7) with such cells; see launch_step_f64.
constexpr int kWideSlots64 = 5;

template <int INTERP, bool BUF>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_step_f64_27(
    const NodeSrc gsrc, double* __restrict__ fout, double* __restrict__ mout, int* __restrict__ niter_out,
    int* __restrict__ slow, const StepArgs a, int cells, int wide_after, int few) {
  constexpr bool WENO = INTERP != 1 && INTERP != 3;
  using Src = typename std::conditional<BUF, NodeBuf, NodeSrc>::type;
  Src src;
  if constexpr (BUF) src = make_nodebuf(gsrc);
  else src = gsrc;
  __shared__ __align__(16) double s_fn[8][28];  // the iterate's populations, per cell
  __shared__ double s_w[28];
  const Grid& g = a.g;
  const int64_t P = g.plane;
  const int lane = threadIdx.x;
  // Lanes of a cell (lane 63 has none).  A 16-byte load takes four neighbouring lanes at a time, so
  // these should want one cache line.  Lagrange-4: a group's seven cells side by side, as its groups'
  // rows mostly differ (64^3 Taylor-Green 14.0 -> 12.1 ms, 100x52x46 with walls 16.9 -> 16.2 ms per step).
  // WENO5, whose groups' rows coincide below half a cell of thermal speed: cells in pairs (weno_slot27;
  // against a cell's nine groups side by side: 128^3 shock-bubble 86.0 -> 82.7 ms, vortex 56.4 ms both).
  const int slot = WENO ? weno_slot27(lane) : lane < 63 ? lane % 7 : 7;
  const int gi = WENO ? (lane < 54 ? lane % 18 / 2 : lane < 63 ? lane - 54 : 0) : lane < 63 ? lane / 7 : 0;
  const int head = WENO ? (slot < 6 ? 18 * (slot / 2) + (slot & 1) : 54) : slot;  // the slot's lane of group 0
  const int GS = WENO ? (slot < 6 ? 2 : 1) : 7;                                   // and from group to group
  const int ey = gi / 3 - 1, ez = gi % 3 - 1;
  constexpr uint64_t kHeads = WENO ? 0x400030000c0003ull : 0x7full;  // group 0 of every slot
  const uint64_t groups = WENO ? (slot < 6 ? 0x15555ull : 0x1ffull) : 0x0102040810204081ull;  // from head on
  if (lane < 28) s_w[lane] = lane < 27 ? a.w[lane] : 0.0;
  const int64_t q0 = xcd_block(blockIdx.x, gridDim.x) * cells;
  const int64_t total = g.ntiles * 64 - q0 < cells ? g.ntiles * 64 - q0 : cells;  // cell slots of the wave
  int64_t next = 0;  // first unstarted slot (the same in every lane)
  bool active = false;
  int64_t cell = 0;
  int x = 0, y = 0, z = 0, niter = 0;
  double c0[4] = {0, 0, 0, 1}, fo[3] = {0, 0, 0};
  int idx[3];
#pragma unroll
  for (int k = 0; k < 3; k++) idx[k] = kIdx27.v[k][ey + 1][ez + 1];
  while (true) {
    const uint64_t want = __ballot(!active) & kHeads;
    if (!active && slot < 7) {
      const int64_t q = next + __popcll(want & ((1ull << head) - 1ull));
      if (q < total && tile_cell(g, (q0 + q) / 64, (int)((q0 + q) % 64), x, y, z)) {
        cell = cell_index(g, x, y, z);
        F64Iter st;
        const bool zero = f64_start(gsrc, cell, a, st);
#pragma unroll
        for (int k = 0; k < 4; k++) c0[k] = st.c0[k];
#pragma unroll
        for (int k = 0; k < 3; k++) fo[k] = zero ? a.w[idx[k]] * 1.0 : gsrc.f[f64_fidx(kD3Q27, idx[k], cell, P)];
        niter = 0;
        active = true;
      }
    }
    next += __popcll(want);
    if (__ballot(active) == 0 && next >= total) break;
    const double uT[4] = {c0[0], c0[1], c0[2], c0[3]};
    const double s = sqrt(uT[3] / a.tlat);
    bool conv = true;
    if (active) {
      double fn[3] = {0, 0, 0};
      f64_group<INTERP>(src, x, y, z, ey, ez, uT, s, a, fn);
#pragma unroll
      for (int k = 0; k < 3; k++) {
        if (fabs(fn[k] - fo[k]) >= a.tol_abs + a.tol_rel * fabs(fn[k])) conv = false;
        fo[k] = fn[k];
        s_fn[slot][idx[k]] = fn[k];
      }
    }
    wave_lds_order();
    // Cell::calcMoments: lane gi of the cell sums moment gi % 5 over the populations in order.  Its
    // factor of population (ex, ey, ez) is wx[ex] + wy[ey] + wz[ez] with the two tables it does not
    // need at zero (adding zero changes neither a factor nor a sum that starts from +0).
    const int mq = gi < 5 ? gi : gi - 5;
    double wx[3], wy[3], wz[3];
#pragma unroll
    for (int e = 0; e < 3; e++) {
      const double vx = s * (double)(e - 1) + uT[0], vy = s * (double)(e - 1) + uT[1], vz = s * (double)(e - 1) + uT[2];
      wx[e] = mq == 0 ? 1.0 : mq == 1 ? vx : mq == 4 ? vx * vx : 0.0;
      wy[e] = mq == 2 ? vy : mq == 4 ? vy * vy : 0.0;
      wz[e] = mq == 3 ? vz : mq == 4 ? vz * vz : 0.0;
    }
    double acc = 0;
#pragma unroll
    for (int i = 0; i < 27; i++) acc += s_fn[slot][i] * (wx[kE27[i][0] + 1] + wy[kE27[i][1] + 1] + wz[kE27[i][2] + 1]);
    const double rho = __shfl(acc, head, 64);
    if (rho != 0) acc /= rho;
    const double m0 = __shfl(acc, head + GS, 64), m1 = __shfl(acc, head + 2 * GS, 64),
                 m2 = __shfl(acc, head + 3 * GS, 64);
    double m3 = __shfl(acc, head + 4 * GS, 64);
    m3 = (m3 - m0 * m0 - m1 * m1 - m2 * m2) * a.inv_dim;
    if (m3 < 0) m3 = uT[3];  // steps.cu:475-478
    const double mn[4] = {m0, m1, m2, m3};
#pragma unroll
    for (int k = 0; k < 4; k++)
      if (fabs(mn[k] - uT[k]) >= a.tol_abs + a.tol_rel * fabs(mn[k])) conv = false;
    const uint64_t bad = (__ballot(!conv) >> head) & groups;
    if (active) {
      niter++;
#pragma unroll
      for (int k = 0; k < 4; k++) c0[k] = mn[k];
      const bool done = bad == 0 || niter >= a.max_iter;
      int e = -1;  // the cell's place in the list of k_step_f64_27_wide
      if (WENO && !done && niter >= wide_after) {
        const bool idle = next >= total && __popcll(__ballot(true) & kHeads) <= kWideSlots64;  // (late cells only)
        if (gi == 0) e = slow_place(slow, idle, few);
        e = __shfl(e, head, 64);
      }
      if (done || e >= 0) {
        // BGK towards rho*w_i (steps.cu:557-564), two populations per lane and store; a cell left to
        // k_step_f64_27_wide stores its iterate as it is
        active = false;
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const int p = gi + 9 * h;
          if (p < 14) {
            double f[2];
#pragma unroll
            for (int k = 0; k < 2; k++) {
              f[k] = s_fn[slot][2 * p + k];
              const double feq = rho * s_w[2 * p + k];
              const double fb = f[k] + a.dtau * (feq - f[k]);
              f[k] = !WENO || done ? fb : f[k];
            }
            if (p < 13) reinterpret_cast<double2*>(fout)[p * P + cell] = make_double2(f[0], f[1]);
            else fout[(p * P + cell) * 2] = f[0];
          }
        }
        if (gi < 5) mout[gi * P + cell] = gi == 0 ? rho : gi == 1 ? m0 : gi == 2 ? m1 : gi == 3 ? m2 : m3;
        if (gi == 5) niter_out[cell] = niter;
        if (WENO && !done && gi == 6) slow[kSlowList + e] = (int)cell;
      }
    }
    wave_lds_order();
  }
}

// The WENO5 cells that k_step_f64_27 left unconverged: one workgroup per cell.
//
// A few cells on shocks and contacts go on to the cap of 100 iterations, and nine lanes take 100 us for
// such an iteration (63 chained steps of one node).  Here the (target, window position, node) transfers
// of an iteration, 1215 or 1350 of them, are spread over the threads and laid down in LDS; the 81
// sub-stencil sums run over them in the order of interp_weno5, one thread each, and one wave forms the
// 27 values and the moments.  Bound by the chain of these parts (128 to 512 threads take the same time
// within 4 %).  Shock-bubble, ms per step before and after: 32^3 10.4 -> 4.1, 64^3 20.5 -> 16.9, 100^3
// 54.4 -> 52.1; 33x18x14 vortex (at most 10 iterations) 0.81 -> 0.65.
constexpr int kWideThreads64 = 256;
template <int VAR>
__global__ __launch_bounds__(kWideThreads64) void k_step_f64_27_wide(const NodeSrc src, double* __restrict__ fout,
                                                                    double* __restrict__ mout,
                                                                    int* __restrict__ niter_out,
                                                                    const int* __restrict__ slow, const StepArgs a) {
  constexpr bool CENTRED = VAR == 1;
  __shared__ double s_T[27 * 5][10];  // target, window position: the nodes (a, b) and (as written) the sample
  __shared__ double s_S[27][3];       // sub-stencil sums
  __shared__ double s_fn[27];         // the iterate, [9 (ey+1) + 3 (ez+1) + ex+1]
  __shared__ double s_g[4];
  __shared__ int s_conv;
  const Grid& g = a.g;
  const int64_t P = g.plane;
  const int tid = threadIdx.x;
  const int count = *slow;
  for (int64_t e0 = blockIdx.x; e0 < count; e0 += gridDim.x) {
    const int64_t cell = slow[kSlowList + e0];
    const int x = (int)(cell % g.nx), y = (int)((cell / g.nx) % g.ny), z = (int)(cell / ((int64_t)g.nx * g.ny));
    double uT[4], rho = 0, fo = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) uT[k] = mout[(k + 1) * P + cell];
    const int ti = tid < 27 ? tid : 0;  // target of a thread of the tail
    const int te = ti / 9 - 1, tz = (ti / 3) % 3 - 1, tx = ti % 3 - 1;
    const int idx = kIdx27.v[tx + 1][te + 1][tz + 1];
    if (tid < 27) fo = fout[f64_fidx(kD3Q27, idx, cell, P)];
    int niter = niter_out[cell];
    bool conv = false;
    while (!conv && niter < a.max_iter) {
      niter++;
      const double s = sqrt(uT[3] / a.tlat);
      // transfers of the nodes (a, b) of every target's window position j, and its sample
      constexpr int NI = CENTRED ? 9 : 10;
#pragma unroll 1
      for (int it = tid; it < 27 * 5 * NI; it += kWideThreads64) {
        const int tj = it / NI, q = it - NI * tj, tg = tj / 5, j = tj - 5 * tg;
        const int ey = tg / 9 - 1, ez = (tg / 3) % 3 - 1, ex = tg % 3 - 1;
        const Tgt27 t = make_tgt27e(ex, ey, ez, uT[0], uT[1], uT[2], uT[3]);
        const double cx = (double)x - (s * (double)ex + uT[0]);
        const double cy = (double)y - (s * (double)ey + uT[1]), cz = (double)z - (s * (double)ez + uT[2]);
        const int r = floor_int(cx + 0.5);
        const int ry = floor_int(cy + 0.5) - (CENTRED ? 1 : 0), rz = floor_int(cz + 0.5) - (CENTRED ? 1 : 0);
        const int yn = q < 9 ? ry + q / 3 : r, zn = q < 9 ? rz + q % 3 : r;
        s_T[tj][q] = transfer27(src, node_off(g, wrapi(r - 2 + j, g.nx), wrapi(yn, g.ny), wrapi(zn, g.nz)), t,
                                a.sqrt_tbase);
      }
      __syncthreads();
      // sums of a target's sub-stencil, in the order of interp_weno5
      if (tid < 81) {
        const int tg = tid / 3, q = tid - 3 * tg;
        const int ey = tg / 9 - 1, ez = (tg / 3) % 3 - 1, ex = tg % 3 - 1;
        const double cx = (double)x - (s * (double)ex + uT[0]);
        const double cy = (double)y - (s * (double)ey + uT[1]), cz = (double)z - (s * (double)ez + uT[2]);
        const int r = floor_int(cx + 0.5);
        const int ry = floor_int(cy + 0.5) - (CENTRED ? 1 : 0), rz = floor_int(cz + 0.5) - (CENTRED ? 1 : 0);
        double Fx[3][2], Fy[3][2], Fz[3][2];
        lag3_factors(cx - (r - 2 + q), Fx);
        lag3_factors(cy - ry, Fy);
        lag3_factors(cz - rz, Fz);
        double S = 0;
#pragma unroll
        for (int ix = 0; ix < 3; ix++) {
          const double p = 1 * Fx[ix][0] * Fx[ix][1];
#pragma unroll
          for (int aa = 0; aa < 3; aa++)
#pragma unroll
            for (int b = 0; b < 3; b++)
              S += p * Fy[aa][0] * Fy[aa][1] * Fz[b][0] * Fz[b][1] * s_T[5 * tg + q + ix][3 * aa + b];
        }
        s_S[tg][q] = S;
      }
      __syncthreads();
      if (tid < 64) {
        double fn = 0;
        if (tid < 27) {
          const double cx = (double)x - (s * (double)tx + uT[0]);
          const int r = floor_int(cx + 0.5);
          double ub[5];
#pragma unroll
          for (int j = 0; j < 5; j++) ub[j] = s_T[5 * tid + j][CENTRED ? 4 : 9];
          fn = weno5_combine_f64<VAR>(cx - r, ub, s_S[tid][0], s_S[tid][1], s_S[tid][2]);
          s_fn[idx] = fn;
        }
        bool same = true;
        if (tid < 27 && fabs(fn - fo) >= a.tol_abs + a.tol_rel * fabs(fn)) same = false;
        fo = fn;
        wave_lds_order();
        // Cell::calcMoments: lane q < 5 sums moment q over the populations in order, as in k_step_f64_27
        const int mq = tid < 5 ? tid : 0;
        double wx[3], wy[3], wz[3];
#pragma unroll
        for (int e = 0; e < 3; e++) {
          const double vx = s * (double)(e - 1) + uT[0], vy = s * (double)(e - 1) + uT[1],
                       vz = s * (double)(e - 1) + uT[2];
          wx[e] = mq == 0 ? 1.0 : mq == 1 ? vx : mq == 4 ? vx * vx : 0.0;
          wy[e] = mq == 2 ? vy : mq == 4 ? vy * vy : 0.0;
          wz[e] = mq == 3 ? vz : mq == 4 ? vz * vz : 0.0;
        }
        double acc = 0;
#pragma unroll
        for (int i = 0; i < 27; i++) acc += s_fn[i] * (wx[kE27[i][0] + 1] + wy[kE27[i][1] + 1] + wz[kE27[i][2] + 1]);
        rho = __shfl(acc, 0, 64);
        if (rho != 0) acc /= rho;
        const double m0 = __shfl(acc, 1, 64), m1 = __shfl(acc, 2, 64), m2 = __shfl(acc, 3, 64);
        double m3 = __shfl(acc, 4, 64);
        m3 = (m3 - m0 * m0 - m1 * m1 - m2 * m2) * a.inv_dim;
        if (m3 < 0) m3 = uT[3];  // steps.cu:475-478
        const double mn[4] = {m0, m1, m2, m3};
#pragma unroll
        for (int k = 0; k < 4; k++)
          if (fabs(mn[k] - uT[k]) >= a.tol_abs + a.tol_rel * fabs(mn[k])) same = false;
        const bool all = __ballot(!same) == 0;
        if (tid == 0) {
#pragma unroll
          for (int k = 0; k < 4; k++) s_g[k] = mn[k];
          s_conv = all;
        }
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 4; k++) uT[k] = s_g[k];
      conv = s_conv != 0;
    }
    // BGK towards rho*w_i (steps.cu:557-564) and the cell's outputs
    if (tid < 27) {
      const double feq = rho * a.w[idx];
      fout[f64_fidx(kD3Q27, idx, cell, P)] = fo + a.dtau * (feq - fo);
    }
    if (tid < 5) mout[tid * P + cell] = tid == 0 ? rho : tid == 1 ? uT[0] : tid == 2 ? uT[1] : tid == 3 ? uT[2] : uT[3];
    if (tid == 5) niter_out[cell] = niter;
    __syncthreads();
  }
}

// Second pass: a fixed grid of waves walks the pending list, every cell resumes its iteration
template <int LAT, int INTERP>
__global__ __launch_bounds__(64) void k_step_f64_rest(const NodeSrc gsrc, double* __restrict__ fout,
                                                      double* __restrict__ mout, int* __restrict__ niter_out,
                                                      Pending pend, const StepArgs a) {
  const NodeSrc& src = gsrc;
  const Grid& g = a.g;
  const int count = *pend.count;
  for (int64_t e = (int64_t)blockIdx.x * 64 + threadIdx.x; e - threadIdx.x < count; e += (int64_t)gridDim.x * 64) {
    if (e >= count) continue;
    const int64_t cell = pend.cell[e];
    const int x = (int)(cell % g.nx);
    const int y = (int)((cell / g.nx) % g.ny);
    const int z = (int)(cell / ((int64_t)g.nx * g.ny));
    F64Iter st;
    for (int k = 0; k < 4; k++) st.c0[k] = pend.g[k * pend.cap + e];
    st.rho0 = pend.res[e];
    st.niter = pend.meta[e];
    // the zero-cell start only matters for the first iteration, which the first pass ran
    f64_iterate<LAT, INTERP>(src, gsrc, fout, cell, x, y, z, false, st, a.max_iter, a);
    f64_finish(fout, mout, niter_out, cell, st, a);
  }
}

// ---------------------------------------------------------------------------------------------
// D3Q125: one block per cell, lane = target population (PonDstepD3Q125, steps.cu:151-250)
//
// A transfer term is W*(gx*gy*gz)*f, four FP64 operations that no two targets share: 125 x 125 x 27 of
// them per cell and iteration are what this step is made of.  Everything else is kept off the lanes:
//   * the basis values of a node depend on (axis, target class, source class) alone: 75 per node, 2025
//     per cell, each formed once by one lane and read by the others from LDS (every lane used to form
//     15 per node);
//   * a node's populations are the same for the whole block: scalar loads put them in SGPRs, which the
//     multiplications read directly (from LDS, 125 broadcast reads per node and wave took as long as
//     the arithmetic).  A node beyond a mirror wall (MIR) is read permuted, through LDS;
//   * lane q of a wave sums moment q % 5 over the populations in order (every lane used to sum all five).
// 40^3 turbulence 20.1 -> 12.4 ms per step, 64^3 82 -> 51 ms; the VALU is busy 93 % of the time, 80 % of
// its instructions being the terms.
template <bool MIR>
__global__ __launch_bounds__(128) void k_step_q125_f64(const double* __restrict__ fin, const double* __restrict__ min,
                                                       double* __restrict__ fout, double* __restrict__ mout,
                                                       int* __restrict__ niter_out, const StepArgs a) {
  constexpr int Q = 125;
  typedef const __attribute__((address_space(4))) double ConstD;
  __shared__ double sf[MIR ? Q : 1];      // MIR: populations of a mirrored node
  __shared__ double sg[27][4];            // the nodes' gauges, the temperature as sqrts(T/1.0)
  __shared__ double sb[27][76];           // basis values g[axis][target class][source class]
  __shared__ double snew[Q];              // cnew.f
  __shared__ int sflag[2];
  const Grid& g = a.g;
  const int64_t P = g.plane;
  const int64_t cell = xcd_block(blockIdx.x, gridDim.x);
  const int k = threadIdx.x;
  const bool lane_ok = k < Q;
  const int x = (int)(cell % g.nx);
  const int y = (int)((cell / g.nx) % g.ny);
  const int z = (int)(cell / ((int64_t)g.nx * g.ny));
  // mirror boundaries (steps.cu:163-190): a node beyond a mirrored face is the mirror image of
  // the cell inside, population k read from the mirrored velocity, the axis velocity negated
  auto node_cell = [&](int n, bool& rx, bool& ry, bool& rz) {
    const int px = mirror_wrap(x - 1 + n / 9, g.nx, MIR && (g.mirror & 1) != 0, rx);
    const int py = mirror_wrap(y - 1 + (n / 3) % 3, g.ny, MIR && (g.mirror & 2) != 0, ry);
    const int pz = mirror_wrap(z - 1 + n % 3, g.nz, MIR && (g.mirror & 4) != 0, rz);
    return cell_index(g, px, py, pz);
  };
  if (k < 108) {
    const int n = k >> 2, d = k & 3;
    bool rx, ry, rz;
    const double v = min[(int64_t)(d + 1) * P + node_cell(n, rx, ry, rz)];
    sg[n][d] = d == 3 ? sqrts_d(v / 1.0) : (d == 0 && rx) || (d == 1 && ry) || (d == 2 && rz) ? -v : v;
  }
  double rho0 = min[cell], c0[4] = {min[P + cell], min[2 * P + cell], min[3 * P + cell], min[4 * P + cell]};
  const bool zero = rho0 == 0 && c0[0] == 0 && c0[1] == 0 && c0[2] == 0 && c0[3] == 0;
  if (zero) { rho0 = 1; c0[3] = a.tlat; }
  double f0 = lane_ok ? (zero ? a.w[k] * 1.0 : fin[f64_fidx(kD3Q125, k, cell, P)]) : 0.0;
  __syncthreads();

  // per-axis class of target k: index into {0,+ec1,-ec1,+ec2,-ec2}
  const int kk = lane_ok ? k : 0;
  const int X[3] = {kk / 25, (kk / 5) % 5, kk % 5};
  int niter = 0;
  while (niter < a.max_iter) {
    niter++;
    const double uT[4] = {c0[0], c0[1], c0[2], c0[3]};
    const double s = sqrt(uT[3] / a.tlat);
    // target constants (structs.cuh:397-416)
    const double S1 = sqrts_d(uT[3] / 1.0);
    const double e1_to = kEc1 * S1, e2_to = kEc2 * S1;
    // basis values of every node: entry (d, X, j) is the product of the four factors b - c over the
    // target nodes c other than X's, in the cyclic order (X+1..X+4)%5 of structs.cuh:432-434, with
    // b - c as b + {-0.0, -e1_to, +e1_to, -e2_to, +e2_to}[c] (b + (-0.0) == b exactly)
    for (int i = k; i < 27 * 75; i += 128) {
      const int n = i / 75, r = i - 75 * n, d = r / 25, Xi = (r / 5) % 5, j = r % 5;
      const double e = j == 0 ? 0.0 : j == 1 ? kEc1 : j == 2 ? -kEc1 : j == 3 ? kEc2 : -kEc2;
      const double u = d == 0 ? uT[0] : d == 1 ? uT[1] : uT[2];
      const double b = (sg[n][d] - u) + e * sg[n][3];
      double f[4];
#pragma unroll
      for (int mm = 1; mm <= 4; mm++) {
        const int c = (Xi + mm) % 5;
        f[mm - 1] = b + (c == 0 ? -0.0 : c == 1 ? -e1_to : c == 2 ? e1_to : c == 3 ? -e2_to : e2_to);
      }
      sb[n][r] = f[0] * f[1] * f[2] * f[3];
    }
    double wv[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
      const double en = kA5[X[d]];
      const double den = en == 0           ? e1_to * e1_to * e2_to * e2_to
                         : fabs(en) == kEc1 ? 2 * e1_to * e1_to * (e1_to * e1_to - e2_to * e2_to)
                                            : 2 * e2_to * e2_to * (e2_to * e2_to - e1_to * e1_to);
      wv[d] = 1. / den;
    }
    const double W = wv[0] * wv[1] * wv[2];
    const double vk[3] = {s * kA5[X[0]] + uT[0], s * kA5[X[1]] + uT[1], s * kA5[X[2]] + uT[2]};
    const double sh[3] = {((double)x - vk[0]) - (double)(x - 1), ((double)y - vk[1]) - (double)(y - 1),
                          ((double)z - vk[2]) - (double)(z - 1)};
    __syncthreads();
    double fpr = 0;
#pragma unroll 1
    for (int n = 0; n < 27; n++) {
      bool rx, ry, rz;
      const int64_t c = node_cell(n, rx, ry, rz);
      ConstD* rec = (ConstD*)(uintptr_t)(fin + c * kF64Q125Doubles);
      const double *bx = &sb[n][5 * X[0]], *by = &sb[n][25 + 5 * X[1]], *bz = &sb[n][50 + 5 * X[2]];
      double gy[5], gz[5];
#pragma unroll
      for (int j = 0; j < 5; j++) { gy[j] = by[j]; gz[j] = bz[j]; }
      auto terms = [&](auto f) {
        double fnew = 0;
#pragma unroll
        for (int jx = 0; jx < 5; jx++) {
          const double gx = bx[jx];
#pragma unroll
          for (int jy = 0; jy < 5; jy++) {
            const double gxy = gx * gy[jy];
#pragma unroll
            for (int jz = 0; jz < 5; jz++) fnew += W * (gxy * gz[jz]) * f[25 * jx + 5 * jy + jz];
          }
        }
        if (!finite_d(fnew)) {
          // a non-finite term: the loop again with such terms dropped (as in terms27)
          fnew = 0;
#pragma unroll 1
          for (int i = 0; i < Q; i++) {
            const double gxy = bx[i / 25] * by[(i / 5) % 5];
            const double fadd = W * (gxy * bz[i % 5]) * f[i];
            if (finite_d(fadd)) fnew += fadd;
          }
        }
        return fnew;
      };
      double fnew;
      if (MIR && (rx || ry || rz)) {  // (the same in the whole block)
        const int kl = 25 * (rx ? kMir5[X[0]] : X[0]) + 5 * (ry ? kMir5[X[1]] : X[1]) + (rz ? kMir5[X[2]] : X[2]);
        __syncthreads();
        if (lane_ok) sf[MIR ? k : 0] = fin[c * kF64Q125Doubles + kl];
        __syncthreads();
        fnew = terms((const double*)sf);
      } else {
        fnew = terms(rec);
      }
      double Fx[2], Fy[2], Fz[2];
      lag3_row(sh[0], n / 9, Fx);
      lag3_row(sh[1], (n / 3) % 3, Fy);
      lag3_row(sh[2], n % 3, Fz);
      fpr += 1 * Fx[0] * Fx[1] * Fy[0] * Fy[1] * Fz[0] * Fz[1] * fnew;
    }
    if (lane_ok) snew[k] = fpr;
    __syncthreads();
    // Cell::calcMoments on the shared cnew in population order, one moment per lane: the factor of
    // population (ix, iy, iz) is wx[ix] + wy[iy] + wz[iz], the tables a lane does not need at zero
    // (as in k_step_f64_27)
    const int mq = (k & 63) % 5;
    double wx[5], wy[5], wz[5];
#pragma unroll
    for (int e = 0; e < 5; e++) {
      const double vx = s * kA5[e] + uT[0], vy = s * kA5[e] + uT[1], vz = s * kA5[e] + uT[2];
      wx[e] = mq == 0 ? 1.0 : mq == 1 ? vx : mq == 4 ? vx * vx : 0.0;
      wy[e] = mq == 2 ? vy : mq == 4 ? vy * vy : 0.0;
      wz[e] = mq == 3 ? vz : mq == 4 ? vz * vz : 0.0;
    }
    double acc = 0;
#pragma unroll
    for (int i = 0; i < Q; i++) acc += snew[i] * (wx[i / 25] + wy[(i / 5) % 5] + wz[i % 5]);
    const double rho = __shfl(acc, 0, 64);
    if (rho != 0) acc /= rho;
    const double m0 = __shfl(acc, 1, 64), m1 = __shfl(acc, 2, 64), m2 = __shfl(acc, 3, 64);
    double m3 = __shfl(acc, 4, 64);
    m3 = (m3 - m0 * m0 - m1 * m1 - m2 * m2) * a.inv_dim;
    if (m3 < 0) m3 = c0[3];
    const double mn[4] = {m0, m1, m2, m3};
    bool conv = true;
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (fabs(mn[q] - c0[q]) >= a.tol_abs + a.tol_rel * fabs(mn[q])) conv = false;
    if (lane_ok && fabs(fpr - f0) >= a.tol_abs + a.tol_rel * fabs(fpr)) conv = false;
    const bool wave_conv = __all(conv);
    if ((threadIdx.x & 63) == 0) sflag[threadIdx.x >> 6] = wave_conv ? 1 : 0;
    __syncthreads();
    const bool all_conv = sflag[0] && sflag[1];
    rho0 = rho;
    c0[0] = m0; c0[1] = m1; c0[2] = m2; c0[3] = m3;
    f0 = fpr;
    __syncthreads();  // sflag, snew and sb are rewritten next iteration
    if (all_conv) break;
  }
  if (lane_ok) {
    const double feq = rho0 * a.w[k];
    f0 += a.dtau * (feq - f0);
    fout[f64_fidx(kD3Q125, k, cell, P)] = f0;
  }
  if (k == 0) {
    mout[cell] = rho0;
    mout[P + cell] = c0[0];
    mout[2 * P + cell] = c0[1];
    mout[3 * P + cell] = c0[2];
    mout[4 * P + cell] = c0[3];
    niter_out[cell] = niter;
  }
}

// ---------------------------------------------------------------------------------------------
// D1Q5 lines (Ny = Nz = 1), short ones: 32 lanes per cell, one lane per (target population,
// stencil node).
//
// A short line's step is one cell's serial chain: a few cells on a shock or contact run to the
// cap of 100 gauge iterations, and with one lane per cell an iteration is ~6000 dependent FP64
// instructions (36 us), so a step took 3.6 ms whatever the length.  Here the 25 (20 for
// Lagrange-4) transfers of an iteration run in 25 lanes at once, the three WENO sub-stencils and
// their weights in three of a target's lanes, and values cross lanes by shuffles; a node's
// populations stay in registers until the lane's node changes.  Every value is the same sequence
// of operations as f64_once gives (bit for bit).  sqrt(|T|)*sign(T) of a node is formed here, so
// the step needs no node-preparation pass and no second pass: it is one launch.  The Sod tube at
// 2000 cells: 3.5 -> 0.155 ms per step (1.5 us per iteration of the slowest cell, ~1000
// instructions of a wave that runs alone on its SIMD: the chain, not the chip, bounds it).
//
// The y/z factors of the tensor weights: off the line's axis every stencil node is the same cell,
// and for uy = uz = 0 the departure point lies on it, so exactly one (a, b) term of the nine
// (sixteen) has weight 1 and the others weight zero.  Adding a zero changes no sum that starts
// from +0, so those terms are left out where the slice terms are finite (0 * inf is not zero).
// Above this length the Lagrange-4 line goes back to one lane per cell (below).
constexpr int64_t kLineCellsLagr4 = 1 << 16;

template <int INTERP>
__global__ __launch_bounds__(64) void k_step_line(const double* __restrict__ fin, const double* __restrict__ min,
                                                  double* __restrict__ fout, double* __restrict__ mout,
                                                  int* __restrict__ niter_out, const StepArgs a) {
  constexpr bool WENO = INTERP == 0 || INTERP == 4;
  constexpr int NN = WENO ? 5 : 4;  // stencil nodes along x
  constexpr int VAR = INTERP == 4 ? 2 : 0;
  const Grid& g = a.g;
  const int64_t P = g.plane;
  const int lane = threadIdx.x, j = lane & 31;
  // lanes past the last (target, node) pair repeat the last target's (they store nothing)
  const int t = j / NN < 4 ? j / NN : 4, nd = j % NN;
  const int base = (lane & 32) + t * NN;  // first lane of the target
  const int64_t cell0 = (int64_t)blockIdx.x * 2 + (lane >> 5);
  const int64_t cell = cell0 < g.n ? cell0 : g.n - 1;
  const int x = (int)cell;
  // a switched-off cell keeps its record (LBMpull, steps.cu:359)
  bool active = cell0 < g.n && !(a.cell_set && a.cell_set[cell] == 0);
  double c0[4] = {min[P + cell], min[2 * P + cell], min[3 * P + cell], min[4 * P + cell]};
  double rho0 = min[cell];
  const bool zero = rho0 == 0 && c0[0] == 0 && c0[1] == 0 && c0[2] == 0 && c0[3] == 0;
  if (zero) { rho0 = 1; c0[3] = a.tlat; }  // steps.cu:360-363
  double fo = zero ? a.w[t] * 1.0 : fin[t * P + cell];
  const double ef = kA5[t];
  int niter = 0;
  int xc = -1;      // node held in (u0x, s0, f): its wrapped coordinate ...
  bool mc = false;  // ... and whether it is held as a mirror image
  double u0x = 0, s0 = 0, f[5] = {0, 0, 0, 0, 0};
  while (__ballot(active) != 0) {
    const double s = sqrt(c0[3] / a.tlat);
    const Tgt5 tg = make_tgt5(t, c0[0], c0[3]);
    const double cx = (double)x - (s * ef + c0[0]);
    const int r = WENO ? floor_int(cx + 0.5) - 2 : floor_int(cx) - 4 / 2 + 1;  // first node
    bool mx = false;
    const int xn = INTERP == 3 ? mirror_wrap(r + nd, g.nx, (g.mirror & 1) != 0, mx) : wrapi(r + nd, g.nx);
    if (xn != xc || mx != mc) {
      xc = xn;
      mc = mx;
      u0x = min[P + xn];
      s0 = sqrts_d(min[4 * P + xn]);
      double v[5];
#pragma unroll
      for (int i = 0; i < 5; i++) v[i] = fin[i * P + xn];
#pragma unroll
      for (int i = 0; i < 5; i++) f[i] = INTERP == 3 && mx ? v[kMir5[i]] : v[i];
      if (INTERP == 3 && mx) u0x = -u0x;
    }
    const double V = transfer5v(u0x, s0, f, tg);
    const double cy = 0.0 - (s * 0.0 + c0[1]), cz = 0.0 - (s * 0.0 + c0[2]);
    const bool on_line = c0[1] == 0 && c0[2] == 0;
    double fn;
    if constexpr (WENO) {
      // lane q = 0, 1, 2 of the target: sub-stencil q (nodes q .. q+2), its sum and weight
      const int q = nd < 2 ? nd : 2;
      const double U[3] = {__shfl(V, base + q, 64), __shfl(V, base + q + 1, 64), __shfl(V, base + q + 2, 64)};
      double Fx[3][2];
      lag3_factors(cx - (r + q), Fx);
      double p[3], S = 0;
      bool plain = on_line;
#pragma unroll
      for (int i = 0; i < 3; i++) {
        p[i] = 1 * Fx[i][0] * Fx[i][1];
        const double v = p[i] * U[i];
        plain = plain && finite_d(v);
        S += v;
      }
      if (!plain) {
        double Fy[3][2], Fz[3][2];
        lag3_factors(cy - floor_int(cy + 0.5), Fy);
        lag3_factors(cz - floor_int(cz + 0.5), Fz);
        S = 0;
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
          for (int b = 0; b < 3; b++)
#pragma unroll
            for (int c = 0; c < 3; c++) S += p[i] * Fy[b][0] * Fy[b][1] * Fz[c][0] * Fz[c][1] * U[i];
      }
      // weno5_combine_f64's weight of this sub-stencil: its three indicators are one expression
      // with other coefficients
      const double cd = cx - (r + 2);
      const double dl = (cd * cd - 3 * cd + 2) / 12., dr = (cd * cd + 3 * cd + 2) / 12.;
      const double dm = VAR == 2 ? 1. - dr - dl : 1. - dl - dr;
      const double dq = q == 0 ? dl : q == 1 ? dm : dr;
      double beta;
      if (VAR == 2) {
        const double kx = q == 2 ? 10 : 4, ky = q == 2 ? 31 : q == 1 ? 13 : 19, kz = q == 1 ? 13 : 25,
                     kw = q == 1 ? 5 : 11, ku = q == 2 ? 19 : q == 1 ? 13 : 31, kv = q == 0 ? 10 : 4;
        beta = (kx * U[0] * U[0] - ky * U[0] * U[1] + kz * U[1] * U[1] + kw * U[0] * U[2] - ku * U[1] * U[2] +
                kv * U[2] * U[2]) / 3.0;
      } else {
        const double kx = q == 0 ? 10 : 4, ky = q == 1 ? 5 : 11, kz = q == 0 ? 31 : q == 1 ? 13 : 19,
                     kw = q == 1 ? 13 : 25, ku = q == 0 ? 19 : q == 1 ? 13 : 31, kv = q == 2 ? 10 : 4;
        beta = (kx * U[2] * U[2] + (ky * U[0] - kz * U[1]) * U[2] + kw * U[1] * U[1] - ku * U[0] * U[1] +
                kv * U[0] * U[0]) / 3.0;
      }
      const double w = dq / ((1e-6 + beta) * (1e-6 + beta));
      const double w0 = __shfl(w, base, 64), w1 = __shfl(w, base + 1, 64), w2 = __shfl(w, base + 2, 64);
      const double wsum = VAR == 2 ? w2 + w1 + w0 : w0 + w1 + w2;
      const double ws = w / wsum * S;
      const double t0 = __shfl(ws, base, 64), t1 = __shfl(ws, base + 1, 64), t2 = __shfl(ws, base + 2, 64);
      fn = VAR == 2 ? t2 + t1 + t0 : t0 + t1 + t2;
    } else {
      double Fx[4][3];
      lag4_factors(cx - r, Fx);
      double p[4], U[4];
      fn = 0;
      bool plain = on_line;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        U[i] = __shfl(V, base + i, 64);
        p[i] = 1 * Fx[i][0] * Fx[i][1] * Fx[i][2];
        const double v = p[i] * U[i];
        plain = plain && finite_d(v);
        fn += v;
      }
      if (!plain) {
        double Fy[4][3], Fz[4][3];
        lag4_factors(cy - (floor_int(cy) - 4 / 2 + 1), Fy);
        lag4_factors(cz - (floor_int(cz) - 4 / 2 + 1), Fz);
        fn = 0;
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
          for (int b = 0; b < 4; b++)
#pragma unroll
            for (int c = 0; c < 4; c++)
              fn += p[i] * Fy[b][0] * Fy[b][1] * Fy[b][2] * Fz[c][0] * Fz[c][1] * Fz[c][2] * U[i];
      }
    }
    // Cell::calcMoments in population order, in every lane
    double rho = 0, m0 = 0, m1 = 0, m2 = 0, m3 = 0;
    const double vy = s * 0.0 + c0[1], vz = s * 0.0 + c0[2];
#pragma unroll
    for (int i = 0; i < 5; i++) {
      const double fi = __shfl(fn, (lane & 32) + i * NN, 64);
      const double vx = s * kA5[i] + c0[0];
      rho += fi;
      m0 += fi * vx;
      m1 += fi * vy;
      m2 += fi * vz;
      m3 += fi * (vx * vx + vy * vy + vz * vz);
    }
    if (rho != 0) { m0 /= rho; m1 /= rho; m2 /= rho; m3 /= rho; }
    m3 = (m3 - m0 * m0 - m1 * m1 - m2 * m2) * a.inv_dim;
    if (m3 < 0) m3 = c0[3];
    const double mn[4] = {m0, m1, m2, m3};
    bool conv = !(fabs(fn - fo) >= a.tol_abs + a.tol_rel * fabs(fn));
#pragma unroll
    for (int k = 0; k < 4; k++)
      if (fabs(mn[k] - c0[k]) >= a.tol_abs + a.tol_rel * fabs(mn[k])) conv = false;
    const uint64_t bad = __ballot(!conv);
    if (active) {
      niter++;
      rho0 = rho;
      c0[0] = m0; c0[1] = m1; c0[2] = m2; c0[3] = m3;
      fo = fn;
      if ((uint32_t)(bad >> (lane & 32)) == 0 || niter >= a.max_iter) {
        // BGK towards rho*w_i (steps.cu:557-564) and the cell's outputs
        active = false;
        if (nd == 0 && j < 5 * NN) {
          const double feq = rho0 * a.w[t];
          double v = fo;
          v += a.dtau * (feq - v);
          fout[t * P + cell] = v;
        }
        if (j == 0) {
          mout[cell] = rho0;
          mout[P + cell] = c0[0];
          mout[2 * P + cell] = c0[1];
          mout[3 * P + cell] = c0[2];
          mout[4 * P + cell] = c0[3];
          niter_out[cell] = niter;
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// host-side launchers

// per-step node data of the load state: D3Q27 the gauge record (ux, uy, uz, P) of every cell, 32
// bytes, D1Q5 the plane of P, with P = sqrt(|T|)*sign(T); empties the step's list of pending cells
__global__ void k_node_prep(const double* __restrict__ m, double* __restrict__ P, int64_t n, int64_t plane,
                            bool record, int* __restrict__ pending_count) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c == 0) *pending_count = 0;
  if (c >= n) return;
  const double Pc = sqrts_d(m[4 * plane + c]);
  if (record) {
    reinterpret_cast<double2*>(P)[2 * c] = make_double2(m[plane + c], m[2 * plane + c]);
    reinterpret_cast<double2*>(P)[2 * c + 1] = make_double2(m[3 * plane + c], Pc);
  } else {
    P[c] = Pc;
  }
}

hipError_t launch_node_prep(int lattice, const double* m, double* P, int64_t n, int64_t plane, int* pending_count,
                            hipStream_t st) {
  hipLaunchKernelGGL(k_node_prep, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, m, P, n, plane,
                     lattice == kD3Q27, pending_count);
  return hipGetLastError();
}

// The line kernel does 3-4 times the work per cell and iteration of the one-lane kernel (lanes of a
// target repeat its tail), and pays where the chip is not full or the iteration counts are uneven.
// WENO5: every line (2^20 cells, the longest: 5.3 -> 1.0 ms on the Sod tube, 3.6 -> 2.9 ms on a
// smooth wave with 3.65 iterations everywhere).  Lagrange-4, one lane per cell and here, on a smooth wave
// with 3 iterations everywhere and on the Sod tube: 32768 cells 0.099 -> 0.070 and 0.26 -> 0.044 ms, 49152
// 0.101 -> 0.101 and 0.27 -> 0.057, 65536 0.102 -> 0.131 and 0.26 -> 0.069; the wave with mirror walls 65536
// 1.61 -> 0.135.  The limit gives the wave's third away for the tube's factor of four.
bool f64_line_step(int lattice, int interp, const Grid& g) {
  return lattice == kD1Q5 && g.ny == 1 && g.nz == 1 && (interp != 1 || g.n <= kLineCellsLagr4);
}

hipError_t launch_step_f64(int lattice, int interp, const double* fin, const double* min, const double* Pin,
                           double* fout, double* mout, int* niter, const Pending& pend, const StepArgs& a,
                           hipStream_t st) {
  if (lattice == kD3Q125) {
    const dim3 nb((unsigned)a.g.n), nt(128);
    if (a.g.mirror) hipLaunchKernelGGL(k_step_q125_f64<true>, nb, nt, 0, st, fin, min, fout, mout, niter, a);
    else hipLaunchKernelGGL(k_step_q125_f64<false>, nb, nt, 0, st, fin, min, fout, mout, niter, a);
    return hipGetLastError();
  }
  // kernel codes: 0 WENO5 as written, 1 Lagrange-4, 2 WENO5 centred, 3 Lagrange-4 with mirror
  // boundaries (its own instantiation, so the periodic kernels carry none of the mirror code),
  // 4 the generic WENO5.  interp is pond_interp (POND_WENO5G = 3).
  const int code = interp == 3 ? 4 : (interp == 1 && a.g.mirror) ? 3 : interp;
  const dim3 nt(64);
  if (f64_line_step(lattice, interp, a.g)) {
    // on a line the centred and as-written WENO5 coincide
    const dim3 nb((unsigned)((a.g.n + 1) / 2));
    if (code == 1) hipLaunchKernelGGL(k_step_line<1>, nb, nt, 0, st, fin, min, fout, mout, niter, a);
    else if (code == 3) hipLaunchKernelGGL(k_step_line<3>, nb, nt, 0, st, fin, min, fout, mout, niter, a);
    else if (code == 4) hipLaunchKernelGGL(k_step_line<4>, nb, nt, 0, st, fin, min, fout, mout, niter, a);
    else hipLaunchKernelGGL(k_step_line<0>, nb, nt, 0, st, fin, min, fout, mout, niter, a);
    return hipGetLastError();
  }
  const NodeSrc src{fin, min, Pin, a.g};
  if (lattice == kD3Q27) {
    // buffer-resource loads while four pair planes fit a 32-bit offset
    const bool buf = (uint64_t)a.g.plane * 8u * 8u <= 0xffffffffull && !a.global_loads;
    // Cells per wave: one per slot, or two where that still leaves several waves for every SIMD (a slot
    // then fills the tail of a slow neighbour).  ms per step with 7, 14, 28 cells: 33x18x14 0.85,
    // 1.09, 1.7; 128^3 vortex 64.9, 65.8, 68; 256x128x128 shock-bubble 183.7, 180.7, 182.
    const int64_t slots = a.g.ntiles * 64;
    int64_t cells = a.refill_chunk > 0 ? 64ll * a.refill_chunk : a.refill_chunk == 0 ? 64 : a.g.n < (1 << 20) ? 7 : 14;
    if (cells > slots) cells = slots;
    const dim3 nb((unsigned)((slots + cells - 1) / cells));
#define POND_LAUNCH(I)                                                                                           \
  do {                                                                                                           \
    if (buf) hipLaunchKernelGGL((k_step_f64_27<I, true>), nb, nt, 0, st, src, fout, mout, niter, pend.count, a, (int)cells, wide_after, few);   \
    else hipLaunchKernelGGL((k_step_f64_27<I, false>), nb, nt, 0, st, src, fout, mout, niter, pend.count, a, (int)cells, wide_after, few);      \
  } while (0)
    // The iteration after which a WENO5 cell goes to k_step_f64_27_wide, early where the grid leaves the
    // chip idle.  ms per step for 5, 6, 8, 12, 16 and never: 33x18x14 vortex 0.64, 0.65, 0.75, 0.84, -,
    // 0.81; shock-bubble 32^3 -, 4.24, 4.10, 4.16, 4.20, 10.4; 64^3 -, 19.5, 17.6, 16.9, 16.9, 20.5;
    // 100^3 -, 55.6, 53.2, 52.1, 52.1, 54.4; 128^3 -, -, 105, 99.7, 99.5, 99.1.
    const int wide_after = a.pass1_iters > 0 ? a.pass1_iters : a.g.n < (1 << 14) ? 6 : a.g.n < (1 << 17) ? 8 : 16;
    // From then on a cell goes when its wave stands idle for it: with no cell left to start and at most
    // kWideSlots64 slots still at such cells.  The workgroups of the chip do 28 iterations per us, the waves
    // with all slots in use 145, so a wave whose cells are all late keeps them; the first 2048 of a step go at
    // once, as a small grid leaves the chip idle anyway.  Tolerance 0 (every cell to the cap), ms per step with every late cell
    // handed over and now: 16^3 18.0, 15.2, 32^3 119, 34, 64^3 877, 185 (with 1024: 11.4, 31, 180, but the
    // 12^3 shock-bubble 1.15 -> 1.29); T = 0.2 with density jumps 16 cells apart 64^3 79.9, 78.3, 96^3 263, 254.
    constexpr int few = 2048;
    const dim3 nw((unsigned)(a.g.n < 1024 ? a.g.n : 1024)), ntw(kWideThreads64);
#define POND_WIDE(V) hipLaunchKernelGGL(k_step_f64_27_wide<V>, nw, ntw, 0, st, src, fout, mout, niter, pend.count, a)
    if (code == 1) {
      POND_LAUNCH(1);
    } else if (code == 3) {
      POND_LAUNCH(3);
    } else if (code == 0) {
      POND_LAUNCH(0);
      POND_WIDE(0);
    } else if (code == 4) {
      POND_LAUNCH(4);
      POND_WIDE(2);
    } else {
      POND_LAUNCH(2);
      POND_WIDE(1);
    }
#undef POND_WIDE
#undef POND_LAUNCH
    return hipGetLastError();
  }
  // D1Q5 off a line and long Lagrange-4 lines: one lane per cell, two passes (the first of eight
  // iterations: 128^3 D3Q27 shock-bubble in this form, K=3 2.98, K=5 3.19, K=8 3.35, single pass 2.86 MLUPS)
  StepArgs b = a;
  if (b.pass1_iters < 0) b.pass1_iters = 8;
  const int64_t w2 = (a.g.n + 63) / 64;
  const dim3 nb1((unsigned)a.g.ntiles), nb2((unsigned)(w2 < 16384 ? w2 : 16384));
#define POND_LAUNCH(I)                                                                                           \
  do {                                                                                                           \
    hipLaunchKernelGGL((k_step_f64<kD1Q5, I>), nb1, nt, 0, st, src, fout, mout, niter, pend, b);                  \
    hipLaunchKernelGGL((k_step_f64_rest<kD1Q5, I>), nb2, nt, 0, st, src, fout, mout, niter, pend, b);             \
  } while (0)
  if (code == 1) POND_LAUNCH(1);
  else if (code == 3) POND_LAUNCH(3);
  else if (code == 4) POND_LAUNCH(4);
  else POND_LAUNCH(0);
#undef POND_LAUNCH
  return hipGetLastError();
}

}  // namespace pond
