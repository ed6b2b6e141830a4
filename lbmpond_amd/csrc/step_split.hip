// step_split.hip -- FP32/FP64-split PonD step for D3Q27 on gfx950.
//
// Same algorithm as the plain path (LBMpull, steps.cu:356-588): fixed-point iteration on the
// cell's gauge (u, T), pull streaming of gauge-transferred populations with WENO5 / Lagrange-4
// interpolation, moments, BGK towards rho*w_i.  Precision split:
//   FP32: population storage, the gauge transfer, interpolation, WENO weights, collide;
//         rho and rho*u summed in FP32 with Kahan compensation;
//   FP64: the energy moment sum f|v|^2, the moment solve (u = m/rho, T = (E/rho - |u|^2)/Dim),
//         the stored temperature, and the gauge-convergence residual.
// The gauge transfer is sum-factorised: the target population's basis is a tensor product of
// per-axis quadratic Lagrange polynomials (structs.cuh:525-548), so
//   f_new(k) = sum_jx Lx[jx] sum_jy Ly[jy] sum_jz Lz[jz] f(jx,jy,jz)
// costs 39 FMAs plus 9 basis values instead of 27 five-factor products.
//
// Convergence (FP32-appropriate; the reference's 1e-10 relative test cannot be met by FP32
// populations): the FP64 gauge residual |du_d| <= tol_rel*sqrt(T) + tol_abs and
// |dT| <= tol_rel*T + tol_abs (defaults 1e-7, 1e-12), or, at the FP32 noise floor, a residual
// below 4 tol_rel that no longer halves from one iteration to the next.  Populations are a
// deterministic function of the gauge, so they converge with it.
//
// Starting gauge: the cell's previous gauge, or (learned initializer) a predicted gauge.  The
// fixed-point iteration has the last word: a prediction that is not finite or not positive in T
// is ignored, and if the residual stops falling before the noise floor, or the cell has not
// converged after kLearnedBudget iterations, it restarts from its previous gauge.
#include "pond_device.h"
#include "step_split.h"

namespace pond {

// per-lane constants of one target population in the current gauge
struct TgtF {
  float u1x, u1y, u1z;     // target gauge velocity, rounded to FP32 ...
  float u1xl, u1yl, u1zl;  // ... and the rounding remainder (u1 = hi + lo to ~2^-48)
  float T1;
  float wx, wy, wz;  // 1/(2T1) or -1/T1 per axis
  float cx, cy, cz;  // e_k*sqrt(T1) per axis
  bool kx, ky, kz;
};

__device__ __forceinline__ TgtF make_tgtf(int k, const double* g) {
  TgtF t;
  t.u1x = (float)g[0]; t.u1y = (float)g[1]; t.u1z = (float)g[2];
  t.u1xl = (float)(g[0] - (double)t.u1x);
  t.u1yl = (float)(g[1] - (double)t.u1y);
  t.u1zl = (float)(g[2] - (double)t.u1z);
  const float T1 = (float)g[3];
  t.T1 = T1;
  const float h = 1.0f / (2.0f * T1), m = -1.0f / T1;
  const float sq1 = sqrtf(fabsf(T1)) * (float)((0.0f < T1) - (T1 < 0.0f));
  const int ex = kE27[k][0], ey = kE27[k][1], ez = kE27[k][2];
  t.wx = ex ? h : m; t.wy = ey ? h : m; t.wz = ez ? h : m;
  t.cx = ex * sq1; t.cy = ey * sq1; t.cz = ez * sq1;
  t.kx = ex != 0; t.ky = ey != 0; t.kz = ez != 0;
  return t;
}

__device__ __forceinline__ int min3(int a, int b, int c) { return min(a, min(b, c)); }
__device__ __forceinline__ int max3(int a, int b, int c) { return max(a, max(b, c)); }

// basis values L[j], j = source component -1,0,+1, of one axis (structs.cuh:530-538)
__device__ __forceinline__ void basis3(float D, float sq0, bool kn, float c, float T1, float w, float L[3]) {
#pragma unroll
  for (int j = 0; j < 3; j++) {
    const float A = D - (float)(j - 1) * sq0;
    const float g = kn ? A * (A - c) : __builtin_fmaf(A, A, -T1);
    L[j] = w * g;
  }
}

// basis3 without the per-axis factor w, the axis kind folded into (c, T): a moving axis
// (kn) passes c = e*sqrt(T1), T = 0 and gets A (A - c); a resting one passes c = 0, T = T1 and
// gets A^2 - T1.  fma(A, A - c, -T) is either, rounded as in basis3, without a select between
// the two forms where the kind is only known at run time.  A_j = D - (j - 1) sq0.
__device__ __forceinline__ void basis3u(float D, float sq0, float c, float T, float G[3]) {
  const float A0 = D + sq0, A1 = D, A2 = D - sq0;
  G[0] = __builtin_fmaf(A0, A0 - c, -T);
  G[1] = __builtin_fmaf(A1, A1 - c, -T);
  G[2] = __builtin_fmaf(A2, A2 - c, -T);
}

// Buffer resources: a load names its plane (or quad plane) through the scalar offset and the
// per-lane address is a single 32-bit offset, where a global load needs a 64-bit per-lane
// address (two VGPRs and a 64-bit add per load).  The resource size is exact, so the hardware
// range check returns 0 rather than reading past the array.  Word 3 (0x00020000) is the
// raw-buffer configuration of the gfx9 family.
constexpr uint32_t kRawBufferWord3 = 0x00020000u;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)(uint32_t)bytes, (int)kRawBufferWord3);
}

// the seven quad planes of the D3Q27 split populations: resource j holds quad planes 2j, 2j+1,
// the quad plane within it is chosen by the scalar offset (plane * 16 bytes each, so up to
// 134,217,727 cells fit the 32-bit offsets)
struct QuadsF {
  __amdgpu_buffer_rsrc_t r[4];
  uint32_t qbytes;  // bytes per quad plane
};

__device__ __forceinline__ QuadsF make_quads(const float* base, int64_t plane) {
  QuadsF q;
  q.qbytes = (uint32_t)(plane * 16);
  for (int j = 0; j < 4; j++) {
    const int cnt = 7 - 2 * j < 2 ? 7 - 2 * j : 2;
    q.r[j] = make_rsrc(base + (int64_t)2 * j * plane * 4, (uint64_t)cnt * q.qbytes);
  }
  return q;
}

// the 27 populations of the cell at byte offset boff of a 4-byte plane (boff = 4 * cell)
__device__ __forceinline__ void load27(const QuadsF& q, uint32_t boff, float f[27]) {
#pragma unroll
  for (int j = 0; j < 7; j++) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(q.r[j >> 1], (int)(boff * 4u), (int)((uint32_t)(j & 1) * q.qbytes), 0);
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (4 * j + e < 27) f[4 * j + e] = __builtin_bit_cast(float, (uint32_t)v[e]);
  }
}

// sum-factorised gauge transfer of the node at byte offset boff to target t.  The gauge
// difference u1 - u0 is formed as (hi - u0) + lo: hi - u0 is exact when the two velocities are
// within a factor of two (Sterbenz), so the difference carries one rounding relative to itself
// rather than one relative to |u1|, which would put a jitter of ulp(|u|) into the velocity
// moment.
__device__ __forceinline__ float transfer27f(const float f[27], float u0x, float u0y, float u0z, float sq0,
                                             const TgtF& t, float sqTb) {
  float Lx[3], Ly[3], Lz[3];
  basis3(((t.u1x - u0x) + t.u1xl) * sqTb, sq0, t.kx, t.cx, t.T1, t.wx, Lx);
  basis3(((t.u1y - u0y) + t.u1yl) * sqTb, sq0, t.ky, t.cy, t.T1, t.wy, Ly);
  basis3(((t.u1z - u0z) + t.u1zl) * sqTb, sq0, t.kz, t.cz, t.T1, t.wz, Lz);
  float out = 0.0f;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    float sy = 0.0f;
#pragma unroll
    for (int b = 0; b < 3; b++) {
      float sz = 0.0f;
#pragma unroll
      for (int c = 0; c < 3; c++) sz = __builtin_fmaf(Lz[c], f[kIdx27.v[a][b][c]], sz);
      sy = __builtin_fmaf(Ly[b], sz, sy);
    }
    out = __builtin_fmaf(Lx[a], sy, out);
  }
  return out;
}

// node side of the load state: the population planes and the node gauges, one 16-byte record
// (ux, uy, uz, sqrt(|T|)*sign(T)) per cell written by k_node_gauge before the step, so a node's
// gauge is one load
struct NodeSrcF {
  QuadsF f;
  __amdgpu_buffer_rsrc_t g4;
  Grid g;
};

__device__ __forceinline__ NodeSrcF make_src(const float* f, const float* g4, const Grid& g) {
  return NodeSrcF{make_quads(f, g.plane), make_rsrc(g4, (uint64_t)g.plane * 16u), g};
}

struct Gauge4 {
  float ux, uy, uz, sq;
};

// gauge record of the cell at byte offset boff of the population planes (4 bytes per cell)
__device__ __forceinline__ Gauge4 ldg4(const NodeSrcF& s, uint32_t boff) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(s.g4, (int)(boff * 4u), 0, 0);
  return Gauge4{__builtin_bit_cast(float, (uint32_t)v[0]), __builtin_bit_cast(float, (uint32_t)v[1]),
                __builtin_bit_cast(float, (uint32_t)v[2]), __builtin_bit_cast(float, (uint32_t)v[3])};
}

__device__ __forceinline__ float node_xfer(const NodeSrcF& s, int64_t c, const TgtF& t, float sqTb) {
  const uint32_t boff = (uint32_t)c * 4u;
  float f[27];
  load27(s.f, boff, f);
  const Gauge4 n = ldg4(s, boff);
  return transfer27f(f, n.ux, n.uy, n.uz, n.sq, t, sqTb);
}

// node_xfer of the node's mirror image on the axes set in mx, my, mz (Cell::mirrX/Y/Z,
// structs.cuh:552-578: the axis velocity negated, every population exchanged with its mirror
// image).  Exchanging the populations along an axis is the same as reversing that axis's basis
// values (sum_j L[j] f[rev j] = sum_j L[rev j] f[j]), so the populations stay in place and only
// the three basis values of a mirrored axis are swapped end for end.
__device__ float node_xfer_mirrored(const NodeSrcF& s, int64_t c, const TgtF& t, float sqTb, bool mx, bool my,
                                    bool mz) {
  const uint32_t boff = (uint32_t)c * 4u;
  float f[27];
  load27(s.f, boff, f);
  const Gauge4 n = ldg4(s, boff);
  float Lx[3], Ly[3], Lz[3];
  basis3(((t.u1x - (mx ? -n.ux : n.ux)) + t.u1xl) * sqTb, n.sq, t.kx, t.cx, t.T1, t.wx, Lx);
  basis3(((t.u1y - (my ? -n.uy : n.uy)) + t.u1yl) * sqTb, n.sq, t.ky, t.cy, t.T1, t.wy, Ly);
  basis3(((t.u1z - (mz ? -n.uz : n.uz)) + t.u1zl) * sqTb, n.sq, t.kz, t.cz, t.T1, t.wz, Lz);
  auto flip = [](bool m, float L[3]) {
    const float a = L[0];
    L[0] = m ? L[2] : L[0];
    L[2] = m ? a : L[2];
  };
  flip(mx, Lx);
  flip(my, Ly);
  flip(mz, Lz);
  float out = 0.0f;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    float sy = 0.0f;
#pragma unroll
    for (int b = 0; b < 3; b++) {
      float sz = 0.0f;
#pragma unroll
      for (int cc = 0; cc < 3; cc++) sz = __builtin_fmaf(Lz[cc], f[kIdx27.v[a][b][cc]], sz);
      sy = __builtin_fmaf(Ly[b], sz, sy);
    }
    out = __builtin_fmaf(Lx[a], sy, out);
  }
  return out;
}

__device__ __forceinline__ void lag3f(float s, float F[3]) {
  // quadratic Lagrange basis on nodes 0,1,2 at s
  F[0] = 0.5f * (s - 1.0f) * (s - 2.0f);
  F[1] = -s * (s - 2.0f);
  F[2] = 0.5f * s * (s - 1.0f);
}

__device__ __forceinline__ void lag4f(float s, float F[4]) {
  // cubic Lagrange basis on nodes 0..3 at s
  const float a = s, b = s - 1.0f, c = s - 2.0f, d = s - 3.0f;
  F[0] = -(b * c * d) * (1.0f / 6.0f);
  F[1] = 0.5f * a * c * d;
  F[2] = -0.5f * a * b * d;
  F[3] = (a * b * c) * (1.0f / 6.0f);
}

// nonlinear WENO5 combination of the three sub-stencil values S at offset c = cx - r from the
// five smoothness samples ub (steps.cu:795-825)
__device__ __forceinline__ float weno5_combine(float c, const float ub[5], const float S[3]) {
  const float d0 = (c * c - 3.f * c + 2.f) * (1.f / 12.f);
  const float d2 = (c * c + 3.f * c + 2.f) * (1.f / 12.f);
  const float d1 = 1.f - d0 - d2;
  // Smoothness indicators in the difference form of Jiang & Shu (J. Comput. Phys. 126, 1996),
  // which expands to exactly the reference's polynomials (steps.cu:801-806).  In FP32 the
  // expanded form cancels terms of size ~25 f^2 down to beta ~ (df)^2, and the rounding of
  // those terms, measured against the 1e-6 regularisation, moves the weights by ~1e-3 from one
  // iteration to the next; the differences carry no such cancellation.
  const float u1 = ub[0], u2 = ub[1], u3 = ub[2], u4 = ub[3], u5 = ub[4];
  const float p0 = u1 - 2.f * u2 + u3, q0 = u1 - 4.f * u2 + 3.f * u3;
  const float p1 = u2 - 2.f * u3 + u4, q1 = u2 - u4;
  const float p2 = u3 - 2.f * u4 + u5, q2 = 3.f * u3 - 4.f * u4 + u5;
  const float b0 = (13.f / 12.f) * p0 * p0 + 0.25f * q0 * q0;
  const float b1 = (13.f / 12.f) * p1 * p1 + 0.25f * q1 * q1;
  const float b2 = (13.f / 12.f) * p2 * p2 + 0.25f * q2 * q2;
  // Weights d_k / (e + b_k)^2, each multiplied by (e + b_min)^2: the same normalised weights,
  // but every factor (e + b_min) / (e + b_k) lies in (0, 1], so large samples (b ~ 1e19 and up,
  // where (e + b)^2 leaves FP32 range and all three weights would round to 0/0) keep finite
  // weights with the largest one equal to d_k.
  const float e = 1e-6f;
  const float em = e + fminf(b0, fminf(b1, b2));
  const float r0 = em / (e + b0), r1 = em / (e + b1), r2 = em / (e + b2);
  const float w0 = d0 * (r0 * r0), w1 = d1 * (r1 * r1), w2 = d2 * (r2 * r2);
  return (w0 * S[0] + w1 * S[1] + w2 * S[2]) / (w0 + w1 + w2);
}


// WENO5 interpolation (propagateWENO<3,5>) in FP32; CENTRED selects the corrected y/z stencil
template <bool CENTRED>
__device__ float interp_weno5f(const NodeSrcF& src, double cx, double cy, double cz, const TgtF& t, float sqTb) {
  const Grid& g = src.g;
  const int r = floor_int(cx + 0.5);
  const int ry = floor_int(cy + 0.5) - (CENTRED ? 1 : 0), rz = floor_int(cz + 0.5) - (CENTRED ? 1 : 0);
  float Fy[3], Fz[3], Fx[3][3];
  lag3f((float)(cy - ry), Fy);
  lag3f((float)(cz - rz), Fz);
#pragma unroll
  for (int k = 0; k < 3; k++) lag3f((float)(cx - (r - 2 + k)), Fx[k]);
  int yy[3], zz[3];
#pragma unroll
  for (int a = 0; a < 3; a++) { yy[a] = wrapi(ry + a, g.ny); zz[a] = wrapi(rz + a, g.nz); }
  const int by = CENTRED ? yy[1] : wrapi(r, g.ny), bz = CENTRED ? zz[1] : wrapi(r, g.nz);
  float S0 = 0.f, S1 = 0.f, S2 = 0.f, ub[5];
  // row offsets of a slice's nodes: the nine of its rows, then (as written) the sample
  constexpr int NN = CENTRED ? 9 : 10;
  uint32_t no[10];
#pragma unroll
  for (int q = 0; q < 9; q++) no[q] = (uint32_t)g.nx * ((uint32_t)yy[q / 3] + (uint32_t)g.ny * (uint32_t)zz[q % 3]);
  no[9] = (uint32_t)g.nx * ((uint32_t)by + (uint32_t)g.ny * (uint32_t)bz);
  for (int xs = 0; xs < 5; xs++) {
    const uint32_t x = (uint32_t)wrapi(r - 2 + xs, g.nx);
    float yzsum = 0.f;  // y/z interpolated value of this x slice
    float zs = 0.f;
    // A node's loads are issued before the transfer of the one before it; left to the compiler, every
    // transfer waited for its own (split WENO5 as written, 64x60x52 12.2 -> 11.0 ms per step, 128x128x64 51.5 -> 45.8).
    float f[2][27];
    Gauge4 n[2];
    auto load = [&](int q) {
      const uint32_t boff = (x + no[q]) * 4u;
      n[q & 1] = ldg4(src, boff);
      load27(src.f, boff, f[q & 1]);
    };
    load(0);
#pragma unroll
    for (int q = 0; q < NN; q++) {
      if (q + 1 < NN) load(q + 1);
      const Gauge4& m = n[q & 1];
      const float T = transfer27f(f[q & 1], m.ux, m.uy, m.uz, m.sq, t, sqTb);
      if (q == (CENTRED ? 4 : 9)) ub[xs] = T;
      if (q == 9) continue;
      zs = __builtin_fmaf(Fz[q % 3], T, q % 3 == 0 ? 0.f : zs);
      if (q % 3 == 2) yzsum = __builtin_fmaf(Fy[q / 3], zs, yzsum);
    }
    if (xs <= 2) S0 = __builtin_fmaf(Fx[0][xs], yzsum, S0);
    if (xs >= 1 && xs <= 3) S1 = __builtin_fmaf(Fx[1][xs - 1], yzsum, S1);
    if (xs >= 2) S2 = __builtin_fmaf(Fx[2][xs - 2], yzsum, S2);
  }
  const float Sv[3] = {S0, S1, S2};
  return weno5_combine((float)(cx - r), ub, Sv);
}

// MIR: mirror boundaries on the axes of g.mirror (steps.cu:1004-1022)
template <bool MIR>
__device__ float interp_lagr4f(const NodeSrcF& src, double cx, double cy, double cz, const TgtF& t, float sqTb) {
  const Grid& g = src.g;
  const int lx = floor_int(cx) - 1, ly = floor_int(cy) - 1, lz = floor_int(cz) - 1;
  float Fx[4], Fy[4], Fz[4];
  lag4f((float)(cx - lx), Fx);
  lag4f((float)(cy - ly), Fy);
  lag4f((float)(cz - lz), Fz);
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
  float out = 0.f;
  for (int ix = 0; ix < 4; ix++) {
    bool rx = false;
    const int x = MIR ? mirror_wrap(lx + ix, g.nx, (g.mirror & 1) != 0, rx) : wrapi(lx + ix, g.nx);
    float ys = 0.f;
#pragma unroll
    for (int a = 0; a < 4; a++) {
      float zs = 0.f;
#pragma unroll
      for (int b = 0; b < 4; b++) {
        const int64_t c = cell_index(g, x, yy[a], zz[b]);
        const float v = MIR && (rx || ry[a] || rz[b]) ? node_xfer_mirrored(src, c, t, sqTb, rx, ry[a], rz[b])
                                                      : node_xfer(src, c, t, sqTb);
        zs = __builtin_fmaf(Fz[b], v, zs);
      }
      ys = __builtin_fmaf(Fy[a], zs, ys);
    }
    out = __builtin_fmaf(Fx[ix], ys, out);
  }
  return out;
}

// WENO5C for the three targets of one (ey, ez) group: ex = -1, 0, +1.  They share the departure
// rows in y and z (same y and z velocity), and their transfer bases differ only along x, so for
// every stencil node the contraction of the 27 source populations over the z and y source
// components, sy[jx] = sum_jy Ly[jy] sum_jz Lz[jz] f(jx,jy,jz), is common to the three:
// 27 loads and 36 FMAs per node, then 3 FMAs and an x basis per target, where three separate
// transfers load the node three times and contract it three times.  The x slices of the three
// five-slice WENO windows are visited once each (their union, at most 5 + |r(-1) - r(+1)|).
// Same interpolation as interp_weno5f<true> per target, with the y/z weights summed in a
// different order.  The x slices are visited two at a time (more loads in flight per lane).
__device__ void interp_group_weno5c(const NodeSrcF& src, int x, int y, int z, double s, const double gc[4], int ey,
                                    int ez, float sqTb, float out[3]) {
  const Grid& g = src.g;
  const float u1x = (float)gc[0], u1y = (float)gc[1], u1z = (float)gc[2];
  const float u1xl = (float)(gc[0] - (double)u1x), u1yl = (float)(gc[1] - (double)u1y),
              u1zl = (float)(gc[2] - (double)u1z);
  const float T1 = (float)gc[3];
  const float h = 1.0f / (2.0f * T1), mm = -1.0f / T1;
  const float sq1 = sqrtf(fabsf(T1)) * (float)((0.0f < T1) - (T1 < 0.0f));
  // y and z: shared rows, Lagrange weights and basis parameters
  const double cy = (double)y - (s * (double)ey + gc[1]), cz = (double)z - (s * (double)ez + gc[2]);
  const int ry = floor_int(cy + 0.5) - 1, rz = floor_int(cz + 0.5) - 1;
  float Fy[3], Fz[3];
  lag3f((float)(cy - ry), Fy);
  lag3f((float)(cz - rz), Fz);
  // row offsets of the stencil rows: node (x, a, b) is cell x + yo[a] + zo[b] (the split
  // path's grids have 32-bit cell indices)
  uint32_t yo[3], zo[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    yo[a] = (uint32_t)wrapi(ry + a, g.ny) * (uint32_t)g.nx;
    zo[a] = (uint32_t)wrapi(rz + a, g.nz) * ((uint32_t)g.nx * (uint32_t)g.ny);
  }
  // y and z basis kinds (basis3u) and factors
  const float cyb = ey ? (float)ey * sq1 : 0.0f, Tyb = ey ? 0.0f : T1;
  const float czb = ez ? (float)ez * sq1 : 0.0f, Tzb = ez ? 0.0f : T1;
  const float wy = ey ? h : mm, wz = ez ? h : mm;
  // x: per target t (ex = t - 1) its window r_t-2 .. r_t+2 and sub-stencil weights
  int r[3];
  float c[3];  // cx - r: sub-stencil k evaluates its quadratic at c + 2 - k
#pragma unroll
  for (int t = 0; t < 3; t++) {
    const double cx = (double)x - (s * (double)(t - 1) + gc[0]);
    r[t] = floor_int(cx + 0.5);
    c[t] = (float)(cx - r[t]);
  }
  const int xlo = min(r[0], min(r[1], r[2])) - 2, xhi = max(r[0], max(r[1], r[2])) + 2;
  // (64-bit difference: for an infinite temperature the windows sit at +-2^30 and the 32-bit
  // difference would overflow)
  if ((int64_t)xhi - (int64_t)xlo > 8) {
    // windows far apart (a gauge with a huge temperature or velocity): target by target, so the
    // loop stays five slices per target whatever the gauge
#pragma unroll 1
    for (int t = 0; t < 3; t++) {
      const int i = kIdx27.v[t][ey + 1][ez + 1];
      const double cx = (double)x - (s * (double)(t - 1) + gc[0]);
      out[t] = interp_weno5f<true>(src, cx, cy, cz, make_tgtf(i, gc), sqTb);
    }
    return;
  }
  // per target and window position j: the middle node's value (smoothness samples) and the
  // slice's y/z sum
  float ub[3][5], yv[3][5];
#pragma unroll
  for (int t = 0; t < 3; t++) {
#pragma unroll
    for (int j = 0; j < 5; j++) ub[t][j] = yv[t][j] = 0.f;
  }
  // contribution of one stencil node (its moments and 27 populations) to the three targets'
  // y/z sums yz (weight wab) and, for the middle node, to their smoothness samples mid
  auto node = [&](float u0x, float u0y, float u0z, float sq0, const float f[27], float wab, bool is_mid, float yz[3],
                  float mid[3]) {
    // basis values without their per-axis factors w: those are constants of the group (y, z)
    // and of the target (x), applied once to the finished window values
    float Ly[3], Lz[3];
    basis3u(((u1y - u0y) + u1yl) * sqTb, sq0, cyb, Tyb, Ly);
    basis3u(((u1z - u0z) + u1zl) * sqTb, sq0, czb, Tzb, Lz);
    float sy[3];
#pragma unroll
    for (int ja = 0; ja < 3; ja++) {
      float acc = 0.f;
#pragma unroll
      for (int jb = 0; jb < 3; jb++) {
        float sz = 0.f;
#pragma unroll
        for (int jc = 0; jc < 3; jc++) sz = __builtin_fmaf(Lz[jc], f[kIdx27.v[ja][jb][jc]], sz);
        acc = __builtin_fmaf(Ly[jb], sz, acc);
      }
      sy[ja] = acc;
    }
    // x basis of the three targets from shared sums: with A_j = Dx - (j - 1) sq0 the moving
    // targets (ex = -1, +1) have g_j = A_j (A_j + sq1), A_j (A_j - sq1) and the resting one
    // A_j^2 - T1, so with P = sum A_j^2 sy_j, Q = sum A_j sy_j, R = sum sy_j the three values
    // are P + sq1 Q, P - T1 R and P - sq1 Q
    const float Dx = ((u1x - u0x) + u1xl) * sqTb;
    const float A0 = Dx + sq0, A1 = Dx, A2 = Dx - sq0;
    const float Q = __builtin_fmaf(A2, sy[2], __builtin_fmaf(A1, sy[1], A0 * sy[0]));
    const float P = __builtin_fmaf(A2, A2 * sy[2], __builtin_fmaf(A1, A1 * sy[1], A0 * (A0 * sy[0])));
    const float R = (sy[0] + sy[1]) + sy[2];
    const float Tt[3] = {__builtin_fmaf(sq1, Q, P), __builtin_fmaf(-T1, R, P), __builtin_fmaf(-sq1, Q, P)};
#pragma unroll
    for (int t = 0; t < 3; t++) {
      yz[t] = __builtin_fmaf(wab, Tt[t], yz[t]);
      if (is_mid) mid[t] = Tt[t];
    }
  };
  // slice xs (its y/z sums yz and middle values mid) enters target t's window at position
  // j = xs - (r_t - 2); the sub-stencil sums are formed once the window is complete
  auto slice = [&](int xs, const float yz[3], const float mid[3]) {
#pragma unroll
    for (int t = 0; t < 3; t++) {
      const int j = xs - (r[t] - 2);
      // (selects with constant indices: the arrays stay in registers)
#pragma unroll
      for (int jj = 0; jj < 5; jj++) {
        const bool at = j == jj;
        ub[t][jj] = at ? mid[t] : ub[t][jj];
        yv[t][jj] = at ? yz[t] : yv[t][jj];
      }
    }
  };
  for (int xs = xlo; xs <= xhi; xs += 2) {
    const int xw = wrapi(xs, g.nx);
    float yz[3] = {0.f, 0.f, 0.f}, mid[3] = {0.f, 0.f, 0.f};
    float yz2[3] = {0.f, 0.f, 0.f}, mid2[3] = {0.f, 0.f, 0.f};
    // slices xs and xs+1 together (the second through the same per-node code)
    const bool two = xs + 1 <= xhi;
    const int xw2 = wrapi(xs + 1, g.nx);
    // one node at a time: its loads are the only ones in flight per lane
#pragma unroll 1
    for (int q = 0; q < 9; q++) {
      const int a = q / 3, b = q - 3 * (q / 3);
      const uint32_t ya = a == 0 ? yo[0] : a == 1 ? yo[1] : yo[2];
      const uint32_t zb = b == 0 ? zo[0] : b == 1 ? zo[1] : zo[2];
      const float fya = a == 0 ? Fy[0] : a == 1 ? Fy[1] : Fy[2];
      const float fzb = b == 0 ? Fz[0] : b == 1 ? Fz[1] : Fz[2];
      const float wab = fya * fzb;
      const uint32_t boff = ((uint32_t)xw + ya + zb) * 4u;
      float f[27];
      load27(src.f, boff, f);
      const Gauge4 n = ldg4(src, boff);
      node(n.ux, n.uy, n.uz, n.sq, f, wab, q == 4, yz, mid);
      if (two) {
        const uint32_t boff2 = ((uint32_t)xw2 + ya + zb) * 4u;
        load27(src.f, boff2, f);
        const Gauge4 n2 = ldg4(src, boff2);
        node(n2.ux, n2.uy, n2.uz, n2.sq, f, wab, q == 4, yz2, mid2);
      }
    }
    slice(xs, yz, mid);
    if (two) slice(xs + 1, yz2, mid2);
  }
  // sub-stencil k (left node r-2+k): quadratic Lagrange weights at c + 2 - k on its nodes
  // m = 0, 1, 2, summed in node order; the window values first take the basis factors
  // w_x(t) w_y w_z left out of the node contributions (the interpolation is linear in them, the
  // WENO weights are not, so they enter before the smoothness indicators)
  const float wyz = wy * wz;
#pragma unroll
  for (int t = 0; t < 3; t++) {
    const float wt = (t != 1 ? h : mm) * wyz;
#pragma unroll
    for (int j = 0; j < 5; j++) {
      ub[t][j] *= wt;
      yv[t][j] *= wt;
    }
    float S[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const float sk = c[t] + (float)(2 - k);
      const float w0 = 0.5f * (sk - 1.0f) * (sk - 2.0f), w1 = -sk * (sk - 2.0f), w2 = 0.5f * sk * (sk - 1.0f);
      S[k] = __builtin_fmaf(w2, yv[t][k + 2], __builtin_fmaf(w1, yv[t][k + 1], __builtin_fmaf(w0, yv[t][k], 0.f)));
    }
    out[t] = weno5_combine(c[t], ub[t], S);
  }
}

// What the three ey groups of an ez pass share of one stencil node: with the node's contraction over
// the z source components, sz[ja][jb] = sum_jc Lz[jc] f(ja, jb, jc), the x basis of the three targets
// is A_j (A_j - c) or A_j^2 - T1 with A_j = Dx - (j-1) sq0, so the x moments R = sum_ja sz, Q = sum_ja
// A_ja sz, P = sum_ja A_ja^2 sz per source y component jb serve every group
struct NodePass {
  float xr[3], xq[3], xp[3];
  float Ay0, Ay1, Ay2;  // the y basis' A_j
};

__device__ __forceinline__ NodePass node_pass(const float f[27], const Gauge4& n, float u1x, float u1xl, float u1y,
                                              float u1yl, float u1z, float u1zl, float sqTb, float czb, float Tzb) {
  NodePass o;
  float Lz[3];
  basis3u(((u1z - n.uz) + u1zl) * sqTb, n.sq, czb, Tzb, Lz);
  float szz[3][3];
#pragma unroll
  for (int ja = 0; ja < 3; ja++)
#pragma unroll
    for (int jb = 0; jb < 3; jb++) {
      float sz = 0.f;
#pragma unroll
      for (int jc = 0; jc < 3; jc++) sz = __builtin_fmaf(Lz[jc], f[kIdx27.v[ja][jb][jc]], sz);
      szz[ja][jb] = sz;
    }
  const float Dy = ((u1y - n.uy) + u1yl) * sqTb;
  const float Dx = ((u1x - n.ux) + u1xl) * sqTb;
  const float A0 = Dx + n.sq, A1 = Dx, A2 = Dx - n.sq;
  const float B0 = A0 * A0, B1 = A1 * A1, B2 = A2 * A2;
#pragma unroll
  for (int jb = 0; jb < 3; jb++) {
    o.xr[jb] = (szz[0][jb] + szz[1][jb]) + szz[2][jb];
    o.xq[jb] = __builtin_fmaf(A2, szz[2][jb], __builtin_fmaf(A1, szz[1][jb], A0 * szz[0][jb]));
    o.xp[jb] = __builtin_fmaf(B2, szz[2][jb], __builtin_fmaf(B1, szz[1][jb], B0 * szz[0][jb]));
  }
  o.Ay0 = Dy + n.sq;
  o.Ay1 = Dy;
  o.Ay2 = Dy - n.sq;
  return o;
}

// the node's values for the three targets of group ey (without the per-axis basis factors): the y
// contraction of the x moments, then P + sq1 Q, P - T1 R and P - sq1 Q
__device__ __forceinline__ void node_group(const NodePass& p, int ey, float sq1, float T1, float Tt[3]) {
  // basis3u of the group: fma(A, A - c, -T) with (c, T) of a moving or resting y axis
  const float cyb = ey ? (float)ey * sq1 : 0.0f, Tyb = ey ? 0.0f : T1;
  const float Ly0 = __builtin_fmaf(p.Ay0, p.Ay0 - cyb, -Tyb), Ly1 = __builtin_fmaf(p.Ay1, p.Ay1 - cyb, -Tyb),
              Ly2 = __builtin_fmaf(p.Ay2, p.Ay2 - cyb, -Tyb);
  const float R = __builtin_fmaf(Ly2, p.xr[2], __builtin_fmaf(Ly1, p.xr[1], Ly0 * p.xr[0]));
  const float Q = __builtin_fmaf(Ly2, p.xq[2], __builtin_fmaf(Ly1, p.xq[1], Ly0 * p.xq[0]));
  const float Pp = __builtin_fmaf(Ly2, p.xp[2], __builtin_fmaf(Ly1, p.xp[1], Ly0 * p.xp[0]));
  Tt[0] = __builtin_fmaf(sq1, Q, Pp);
  Tt[1] = __builtin_fmaf(-T1, R, Pp);
  Tt[2] = __builtin_fmaf(-sq1, Q, Pp);
}

// WENO5C for the nine targets that share ez (ey, ex = -1, 0, 1): one pass over the union of
// their stencil nodes.  Their departure points share the z rows, and the x windows depend on ex
// only; the y rows of the three ey groups differ by at most a row or two (they coincide wherever
// the thermal speed is below half a cell per step).  So each node of the union (x window union ×
// y row union × 3 z rows) is loaded once for all nine targets instead of once per group, and its
// contraction over the z source components, sz[ja][jb] = sum_jc Lz[jc] f(ja, jb, jc), is formed
// once and shared by the three ey groups; each group whose three rows contain the node then
// contracts over y with its own basis and adds to its three targets as interp_group_weno5c
// does.  The three sub-stencil sums of each target are accumulated slice by slice (a slice's
// y/z sum enters every sub-stencil whose window holds it), so only the five smoothness samples
// of a window are kept.  The values go to o[3 (ey+1) + ex+1] (LDS).  Windows or rows far apart (absurd gauges) fall back to
// interp_group_weno5c per group, which bounds the loops whatever the gauge.
__device__ __forceinline__ void interp_pass_weno5c(const NodeSrcF& src, int x, int y, int z, double s,
                                                   const double gc[4], int ez, float sqTb, float* o) {
  const Grid& g = src.g;
  const float u1x = (float)gc[0], u1y = (float)gc[1], u1z = (float)gc[2];
  const float u1xl = (float)(gc[0] - (double)u1x), u1yl = (float)(gc[1] - (double)u1y),
              u1zl = (float)(gc[2] - (double)u1z);
  const float T1 = (float)gc[3];
  const float h = 1.0f / (2.0f * T1), mm = -1.0f / T1;
  const float sq1 = sqrtf(fabsf(T1)) * (float)((0.0f < T1) - (T1 < 0.0f));
  // z: the pass's rows, Lagrange weights and basis parameters
  const double cz = (double)z - (s * (double)ez + gc[2]);
  const int rz = floor_int(cz + 0.5) - 1;
  float Fz[3];
  lag3f((float)(cz - rz), Fz);
  const float czb = ez ? (float)ez * sq1 : 0.0f, Tzb = ez ? 0.0f : T1;
  const float wz = ez ? h : mm;
  // y: rows and weights of the three groups ey = e - 1
  int ry[3];
  float Fy[3][3];
  double cyv[3];
#pragma unroll
  for (int e = 0; e < 3; e++) {
    cyv[e] = (double)y - (s * (double)(e - 1) + gc[1]);
    ry[e] = floor_int(cyv[e] + 0.5) - 1;
    lag3f((float)(cyv[e] - ry[e]), Fy[e]);
  }
  // x: per target t (ex = t - 1) its window r_t-2 .. r_t+2 (the same for the three groups)
  int r[3];
  float c[3];
#pragma unroll
  for (int t = 0; t < 3; t++) {
    const double cx = (double)x - (s * (double)(t - 1) + gc[0]);
    r[t] = floor_int(cx + 0.5);
    c[t] = (float)(cx - r[t]);
  }
  const int xlo = min(r[0], min(r[1], r[2])) - 2, xhi = max(r[0], max(r[1], r[2])) + 2;
  const int ylo = min(ry[0], min(ry[1], ry[2])), yhi = max(ry[0], max(ry[1], ry[2])) + 2;
  // (64-bit differences: an infinite temperature puts the windows at +-2^30)
  if ((int64_t)xhi - (int64_t)xlo > 8 || (int64_t)yhi - (int64_t)ylo > 4) {
#pragma unroll 1
    for (int e = 0; e < 3; e++) {
      float f3[3];
      interp_group_weno5c(src, x, y, z, s, gc, e - 1, ez, sqTb, f3);
#pragma unroll
      for (int t = 0; t < 3; t++) o[3 * e + t] = f3[t];
    }
    return;
  }
  uint32_t zo[3];
#pragma unroll
  for (int b = 0; b < 3; b++) zo[b] = (uint32_t)wrapi(rz + b, g.nz) * ((uint32_t)g.nx * (uint32_t)g.ny);
  // per group e and target t: the three sub-stencil sums, accumulated slice by slice, and the
  // smoothness samples at the five window positions (the middle node of each slice).  The
  // samples live in LDS, one column per lane (the kernels calling this run 64-lane blocks), at
  // the window position the slice has for the target: every position of every target and group
  // is written once (the slices span each target's window, the rows each group's middle row),
  // so nothing needs clearing.
  __shared__ float s_ub[45][64];
  const int lane = (int)threadIdx.x;
  float Sk[3][3][3];
#pragma unroll
  for (int e = 0; e < 3; e++)
#pragma unroll
    for (int t = 0; t < 3; t++)
#pragma unroll
      for (int k = 0; k < 3; k++) Sk[e][t][k] = 0.f;
  // target t's window position of slice xs is j = xs - (r_t - 2); sub-stencil k holds positions
  // k .. k+2, with the quadratic Lagrange weights at sk = c_t + 2 - k.
  //
  // The (slice, row) steps run as one loop whose node loads are one step ahead: node b of the
  // next step (the next row of the slice, or the first row of the next slice) is loaded into
  // the registers of node b of the current step once that node's contributions are added, so a
  // load has the rest of the step (about two nodes of arithmetic) to arrive in.  The loads are
  // unconditional (the step after the last loads three wrapped, unused nodes), so no lane has
  // to keep a node it has used.  The arithmetic and its order are those of a plain slice/row
  // loop.
  float fb[3][27];
  Gauge4 nb[3];
  {
    const uint32_t o0 = (uint32_t)wrapi(xlo, g.nx) + (uint32_t)wrapi(ylo, g.ny) * (uint32_t)g.nx;
#pragma unroll
    for (int b = 0; b < 3; b++) {
      const uint32_t zb = b == 0 ? zo[0] : b == 1 ? zo[1] : zo[2];
      load27(src.f, (o0 + zb) * 4u, fb[b]);
      nb[b] = ldg4(src, (o0 + zb) * 4u);
    }
  }
  float yz[3][3];
#pragma unroll
  for (int e = 0; e < 3; e++)
#pragma unroll
    for (int t = 0; t < 3; t++) yz[e][t] = 0.f;
  int xs = xlo, yr = ylo;
#pragma unroll 1
  while (true) {
    int jt[3];
#pragma unroll
    for (int t = 0; t < 3; t++) jt[t] = xs - (r[t] - 2);
    const bool last_row = yr == yhi;
    const int xn = last_row ? xs + 1 : xs, yn = last_row ? ylo : yr + 1;
    const uint32_t on = (uint32_t)wrapi(xn, g.nx) + (uint32_t)wrapi(yn, g.ny) * (uint32_t)g.nx;
    {
      // the row's place in each group's three rows (outside: the group skips the node)
      int ya[3];
#pragma unroll
      for (int e = 0; e < 3; e++) ya[e] = yr - ry[e];
#pragma unroll
      for (int b = 0; b < 3; b++) {
        const uint32_t zb = b == 0 ? zo[0] : b == 1 ? zo[1] : zo[2];
        const float fzb = b == 0 ? Fz[0] : b == 1 ? Fz[1] : Fz[2];
        const NodePass np = node_pass(fb[b], nb[b], u1x, u1xl, u1y, u1yl, u1z, u1zl, sqTb, czb, Tzb);
#pragma unroll
        for (int e = 0; e < 3; e++) {
          const int a = ya[e];
          if (a < 0 || a > 2) continue;
          float Tt[3];
          node_group(np, e - 1, sq1, T1, Tt);
          const float fya = a == 0 ? Fy[e][0] : a == 1 ? Fy[e][1] : Fy[e][2];
          const float wab = fya * fzb;
#pragma unroll
          for (int t = 0; t < 3; t++) yz[e][t] = __builtin_fmaf(wab, Tt[t], yz[e][t]);
          // the smoothness samples are the middle node's values: the middle z row (b, uniform
          // across the wave) and the group's middle y row
          if (b == 1 && a == 1) {
#pragma unroll
            for (int t = 0; t < 3; t++)
              if (jt[t] >= 0 && jt[t] <= 4) s_ub[(e * 3 + t) * 5 + jt[t]][lane] = Tt[t];
          }
        }
        // node b of this step is used up: load node b of the next step in its place
        load27(src.f, (on + zb) * 4u, fb[b]);
        nb[b] = ldg4(src, (on + zb) * 4u);
      }
    }
    if (last_row) {
      // the slice's y/z sums into the sub-stencil sums whose window holds it
#pragma unroll
      for (int t = 0; t < 3; t++) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
          const float sk = c[t] + (float)(2 - k);
          const int m = jt[t] - k;  // node of sub-stencil k, 0..2 inside it
          const float wk = m == 0 ? 0.5f * (sk - 1.0f) * (sk - 2.0f) : m == 1 ? -sk * (sk - 2.0f) : 0.5f * sk * (sk - 1.0f);
          const bool in = m >= 0 && m <= 2;
#pragma unroll
          for (int e = 0; e < 3; e++) Sk[e][t][k] = in ? __builtin_fmaf(wk, yz[e][t], Sk[e][t][k]) : Sk[e][t][k];
        }
      }
#pragma unroll
      for (int e = 0; e < 3; e++)
#pragma unroll
        for (int t = 0; t < 3; t++) yz[e][t] = 0.f;
      if (xn > xhi) break;
    }
    xs = xn;
    yr = yn;
  }
  // as in interp_group_weno5c: the basis factors, the sub-stencil sums, the WENO combination
#pragma unroll
  for (int e = 0; e < 3; e++) {
    const float wyz = ((e != 1) ? h : mm) * wz;
#pragma unroll
    for (int t = 0; t < 3; t++) {
      const float wt = (t != 1 ? h : mm) * wyz;
      float ubt[5], S[3];
#pragma unroll
      for (int j = 0; j < 5; j++) ubt[j] = s_ub[(e * 3 + t) * 5 + j][lane] * wt;
#pragma unroll
      for (int k = 0; k < 3; k++) S[k] = Sk[e][t][k] * wt;
      o[3 * e + t] = weno5_combine(c[t], ubt, S);
    }
  }
}

__device__ __forceinline__ void kahan_add(float& s, float& c, float v) {
  const float y = v - c;
  const float t = s + y;
  c = (t - s) - y;
  s = t;
}

// node gauge record of every cell for the node side of the transfer: (ux, uy, uz) and
// sqrt(|T|)*sign(T) in FP32, 16 bytes per cell
// Node gauge records of a D3Q27 split state, and its non-finite node data.  The reference
// transfer drops every term w*g*f that is NaN or infinite (structs.cuh:542), so a node with
// non-finite data adds only its finite terms to an interpolation instead of turning the whole
// neighbourhood NaN.  With a finite gauge (finite basis values) a term is non-finite exactly
// when its population is, and with a non-finite gauge every term of the node is.  So before the
// step reads the state as nodes, a non-finite population is set to zero, and a node with a
// non-finite gauge gets all-zero populations and a zero gauge record (zero gauge: finite basis
// values, so the node adds nothing).  This rewrites the load state, which the step consumes: its
// cells are updated from their own moments (m, T, unchanged here) and the rewritten populations
// are read only as nodes.  FP32 ranges: a population or gauge beyond FP32 range is already
// infinite in the split state.
__global__ void k_node_gauge(float* __restrict__ f, const float* __restrict__ m, const double* __restrict__ T,
                             float* __restrict__ g4, int64_t n, int64_t plane, int* __restrict__ count) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c == 0) *count = 0;  // the step's list of pending cells
  if (c >= n) return;
  const double t = T[c];
  float4 v;
  v.x = m[plane + c];
  v.y = m[2 * plane + c];
  v.z = m[3 * plane + c];
  v.w = (float)(sqrt(fabs(t)) * (double)((0.0 < t) - (t < 0.0)));
  const bool gok = isfinite(v.x) && isfinite(v.y) && isfinite(v.z) && isfinite(v.w);
  float4 q[7];
  bool ok = gok;
#pragma unroll
  for (int j = 0; j < 7; j++) {
    q[j] = reinterpret_cast<const float4*>(f)[j * plane + c];
    ok = ok && isfinite(q[j].x) && isfinite(q[j].y) && isfinite(q[j].z) && (j == 6 || isfinite(q[j].w));
  }
  if (!ok) {
    auto fix = [gok](float x) { return gok && isfinite(x) ? x : 0.0f; };
#pragma unroll
    for (int j = 0; j < 7; j++) {
      float4 r = make_float4(fix(q[j].x), fix(q[j].y), fix(q[j].z), j == 6 ? q[j].w : fix(q[j].w));
      reinterpret_cast<float4*>(f)[j * plane + c] = r;
    }
    if (!gok) v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
  reinterpret_cast<float4*>(g4)[c] = v;
}

// iterations a predicted starting gauge gets to converge before the cell falls back to its
// previous gauge.  Cells that need this many are the ill-conditioned ones (slow contraction at
// contact discontinuities), whose converged state can depend on the starting point.
constexpr int kLearnedBudget = 12;
// SplitArgs::learned_trust: the largest predicted change (in thermal units: du/sqrt(T), dT/T)
// used as a start.  Larger changes sit on shocks and contact layers, where the gauge map can have
// separate fixed points and a start far from the previous gauge may settle on another one than
// the reference reaches.

// Lagrange-4 (propagate<4>, steps.cu:986-1036) for the nine targets that share ez, in one pass
// over the union of their stencil nodes, as interp_pass_weno5c does for WENO5C: the z rows
// (floor(cz)-1 .. +2) are common, the x windows depend on ex only, and the y rows of the three ey
// groups differ by at most a row or two.  Each node of the union is loaded once, its z
// contraction formed once for the three groups; each group whose four rows hold the node
// contracts over y, and each of its targets whose four x slices hold the node adds the node's
// value with its tensor Lagrange weight.  The per-axis basis factors w (1/(2T1) or -1/T1) are
// applied to the finished sums.  MIR: mirror boundaries on the axes of g.mirror (a node beyond
// a mirrored face is the mirror image of the cell inside).  Windows or rows far apart (absurd
// gauges) fall back to interp_lagr4f per target.  The values go to o[3 (ey+1) + ex+1] (LDS).
template <bool MIR>
__device__ __forceinline__ void interp_pass_lagr4(const NodeSrcF& src, int x, int y, int z, double s,
                                                  const double gc[4], int ez, float sqTb, float* o) {
  const Grid& g = src.g;
  const float u1x = (float)gc[0], u1y = (float)gc[1], u1z = (float)gc[2];
  const float u1xl = (float)(gc[0] - (double)u1x), u1yl = (float)(gc[1] - (double)u1y),
              u1zl = (float)(gc[2] - (double)u1z);
  const float T1 = (float)gc[3];
  const float h = 1.0f / (2.0f * T1), mm = -1.0f / T1;
  const float sq1 = sqrtf(fabsf(T1)) * (float)((0.0f < T1) - (T1 < 0.0f));
  const double cz = (double)z - (s * (double)ez + gc[2]);
  const int lz = floor_int(cz) - 1;
  float Fz[4];
  lag4f((float)(cz - lz), Fz);
  const float czb = ez ? (float)ez * sq1 : 0.0f, Tzb = ez ? 0.0f : T1;
  const float wz = ez ? h : mm;
  int ly[3], lx[3];
  float Fy[3][4], Fx[3][4];
  double cxv[3], cyv[3];
#pragma unroll
  for (int e = 0; e < 3; e++) {
    cyv[e] = (double)y - (s * (double)(e - 1) + gc[1]);
    ly[e] = floor_int(cyv[e]) - 1;
    lag4f((float)(cyv[e] - ly[e]), Fy[e]);
    cxv[e] = (double)x - (s * (double)(e - 1) + gc[0]);
    lx[e] = floor_int(cxv[e]) - 1;
    lag4f((float)(cxv[e] - lx[e]), Fx[e]);
  }
  const int xlo = min(lx[0], min(lx[1], lx[2])), xhi = max(lx[0], max(lx[1], lx[2])) + 3;
  const int ylo = min(ly[0], min(ly[1], ly[2])), yhi = max(ly[0], max(ly[1], ly[2])) + 3;
  if ((int64_t)xhi - (int64_t)xlo > 6 || (int64_t)yhi - (int64_t)ylo > 6) {
#pragma unroll 1
    for (int q = 0; q < 9; q++) {
      const int e = q / 3, t = q % 3;
      const int i = kIdx27.v[t][e][ez + 1];
      o[q] = interp_lagr4f<MIR>(src, cxv[t], cyv[e], cz, make_tgtf(i, gc), sqTb);
    }
    return;
  }
  float acc[3][3];
#pragma unroll
  for (int e = 0; e < 3; e++)
#pragma unroll
    for (int t = 0; t < 3; t++) acc[e][t] = 0.f;
  // cell of node (xs, yr, lz + b) = row_cell(xs, yr) + zo[b], its mirror image where it lies beyond a
  // mirrored face (wrapped once per step and per pass, not at every node: 150x101x94 8.52 -> 8.10 ms)
  uint32_t zo[4];
  bool rz[4] = {false, false, false, false};
#pragma unroll
  for (int b = 0; b < 4; b++)
    zo[b] = (uint32_t)(MIR ? mirror_wrap(lz + b, g.nz, (g.mirror & 4) != 0, rz[b]) : wrapi(lz + b, g.nz)) *
            ((uint32_t)g.nx * (uint32_t)g.ny);
  auto row_cell = [&](int xs_, int yr_) -> uint32_t {
    bool rv;
    const int xw = MIR ? mirror_wrap(xs_, g.nx, (g.mirror & 1) != 0, rv) : wrapi(xs_, g.nx);
    const int yw = MIR ? mirror_wrap(yr_, g.ny, (g.mirror & 2) != 0, rv) : wrapi(yr_, g.ny);
    return (uint32_t)xw + (uint32_t)yw * (uint32_t)g.nx;
  };
  // The (slice, row) steps run as one loop whose node loads are one step ahead, as in
  // interp_pass_weno5c: node b of the next step is loaded into the registers of node b of the
  // current step once its contributions are added (unconditionally: the step after the last
  // loads four wrapped, unused nodes).  The arithmetic and its order are those of a plain
  // slice/row loop.
  float fb[4][27];
  Gauge4 nb[4];
#pragma unroll
  for (int b = 0; b < 4; b++) {
    const uint32_t boff = (row_cell(xlo, ylo) + zo[b]) * 4u;
    load27(src.f, boff, fb[b]);
    nb[b] = ldg4(src, boff);
  }
  int xs = xlo, yr = ylo;
#pragma unroll 1
  while (true) {
    bool rx = false, ryf = false;
    if (MIR) {
      mirror_wrap(xs, g.nx, (g.mirror & 1) != 0, rx);
      mirror_wrap(yr, g.ny, (g.mirror & 2) != 0, ryf);
    }
    // the slice's Lagrange weight in each target's four x slices (0 outside), the row's in each
    // group's four rows
    float wx[3], wy[3];
#pragma unroll
    for (int t = 0; t < 3; t++) {
      const int m = xs - lx[t];
      wx[t] = m == 0 ? Fx[t][0] : m == 1 ? Fx[t][1] : m == 2 ? Fx[t][2] : m == 3 ? Fx[t][3] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < 3; e++) {
      const int a = yr - ly[e];
      wy[e] = a == 0 ? Fy[e][0] : a == 1 ? Fy[e][1] : a == 2 ? Fy[e][2] : a == 3 ? Fy[e][3] : 0.f;
    }
    const bool last_row = yr == yhi;
    const int xn = last_row ? xs + 1 : xs, yn = last_row ? ylo : yr + 1;
    const uint32_t on = row_cell(xn, yn);
#pragma unroll
    for (int b = 0; b < 4; b++) {
      const bool rzf = rz[b];
      const float fzb = b == 0 ? Fz[0] : b == 1 ? Fz[1] : b == 2 ? Fz[2] : Fz[3];
      Gauge4 n = nb[b];
      // a node beyond a mirrored face is the mirror image of the cell inside
      // (Cell::mirrX/Y/Z, structs.cuh:552-578): its axis velocity negated, and its populations
      // exchanged with their mirror images, which is the same as reversing that axis's basis
      // values (node_xfer_mirrored)
      if (MIR) {
        n.ux = rx ? -n.ux : n.ux;
        n.uy = ryf ? -n.uy : n.uy;
        n.uz = rzf ? -n.uz : n.uz;
      }
      auto flip = [](bool m, float L[3]) {
        const float a = L[0];
        L[0] = m ? L[2] : L[0];
        L[2] = m ? a : L[2];
      };
      float Lz[3];
      basis3u(((u1z - n.uz) + u1zl) * sqTb, n.sq, czb, Tzb, Lz);
      if (MIR) flip(rzf, Lz);
      float szz[3][3];
#pragma unroll
      for (int ja = 0; ja < 3; ja++)
#pragma unroll
        for (int jb = 0; jb < 3; jb++) {
          float sz = 0.f;
#pragma unroll
          for (int jc = 0; jc < 3; jc++) sz = __builtin_fmaf(Lz[jc], fb[b][kIdx27.v[ja][jb][jc]], sz);
          szz[ja][jb] = sz;
        }
      const float Dy = ((u1y - n.uy) + u1yl) * sqTb;
      const float Dx = ((u1x - n.ux) + u1xl) * sqTb;
      float A0 = Dx + n.sq, A1 = Dx, A2 = Dx - n.sq;
      if (MIR) {
        const float a = A0;
        A0 = rx ? A2 : A0;
        A2 = rx ? a : A2;
      }
      // x moments of the z sums, common to the three groups (as in interp_pass_weno5c)
      const float B0 = A0 * A0, B1 = A1 * A1, B2 = A2 * A2;
      float xr[3], xq[3], xp[3];
#pragma unroll
      for (int jb = 0; jb < 3; jb++) {
        xr[jb] = (szz[0][jb] + szz[1][jb]) + szz[2][jb];
        xq[jb] = __builtin_fmaf(A2, szz[2][jb], __builtin_fmaf(A1, szz[1][jb], A0 * szz[0][jb]));
        xp[jb] = __builtin_fmaf(B2, szz[2][jb], __builtin_fmaf(B1, szz[1][jb], B0 * szz[0][jb]));
      }
#pragma unroll
      for (int e = 0; e < 3; e++) {
        if (wy[e] == 0.f) continue;
        const int ey = e - 1;
        float Ly[3];
        basis3u(Dy, n.sq, ey ? (float)ey * sq1 : 0.0f, ey ? 0.0f : T1, Ly);
        if (MIR) flip(ryf, Ly);
        const float R = __builtin_fmaf(Ly[2], xr[2], __builtin_fmaf(Ly[1], xr[1], Ly[0] * xr[0]));
        const float Q = __builtin_fmaf(Ly[2], xq[2], __builtin_fmaf(Ly[1], xq[1], Ly[0] * xq[0]));
        const float Pp = __builtin_fmaf(Ly[2], xp[2], __builtin_fmaf(Ly[1], xp[1], Ly[0] * xp[0]));
        const float Tt[3] = {__builtin_fmaf(sq1, Q, Pp), __builtin_fmaf(-T1, R, Pp), __builtin_fmaf(-sq1, Q, Pp)};
        const float wyz = wy[e] * fzb;
#pragma unroll
        for (int t = 0; t < 3; t++) acc[e][t] = __builtin_fmaf(wx[t] * wyz, Tt[t], acc[e][t]);
      }
      // node b of this step is used up: load node b of the next step in its place
      const uint32_t boff = (on + zo[b]) * 4u;
      load27(src.f, boff, fb[b]);
      nb[b] = ldg4(src, boff);
    }
    if (last_row && xn > xhi) break;
    xs = xn;
    yr = yn;
  }
#pragma unroll
  for (int e = 0; e < 3; e++) {
    const float wyz = ((e != 1) ? h : mm) * wz;
#pragma unroll
    for (int t = 0; t < 3; t++)
      o[3 * e + t] = acc[e][t] * ((t != 1 ? h : mm) * wyz);
  }
}

// Iteration state of one cell, carried from the first pass to the second.
struct SplitIter {
  double gc[4];      // current gauge (u, T)
  double res_prev;   // residual of the previous iteration
  double rho;        // density of the last iterate
  int niter;         // iterations so far, reported
  int base;          // iterations spent on a predicted start that was abandoned
  bool learned;      // started from the predicted gauge and not yet fallen back
  bool contracted;   // a residual has fallen since the current start
};

// previous gauge of the cell (the plain start); an all-zero cell is reset as in steps.cu:360-363
__device__ __forceinline__ void split_prev_gauge(const float* __restrict__ min, const double* __restrict__ Tin,
                                                 int64_t P, int64_t cell, double tlat, double gp[4], double& rho0) {
  rho0 = min[cell];
  gp[0] = min[P + cell]; gp[1] = min[2 * P + cell]; gp[2] = min[3 * P + cell]; gp[3] = Tin[cell];
  if (rho0 == 0 && gp[0] == 0 && gp[1] == 0 && gp[2] == 0 && gp[3] == 0) { rho0 = 1; gp[3] = tlat; }
}

// moments in the frame of the current gauge: A = sum f, B = sum f xi (compensated, FP32) and
// C = sum f |xi|^2 (FP64)
struct SplitSums {
  float as = 0.f, ac = 0.f, bxs = 0.f, bxc = 0.f, bys = 0.f, byc = 0.f, bzs = 0.f, bzc = 0.f;
  double cs = 0.0;
  __device__ __forceinline__ void add(int ex, int ey, int ez, float fn) {
    kahan_add(as, ac, fn);
    kahan_add(bxs, bxc, (float)ex * fn);
    kahan_add(bys, byc, (float)ey * fn);
    kahan_add(bzs, bzc, (float)ez * fn);
    cs += (double)fn * (double)(ex * ex + ey * ey + ez * ez);
  }
};

// The end of one fixed-point iteration of one cell, from the sums over its new populations (s: the
// lattice scale of the gauge they were formed in): true when it has converged.
__device__ __forceinline__ bool split27_update(const SplitSums& q, double s, int64_t cell,
                                               const float* __restrict__ min, const double* __restrict__ Tin,
                                               SplitIter& st, const SplitArgs& a) {
  const int64_t P = a.g.plane;
  double* gc = st.gc;
  st.niter++;
  {
    // FP64 moment solve (Cell::calcMoments, structs.cuh:315-342) restated in the gauge frame:
    // with v = u_g + s xi, sum f v / rho = u_g + s B/rho and
    // (sum f |v|^2/rho - |u|^2)/Dim = s^2 (C - |B|^2/rho) / (rho Dim).  This is the same
    // algebra without the cancellation of |u|^2 against sum f |v|^2 / rho, which at Mach 1
    // and above would amplify the FP32 rounding of the populations several times.
    const double rho = (double)q.as - (double)q.ac;
    const double cs = q.cs;
    st.rho = rho;
    const double B[3] = {(double)q.bxs - (double)q.bxc, (double)q.bys - (double)q.byc, (double)q.bzs - (double)q.bzc};
    double m[4];
    if (rho != 0) {
      const double ir = 1.0 / rho;
      for (int k = 0; k < 3; k++) m[k] = gc[k] + s * (B[k] * ir);
      m[3] = s * s * (cs - (B[0] * B[0] + B[1] * B[1] + B[2] * B[2]) * ir) * ir * a.inv_dim;
    } else {  // no division by rho (structs.cuh:329): u = sum f v, T = (sum f |v|^2 - |u|^2)/Dim
      for (int k = 0; k < 3; k++) m[k] = s * B[k];
      m[3] = (2.0 * s * (gc[0] * B[0] + gc[1] * B[1] + gc[2] * B[2]) + s * s * cs - (m[0] * m[0] + m[1] * m[1] + m[2] * m[2])) *
             a.inv_dim;
    }
    if (m[3] < 0) m[3] = gc[3];
    // FP64 gauge residual, scaled by the thermal speed and the temperature
    const double sth = sqrt(fabs(m[3]));
    double res = 0;
    bool conv = true;
    for (int k = 0; k < 4; k++) {
      const double scale = k < 3 ? sth : fabs(m[3]);
      const double d = fabs(m[k] - gc[k]);
      // a NaN difference counts as converged, as in the reference's test (steps.cu:58-75,
      // which fails only on difference >= tolerance), so a cell with non-finite data stops at once
      if (d > a.tol_rel * scale + a.tol_abs) conv = false;
      const double rk = d / (scale + 1e-300);
      if (res == res && !(rk <= res)) res = rk;  // NaN propagates (fmax would drop it)
    }
    // FP32 populations leave a noise floor near the tolerance (interpolation rounding of a few
    // 1e-7 per population): a residual below 4 tol that has stopped falling has reached it.  A
    // residual that still falls, however slowly, keeps iterating down to tol.
    // (A predicted start must first show a falling residual: one that lands in the noise band
    // at once may sit next to a fixed point the previous-gauge start does not reach.)
    if (!conv && st.niter - st.base > 1 && res <= 4.0 * a.tol_rel && res >= st.res_prev &&
        (!st.learned || st.contracted))
      conv = true;
    if (st.niter - st.base > 1 && res < st.res_prev) st.contracted = true;
    // (a NaN iterate from a predicted start is not accepted: the cell falls back)
    if (conv && !(st.learned && res != res)) {
      for (int k = 0; k < 4; k++) gc[k] = m[k];
      return true;
    }
    if (st.learned && (res != res || (st.niter > 1 && !(res < st.res_prev)) || st.niter == kLearnedBudget)) {
      // the predicted start does not contract (or not within the budget): restart from the
      // previous gauge (read again from the step's input, which the step does not write, so
      // no lane carries it through its iterations), so the cell ends where the plain method
      // ends
      double gp[4], rho0;
      split_prev_gauge(min, Tin, P, cell, a.tlat, gp, rho0);
      for (int k = 0; k < 4; k++) gc[k] = gp[k];
      st.learned = false;
      st.contracted = false;
      st.res_prev = 0;
      st.base = st.niter;
      return false;
    }
    st.res_prev = res;
    for (int k = 0; k < 4; k++) gc[k] = m[k];
  }
  return false;
}

// One iteration of one cell with the WENO5 as written, target by target; the iterate's populations are
// left in fout.
__device__ __forceinline__ bool split27_once(const NodeSrcF& src, float* __restrict__ fout, int64_t cell, int x,
                                             int y, int z, const float* __restrict__ min,
                                             const double* __restrict__ Tin, SplitIter& st, const SplitArgs& a) {
  const float sqTb = (float)a.sqrt_tbase;
  const double* gc = st.gc;
  const double s = sqrt(gc[3] / a.tlat);
  SplitSums sums;
  for (int i = 0; i < 27; i++) {
    const int ex = kE27[i][0], ey = kE27[i][1], ez = kE27[i][2];
    const double vx = s * (double)ex + gc[0];
    const double vy = s * (double)ey + gc[1];
    const double vz = s * (double)ez + gc[2];
    const TgtF t = make_tgtf(i, gc);
    const double cx = (double)x - vx, cy = (double)y - vy, cz = (double)z - vz;
    const float fn = interp_weno5f<false>(src, cx, cy, cz, t, sqTb);
    fout[split27_fidx(i, cell, a.g.plane)] = fn;
    sums.add(ex, ey, ez, fn);
  }
  return split27_update(sums, s, cell, min, Tin, st, a);
}

// Fixed-point iterations of one cell from state st until it converges (true), its count
// reaches stop_at, or its count since its current start reaches the cap (false).  A cell that
// abandons a predicted start gets the full cap from its previous gauge, so a cell that does
// not converge ends on the same iterate as without the prediction.  The iterate's populations
// are left in fout.
__device__ bool split27_iterate(const NodeSrcF& src, float* __restrict__ fout, int64_t cell, int x, int y, int z,
                                const float* __restrict__ min, const double* __restrict__ Tin, SplitIter& st,
                                int stop_at, const SplitArgs& a) {
  while (st.niter < stop_at && st.niter - st.base < a.max_iter)
    if (split27_once(src, fout, cell, x, y, z, min, Tin, st, a)) return true;
  return false;
}

// BGK in FP32 (steps.cu:557-564) on the iterate left in fout, and the cell's outputs
__device__ __forceinline__ void split27_finish(float* __restrict__ fout, float* __restrict__ mout,
                                               double* __restrict__ Tout, int* __restrict__ niter_out, int64_t cell,
                                               const SplitIter& st, const SplitArgs& a) {
  const int64_t P = a.g.plane;
  const float rf = (float)st.rho, dt = (float)a.dtau;
  for (int i = 0; i < 27; i++) {
    const int64_t o = split27_fidx(i, cell, P);
    float f = fout[o];
    f = __builtin_fmaf(dt, rf * a.w[i] - f, f);
    fout[o] = f;
  }
  mout[cell] = rf;
  mout[P + cell] = (float)st.gc[0];
  mout[2 * P + cell] = (float)st.gc[1];
  mout[3 * P + cell] = (float)st.gc[2];
  Tout[cell] = st.gc[3];
  niter_out[cell] = st.niter;
}

// A predicted start is taken only in cells whose previous step took kLearnedPrevMin ..
// kLearnedPrevMax iterations (step_split.h).  Where the gauge map contracts slowly (cells that
// needed more, on shocks and contact layers) it can have a second fixed point near the first,
// and a start from elsewhere may settle there: on the 384^3 shock-bubble, one step from the same
// FP64 state, ungated predicted starts left 13-189 cells per step 1e-4 to 2e-3 (relative, u and
// T) away from the FP64 step, all in cells whose FP64 step needed 9-10 iterations; with an upper
// bound of 8 previous iterations 76-78 cells were still up to 1.7e-3 off; with 4 or 6 every cell
// stayed within the plain start's 2e-7.  On the 64^3 shock-bubble (sharper fronts per cell) an
// upper bound of 6 left cells 5.8e-5 off at step 12, and 4 kept every cell within 3e-7 through
// step 12.  Below: a cell that took one or two iterations gains
// nothing (a prediction lands within the 1e-7 tolerance of the fixed point only by chance, so
// such a cell takes as many iterations from it; windows from 1, 2 or 3 gave the same counts).

// Starting state of a cell: its previous gauge, or the predicted one where a prediction is
// given, finite, not all zero, has T > 0, lies within the trust radius and the cell's previous
// step took kLearnedPrevMin .. kLearnedPrevMax iterations (niter_prev: the counts of the previous step,
// which this step overwrites cell by cell after reading).
__device__ __forceinline__ void split27_start(const float* __restrict__ min, const double* __restrict__ Tin,
                                              const float* __restrict__ guess, const int* __restrict__ niter_prev,
                                              int64_t cell, SplitIter& st, const SplitArgs& a) {
  const int64_t P = a.g.plane;
  double gp[4], rho0;
  split_prev_gauge(min, Tin, P, cell, a.tlat, gp, rho0);
  for (int k = 0; k < 4; k++) st.gc[k] = gp[k];
  st.res_prev = 0;
  st.rho = rho0;
  st.niter = 0;
  st.base = 0;
  st.learned = false;
  st.contracted = false;
  // (the previous count is tested first, so the prediction is read only where it may be taken)
  if (guess && niter_prev[cell] >= kLearnedPrevMin && niter_prev[cell] <= kLearnedPrevMax) {
    // decode the predicted increment: (du/sqrt(T), dT/T) relative to the previous gauge
    const double sq = sqrt(gp[3]);
    const float p0 = guess[cell], p1 = guess[P + cell], p2 = guess[2 * P + cell], p3 = guess[3 * P + cell];
    const double q[4] = {gp[0] + sq * p0, gp[1] + sq * p1, gp[2] + sq * p2, gp[3] * (1.0 + (double)p3)};
    const float pmax = fmaxf(fmaxf(fabsf(p0), fabsf(p1)), fmaxf(fabsf(p2), fabsf(p3)));
    // (a prediction of no change at all is the previous-gauge start, with its stopping rules)
    if (isfinite(q[0]) && isfinite(q[1]) && isfinite(q[2]) && isfinite(q[3]) && q[3] > 0 && pmax <= a.learned_trust &&
        pmax > 0.0f) {
      for (int k = 0; k < 4; k++) st.gc[k] = q[k];
      st.learned = true;
    }
  }
}

// The WENO5 as written (unstable in 3D; kept for parity runs): one lane per cell.  First pass: every
// cell iterates up to a.pass1_iters times.  A wave runs as long as its slowest cell, and on contact
// discontinuities and shocks a thin layer of cells needs several times the mean, so cells still
// unconverged after the first pass are appended to a list (wave-aggregated: one atomic per wave) and
// finished by k_step_split27_rest, whose waves hold only such cells.  Each cell's arithmetic is the
// same as in a single pass.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_step_split27_written(
    const float* __restrict__ fin, const float* __restrict__ min, const double* __restrict__ Tin,
    const float* __restrict__ g4in, float* __restrict__ fout, float* __restrict__ mout, double* __restrict__ Tout,
    int* __restrict__ niter_out, const float* __restrict__ guess, SplitPending pend, const SplitArgs a) {
  const Grid& g = a.g;
  int x, y, z;
  const bool live = tile_cell(g, xcd_block(blockIdx.x, gridDim.x), threadIdx.x, x, y, z);
  bool pending = false;
  SplitIter st;
  const int64_t cell = live ? cell_index(g, x, y, z) : 0;
  if (live) {
    split27_start(min, Tin, guess, niter_out, cell, st, a);
    const NodeSrcF src = make_src(fin, g4in, g);
    const bool conv = split27_iterate(src, fout, cell, x, y, z, min, Tin, st, a.pass1_iters, a);
    pending = !conv && st.niter - st.base < a.max_iter;
    if (!pending) split27_finish(fout, mout, Tout, niter_out, cell, st, a);
  }
  // append the pending cells of this wave to the list
  bool any;
  const int64_t e = pending_slot(pend, pending, any);
  if (pending) {
    pend.cell[e] = (int)cell;
    for (int k = 0; k < 4; k++) pend.g[k * pend.cap + e] = st.gc[k];
    pend.res[e] = st.res_prev;
    pend.meta[e] = st.niter | (st.base << 8) | (st.learned ? 0x10000 : 0) | (st.contracted ? 0x20000 : 0);
  }
}

// Second pass: a fixed grid of waves walks the pending list; every cell resumes its iteration
// where the first pass left it.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_step_split27_rest(
    const float* __restrict__ fin, const float* __restrict__ min, const double* __restrict__ Tin,
    const float* __restrict__ g4in, float* __restrict__ fout, float* __restrict__ mout, double* __restrict__ Tout,
    int* __restrict__ niter_out, SplitPending pend, const SplitArgs a) {
  const Grid& g = a.g;
  const int count = *pend.count;
  const NodeSrcF src = make_src(fin, g4in, g);
  for (int64_t e = (int64_t)blockIdx.x * 64 + threadIdx.x; e - threadIdx.x < count; e += (int64_t)gridDim.x * 64) {
    if (e >= count) continue;
    const int64_t cell = pend.cell[e];
    const int x = (int)(cell % g.nx);
    const int y = (int)((cell / g.nx) % g.ny);
    const int z = (int)(cell / ((int64_t)g.nx * g.ny));
    double gp[4], rho0;
    split_prev_gauge(min, Tin, g.plane, cell, a.tlat, gp, rho0);
    SplitIter st;
    for (int k = 0; k < 4; k++) st.gc[k] = pend.g[k * pend.cap + e];
    st.res_prev = pend.res[e];
    st.rho = rho0;
    const int meta = pend.meta[e];
    st.niter = meta & 0xff;
    st.base = (meta >> 8) & 0xff;
    st.learned = (meta & 0x10000) != 0;
    st.contracted = (meta & 0x20000) != 0;
    split27_iterate(src, fout, cell, x, y, z, min, Tin, st, 0x7fffffff, a);
    split27_finish(fout, mout, Tout, niter_out, cell, st, a);
  }
}

// A cell late in its iterations goes to k_step_split27_wide where its wave has no cell left to start and no
// more than this many slots (of 21) with such cells; see launch_step_split.
constexpr int kWideSlots = 5;

// WENO5C and Lagrange-4 (INTERP 2, 1; 3: Lagrange-4 with mirror walls): three lanes per cell, lane =
// ez pass of nine targets, 21 cells per wave.
//
// With one lane per cell (its three passes one after the other) a wave spanned 64 cells: a third of
// its lane-iterations went to row ends waiting for the last slow cells, each pass fetched the same
// neighbourhood again, and a cell at the cap of 100 iterations took 17 ms by itself.  Side by side,
// the passes of a cell share their node loads (the lanes ask for the same cache lines wherever their z
// rows coincide), the iterate stays in LDS instead of going through global memory, and a slot takes the
// next cell of the wave's run when its own has converged.  Each cell's arithmetic and its order are the
// same (bit for bit).  Per step, before and after: 256^3 vortex 65.3 -> 39.6 ms, 256^3 shock-bubble
// 107 -> 69.7 ms, 32^3 shock-bubble 16.9 -> 5.6 ms; Lagrange-4 192^3 Taylor-Green 81 -> 37.5 ms,
// 150x101x94 22.0 -> 8.1 ms.  Bound by VALU issue: 256^3 vortex busy 86 % (57 of 64 lanes; texture-address
// unit 73 %), 150x101x94 90 % (44 lanes: windows and rows that differ between the cells of a wave).
// Two waves per SIMD (256 registers): with more registers the load latency would be left unhidden.
template <int INTERP>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_step_split27_cells(
    const float* __restrict__ fin, const float* __restrict__ min, const double* __restrict__ Tin,
    const float* __restrict__ g4in, float* __restrict__ fout, float* __restrict__ mout, double* __restrict__ Tout,
    int* __restrict__ niter_out, const float* __restrict__ guess, int* __restrict__ slow, const SplitArgs a, int cells,
    int wide_after, int few) {
  constexpr int FS = 28;
  __shared__ __align__(16) float s_f[22][FS];  // the iterate's populations, [cell][9 (ez+1) + 3 (ey+1) + ex+1]
  __shared__ float s_w[FS];
  const Grid& g = a.g;
  const int64_t P = g.plane;
  const int lane = threadIdx.x;
  // Lanes of a cell (lane 63 has none).  A 16-byte load takes four neighbouring lanes at a time, so
  // these should want one cache line.  Lagrange-4: a pass's 21 cells side by side, as its passes' rows
  // mostly differ (floor(z) moves with ez): with a cell's passes side by side, 192^3 took 37.3 instead of
  // 29.3 ms per step, the 128^3 shock-bubble 15.3 instead of 12.6 ms.  WENO5C: twelve lanes per four cells
  // (two cells by two passes, the third pass of all four, the other two by two), as its passes' rows
  // coincide below half a cell of thermal speed and differ above (against a cell's passes side by side:
  // 256^3 shock-bubble 70.2 -> 67.0 ms, vortex 40.1 -> 40.4 ms; as Lagrange-4: 66.7 and 41.3 ms).
  constexpr bool BLOCKS = INTERP == 2;
  const int l12 = lane % 12;
  const int slot = BLOCKS ? (lane < 60 ? 4 * (lane / 12) + (int)((0xeee444u >> (2 * l12)) & 3) : lane < 63 ? 20 : 21)
                          : (lane < 63 ? lane % 21 : 21);
  const int pz = BLOCKS ? (lane < 60 ? (int)((0x50aa50u >> (2 * l12)) & 3) : (lane - 60) % 3) : lane < 63 ? lane / 21 : 0;
  // the slot's lane of the first pass
  const int head = BLOCKS ? (slot < 20 ? 12 * (slot / 4) + (slot & 1) + 4 * (slot & 2) : 60) : slot;
  constexpr uint64_t kHeads = BLOCKS ? 0x1303303303303303ull : 0x1fffffull;
  if (lane < FS) s_w[lane] = lane < 27 ? a.w[lane] : 0.f;
  const int64_t q0 = xcd_block(blockIdx.x, gridDim.x) * cells;
  const int64_t total = g.ntiles * 64 - q0 < cells ? g.ntiles * 64 - q0 : cells;  // cell slots of the wave
  const NodeSrcF src = make_src(fin, g4in, g);
  int64_t next = 0;  // first unstarted slot (the same in every lane)
  bool active = false;
  int64_t cell = 0;
  int x = 0, y = 0, z = 0;
  SplitIter st;
  while (true) {
    if constexpr (INTERP == 2) {
      const bool late = active && st.niter >= wide_after;
      const bool idle = next >= total && __popcll(__ballot(late) & kHeads) <= kWideSlots;
      if (late) {
        int e = -1;  // the cell's place in the list of k_step_split27_wide
        if (pz == 0) e = slow_place(slow, idle, few);
        e = __shfl(e, head, 64);
        if (e >= 0) {
          // its state goes with it in three of the cell's output quads (arguments for separate arrays
          // cost the pass scratch registers: 39.7 -> 49.8 ms on the 256^3 vortex)
          active = false;
          const int64_t meta =
              st.niter | ((int64_t)st.base << 32) | (st.learned ? 1ll << 48 : 0) | (st.contracted ? 1ll << 49 : 0);
          reinterpret_cast<double2*>(fout)[pz * P + cell] =
              make_double2(pz == 0 ? st.gc[0] : pz == 1 ? st.gc[2] : st.res_prev,
                           pz == 0 ? st.gc[1] : pz == 1 ? st.gc[3] : __longlong_as_double(meta));
          if (pz == 0) slow[kSlowList + e] = (int)cell;
        }
      }
    }
    const uint64_t want = __ballot(!active) & kHeads;
    if (!active && slot < 21) {
      const int64_t q = next + __popcll(want & ((1ull << head) - 1ull));
      // (a slot outside the grid, in a ragged last tile, is used up without a cell)
      if (q < total && tile_cell(g, (q0 + q) / 64, (int)((q0 + q) % 64), x, y, z)) {
        cell = cell_index(g, x, y, z);
        split27_start(min, Tin, guess, niter_out, cell, st, a);
        active = true;
      }
    }
    next += __popcll(want);
    if (__ballot(active) == 0 && next >= total) break;
    double s = 0;
    if (active) {
      s = sqrt(st.gc[3] / a.tlat);
      float* o = &s_f[slot][9 * pz];
      if constexpr (INTERP == 2) interp_pass_weno5c(src, x, y, z, s, st.gc, pz - 1, (float)a.sqrt_tbase, o);
      else interp_pass_lagr4<INTERP == 3>(src, x, y, z, s, st.gc, pz - 1, (float)a.sqrt_tbase, o);
    }
    wave_lds_order();
    if (active) {
      // the cell's sums in the order (ey, ez, ex), in each of its lanes
      float f[FS];
#pragma unroll
      for (int q = 0; q < 7; q++) {
        const float4 v = *reinterpret_cast<const float4*>(&s_f[slot][4 * q]);
        f[4 * q] = v.x; f[4 * q + 1] = v.y; f[4 * q + 2] = v.z; f[4 * q + 3] = v.w;
      }
      SplitSums sums;
#pragma unroll
      for (int ey = 0; ey < 3; ey++)
#pragma unroll
        for (int ez = 0; ez < 3; ez++)
#pragma unroll
          for (int ex = 0; ex < 3; ex++) sums.add(ex - 1, ey - 1, ez - 1, f[9 * ez + 3 * ey + ex]);
      if (split27_update(sums, s, cell, min, Tin, st, a) || st.niter - st.base >= a.max_iter) {
        // BGK in FP32 (steps.cu:557-564) and the cell's outputs: quad planes pz, pz + 3, pz + 6
        active = false;
        const float rf = (float)st.rho, dt = (float)a.dtau;
#pragma unroll
        for (int q = 0; q < 7; q++) {
          if (q % 3 != pz) continue;
          float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const int i = 4 * q + e;
            if (i < 27) {
              const float fi = f[9 * (kE27[i][2] + 1) + 3 * (kE27[i][1] + 1) + kE27[i][0] + 1];
              v[e] = __builtin_fmaf(dt, rf * s_w[i] - fi, fi);
            }
          }
          reinterpret_cast<float4*>(fout)[q * P + cell] = make_float4(v[0], v[1], v[2], v[3]);
        }
        if (pz == 0) {
          mout[cell] = rf;
          mout[P + cell] = (float)st.gc[0];
        } else if (pz == 1) {
          mout[2 * P + cell] = (float)st.gc[1];
          mout[3 * P + cell] = (float)st.gc[2];
        } else {
          Tout[cell] = st.gc[3];
          niter_out[cell] = st.niter;
        }
      }
    }
    wave_lds_order();
  }
}

// The WENO5C cells that k_step_split27_cells left unconverged: one workgroup per cell.
//
// A few cells on shocks and contacts go on to the cap of 100 iterations.  Three lanes take 50 us for such
// an iteration (63 chained steps of three nodes), so on grids up to 128^3 they held up the whole step.
// Here the nodes of the three passes are spread over the threads (189 for a seven-slice window on
// three rows), their values for the targets laid down in LDS, and the sums over them run target
// by target in the pass's order, so every value is the one the pass gives.  6.5 us per iteration, bound by the
// chain of its six dependent parts (8.5 us with one wave per cell and three nodes per lane).
// Shock-bubble, ms per step before and after: 32^3 5.6 -> 1.0, 64^3 6.7 -> 2.5, 128^3 14.5 -> 11.6.
//
// Every thread of the group forms the same sums and the same gauge from LDS, so the group leaves its
// loop together and each barrier is met by all.
constexpr int kWideThreads = 256;
__global__ __launch_bounds__(kWideThreads) void k_step_split27_wide(
    const float* __restrict__ fin, const float* __restrict__ min, const double* __restrict__ Tin,
    const float* __restrict__ g4in, float* __restrict__ fout, float* __restrict__ mout, double* __restrict__ Tout,
    int* __restrict__ niter_out, const int* __restrict__ slow, const SplitArgs a) {
  constexpr int MS = 9, MR = 5;             // most slices and rows of a pass
  __shared__ float s_T[3 * MS * MR * 3][9];  // a node's values for the targets 3 e + t
  __shared__ float s_yz[27][MS];            // y/z sums of a target's slices
  __shared__ float s_f[28];                 // the iterate, [9 (ez+1) + 3 (ey+1) + ex+1]
  __shared__ float s_Fy[9], s_Fz[9];
  const Grid& g = a.g;
  const int64_t P = g.plane;
  const int lane = threadIdx.x;
  const NodeSrcF src = make_src(fin, g4in, g);
  const float sqTb = (float)a.sqrt_tbase;
  const int count = *slow;
  for (int64_t e0 = blockIdx.x; e0 < count; e0 += gridDim.x) {
    const int64_t cell = slow[kSlowList + e0];
    const int x = (int)(cell % g.nx);
    const int y = (int)((cell / g.nx) % g.ny);
    const int z = (int)(cell / ((int64_t)g.nx * g.ny));
    const double2* so = reinterpret_cast<const double2*>(fout) + cell;
    const double2 g01 = so[0], g23 = so[P], rm = so[2 * P];
    const int64_t meta = __double_as_longlong(rm.y);
    SplitIter st;
    st.gc[0] = g01.x;
    st.gc[1] = g01.y;
    st.gc[2] = g23.x;
    st.gc[3] = g23.y;
    st.res_prev = rm.x;
    st.rho = 0;
    st.niter = (int)(meta & 0x7fffffff);
    st.base = (int)((meta >> 32) & 0xffff);  // (at most kLearnedBudget)
    st.learned = (meta >> 48) & 1;
    st.contracted = (meta >> 49) & 1;
    bool conv = false;
    while (!conv && st.niter - st.base < a.max_iter) {
      const double* gc = st.gc;
      const double s = sqrt(gc[3] / a.tlat);
      // the pass's constants (interp_pass_weno5c)
      const float u1x = (float)gc[0], u1y = (float)gc[1], u1z = (float)gc[2];
      const float u1xl = (float)(gc[0] - (double)u1x), u1yl = (float)(gc[1] - (double)u1y),
                  u1zl = (float)(gc[2] - (double)u1z);
      const float T1 = (float)gc[3];
      const float h = 1.0f / (2.0f * T1), mm = -1.0f / T1;
      const float sq1 = sqrtf(fabsf(T1)) * (float)((0.0f < T1) - (T1 < 0.0f));
      int rz[3], ry[3], r[3];
      float c[3];
#pragma unroll
      for (int q = 0; q < 3; q++) {
        const double cz = (double)z - (s * (double)(q - 1) + gc[2]), cy = (double)y - (s * (double)(q - 1) + gc[1]);
        const double cx = (double)x - (s * (double)(q - 1) + gc[0]);
        rz[q] = floor_int(cz + 0.5) - 1;
        ry[q] = floor_int(cy + 0.5) - 1;
        r[q] = floor_int(cx + 0.5);
        c[q] = (float)(cx - r[q]);
        float Fz[3], Fy[3];
        lag3f((float)(cz - rz[q]), Fz);
        lag3f((float)(cy - ry[q]), Fy);
        if (lane == 0) {
#pragma unroll
          for (int m = 0; m < 3; m++) { s_Fz[3 * q + m] = Fz[m]; s_Fy[3 * q + m] = Fy[m]; }
        }
      }
      const int xlo = min3(r[0], r[1], r[2]) - 2, xhi = max3(r[0], r[1], r[2]) + 2;
      const int ylo = min3(ry[0], ry[1], ry[2]), yhi = max3(ry[0], ry[1], ry[2]) + 2;
      __syncthreads();
      if ((int64_t)xhi - (int64_t)xlo > MS - 1 || (int64_t)yhi - (int64_t)ylo > MR - 1) {
        if (lane < 9) {
          float f3[3];
          interp_group_weno5c(src, x, y, z, s, gc, lane % 3 - 1, lane / 3 - 1, sqTb, f3);
#pragma unroll
          for (int t = 0; t < 3; t++) s_f[3 * lane + t] = f3[t];
        }
      } else {
        const int nsl = xhi - xlo + 1, nrw = yhi - ylo + 1;
        for (int it = lane; it < 9 * nsl * nrw; it += kWideThreads) {
          const int st3 = it / 3, b = it - 3 * st3, sl3 = st3 / nrw, rw = st3 - nrw * sl3;
          const int ez = (sl3 >= nsl) + (sl3 >= 2 * nsl), sl = sl3 - nsl * ez;
          const int rzi = ez == 0 ? rz[0] : ez == 1 ? rz[1] : rz[2];
          const uint32_t off = ((uint32_t)wrapi(xlo + sl, g.nx) + (uint32_t)wrapi(ylo + rw, g.ny) * (uint32_t)g.nx +
                                (uint32_t)wrapi(rzi + b, g.nz) * ((uint32_t)g.nx * (uint32_t)g.ny)) * 4u;
          float f[27];
          load27(src.f, off, f);
          const float czb = ez != 1 ? (float)(ez - 1) * sq1 : 0.0f, Tzb = ez != 1 ? 0.0f : T1;
          const NodePass np = node_pass(f, ldg4(src, off), u1x, u1xl, u1y, u1yl, u1z, u1zl, sqTb, czb, Tzb);
#pragma unroll
          for (int e = 0; e < 3; e++) {
            float Tt[3];
            node_group(np, e - 1, sq1, T1, Tt);
#pragma unroll
            for (int t = 0; t < 3; t++) s_T[it][3 * e + t] = Tt[t];
          }
        }
        __syncthreads();
        // y/z sums of every target's slices
        for (int ch = lane; ch < 27 * nsl; ch += kWideThreads) {
          const int sl = ch / 27, tg = ch - 27 * sl, ez = tg / 9, et = tg - 9 * ez, e = et / 3;
          const int rye = e == 0 ? ry[0] : e == 1 ? ry[1] : ry[2];
          float yz = 0.f;
          for (int aa = 0; aa < 3; aa++) {  // the group's three rows
            const int it = (ez * nsl + sl) * nrw + (rye + aa - ylo);
#pragma unroll
            for (int b = 0; b < 3; b++) {
              const float wab = s_Fy[3 * e + aa] * s_Fz[3 * ez + b];
              yz = __builtin_fmaf(wab, s_T[3 * it + b][et], yz);
            }
          }
          s_yz[tg][sl] = yz;
        }
        __syncthreads();
        // sub-stencil sums, smoothness samples and the WENO combination, one lane per target
        if (lane < 27) {
          const int ez = lane / 9, et = lane - 9 * ez, e = et / 3, t = et - 3 * e;
          const int rt = t == 0 ? r[0] : t == 1 ? r[1] : r[2], rye = e == 0 ? ry[0] : e == 1 ? ry[1] : ry[2];
          const float ct = t == 0 ? c[0] : t == 1 ? c[1] : c[2];
          const float wz = ez != 1 ? h : mm;
          const float wyz = ((e != 1) ? h : mm) * wz;
          const float wt = (t != 1 ? h : mm) * wyz;
          const int sl0 = (rt - 2) - xlo;  // the window's first slice
          float S[3], ub[5];
#pragma unroll
          for (int k = 0; k < 3; k++) {
            const float sk = ct + (float)(2 - k);
            const float w0 = 0.5f * (sk - 1.0f) * (sk - 2.0f), w1 = -sk * (sk - 2.0f), w2 = 0.5f * sk * (sk - 1.0f);
            float v = 0.f;
            v = __builtin_fmaf(w0, s_yz[lane][sl0 + k], v);
            v = __builtin_fmaf(w1, s_yz[lane][sl0 + k + 1], v);
            v = __builtin_fmaf(w2, s_yz[lane][sl0 + k + 2], v);
            S[k] = v * wt;
          }
#pragma unroll
          for (int j = 0; j < 5; j++) ub[j] = s_T[3 * ((ez * nsl + sl0 + j) * nrw + (rye + 1 - ylo)) + 1][et] * wt;
          s_f[lane] = weno5_combine(ct, ub, S);
        }
      }
      __syncthreads();
      SplitSums sums;
#pragma unroll
      for (int ey = 0; ey < 3; ey++)
#pragma unroll
        for (int ez = 0; ez < 3; ez++)
#pragma unroll
          for (int ex = 0; ex < 3; ex++) sums.add(ex - 1, ey - 1, ez - 1, s_f[9 * ez + 3 * ey + ex]);
      conv = split27_update(sums, s, cell, min, Tin, st, a);
    }
    // BGK in FP32 (steps.cu:557-564) and the cell's outputs
    const float rf = (float)st.rho, dt = (float)a.dtau;
    if (lane < 27) {
      const int ex = kE27[lane][0], ey = kE27[lane][1], ez = kE27[lane][2];
      const float fi = s_f[9 * (ez + 1) + 3 * (ey + 1) + ex + 1];
      fout[split27_fidx(lane, cell, P)] = __builtin_fmaf(dt, rf * a.w[lane] - fi, fi);
    }
    if (lane < 4) mout[lane * P + cell] = lane == 0 ? rf : (float)(lane == 1 ? st.gc[0] : lane == 2 ? st.gc[1] : st.gc[2]);
    if (lane == 4) Tout[cell] = st.gc[3];
    if (lane == 5) niter_out[cell] = st.niter;
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------------------------
// D3Q125 split step: 32 lanes per cell, lane = stencil node (PonDstepD3Q125, steps.cu:151-250: the
// fixed 3x3x3 neighbourhood, 27 nodes), two cells per wave.
//
// Transfer of node n to target k (structs.cuh:396-524): per axis the target's quartic Lagrange
// basis on the target nodes {0, +-ec1 S1, +-ec2 S1} evaluated at the five source velocities
// (u0 - u1) + a_j S0, so f_new(k) = sum_jx Lx sum_jy Ly sum_jz Lz f(jx,jy,jz).  Interpolation on the
// fixed stencil coord-1..coord+1 with the quadratic Lagrange weights, also sum-factorised.
// Moments in the frame of the current gauge (A = sum f, B = sum f xi, C = sum f |xi|^2) are FP64
// sums; the moment solve, the residual and the stopping rules are those of the D3Q27 split step.
//
// A node's transfer to all 125 targets is three contractions of 625 FMAs over its own data, so
// one lane holds the node's 125 populations in registers and contracts them in place, one axis
// after the other: no exchange, no barrier, no LDS operand.  Then, one ky slab of 25 targets at a
// time, the lanes lay their transferred values down in LDS and 25 lanes of the cell sum them over
// the 27 nodes with the interpolation weights of their target.  With a lane per target instead
// (128 lanes per cell, the contractions through LDS, two barriers per node) the step was bound by
// its 30 LDS reads for every 15 FMAs: 96^3 turbulence 26.0 -> 7.7 ms per step, 160^3 122 -> 36 ms.
// Bound now by VALU issue (75 % of the cycles, 3400 instructions per iteration of a wave, 1875 of
// them the contractions); the texture-address unit is 50 % busy.
//
// A wave owns `chunk` consecutive cells; a half whose cell is done takes the next one, so cells
// that need more iterations hold up nobody but themselves.
constexpr double kA5d[5] = {0.0, kEc1, -kEc1, kEc2, -kEc2};

// target node m of one axis, {0, +e1, -e1, +e2, -e2}[m], as selects (m varies per lane)
__device__ __forceinline__ double node5(int m, double e1, double e2) {
  return m == 0 ? 0.0 : m == 1 ? e1 : m == 2 ? -e1 : m == 3 ? e2 : -e2;
}

// v of the lane a DPP control takes it from (a cross-lane move in the VALU, no LDS round trip)
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, 0xf, 0xf, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// sum of v over the 32 lanes of each half of the wave, in every lane, added pairwise at distances
// 16, 8, 4, 2, 1 (after the first two additions the values repeat with period 8, so a rotation by
// 4 within the row pairs the lanes at distance 4)
__device__ __forceinline__ double half_sum(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  // each row of 16 lanes and its neighbour row, side by side in both
  const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)u, (uint32_t)u, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)(u >> 32), (uint32_t)(u >> 32), false, false);
  v = __builtin_bit_cast(double, ((uint64_t)hi[0] << 32) | lo[0]) +
      __builtin_bit_cast(double, ((uint64_t)hi[1] << 32) | lo[1]);
  v += dpp_d<0x128>(v);  // row_ror:8
  v += dpp_d<0x124>(v);  // row_ror:4
  v += dpp_d<0x4e>(v);   // quad_perm [2, 3, 0, 1]
  v += dpp_d<0xb1>(v);   // quad_perm [1, 0, 3, 2]
  return v;
}

// one axis' basis values L[target class][source class] of a node: du = u0 - u1 in the axis,
// s0 its sqrt(|T|)*sign(T), target nodes {0, +-e1, +-e2} and factors bw
__device__ __forceinline__ void basis125(float du, float s0, float e1, float e2, const float (&bw)[5],
                                         float (&L)[5][5]) {
#pragma unroll
  for (int jj = 0; jj < 5; jj++) {
    const float bv = du + (float)kA5d[jj] * s0;
    const float D0 = bv, D1 = bv - e1, D2 = bv + e1, D3 = bv - e2, D4 = bv + e2;
    const float D01 = D0 * D1, D012 = D01 * D2;
    L[0][jj] = bw[0] * (((D1 * D2) * D3) * D4);
    L[1][jj] = bw[1] * (((D0 * D2) * D3) * D4);
    L[2][jj] = bw[2] * ((D01 * D3) * D4);
    L[3][jj] = bw[3] * (D012 * D4);
    L[4][jj] = bw[4] * (D012 * D3);
  }
}

// five values at distance `st` in f contracted with L in place (one axis of a node's populations)
template <int ST>
__device__ __forceinline__ void contract125(float* f, const float (&L)[5][5]) {
  float o[5];
#pragma unroll
  for (int k = 0; k < 5; k++) {
    float t = 0.f;
#pragma unroll
    for (int jj = 0; jj < 5; jj++) t = __builtin_fmaf(L[k][jj], f[jj * ST], t);
    o[k] = t;
  }
#pragma unroll
  for (int k = 0; k < 5; k++) f[k * ST] = o[k];
}

__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_step_split125(
    const float* __restrict__ fin, const float* __restrict__ min, const double* __restrict__ Tin,
    float* __restrict__ fout, float* __restrict__ mout, double* __restrict__ Tout, int* __restrict__ niter_out,
    const float* __restrict__ guess, const SplitArgs a, int chunk) {
  constexpr int Q = 125, NSTR = 28, CSTR = 27 * NSTR + 44;  // strides that spread the banks
  __shared__ __align__(16) float st[2][CSTR];  // a ky slab: [cell half][node][5 kx + kz]
  __shared__ __align__(16) float sfn[2][128];  // the iterate, by population
  __shared__ __align__(16) double sxi[128][4]; // xi_x, xi_y, xi_z, |xi|^2 of each population
  __shared__ __align__(16) float sw[128];
  const Grid& g = a.g;
  const int64_t P = g.plane;
  const int lane = threadIdx.x, h = lane >> 5, j = lane & 31;
  const int n = j < 27 ? j : 26;  // lanes 27..31 repeat node 26 (they store nothing)
  for (int k = lane; k < 128; k += 64) {
    const double xv = k < Q ? kA5d[k / 25] : 0.0, yv = k < Q ? kA5d[(k / 5) % 5] : 0.0, zv = k < Q ? kA5d[k % 5] : 0.0;
    sxi[k][0] = xv;
    sxi[k][1] = yv;
    sxi[k][2] = zv;
    sxi[k][3] = xv * xv + yv * yv + zv * zv;
    sw[k] = k < Q ? a.w[k] : 0.f;
    sfn[0][k] = sfn[1][k] = 0.f;
  }
  wave_lds_order();
  const int64_t c_first = xcd_block(blockIdx.x, gridDim.x) * chunk;
  const int total = (int)(g.n - c_first < chunk ? g.n - c_first : chunk);
  int next = 0;
  // target of this lane in a ky slab (lanes 25..31 repeat one)
  const int kx = j < 25 ? j / 5 : 4, kz = j % 5;
  const double xax = node5(kx, kEc1, kEc2), xaz = node5(kz, kEc1, kEc2);
  bool active = false, dirty = false, fresh = false;
  int64_t cell = c_first;
  int x = 0, y = 0, z = 0;
  bool rx = false, ry = false, rz = false;
  int64_t rec = 0;                              // the node's populations: index of its record ...
  float nux = 0, nuy = 0, nuz = 0, ns0 = 0;     // ... and gauge
  bool gok = true;
  double gc[4] = {0, 0, 0, 1}, res_prev = 0, rho = 0;
  int niter = 0, base = 0;  // base: iterations spent on an abandoned predicted start
  bool learned = false, contracted = false;  // contracted: a residual has fallen since the current start
  auto prev_gauge = [&](double gp[4], double& rho0) {
    rho0 = min[cell];
    gp[0] = min[P + cell]; gp[1] = min[2 * P + cell]; gp[2] = min[3 * P + cell]; gp[3] = Tin[cell];
    if (rho0 == 0 && gp[0] == 0 && gp[1] == 0 && gp[2] == 0 && gp[3] == 0) { rho0 = 1; gp[3] = a.tlat; }
  };
  while (true) {
    const uint64_t want = __ballot(!active);
    if (!active) {
      const int slot = next + (h && (want & 1) ? 1 : 0);
      if (slot < total) {
        active = fresh = true;
        cell = c_first + slot;
        x = (int)(cell % g.nx);
        y = (int)((cell / g.nx) % g.ny);
        z = (int)(cell / ((int64_t)g.nx * g.ny));
        // mirror boundaries (steps.cu:163-190): a node beyond a mirrored face is the mirror image of
        // the cell inside, population k read from the mirrored velocity, the axis velocity negated
        const int px = mirror_wrap(x - 1 + n / 9, g.nx, (g.mirror & 1) != 0, rx);
        const int py = mirror_wrap(y - 1 + (n / 3) % 3, g.ny, (g.mirror & 2) != 0, ry);
        const int pz = mirror_wrap(z - 1 + n % 3, g.nz, (g.mirror & 4) != 0, rz);
        const int64_t c = cell_index(g, px, py, pz);
        rec = c * kSplit125Floats;
        nux = rx ? -min[P + c] : min[P + c];
        nuy = ry ? -min[2 * P + c] : min[2 * P + c];
        nuz = rz ? -min[3 * P + c] : min[3 * P + c];
        const double t = Tin[c];
        ns0 = (float)(sqrt(fabs(t)) * (double)((0.0 < t) - (t < 0.0)));
        // non-finite data as in k_node_gauge (the reference drops non-finite transfer terms,
        // structs.cuh:516): a non-finite population counts as zero, a node with a non-finite gauge
        // as all zeros with a zero gauge
        gok = isfinite(nux) && isfinite(nuy) && isfinite(nuz) && isfinite(ns0);
        if (!gok) nux = nuy = nuz = ns0 = 0.f;
        double gp[4], rho0;
        prev_gauge(gp, rho0);
        for (int d = 0; d < 4; d++) gc[d] = gp[d];
        learned = contracted = false;
        niter = base = 0;
        res_prev = 0;
        rho = rho0;
        if (guess) {
          const double sq = sqrt(gp[3]);
          const float p0 = guess[cell], p1 = guess[P + cell], p2 = guess[2 * P + cell], p3 = guess[3 * P + cell];
          const double q[4] = {gp[0] + sq * p0, gp[1] + sq * p1, gp[2] + sq * p2, gp[3] * (1.0 + (double)p3)};
          const float pmax = fmaxf(fmaxf(fabsf(p0), fabsf(p1)), fmaxf(fabsf(p2), fabsf(p3)));
          if (isfinite(q[0]) && isfinite(q[1]) && isfinite(q[2]) && isfinite(q[3]) && q[3] > 0 &&
              pmax <= a.learned_trust && pmax > 0.0f && niter_out[cell] >= kLearnedPrevMin &&
              niter_out[cell] <= kLearnedPrevMax) {
            for (int d = 0; d < 4; d++) gc[d] = q[d];
            learned = true;
          }
        }
      }
    }
    next += ((want & 1) ? 1 : 0) + ((want >> 32 & 1) ? 1 : 0);
    if (__ballot(active) == 0) break;

    // the node's populations (read again in every iteration: kept, they would take the registers of
    // a second wave; the empty asm keeps the loads from being lifted out of the loop)
    float f[128];
    {
      int64_t r = rec;
      asm volatile("" : "+v"(r));
#pragma unroll
      for (int q = 0; q < 32; q++) {
        const float4 v = reinterpret_cast<const float4*>(fin + r)[q];
        f[4 * q] = v.x; f[4 * q + 1] = v.y; f[4 * q + 2] = v.z; f[4 * q + 3] = v.w;
      }
    }
    const double s = sqrt(gc[3] / a.tlat);
    // target basis constants (structs.cuh:397-416)
    const double S1 = sqrt(fabs(gc[3])) * (double)((0.0 < gc[3]) - (gc[3] < 0.0));
    const double e1 = kEc1 * S1, e2 = kEc2 * S1;
    const float e1f = (float)e1, e2f = (float)e2;
    float bw[5];
    {
      // the factor of target class m in lane m of the half
      const int m = j < 5 ? j : 4;
      const double xn = node5(m, e1, e2);
      double den = 1.0;
#pragma unroll
      for (int q = 0; q < 4; q++) den *= xn - node5(q < m ? q : q + 1, e1, e2);
      const float b = (float)(1.0 / den);
#pragma unroll
      for (int k = 0; k < 5; k++) bw[k] = __shfl(b, (lane & 32) + k, 64);
    }
    if (__ballot(fresh) != 0) {
      // 0 * v is NaN for a non-finite v
      float zz[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < Q; q++) zz[q % 5] = __builtin_fmaf(f[q], 0.f, zz[q % 5]);
      const float zs = ((zz[0] + zz[1]) + (zz[2] + zz[3])) + zz[4];
      if (fresh) dirty = !gok || zs != zs;
      fresh = false;
    }
    if (__ballot(dirty) != 0) {
#pragma unroll
      for (int q = 0; q < Q; q++) f[q] = gok && isfinite(f[q]) ? f[q] : 0.0f;
    }
    if (g.mirror) {
      auto swap = [](bool m, float& p, float& q) {
        const float t = p;
        p = m ? q : p;
        q = m ? t : q;
      };
      if (__ballot(rx) != 0) {
#pragma unroll
        for (int q = 0; q < 25; q++) { swap(rx, f[25 + q], f[50 + q]); swap(rx, f[75 + q], f[100 + q]); }
      }
      if (__ballot(ry) != 0) {
#pragma unroll
        for (int q = 0; q < 25; q++) {
          float* p = f + 25 * (q / 5) + q % 5;
          swap(ry, p[5], p[10]);
          swap(ry, p[15], p[20]);
        }
      }
      if (__ballot(rz) != 0) {
#pragma unroll
        for (int q = 0; q < 25; q++) { swap(rz, f[5 * q + 1], f[5 * q + 2]); swap(rz, f[5 * q + 3], f[5 * q + 4]); }
      }
    }
    const float u1x = (float)gc[0], u1y = (float)gc[1], u1z = (float)gc[2];
    const float u1xl = (float)(gc[0] - (double)u1x), u1yl = (float)(gc[1] - (double)u1y),
                u1zl = (float)(gc[2] - (double)u1z);
    float L[5][5];
    basis125((nuz - u1z) - u1zl, ns0, e1f, e2f, bw, L);
#pragma unroll
    for (int q = 0; q < 25; q++) contract125<1>(f + 5 * q, L);
    basis125((nuy - u1y) - u1yl, ns0, e1f, e2f, bw, L);
#pragma unroll
    for (int q = 0; q < 25; q++) contract125<5>(f + 25 * (q / 5) + q % 5, L);
    basis125((nux - u1x) - u1xl, ns0, e1f, e2f, bw, L);
    // departure point on the fixed stencil coord-1..coord+1 (steps.cu:163,207-208)
    float Fx[3], Fz[3];
    lag3f((float)(((double)x - (s * xax + gc[0])) - (double)(x - 1)), Fx);
    lag3f((float)(((double)z - (s * xaz + gc[2])) - (double)(z - 1)), Fz);
#pragma unroll
    for (int ky = 0; ky < 5; ky++) {
#pragma unroll
      for (int q = 0; q < 5; q++) contract125<25>(f + 5 * ky + q, L);
      wave_lds_order();  // the previous slab's reads are done
      if (j < 27) {
        float* o = &st[h][n * NSTR];
        float v[28];
#pragma unroll
        for (int q = 0; q < 25; q++) v[q] = f[25 * (q / 5) + 5 * ky + q % 5];
        v[25] = v[26] = v[27] = 0.f;
#pragma unroll
        for (int q = 0; q < 7; q++) *reinterpret_cast<float4*>(o + 4 * q) = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
      }
      wave_lds_order();
      float Fy[3];
      lag3f((float)(((double)y - (s * kA5d[ky] + gc[1])) - (double)(y - 1)), Fy);
      // the stencil sums of the fixed 3x3x3 neighbourhood: z inner, then y, then x
      const float* t = &st[h][5 * kx + kz];
      float acc = 0.f;
#pragma unroll
      for (int ia = 0; ia < 3; ia++) {
        float accy = 0.f;
#pragma unroll
        for (int ib = 0; ib < 3; ib++) {
          float accz = 0.f;
#pragma unroll
          for (int ic = 0; ic < 3; ic++) accz = __builtin_fmaf(Fz[ic], t[(9 * ia + 3 * ib + ic) * NSTR], accz);
          accy = __builtin_fmaf(Fy[ib], accz, accy);
        }
        acc = __builtin_fmaf(Fx[ia], accy, acc);
      }
      if (j < 25) sfn[h][25 * kx + 5 * ky + kz] = acc;
    }
    wave_lds_order();
    // moments in the frame of the current gauge, FP64 sums over the populations: pairs 32 apart, then
    // the halves' tree, populations 0..63 and 64..127 separately
    double mom[5];
    {
      double lo[5], hi[5];
#pragma unroll
      for (int b = 0; b < 4; b++) {
        const int k = j + 32 * b;
        const double fd = (double)sfn[h][k];
        const double v[5] = {fd, fd * sxi[k][0], fd * sxi[k][1], fd * sxi[k][2], fd * sxi[k][3]};
#pragma unroll
        for (int q = 0; q < 5; q++) {
          if (b == 0) lo[q] = v[q];
          if (b == 1) lo[q] += v[q];
          if (b == 2) hi[q] = v[q];
          if (b == 3) hi[q] += v[q];
        }
      }
#pragma unroll
      for (int q = 0; q < 5; q++) mom[q] = half_sum(lo[q]) + half_sum(hi[q]);
    }
    bool done = false;
    if (active) {
      niter++;
      rho = mom[0];
      const double B[3] = {mom[1], mom[2], mom[3]}, C = mom[4];
      double m[4];
      if (rho != 0) {
        const double ir = 1.0 / rho;
        for (int d = 0; d < 3; d++) m[d] = gc[d] + s * (B[d] * ir);
        m[3] = s * s * (C - (B[0] * B[0] + B[1] * B[1] + B[2] * B[2]) * ir) * ir * a.inv_dim;
      } else {
        for (int d = 0; d < 3; d++) m[d] = s * B[d];
        m[3] = (2.0 * s * (gc[0] * B[0] + gc[1] * B[1] + gc[2] * B[2]) + s * s * C - (m[0] * m[0] + m[1] * m[1] + m[2] * m[2])) *
               a.inv_dim;
      }
      if (m[3] < 0) m[3] = gc[3];
      const double sth = sqrt(fabs(m[3]));
      double res = 0;
      bool conv = true;
      for (int d = 0; d < 4; d++) {
        const double scale = d < 3 ? sth : fabs(m[3]);
        const double dd = fabs(m[d] - gc[d]);
        if (dd > a.tol_rel * scale + a.tol_abs) conv = false;  // NaN: converged, as in the D3Q27 step
        const double rk = dd / (scale + 1e-300);
        if (res == res && !(rk <= res)) res = rk;  // NaN propagates (fmax would drop it)
      }
      if (!conv && niter - base > 1 && res <= 4.0 * a.tol_rel && res >= res_prev && (!learned || contracted)) conv = true;
      if (niter - base > 1 && res < res_prev) contracted = true;
      // (unlike the D3Q27 step, no fallback from a predicted start on a NaN residual)
      if (!conv && learned && ((niter > 1 && !(res < res_prev)) || niter == kLearnedBudget)) {
        double rho0;
        prev_gauge(gc, rho0);
        learned = contracted = false;
        res_prev = 0;
        base = niter;
      } else {
        res_prev = res;
        for (int d = 0; d < 4; d++) gc[d] = m[d];
      }
      done = conv || niter - base >= a.max_iter;
    }
    if (done) {
      // BGK on the iterate, four populations per lane: the cell's record in one store
      active = false;
      const float rf = (float)rho, dt = (float)a.dtau;
      float4 o;
      float* ov = &o.x;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const float v = sfn[h][4 * j + q];
        ov[q] = __builtin_fmaf(dt, rf * sw[4 * j + q] - v, v);
      }
      reinterpret_cast<float4*>(fout + cell * kSplit125Floats)[j] = o;
      if (j == 0) {
        mout[cell] = rf;
        mout[P + cell] = (float)gc[0];
        mout[2 * P + cell] = (float)gc[1];
        mout[3 * P + cell] = (float)gc[2];
        Tout[cell] = gc[3];
        niter_out[cell] = niter;
      }
    }
    wave_lds_order();
  }
}

hipError_t launch_node_gauge(float* f, const float* m, const double* T, float* g4, int64_t n, int64_t plane,
                             int* pending_count, hipStream_t st) {
  hipLaunchKernelGGL(k_node_gauge, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, f, m, T, g4, n, plane,
                     pending_count);
  return hipGetLastError();
}

hipError_t launch_step_split(int lattice, int interp, const SplitPtrs& in, const SplitPtrs& out, const float* g4,
                             int* niter, const float* guess, const SplitPending& pend, const SplitArgs& a,
                             hipStream_t st) {
  if (lattice == kD3Q125) {
    // Consecutive cells per wave: four, or two (one per half) where that would leave SIMDs without a
    // wave.  Turbulence, ms per step with chunks of 2, 4, 8, 16, 32: 16^3 0.086, 0.104, 0.142, 0.229,
    // 0.425; 32^3 0.359, 0.352, 0.346, 0.324, 0.484; 96^3 7.82, 7.63, 7.70, 7.72, 7.78.
    const int chunk = a.g.n < 8192 ? 2 : 4;
    hipLaunchKernelGGL(k_step_split125, dim3((unsigned)((a.g.n + chunk - 1) / chunk)), dim3(64), 0, st, in.f, in.m, in.T,
                       out.f, out.m, out.T, niter, guess, a, chunk);
    return hipGetLastError();
  }
  if (lattice != kD3Q27) return hipErrorInvalidValue;
  if (interp != 0) {
    const int64_t slots = a.g.ntiles * 64;
    // Cells per wave.  By x rows (row patches, or linear order with WENO5C): whole rows, at least 128
    // (64) cells, so that the waves resident on an XCD cover a compact patch of rows, but not so many
    // that SIMDs go without two waves, and on small grids one cell per slot.  Lagrange-4 in linear order: one or two cells per slot (the waves
    // in flight then cover fewer planes, and more of them even out the last round).  ms per step, with 21,
    // 42, 64, 128, 192, 256, 384 cells, WENO5C vortex in patches: 64^3 1.03, 0.98, 0.86, 0.84, 1.10, 1.36,
    // 1.96; 128^3 6.79, 6.24, 5.95, 5.43, 5.66, 5.36, 5.73; 192^3 22.4, 20.4, 19.2, 17.8, 17.0, 17.5, 16.9.
    // In linear order with 21, 64, 128 cells and one row: 50x40x30 0.40, 0.49, 0.75, -; 100x60x50 1.19, 1.10, 1.28, 1.10; 100x90x80 2.60,
    // 2.26, 2.27, 2.16; 150x101x94 4.76, 4.35, 4.18, 3.88 (shock-bubble 9.68, 8.36, 8.26, 7.60); 250x200x180
    // -, 25.9, 23.3, 22.4.  Lagrange-4 with 21, 42, 128 cells: Taylor-Green 150x101x94 7.81, 8.50, 10.4;
    // 250x200x180 44.5, 46.2, 48.7; shock-bubble 9.94, 9.55, 11.0 and 55.8, 51.1, 53.3.
    int64_t cells;
    if (a.refill_chunk >= 0) {
      cells = a.refill_chunk > 0 ? 64ll * a.refill_chunk : 64;
    } else if (interp == 2 && a.g.n < (1 << 17)) {
      cells = 21;
    } else if (a.g.rp > 0 || (interp == 2 && a.g.nx <= 512)) {
      const int64_t least = a.g.rp > 0 ? 128 : 64;
      cells = a.g.nx * ((least + a.g.nx - 1) / a.g.nx);
      // (Lagrange-4 four waves: 64^3 Taylor-Green 1.53 -> 1.45 ms with 64 cells, 128x52x52 2.74 -> 2.31)
      while (cells > 21 && slots / cells < (interp == 2 ? 2048 : 4096)) cells /= 2;
      if (cells < 21) cells = 21;
    } else if (interp == 2) {
      cells = 128;
    } else {
      cells = a.g.n >= (1 << 22) ? 42 : 21;
    }
    if (cells > slots) cells = slots;
    const dim3 nb((unsigned)((slots + cells - 1) / cells));
#define POND_LAUNCH(I)                                                                                             \
  hipLaunchKernelGGL(k_step_split27_cells<I>, nb, dim3(64), 0, st, in.f, in.m, in.T, g4, out.f, out.m, out.T, niter, \
                     guess, pend.count, a, (int)cells, wide_after, few)
    // The iteration after which a cell goes to k_step_split27_wide.  A workgroup there serves a cell's
    // iteration eight times sooner, but the chip gets through far fewer of them: early where the
    // cells kernel leaves it idle.  ms per step for 4, 6, 8, 12, 16 and never, shock-bubble: 32^3 1.03, 0.98,
    // 1.02, 1.18, 1.36, 5.29; 64^3 2.99, 2.67, 2.54, 2.53, 2.59, 6.70; 128^3 14.2, 12.9, 11.97, 11.61,
    // 11.60, 14.5; 256^3 -, 73.9, 70.7, 69.5, 69.4, 69.8 (vortex, at most 10 iterations: 41.4, 39.82,
    // 39.78, -, -, 39.74).
    const int wide_after = a.pass1_iters > 0 ? a.pass1_iters : a.g.n < (1 << 19) ? 8 : 16;
    // From then on a cell goes when its wave stands idle for it: with no cell left to start and at most
    // kWideSlots slots still at such cells.  The workgroups of the chip do 80 iterations per us, the waves
    // with all slots in use 900, so a wave whose cells are all late keeps them.  Only the first `few` of a
    // step go at once: a small grid leaves the chip idle anyway.  Tolerance 0 (every cell to the cap), ms per
    // step with every late cell handed over and now: 64^3 250, 33, 128^3 1840, 208; tolerance 1.4e-8 (a third
    // of the cells past 16 iterations): 64^3 53, 15, 128^3 320, 85; T = 0.2 with density jumps 16 cells apart:
    // 64^3 17.9, 16.7, 128^3 102, 99, 200^3 443, 503 (one lane per cell: 951).  32^3 with few = 4096, 8192 and
    // 16384: tolerance 0 9.7, 14.9, 21 (all handed over 31.4), 2e-8 2.23, 2.05, 2.04.
    const int few = a.g.n < (1 << 16) ? 8192 : 4096;
    if (interp == 2) {
      POND_LAUNCH(2);
      const unsigned nw = (unsigned)(a.g.n < 1024 ? a.g.n : 1024);
      hipLaunchKernelGGL(k_step_split27_wide, dim3(nw), dim3(kWideThreads), 0, st, in.f, in.m, in.T, g4, out.f, out.m, out.T, niter,
                         pend.count, a);
    } else if (a.g.mirror) {
      POND_LAUNCH(3);
    } else {
      POND_LAUNCH(1);
    }
#undef POND_LAUNCH
    return hipGetLastError();
  }
  // By default the first pass goes to the end (192^3 shock-bubble: K=3 7.6, K=8 8.9, single pass 11.5
  // MLUPS: the second, with one lane per cell too, runs alone after the first and a few slowly
  // converging cells make a tail).
  SplitArgs b = a;
  b.pass1_iters = a.pass1_iters < 0 ? 1 << 30 : a.pass1_iters < 255 ? a.pass1_iters : 255;  // (8 bits in the list)
  // second-pass grid: enough waves to fill the chip several times, never more than the cells
  const int64_t w2 = (a.g.n + 63) / 64;
  const unsigned blocks2 = (unsigned)(w2 < 16384 ? w2 : 16384);
  hipLaunchKernelGGL(k_step_split27_written, dim3((unsigned)a.g.ntiles), dim3(64), 0, st, in.f, in.m, in.T, g4, out.f,
                     out.m, out.T, niter, guess, pend, b);
  hipLaunchKernelGGL(k_step_split27_rest, dim3(blocks2), dim3(64), 0, st, in.f, in.m, in.T, g4, out.f, out.m, out.T,
                     niter, pend, b);
  return hipGetLastError();
}

}  // namespace pond
