// Regular (non-singular) pair integrals shared by the assembly kernels: the Stokeslet and
// stresslet moments of one (collocation point, element) pair with one quadrature rule.
#pragma once
#include "andr_internal.h"

// quadrature table of this translation unit: l1, l2, l3, w per point (see andr_rule)
static __constant__ double c_qd[ANDR_QTAB_N][4];
static __constant__ float c_qf[ANDR_QTAB_N][4];

static inline int andr_upload_rules_here(andr_ctx *ctx, const double *tab, const float *tabf) {
  ANDR_HIP(ctx, hipMemcpyToSymbol(HIP_SYMBOL(c_qd), tab, sizeof(double) * 4 * ANDR_QTAB_N));
  ANDR_HIP(ctx, hipMemcpyToSymbol(HIP_SYMBOL(c_qf), tabf, sizeof(float) * 4 * ANDR_QTAB_N));
  return ANDR_OK;
}


// 1 / sqrt(x) in FP64 for 0 < x < infinity: the hardware estimate (v_rsq_f64, error e below 2^-20) and one step of
// third order (Householder), which leaves e^3: five operations against the some twenty of a division and
// a square root in their general forms. ENDS: 0 and infinity too, whose estimates, infinity and 0, stand (e is no
// number there, its minimum with anything the other).
template <bool ENDS = false>
__device__ inline double rsqrt64(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double e = fma(-x * y, y, 1.0);
  if constexpr (ENDS) e = fmin(e, 0.5);
  return fma(y * e, fma(0.375, e, 0.5), y);
}

// The regular integrals of one triangle seen from s, in FP64 with pressure (Triangle_3DStokesInt,
// src/lib_Stokes.f90:2341-2446, with StokesKernel :2450-2544): Stokeslet Gs, pressure vector pG,
// stresslet moments Tv and pressure moments pT per vertex, for the normal (nx, ny, nz) and area A.
// r.n is one number per flat element, so the sums are the moments of r_i r_j / r^5, r_i / r^5 and 1 / r^3
// with the shape functions, and the normal comes in once at the end: 73 FP64 operations a
// point (1082 rows of 720 triangles with k_stokes_rows: 1361 -> 386 us, with the turns of its workgroup).
__device__ inline void stokes_tri_full(const double s[3], const double *x1, const double *x2, const double *x3,
                                       double nx, double ny, double nz, double A, int qoff, int nq, double Gs[6],
                                       double pG[3], double Tv[6][3], double pT[3][3]) {
  const double d[3] = {x3[0] - s[0], x3[1] - s[1], x3[2] - s[2]};
  const double xa[3] = {x1[0] - x3[0], x1[1] - x3[1], x1[2] - x3[2]};
  const double xb[3] = {x2[0] - x3[0], x2[1] - x3[1], x2[2] - x3[2]};
  double g1 = 0.0, g3[6] = {0, 0, 0, 0, 0, 0}, p3[3] = {0, 0, 0}, m3[3] = {0, 0, 0};
  double t[6][3] = {{0}}, m5[3][3] = {{0}};
  for (int q = 0; q < nq; ++q) {
    const double l[3] = {c_qd[qoff + q][0], c_qd[qoff + q][1], c_qd[qoff + q][2]};
    const double w = c_qd[qoff + q][3];
    double r[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) r[c] = d[c] + l[0] * xa[c] + l[1] * xb[c];
    const double rr[6] = {r[0] * r[0], r[0] * r[1], r[0] * r[2], r[1] * r[1], r[1] * r[2], r[2] * r[2]};
    const double ir = rsqrt64(rr[0] + rr[3] + rr[5]);
    const double ir2 = ir * ir, w1 = w * ir, w3 = w1 * ir2, w5 = w3 * ir2;
    g1 += w1;
#pragma unroll
    for (int k = 0; k < 6; ++k) g3[k] += w3 * rr[k];
#pragma unroll
    for (int k = 0; k < 3; ++k) p3[k] += w3 * r[k];
#pragma unroll
    for (int v = 0; v < 3; ++v) {
      const double wl = w5 * l[v];
      m3[v] += w3 * l[v];
#pragma unroll
      for (int k = 0; k < 6; ++k) t[k][v] += wl * rr[k];
#pragma unroll
      for (int k = 0; k < 3; ++k) m5[k][v] += wl * r[k];
    }
  }
  const double n[3] = {nx, ny, nz}, rn = d[0] * nx + d[1] * ny + d[2] * nz;
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    Gs[k] = A * ((k == 0 || k == 3 || k == 5) ? g1 + g3[k] : g3[k]);
#pragma unroll
    for (int v = 0; v < 3; ++v) Tv[k][v] = -6.0 * A * rn * t[k][v];
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    pG[k] = 2.0 * A * p3[k];
#pragma unroll
    for (int v = 0; v < 3; ++v) pT[k][v] = 4.0 * A * (3.0 * rn * m5[k][v] - n[k] * m3[v]);
  }
}

// Gs: Stokeslet block (FP64); Tv: stresslet moments per vertex, in the quadrature type CT
template <class CT>
__device__ inline void stokes_pair_regular(const double s[3], const double *x1, const double *x2, const double *x3,
                                           double nx, double ny, double nz, double area, int qoff, int nq,
                                           double Gs[6], CT Tv[6][3]) {
  // relative geometry formed in FP64, quadrature in CT
  const CT d0 = (CT)(x3[0] - s[0]), d1 = (CT)(x3[1] - s[1]), d2 = (CT)(x3[2] - s[2]);
  const CT a0 = (CT)(x1[0] - x3[0]), a1 = (CT)(x1[1] - x3[1]), a2 = (CT)(x1[2] - x3[2]);
  const CT b0 = (CT)(x2[0] - x3[0]), b1 = (CT)(x2[1] - x3[1]), b2 = (CT)(x2[2] - x3[2]);
  const CT n0 = (CT)nx, n1 = (CT)ny, n2 = (CT)nz;
  CT g[6] = {0, 0, 0, 0, 0, 0};
  CT t[6][3] = {{0}};
  for (int q = 0; q < nq; ++q) {
    CT l1, l2, l3, w;
    if constexpr (sizeof(CT) == 8) {
      l1 = c_qd[qoff + q][0]; l2 = c_qd[qoff + q][1]; l3 = c_qd[qoff + q][2]; w = c_qd[qoff + q][3];
    } else {
      l1 = c_qf[qoff + q][0]; l2 = c_qf[qoff + q][1]; l3 = c_qf[qoff + q][2]; w = c_qf[qoff + q][3];
    }
    const CT rx = d0 + l1 * a0 + l2 * b0;
    const CT ry = d1 + l1 * a1 + l2 * b1;
    const CT rz = d2 + l1 * a2 + l2 * b2;
    const CT rxx = rx * rx, rxy = rx * ry, rxz = rx * rz, ryy = ry * ry, ryz = ry * rz, rzz = rz * rz;
    CT ir;
    if constexpr (sizeof(CT) == 8) ir = rsqrt(rxx + ryy + rzz);
    else ir = __frsqrt_rn(rxx + ryy + rzz);
    const CT ir2 = ir * ir, ir3 = ir2 * ir;
    const CT wir = w * ir, wir3 = w * ir3;
    g[0] += wir + rxx * wir3;
    g[1] += rxy * wir3;
    g[2] += rxz * wir3;
    g[3] += wir + ryy * wir3;
    g[4] += ryz * wir3;
    g[5] += wir + rzz * wir3;
    const CT ct = (CT)(-6.0) * ir2 * ir3 * (rx * n0 + ry * n1 + rz * n2);
    const CT wc[3] = {w * l1 * ct, w * l2 * ct, w * l3 * ct};
    const CT rr[6] = {rxx, rxy, rxz, ryy, ryz, rzz};
#pragma unroll
    for (int k = 0; k < 6; ++k)
#pragma unroll
      for (int v = 0; v < 3; ++v) t[k][v] += wc[v] * rr[k];
  }
  const CT ca = (CT)area;
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    Gs[k] = (double)g[k] * area;
#pragma unroll
    for (int v = 0; v < 3; ++v) Tv[k][v] = t[k][v] * ca;
  }
}

// As stokes_pair_regular, with the stresslet moments summed over the vertices: Ts[k] = sum_v Tv[k][v]
// (the shape functions sum to one, so the vertex weights drop out of the quadrature loop). Enough for
// a velocity field that is affine over the element (a rigid motion of all three vertices): then
// sum_v Tv[k][v] u(x_v) = int T_k u(x), and the rotation terms reduce to Ts and the collocation point
// (the third moments int T_{c,i} r_j enter the rotations antisymmetrised in (i, j), where
// T_{c,i} r_j = t r_c r_i r_j cancels at every quadrature point).
template <class CT>
__device__ inline void stokes_pair_sum(const double s[3], const double *x1, const double *x2, const double *x3,
                                       double nx, double ny, double nz, double area, int qoff, int nq, double Gs[6],
                                       CT Ts[6]) {
  const CT d0 = (CT)(x3[0] - s[0]), d1 = (CT)(x3[1] - s[1]), d2 = (CT)(x3[2] - s[2]);
  const CT a0 = (CT)(x1[0] - x3[0]), a1 = (CT)(x1[1] - x3[1]), a2 = (CT)(x1[2] - x3[2]);
  const CT b0 = (CT)(x2[0] - x3[0]), b1 = (CT)(x2[1] - x3[1]), b2 = (CT)(x2[2] - x3[2]);
  const CT n0 = (CT)nx, n1 = (CT)ny, n2 = (CT)nz;
  CT g[6] = {0, 0, 0, 0, 0, 0};
  CT t[6] = {0, 0, 0, 0, 0, 0};
  for (int q = 0; q < nq; ++q) {
    CT l1, l2, w;
    if constexpr (sizeof(CT) == 8) {
      l1 = c_qd[qoff + q][0]; l2 = c_qd[qoff + q][1]; w = c_qd[qoff + q][3];
    } else {
      l1 = c_qf[qoff + q][0]; l2 = c_qf[qoff + q][1]; w = c_qf[qoff + q][3];
    }
    const CT rx = d0 + l1 * a0 + l2 * b0;
    const CT ry = d1 + l1 * a1 + l2 * b1;
    const CT rz = d2 + l1 * a2 + l2 * b2;
    const CT rxx = rx * rx, rxy = rx * ry, rxz = rx * rz, ryy = ry * ry, ryz = ry * rz, rzz = rz * rz;
    CT ir;
    if constexpr (sizeof(CT) == 8) ir = rsqrt(rxx + ryy + rzz);
    else ir = __frsqrt_rn(rxx + ryy + rzz);
    const CT ir2 = ir * ir, ir3 = ir2 * ir;
    const CT wir = w * ir, wir3 = w * ir3;
    g[0] += wir + rxx * wir3;
    g[1] += rxy * wir3;
    g[2] += rxz * wir3;
    g[3] += wir + ryy * wir3;
    g[4] += ryz * wir3;
    g[5] += wir + rzz * wir3;
    const CT wc = (CT)(-6.0) * wir3 * ir2 * (rx * n0 + ry * n1 + rz * n2);
    t[0] += wc * rxx;
    t[1] += wc * rxy;
    t[2] += wc * rxz;
    t[3] += wc * ryy;
    t[4] += wc * ryz;
    t[5] += wc * rzz;
  }
  const CT ca = (CT)area;
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    Gs[k] = (double)g[k] * area;
    Ts[k] = t[k] * ca;
  }
}

