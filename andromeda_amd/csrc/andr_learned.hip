// Learned Gauss-order selection (no counterpart in the reference, which integrates every regular
// pair with one fixed rule, src/lib_Stokes.f90:2341-2446).
//
// A small network (6 -> 64 -> 64 -> 64 -> 8, ReLU) predicts, for a near-field (collocation point,
// element) pair, the cheapest triangle rule that reproduces the fixed-order integral: classes
// 0..6 are the Dunavant rules with 3, 4, 6, 7, 12, 13 and 19 points, class 7 the mesh's own
// fixed-order rule. Far pairs take a rule from a distance table calibrated on the same labels.
// Labels are produced here from FP64 integrals (the fixed-order rule is the reference), the network
// is trained here (forward, backward and Adam kernels), and inference runs in a classification
// pass before the assembly with BF16 weights in LDS and FP32 accumulation.
#include "andr_learned.h"
#include "andr_pairs.h"
#include "andr_prof.h"
#include "andr_singular.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <random>
#include <vector>

namespace {

constexpr int NIN = 6, NH = 64, NOUT = 8;
constexpr int P_W1 = 0, P_B1 = P_W1 + NIN * NH, P_W2 = P_B1 + NH, P_B2 = P_W2 + NH * NH, P_W3 = P_B2 + NH,
              P_B3 = P_W3 + NH * NH, P_W4 = P_B3 + NH, P_B4 = P_W4 + NH * NOUT, NPARAM = P_B4 + NOUT;
static_assert(NPARAM == ANDR_MLP_NPARAM, "parameter layout");
constexpr int NCLS_DUN = 7;   // Dunavant classes; class 7 = fixed-order rule
constexpr int DUN_ID0 = 6;    // rule id of the first Dunavant rule in the quadrature table

// ---- pair geometry and features ---------------------------------------------------------------
struct PairGeo {
  double dh;      // distance from the collocation point to the element centroid / longest edge
  double aspect;  // longest edge^2 / (2 area)
  double cosn;    // cosine of the angle between the two element normals
};

__device__ inline PairGeo pair_geo(const double s[3], const double ns[3], const double *x1, const double *x2,
                                   const double *x3, const double ne[3], double area) {
  PairGeo p;
  const double c[3] = {(x1[0] + x2[0] + x3[0]) / 3.0, (x1[1] + x2[1] + x3[1]) / 3.0, (x1[2] + x2[2] + x3[2]) / 3.0};
  const double d = sqrt((s[0] - c[0]) * (s[0] - c[0]) + (s[1] - c[1]) * (s[1] - c[1]) + (s[2] - c[2]) * (s[2] - c[2]));
  auto l2 = [](const double *a, const double *b) {
    return (a[0] - b[0]) * (a[0] - b[0]) + (a[1] - b[1]) * (a[1] - b[1]) + (a[2] - b[2]) * (a[2] - b[2]);
  };
  const double L2 = fmax(l2(x1, x2), fmax(l2(x2, x3), l2(x3, x1)));
  p.dh = d / sqrt(L2);
  p.aspect = L2 / (2.0 * area);
  p.cosn = ns[0] * ne[0] + ns[1] * ne[1] + ns[2] * ne[2];
  return p;
}

__device__ inline void features(const PairGeo &p, int kernel, float f[NIN]) {
  f[0] = logf((float)p.dh);  // the network takes FP32 inputs; FP32 logarithms are as good here
  f[1] = logf((float)p.aspect);
  f[2] = (float)p.cosn;
  f[3] = kernel == 0 ? 1.f : 0.f;
  f[4] = kernel == 1 ? 1.f : 0.f;
  f[5] = kernel == 2 ? 1.f : 0.f;
}

__device__ inline int far_bin(double dh, double near_ratio) {
  int b = (int)floor(2.0 * log2(dh / near_ratio));
  return b < 0 ? 0 : (b > ANDR_FAR_BINS - 1 ? ANDR_FAR_BINS - 1 : b);
}

// Laplace pair in FP64: out = {G, H1, H2, H3} (BemKernel, r = s - f)
__device__ inline void lap_pair(const double s[3], const double *x1, const double *x2, const double *x3,
                                const double n[3], double area, int qoff, int nq, double out[4]) {
  double g = 0, h1 = 0, h2 = 0, h3 = 0;
  for (int q = 0; q < nq; ++q) {
    const double l1 = c_qd[qoff + q][0], l2 = c_qd[qoff + q][1], l3 = c_qd[qoff + q][2], w = c_qd[qoff + q][3];
    const double rx = s[0] - (l1 * x1[0] + l2 * x2[0] + l3 * x3[0]);
    const double ry = s[1] - (l1 * x1[1] + l2 * x2[1] + l3 * x3[1]);
    const double rz = s[2] - (l1 * x1[2] + l2 * x2[2] + l3 * x3[2]);
    const double ira = rsqrt(rx * rx + ry * ry + rz * rz);
    const double fg = (0.25 / ANDR_PI) * ira;
    const double fh = (rx * n[0] + ry * n[1] + rz * n[2]) * ira * ira * fg;
    g += w * fg;
    h1 += w * fh * l1;
    h2 += w * fh * l2;
    h3 += w * fh * l3;
  }
  out[0] = g * area;
  out[1] = h1 * area;
  out[2] = h2 * area;
  out[3] = h3 * area;
}

// values of one kernel family with one rule: Laplace 4, Stokes-G 6, Stokes-H 18
__device__ inline int kernel_values(int kernel, const double s[3], const double *x1, const double *x2,
                                    const double *x3, const double n[3], double area, int qoff, int nq,
                                    double v[18]) {
  if (kernel == 0) {
    lap_pair(s, x1, x2, x3, n, area, qoff, nq, v);
    return 4;
  }
  double G[6], T[6][3];
  stokes_pair_regular<double>(s, x1, x2, x3, n[0], n[1], n[2], area, qoff, nq, G, T);
  if (kernel == 1) {
    for (int i = 0; i < 6; ++i) v[i] = G[i];
    return 6;
  }
  for (int k = 0; k < 6; ++k)
    for (int t = 0; t < 3; ++t) v[3 * k + t] = T[k][t];
  return 18;
}

// smallest Dunavant class whose values agree with the fixed-order values to rel_tol, else 7
__device__ inline int pair_label(int kernel, const double s[3], const double *x1, const double *x2, const double *x3,
                                 const double n[3], double area, int qoff_ref, int nq_ref, const int *dun_off,
                                 const int *dun_n, double rel_tol) {
  double ref[18], v[18];
  const int nv = kernel_values(kernel, s, x1, x2, x3, n, area, qoff_ref, nq_ref, ref);
  double scale = 0.0;
  for (int i = 0; i < nv; ++i) scale = fmax(scale, fabs(ref[i]));
  for (int c = 0; c < NCLS_DUN; ++c) {
    kernel_values(kernel, s, x1, x2, x3, n, area, dun_off[c], dun_n[c], v);
    double err = 0.0;
    for (int i = 0; i < nv; ++i) err = fmax(err, fabs(v[i] - ref[i]));
    if (err <= rel_tol * scale) return c;
  }
  return NCLS_DUN;
}

struct RuleTab {
  int off[8], n[8];
};

// deterministic 32-bit hash of a pair (subsampling of the training records)
__device__ inline uint32_t pair_hash(uint32_t r, uint32_t e) {
  uint32_t h = r * 0x9E3779B1u ^ (e + 0x7F4A7C15u) * 0x85EBCA77u;
  h ^= h >> 16;
  h *= 0x7FEB352Du;
  h ^= h >> 15;
  h *= 0x846CA68Bu;
  h ^= h >> 16;
  return h;
}

// one block per centroid row. mode 0: near pairs with hash <= keep -> (features, label) records,
// three per pair (one per kernel); mode 1: far pairs -> bin maxima; mode 2: count near records.
__global__ __launch_bounds__(256) void k_pair_labels(BodyGeom g, int qoff_ref, int nq_ref, RuleTab rt,
                                                     double near_ratio, double rel_tol, int mode, uint32_t keep,
                                                     int64_t max_pairs, float *__restrict__ feats,
                                                     int *__restrict__ labels,
                                                     unsigned long long *__restrict__ counter,
                                                     int *__restrict__ far_max) {
  const int r = blockIdx.x;
  const int ne = g.ne;
  const double s[3] = {g.cen[3 * r], g.cen[3 * r + 1], g.cen[3 * r + 2]};
  const double ns[3] = {g.nrm[3 * r], g.nrm[3 * r + 1], g.nrm[3 * r + 2]};
  for (int e = threadIdx.x; e < ne; e += blockDim.x) {
    if (e == r) continue;
    const double *x1 = g.xyz + 3 * g.con[3 * e], *x2 = g.xyz + 3 * g.con[3 * e + 1], *x3 = g.xyz + 3 * g.con[3 * e + 2];
    const double n[3] = {g.nrm[3 * e], g.nrm[3 * e + 1], g.nrm[3 * e + 2]};
    const PairGeo pg = pair_geo(s, ns, x1, x2, x3, n, g.area[e]);
    if (mode == 2 && pg.dh < near_ratio) {
      atomicAdd(counter, 3ull);
    } else if (mode == 0 && pg.dh < near_ratio && pair_hash(r, e) <= keep) {
      for (int kernel = 0; kernel < 3; ++kernel) {
        const int lab = pair_label(kernel, s, x1, x2, x3, n, g.area[e], qoff_ref, nq_ref, rt.off, rt.n, rel_tol);
        const unsigned long long idx = atomicAdd(counter, 1ull);
        if ((int64_t)idx < max_pairs) {
          float f[NIN];
          features(pg, kernel, f);
          for (int i = 0; i < NIN; ++i) feats[idx * NIN + i] = f[i];
          labels[idx] = lab;
        }
      }
    } else if (mode == 1 && pg.dh >= near_ratio && pg.dh < near_ratio * 256.0) {
      const int b = far_bin(pg.dh, near_ratio);
      int lab = pair_label(1, s, x1, x2, x3, n, g.area[e], qoff_ref, nq_ref, rt.off, rt.n, rel_tol);
      lab = max(lab, pair_label(2, s, x1, x2, x3, n, g.area[e], qoff_ref, nq_ref, rt.off, rt.n, rel_tol));
      atomicMax(far_max + b, lab);
    }
  }
}

// ---- the network in FP32 on the matrix cores (v_mfma_f32_16x16x4f32), row-major ------------------
// Lane layout of one 16x16x4 step: lane 16 g + i supplies A[i][g] and B[g][i] and, after the K
// loop, holds C[4 g + v][i], v = 0..3. Inside a 16-deep K block, step t gives lane group g the index
// k0 + 4 g + t on both operands (one permutation of K, so every k is summed once); the four steps
// go to four accumulators, added at the end. Out-of-range rows, columns and k read as 0.
typedef float f32x4 __attribute__((ext_vector_type(4)));

// A 64-thread wave owns 16 of the 64 columns of every layer. wf: B operand of a forward layer,
// W[16 kb + 4 g + t][col]; wt: of a backward one, W[col][16 kb + 4 g + t] (ldw a multiple of four and the
// parameters of each layer on 16 bytes, so four k of a row are one load).
template <int K>
__device__ inline void wf(const float *__restrict__ W, int ldw, int col, bool cok, int g, f32x4 b[(K + 15) / 16]) {
#pragma unroll
  for (int kb = 0; kb < (K + 15) / 16; ++kb)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int k = 16 * kb + 4 * g + t;
      const float x = W[(size_t)(k < K ? k : 0) * ldw + (cok ? col : 0)];
      b[kb][t] = (k < K && cok) ? x : 0.f;
    }
}
template <int K>
__device__ inline void wt(const float *__restrict__ W, int ldw, int col, int g, f32x4 b[(K + 15) / 16]) {
#pragma unroll
  for (int kb = 0; kb < (K + 15) / 16; ++kb) {
    const int k = 16 * kb + 4 * g;
    const f32x4 x = *(const f32x4 *)(W + (size_t)col * ldw + (k < K ? k : 0));
    b[kb] = k < K ? x : f32x4{0.f, 0.f, 0.f, 0.f};
  }
}

// C tile of 16 samples: A from LDS (rows of MT_LD floats), B in registers; returns (+ bias)
constexpr int MT_LD = NH + 4;
template <int KB>
__device__ inline f32x4 mlp_tile(const float *__restrict__ A, const f32x4 b[KB], int g, int i, float bias) {
  f32x4 acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const f32x4 a = *(const f32x4 *)(A + i * MT_LD + 16 * kb + 4 * g);
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], b[kb][t], acc[t], 0, 0, 0);
  }
  f32x4 z;
#pragma unroll
  for (int v = 0; v < 4; ++v) z[v] = (acc[0][v] + acc[1][v]) + (acc[2][v] + acc[3][v]) + bias;
  return z;
}

// What a minibatch leaves for the weight gradients: inputs and outputs' gradients of the four layers (M rows each).
struct MlpAct {
  float *X, *H1, *H2, *H3, *D1, *D2, *D3, *D4;
};

// Forward pass of M samples (rows idx[m] of X and lab, or m itself): Z_l = H_(l-1) W_l + b_l, H_l = relu(Z_l),
// then the softmax of the logits into P; with GRAD the mean cross-entropy's gradient goes back through the
// layers instead: loss (per sample) and everything that the weight gradients read into `act`.
// Latency bound on a minibatch (a chain of seven layers for each 16 samples), so one launch keeps the tile in
// LDS with all weights of the wave's columns loaded ahead into registers: 8.4 us for 1024 samples, where a launch
// per layer (gather, four forward, softmax, three backward, each through memory) cost 6 to 9 us nine times.
template <bool GRAD>
__global__ __launch_bounds__(256) void k_mlp(int M, const int *__restrict__ idx, const float *__restrict__ X,
                                             const int *__restrict__ lab, const float *__restrict__ p,
                                             float *__restrict__ P, float *__restrict__ loss, MlpAct act, float scale) {
  __shared__ __align__(16) float T[2][16 * MT_LD];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, g = lane >> 4, i = lane & 15;
  const int col = 16 * w + i;
  f32x4 w1[1], w2[4], w3[4], w4[4], t4[1], t3[4], t2[4];
  wf<NIN>(p + P_W1, NH, col, true, g, w1);
  wf<NH>(p + P_W2, NH, col, true, g, w2);
  wf<NH>(p + P_W3, NH, col, true, g, w3);
  wf<NH>(p + P_W4, NOUT, i, i < NOUT, g, w4);  // every wave holds the one tile of the output layer
  if (GRAD) {
    wt<NOUT>(p + P_W4, NOUT, col, g, t4);
    wt<NH>(p + P_W3, NH, col, g, t3);
    wt<NH>(p + P_W2, NH, col, g, t2);
  }
  const float b1 = p[P_B1 + col], b2 = p[P_B2 + col], b3 = p[P_B3 + col], b4 = p[P_B4 + (i & (NOUT - 1))];
  const int ntiles = (M + 15) >> 4;
  for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int m0 = 16 * tile;
    // lane (s, k) of the first two waves: input k and, later, logit k of sample s
    const int s = tid >> 3, k = tid & 7, ms = m0 + s;
    const bool sok = tid < 128 && ms < M;
    const int src = sok ? (idx ? idx[ms] : ms) : 0;
    int ls = -1;
    if (tid < 128) {
      const float x = sok && k < NIN ? X[(size_t)src * NIN + k] : 0.f;
      if (sok && lab) ls = lab[src];
      T[0][s * MT_LD + k] = x;
      T[0][s * MT_LD + 8 + k] = 0.f;
      if (GRAD && act.X && sok && k < NIN) act.X[(size_t)ms * NIN + k] = x;
    }
    __syncthreads();
    // H of a layer into the other tile and, for the weight gradients, to memory
    auto put = [&](float *dst, float *glob, f32x4 h) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        dst[(4 * g + v) * MT_LD + col] = h[v];
        if (GRAD && m0 + 4 * g + v < M) glob[(size_t)(m0 + 4 * g + v) * NH + col] = h[v];
      }
      __syncthreads();
    };
    auto relu = [](f32x4 z) {
#pragma unroll
      for (int v = 0; v < 4; ++v) z[v] = fmaxf(z[v], 0.f);
      return z;
    };
    auto where = [](f32x4 z, f32x4 h) {  // the ReLU's backward: h > 0 where its input was
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (!(h[v] > 0.f)) z[v] = 0.f;
      return z;
    };
    const f32x4 h1 = relu(mlp_tile<1>(T[0], w1, g, i, b1));
    put(T[1], act.H1, h1);
    const f32x4 h2 = relu(mlp_tile<4>(T[1], w2, g, i, b2));
    put(T[0], act.H2, h2);
    const f32x4 h3 = relu(mlp_tile<4>(T[0], w3, g, i, b3));
    put(T[1], act.H3, h3);
    if (w == 0) {
      const f32x4 z = mlp_tile<4>(T[1], w4, g, i, b4);
      if (i < NOUT)
#pragma unroll
        for (int v = 0; v < 4; ++v) T[0][(4 * g + v) * MT_LD + i] = z[v];
    }
    __syncthreads();
    if (w < 2) {  // softmax cross-entropy, a lane per logit; the sum runs over the logits in order
      const float *z = &T[0][s * MT_LD];
      const float zk = z[k];
      float mx = z[0];
#pragma unroll
      for (int j = 1; j < NOUT; ++j) mx = fmaxf(mx, z[j]);
      const float ek = expf(zk - mx);
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < NOUT; ++j) sum += __shfl(ek, (lane & ~7) + j, 64);
      const float pk = ek / sum;
      if (P && sok) P[(size_t)ms * NOUT + k] = pk;
      if (GRAD) {
        const float d = (pk - (ls == k ? 1.f : 0.f)) * scale;
        if (sok && ls == k) loss[ms] = -(zk - mx - logf(sum));
        T[1][s * MT_LD + k] = sok ? d : 0.f;
        T[1][s * MT_LD + 8 + k] = 0.f;
        if (sok) act.D4[(size_t)ms * NOUT + k] = d;
      }
    }
    __syncthreads();
    if (GRAD) {
      const f32x4 d3 = where(mlp_tile<1>(T[1], t4, g, i, 0.f), h3);
      put(T[0], act.D3, d3);
      const f32x4 d2 = where(mlp_tile<4>(T[0], t3, g, i, 0.f), h2);
      put(T[1], act.D2, d2);
      const f32x4 d1 = where(mlp_tile<4>(T[1], t2, g, i, 0.f), h1);
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (m0 + 4 * g + v < M) act.D1[(size_t)(m0 + 4 * g + v) * NH + col] = d1[v];
    }
  }
}

struct AdamStep {
  float *m, *v;  // moments; the parameters move when m is set, else the gradient is written
  float lr, b1, b2, eps, c1, c2;
};

// Weight and bias gradients of all layers, G = A^T D (A: M x NI, D: M x NO, row-major) and the column sums of
// D, and the Adam step with them. One 1024-thread block per 16x16 tile of a G: its 16 waves take the samples
// 16 at a time in turn, four turns' loads together, and their partial tiles are added in a fixed order through
// LDS, a wave per row of the lanes' results. The blocks of the first row of tiles (tm = 0) also take the bias.
// Latency bound on a minibatch: 6.5 us for 1024 samples, where the four layers and Adam's step were five launches of
// 6 to 9 us in a row. A minibatch with its host share went from 98 to 19 us.
constexpr int WG_WAVES = 16, WG_TURNS = 4;
constexpr int WG_BLOCKS = 4 + 16 + 16 + 4;
__global__ __launch_bounds__(1024) void k_mlp_update(int M, MlpAct act, float *__restrict__ p, float *__restrict__ grad,
                                                     AdamStep ad) {
  __shared__ float part[WG_WAVES][5][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int bid = blockIdx.x;
  const int layer = bid < 4 ? 0 : bid < 20 ? 1 : bid < 36 ? 2 : 3;
  const int tile = bid - (layer == 0 ? 0 : layer == 1 ? 4 : layer == 2 ? 20 : 36);
  const int NI = layer == 0 ? NIN : NH, NO = layer == 3 ? NOUT : NH;
  const float *__restrict__ A = layer == 0 ? act.X : layer == 1 ? act.H1 : layer == 2 ? act.H2 : act.H3;
  const float *__restrict__ D = layer == 0 ? act.D1 : layer == 1 ? act.D2 : layer == 2 ? act.D3 : act.D4;
  const int pw = layer == 0 ? P_W1 : layer == 1 ? P_W2 : layer == 2 ? P_W3 : P_W4;
  const int pb = layer == 0 ? P_B1 : layer == 1 ? P_B2 : layer == 2 ? P_B3 : P_B4;
  const int tiles_n = (NO + 15) >> 4;
  const int tm = tile / tiles_n, tn = tile - tm * tiles_n;
  const int g = lane >> 4, i = lane & 15;
  const int row = 16 * tm + i, col = 16 * tn + i;
  const bool rok = row < NI, cok = col < NO;
  const float *__restrict__ Ar = A + (rok ? row : 0), *__restrict__ Dc = D + (cok ? col : 0);
  f32x4 acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float cs = 0.f;  // this lane's share of the column sum of D
  for (int m0 = 16 * w; m0 < M; m0 += 16 * WG_WAVES * WG_TURNS) {
    f32x4 a[WG_TURNS], d[WG_TURNS];
#pragma unroll
    for (int u = 0; u < WG_TURNS; ++u)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int m = m0 + 16 * WG_WAVES * u + 4 * g + t;
        const size_t mm = m < M ? m : 0;
        a[u][t] = Ar[mm * NI];
        d[u][t] = Dc[mm * NO];
      }
#pragma unroll
    for (int u = 0; u < WG_TURNS; ++u) {
      if (m0 + 16 * WG_WAVES * u >= M) break;  // uniform over the wave
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const bool mok = m0 + 16 * WG_WAVES * u + 4 * g + t < M;
        const float av = rok && mok ? a[u][t] : 0.f, dv = cok && mok ? d[u][t] : 0.f;
        cs += dv;
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, dv, acc[t], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) part[w][v][lane] = (acc[0][v] + acc[1][v]) + (acc[2][v] + acc[3][v]);
  part[w][4][lane] = cs;
  __syncthreads();
  if (w > 4) return;
  float gg = 0.f;
#pragma unroll
  for (int u = 0; u < WG_WAVES; ++u) gg += part[u][w][lane];
  int t;
  bool ok;
  if (w < 4) {
    const int r = 16 * tm + 4 * g + w;
    ok = cok && r < NI;
    t = pw + r * NO + col;
  } else {
    // the column sum: the four lane groups hold sums over disjoint samples (all lanes take part)
    gg += __shfl_xor(gg, 16, 64);
    gg += __shfl_xor(gg, 32, 64);
    ok = cok && tm == 0 && g == 0;
    t = pb + col;
  }
  if (!ok) return;
  if (!ad.m) {
    grad[t] = gg;
    return;
  }
  const float mm = ad.b1 * ad.m[t] + (1.f - ad.b1) * gg;
  const float vv = ad.b2 * ad.v[t] + (1.f - ad.b2) * gg * gg;
  ad.m[t] = mm;
  ad.v[t] = vv;
  p[t] -= ad.lr * (mm / ad.c1) / (sqrtf(vv / ad.c2) + ad.eps);
}

// Buffers of one forward/backward pass on a minibatch of at most b samples.
struct MlpWork {
  DevBuf<float> buf;
  MlpAct act{};
  int alloc(andr_ctx *ctx, int b) {
    const size_t B = ((size_t)b + 3) / 4 * 4;
    if (buf.call_alloc(B * (NIN + 6 * NH + NOUT), ctx)) return 1;
    float *q = buf.p;
    for (float **h : {&act.H1, &act.H2, &act.H3, &act.D1, &act.D2, &act.D3}) {
      *h = q;
      q += B * NH;
    }
    act.D4 = q;
    act.X = q + B * NOUT;
    return 0;
  }
};

// blocks of k_mlp: more tiles than four blocks per CU share the weights in a block's registers
int mlp_blocks(int M) { return std::min((M + 15) / 16, 1024); }

// loss and gradients of the mean cross-entropy over M samples, then the step of `ad` (or the gradient out)
void mlp_step(hipStream_t st, int M, const int *idx, const float *X, const int *lab, float *p, MlpWork &w,
              float *loss, float *grad, const AdamStep &ad) {
  hipLaunchKernelGGL(k_mlp<true>, dim3(mlp_blocks(M)), dim3(256), 0, st, M, idx, X, lab, p, (float *)nullptr, loss,
                     w.act, 1.f / (float)M);
  hipLaunchKernelGGL(k_mlp_update, dim3(WG_BLOCKS), dim3(64 * WG_WAVES), 0, st, M, w.act, p, grad, ad);
}

// ---- inference inside the assembly: BF16 matrix cores, FP32 accumulation --------------------------
// The network runs transposed, H^T = W^T X^T: hidden units are the M dimension and pairs the N
// dimension of v_mfma_f32_16x16x16bf16_1k. With that orientation the accumulator tile of one layer
// (lane (g, c) holds rows 4g..4g+3 of a 16-row block for pair c) is, after bias, ReLU and rounding
// to BF16, exactly the B operand (rows 4g..4g+3 of a 16-deep K block, column c) of the next layer:
// the activations never leave the registers. Each wave keeps the 40 weight tiles (A operands) in
// registers, collects the near pairs of its row in an LDS queue and evaluates them 64 at a time
// (4 column blocks of 16 pairs), for the Stokes-G and Stokes-H kernel ids.
typedef short bf16x4 __attribute__((ext_vector_type(4)));

__device__ inline short f2bf(float x) {  // round to nearest even (v_cvt_pk_bf16_f32)
  return __builtin_bit_cast(short, (__bf16)x);
}

constexpr int CLS_THREADS = 256, CLS_WAVES = CLS_THREADS / 64, CLS_Q = 128;
// rows from which k_classify gives each wave one: 1280 rows 91 us either way, 2000 rows 108 (139 with a block
// a row), 3920 196 (248); but 500 rows 76 (46)
constexpr int CLS_WAVE_ROWS = 1536;

// lane (g, i): A[m = 16 mt + i][k = 16 kt + 4 g + t] = W[in = 16 kt + 4 g + t][out = 16 mt + i]
// (0 outside the layer). The 40 tiles are packed on the host when the model is set, lane by lane in
// operand order: tile index CLS_T_* + ..., then lane, then t (the A operand of one lane).
constexpr int CLS_T_W1 = 0, CLS_T_W2 = 4, CLS_T_W3 = 20, CLS_T_W4 = 36, CLS_NTILES = 40;
// the device model buffer: FP32 parameters, BF16 parameters, far table, rule sizes, then the packed
// tiles (16-byte aligned)
constexpr size_t model_tiles_off() {
  return (NPARAM * (sizeof(uint16_t) + sizeof(float)) + ANDR_FAR_BINS * sizeof(int) + 8 * sizeof(int) + 15) / 16 * 16;
}
static void pack_tile(const uint16_t *w, int nin, int nout, int mt, int kt, uint16_t *out) {
  for (int lane = 0; lane < 64; ++lane) {
    const int g = lane >> 4, i = lane & 15;
    for (int t = 0; t < 4; ++t) {
      const int in = 16 * kt + 4 * g + t, o = 16 * mt + i;
      out[lane * 4 + t] = (in < nin && o < nout) ? w[in * nout + o] : (uint16_t)0;
    }
  }
}

// bias + ReLU + BF16 of an accumulator tile -> B operand of the next layer
__device__ inline bf16x4 act_tile(f32x4 c, const float *bias, int mt, int g) {
  bf16x4 r;
#pragma unroll
  for (int v = 0; v < 4; ++v) r[v] = f2bf(fmaxf(c[v] + bias[16 * mt + 4 * g + v], 0.f));
  return r;
}

// logits of 16 pairs (column block) for one kernel id; returns in lanes g == 0 the class and the
// rule class of pair c (quantile decision, see below)
__device__ inline void mlp_block(const bf16x4 *lt /* this lane's entry of tile 0, in LDS */, const float *sb,
                                 const float *feat /* [16][3] */, int kernel, int g, int c, float min_conf, int *cls,
                                 float *conf) {
  bf16x4 x;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int f = 4 * g + t;  // feature index
    float v = 0.f;
    if (f < 3) v = feat[3 * c + f];
    else if (f == 3 + kernel) v = 1.f;
    x[t] = f2bf(v);
  }
  bf16x4 h1[4], h2[4];
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(lt[(CLS_T_W1 + mt) * 64], x, acc, 0, 0, 0);
    h1[mt] = act_tile(acc, sb + 0, mt, g);
  }
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(lt[(CLS_T_W2 + 4 * mt + kt) * 64], h1[kt], acc, 0, 0, 0);
    h2[mt] = act_tile(acc, sb + NH, mt, g);
  }
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(lt[(CLS_T_W3 + 4 * mt + kt) * 64], h2[kt], acc, 0, 0, 0);
    h1[mt] = act_tile(acc, sb + 2 * NH, mt, g);
  }
  f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kt = 0; kt < 4; ++kt) z = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(lt[(CLS_T_W4 + kt) * 64], h1[kt], z, 0, 0, 0);
  // classes 4g + v; lanes g = 0 hold classes 0..3 of pair c, lanes g = 1 classes 4..7
  float zz[8];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const float mine = z[v] + (g < 2 ? sb[3 * NH + 4 * g + v] : 0.f);
    const float other = __shfl_xor(mine, 16, 64);
    zz[v] = g == 0 ? mine : other;
    zz[4 + v] = g == 0 ? other : mine;
  }
  // The classes are ordered (a rule that is good enough stays good enough for every larger class),
  // so the decision is a quantile of the predicted label distribution: the smallest class whose
  // cumulative probability reaches min_conf. *conf is 1 when that happens below the last class.
  float mx = zz[0];
#pragma unroll
  for (int o = 1; o < NOUT; ++o) mx = fmaxf(mx, zz[o]);
  float e[NOUT], sum = 0.f;
#pragma unroll
  for (int o = 0; o < NOUT; ++o) {
    e[o] = __expf(zz[o] - mx);  // the quantile decision needs no last-ulp exponentials
    sum += e[o];
  }
  const float target = min_conf * sum;
  float cum = 0.f;
  int pick = NOUT - 1;
  bool found = false;
#pragma unroll
  for (int o = 0; o < NOUT; ++o) {
    cum += e[o];
    if (!found && cum >= target) {
      pick = o;
      found = true;
    }
  }
  *cls = pick;
  *conf = found ? 1.f : 0.f;
}

// Rule class of every pair of a row: a wave per (job, row) (WROW), or the block's four waves a row in turn where
// the rows are too few to fill the chip. Latency of the batches: near pairs are few (of the order of a hundred a
// row), so four waves of a row end with a quarter-full batch each, and every row pays for the network's tiles
// in LDS. 40 bodies, 102752 rows: 4.9 -> 3.0 ms with a wave per row.
template <bool WROW>
__global__ __launch_bounds__(CLS_THREADS, 3) void k_classify(const SysJob *__restrict__ jobs,
                                                          const int2 *__restrict__ rowmap, int nrows,
                                                          const bf16x4 *__restrict__ tiles, const float *__restrict__ wf,
                                                          const int *__restrict__ far_table,
                                                          double near_ratio,
                                                          float min_conf, unsigned long long *__restrict__ stats) {
  __shared__ float sb[3 * NH + NOUT];                 // biases b1, b2, b3, b4
  __shared__ int sfar[ANDR_FAR_BINS];
  __shared__ int qe[CLS_WAVES][CLS_Q];                // queued near pairs: element
  __shared__ float qf[CLS_WAVES][64][3];              // three geometric features of a batch
  __shared__ int qres[CLS_WAVES][64][2];              // class per kernel of a processed batch
  __shared__ bf16x4 s_tiles[CLS_NTILES * 64];  // the network's operand tiles, shared by the block's waves
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int g = lane >> 4, c = lane & 15;
  for (int i = threadIdx.x; i < NH; i += blockDim.x) {
    sb[i] = wf[P_B1 + i];
    sb[NH + i] = wf[P_B2 + i];
    sb[2 * NH + i] = wf[P_B3 + i];
  }
  if (threadIdx.x < NOUT) sb[3 * NH + threadIdx.x] = wf[P_B4 + threadIdx.x];
  if (threadIdx.x < ANDR_FAR_BINS) sfar[threadIdx.x] = far_table[threadIdx.x];
  // the operand tiles (packed lane by lane when the model was set) into LDS: the four waves use the
  // same tiles, and registers stay free for occupancy
  for (int i = threadIdx.x; i < CLS_NTILES * 64; i += blockDim.x) s_tiles[i] = tiles[i];
  const bf16x4 *lt = s_tiles + lane;
  __syncthreads();
  const int row = WROW ? blockIdx.x * CLS_WAVES + __builtin_amdgcn_readfirstlane(wid) : blockIdx.x;
  if (row >= nrows) return;  // no barriers of the block below
  const int2 jr = rowmap[row];
  const SysJob &J = jobs[jr.x];
  const BodyGeom &g_ = J.g;
  const int r = jr.y, ne = g_.ne;
  uint8_t *crow = J.cls + (size_t)r * ne;
  const float inv_nr2 = (float)(1.0 / (near_ratio * near_ratio));
  const float4 sr = g_.cenl[r];
  unsigned pts = 0, nl = 0, nf = 0;  // per lane and row: at most 8000 x 126 points
  int qn = 0;  // queue length (wave-uniform)
  // classify the first `cnt` queued pairs (all lanes take part: the matrix cores need a full wave)
  // rule points of a class: Dunavant sizes {3,4,6,7,12,13,19} (6 bits each), the fixed rule's J.nq
  auto npts = [&](int cl) { return cl == NCLS_DUN ? J.nq : (int)((0x1334C1C6103ull >> (6 * cl)) & 63); };
  auto run_batch = [&](int cnt) {
    // the features of the batch's pairs, one per lane (the FP64 pair geometry with every lane busy);
    // unused slots get harmless features
    {
      float f0 = 0.f, f1 = 0.f, f2 = 1.f;
      if (lane < cnt) {
        const int e = qe[wid][lane];
        const double *x1 = g_.xyz + 3 * g_.con[3 * e], *x2 = g_.xyz + 3 * g_.con[3 * e + 1],
                     *x3 = g_.xyz + 3 * g_.con[3 * e + 2];
        const double n[3] = {g_.nrm[3 * e], g_.nrm[3 * e + 1], g_.nrm[3 * e + 2]};
        float f[NIN];
        // the row's centroid and normal, read here (not held in registers through the scan)
        const double s[3] = {g_.cen[3 * r], g_.cen[3 * r + 1], g_.cen[3 * r + 2]};
        const double ns[3] = {g_.nrm[3 * r], g_.nrm[3 * r + 1], g_.nrm[3 * r + 2]};
        features(pair_geo(s, ns, x1, x2, x3, n, g_.area[e]), 0, f);
        f0 = f[0];
        f1 = f[1];
        f2 = f[2];
      }
      qf[wid][lane][0] = f0;
      qf[wid][lane][1] = f1;
      qf[wid][lane][2] = f2;
      __builtin_amdgcn_wave_barrier();
    }
    for (int blk = 0; blk < 4; ++blk) {
      if (16 * blk >= cnt) break;  // uniform
      const float *feat = &qf[wid][16 * blk][0];
      int a, b;
      float ca, cb;  // whether the quantile was reached below the last class (unused here)
      mlp_block(lt, sb, feat, 1, g, c, min_conf, &a, &ca);
      mlp_block(lt, sb, feat, 2, g, c, min_conf, &b, &cb);
      if (g == 0) {
        qres[wid][16 * blk + c][0] = a;
        qres[wid][16 * blk + c][1] = b;
      }
    }
    __builtin_amdgcn_wave_barrier();
    if (lane < cnt) {
      const int a = qres[wid][lane][0], b = qres[wid][lane][1];
      uint8_t cl;
      if (a == NCLS_DUN || b == NCLS_DUN) {
        cl = NCLS_DUN;
        ++nf;
      } else {
        cl = (uint8_t)max(a, b);
        ++nl;
      }
      pts += npts(cl);
      crow[qe[wid][lane]] = cl;
    }
    __builtin_amdgcn_wave_barrier();
  };
  // scan the row (or every fourth group of 64 elements of it); near pairs are queued and
  // classified 64 at a time, the rest of the queue once the scan is done (one batch call site)
  int base = WROW ? 0 : wid * 64;
  for (;;) {
    if (base < ne) {
      const int e = base + lane;
      bool near = false;
      if (e < ne) {
        // far test on squared distances from the stored centroid and longest edge (FP32): dh >=
        // near_ratio is d^2 >= near_ratio^2 L^2, and the half-octave bin floor(2 log2(dh / near_ratio))
        // is the binary exponent of d^2 / (near_ratio^2 L^2)
        const float4 ce = g_.cenl[e];
        const float dx = sr.x - ce.x, dy = sr.y - ce.y, dz = sr.z - ce.z;
        const float q = (dx * dx + dy * dy + dz * dz) * ce.w * inv_nr2;
        if (e == r) {
          crow[e] = NCLS_DUN;
        } else if (q >= 1.f) {
          const int cl = sfar[min(ilogbf(q), ANDR_FAR_BINS - 1)];
          crow[e] = (uint8_t)cl;
          pts += npts(cl);
        } else {
          near = true;  // queued: its features are formed in the batch, all lanes busy
        }
      }
      const unsigned long long m = __ballot(near);
      const int pos = qn + __popcll(m & ((1ull << lane) - 1ull));
      if (near) qe[wid][pos] = e;
      qn += __popcll(m);
      base += WROW ? 64 : CLS_THREADS;
      __builtin_amdgcn_wave_barrier();
    }
    const bool scanned = base >= ne;  // uniform over the wave
    if (qn >= 64 || (scanned && qn > 0)) {
      const int cnt = min(qn, 64);
      run_batch(cnt);
      qn -= cnt;
      // move the rest (< 64) to the front
      const int te = lane < qn ? qe[wid][64 + lane] : 0;
      __builtin_amdgcn_wave_barrier();
      if (lane < qn) qe[wid][lane] = te;
      __builtin_amdgcn_wave_barrier();
    } else if (scanned) {
      break;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    pts += __shfl_xor(pts, o, 64);
    nl += __shfl_xor(nl, o, 64);
    nf += __shfl_xor(nf, o, 64);
  }
  if (lane < 3) atomicAdd(stats + 3 * (size_t)jr.x + lane, (unsigned long long)(lane == 0 ? pts : lane == 1 ? nl : nf));
}

RuleTab dunavant_tab(int qoff_fixed, int nq_fixed) {
  RuleTab t;
  for (int c = 0; c < NCLS_DUN; ++c) {
    QuadRule q = andr_rule(DUN_ID0 + c);
    t.off[c] = q.offset;
    t.n[c] = q.npts;
  }
  t.off[NCLS_DUN] = qoff_fixed;
  t.n[NCLS_DUN] = nq_fixed;
  return t;
}

}  // namespace

// ---- C-ABI -----------------------------------------------------------------------------------------
static int labels_common(andr_ctx *ctx, const andr_mesh *mesh, double near_ratio, double rel_tol, int mode,
                         int64_t max_pairs, float *features_out, int32_t *labels_out, int64_t *npairs,
                         int32_t *far_table) {
  if (!ctx) return ANDR_ERR_ARG;
  if (!(near_ratio > 0.0) || !(rel_tol > 0.0)) return andr_fail(ctx, ANDR_ERR_ARG, "near_ratio and rel_tol must be > 0");
  if (mesh && mesh->nvert == 4) return andr_fail(ctx, ANDR_ERR_ARG, "quadrature training takes triangle meshes");
  ANDR_HIP(ctx, hipSetDevice(ctx->device));
  DevBody b;
  int rc = andr_body_upload(ctx, mesh, b, false);
  if (rc) return rc;
  const QuadRule ref = andr_rule(b.itri);
  RuleTab rt = dunavant_tab(ref.offset, ref.npts);
  DevBuf<float> df;
  DevBuf<int> dl, dfar;
  DevBuf<unsigned long long> cnt;
  const int64_t mp = mode == 0 ? std::max<int64_t>(max_pairs, 1) : 1;
  andr_pool_headroom(ctx);  // the label kernel's private arrays: others may have filled the device meanwhile
  if (df.call_alloc((size_t)mp * 6, ctx) || dl.call_alloc(mp, ctx) || dfar.alloc(ANDR_FAR_BINS, ctx) ||
      cnt.alloc(1, ctx))
    return andr_fail(ctx, ANDR_ERR_ALLOC, "training pair buffers");
  uint32_t keep = 0xFFFFFFFFu;
  unsigned long long n = 0;
  if (mode == 0) {  // count first; sample the pairs uniformly when they exceed max_pairs
    ANDR_HIP(ctx, hipMemsetAsync(cnt.p, 0, sizeof(unsigned long long), ctx->stream));
    hipLaunchKernelGGL(k_pair_labels, dim3(b.g.ne), dim3(256), 0, ctx->stream, b.g, ref.offset, ref.npts, rt,
                       near_ratio, rel_tol, 2, keep, mp, df.p, dl.p, cnt.p, dfar.p);
    ANDR_HIP(ctx, hipGetLastError());
    ANDR_HIP(ctx, hipMemcpyAsync(&n, cnt.p, sizeof(n), hipMemcpyDeviceToHost, ctx->stream));
    ANDR_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if ((double)n > (double)max_pairs)
      keep = (uint32_t)std::min(4294967295.0, 0.97 * (double)max_pairs / (double)n * 4294967296.0);
  }
  ANDR_HIP(ctx, hipMemsetAsync(cnt.p, 0, sizeof(unsigned long long), ctx->stream));
  ANDR_HIP(ctx, hipMemsetAsync(dfar.p, 0xff, sizeof(int) * ANDR_FAR_BINS, ctx->stream));  // -1: bin not seen
  hipLaunchKernelGGL(k_pair_labels, dim3(b.g.ne), dim3(256), 0, ctx->stream, b.g, ref.offset, ref.npts, rt, near_ratio,
                     rel_tol, mode, keep, mp, df.p, dl.p, cnt.p, dfar.p);
  ANDR_HIP(ctx, hipGetLastError());
  ANDR_HIP(ctx, hipMemcpyAsync(&n, cnt.p, sizeof(n), hipMemcpyDeviceToHost, ctx->stream));
  ANDR_HIP(ctx, hipStreamSynchronize(ctx->stream));
  if (mode == 0) {
    const int64_t k = std::min<int64_t>((int64_t)n, max_pairs);
    if (k > 0) {
      ANDR_HIP(ctx, hipMemcpy(features_out, df.p, sizeof(float) * 6 * k, hipMemcpyDeviceToHost));
      ANDR_HIP(ctx, hipMemcpy(labels_out, dl.p, sizeof(int) * k, hipMemcpyDeviceToHost));
    }
    if (npairs) *npairs = k;
  } else {
    ANDR_HIP(ctx, hipMemcpy(far_table, dfar.p, sizeof(int) * ANDR_FAR_BINS, hipMemcpyDeviceToHost));
  }
  return ANDR_OK;
}

extern "C" int andr_quad_training_pairs(andr_ctx *ctx, const andr_mesh *mesh, double near_ratio, double rel_tol,
                                        int64_t max_pairs, float *features_out, int32_t *labels_out, int64_t *npairs) {
  if (!features_out || !labels_out || max_pairs <= 0) return andr_fail(ctx, ANDR_ERR_ARG, "output buffers");
  return labels_common(ctx, mesh, near_ratio, rel_tol, 0, max_pairs, features_out, labels_out, npairs, nullptr);
}

extern "C" int andr_quad_far_calibration(andr_ctx *ctx, const andr_mesh *mesh, double near_ratio, double rel_tol,
                                         int32_t *far_table) {
  if (!far_table) return andr_fail(ctx, ANDR_ERR_ARG, "far_table");
  return labels_common(ctx, mesh, near_ratio, rel_tol, 1, 0, nullptr, nullptr, nullptr, far_table);
}

extern "C" int andr_mlp_loss_grad(andr_ctx *ctx, int64_t npairs, const float *features, const int32_t *labels,
                                  const float *params, float *loss, float *grad) {
  if (!ctx || npairs <= 0 || npairs > (1 << 24) || !features || !labels || !params || !grad)
    return ctx ? andr_fail(ctx, ANDR_ERR_ARG, "andr_mlp_loss_grad arguments") : ANDR_ERR_ARG;
  ANDR_HIP(ctx, hipSetDevice(ctx->device));
  const int M = (int)npairs;
  for (int64_t i = 0; i < npairs; ++i)
    if (labels[i] < 0 || labels[i] >= NOUT) return andr_fail(ctx, ANDR_ERR_ARG, "label out of range");
  MlpWork w;
  DevBuf<float> X, p, gr, dloss;
  DevBuf<int> L;
  if (w.alloc(ctx, M) || X.call_alloc((size_t)M * NIN, ctx) || p.alloc(NPARAM, ctx) || gr.alloc(NPARAM, ctx) ||
      dloss.call_alloc(M, ctx) || L.call_alloc(M, ctx))
    return andr_fail(ctx, ANDR_ERR_ALLOC, "MLP buffers");
  hipStream_t st = ctx->stream;
  ANDR_HIP(ctx, hipMemcpyAsync(X.p, features, sizeof(float) * M * NIN, hipMemcpyHostToDevice, st));
  ANDR_HIP(ctx, hipMemcpyAsync(L.p, labels, sizeof(int) * M, hipMemcpyHostToDevice, st));
  ANDR_HIP(ctx, hipMemcpyAsync(p.p, params, sizeof(float) * NPARAM, hipMemcpyHostToDevice, st));
  mlp_step(st, M, nullptr, X.p, L.p, p.p, w, dloss.p, gr.p, AdamStep{});
  ANDR_HIP(ctx, hipGetLastError());
  std::vector<float> hl(M);
  ANDR_HIP(ctx, hipMemcpyAsync(hl.data(), dloss.p, sizeof(float) * M, hipMemcpyDeviceToHost, st));
  ANDR_HIP(ctx, hipMemcpyAsync(grad, gr.p, sizeof(float) * NPARAM, hipMemcpyDeviceToHost, st));
  ANDR_HIP(ctx, hipStreamSynchronize(st));
  double s = 0.0;
  for (float v : hl) s += v;
  if (loss) *loss = (float)(s / M);
  return ANDR_OK;
}

extern "C" int andr_mlp_infer(andr_ctx *ctx, int64_t npairs, const float *features, const float *params, float *probs) {
  if (!ctx || npairs <= 0 || !features || !params || !probs)
    return ctx ? andr_fail(ctx, ANDR_ERR_ARG, "andr_mlp_infer arguments") : ANDR_ERR_ARG;
  ANDR_HIP(ctx, hipSetDevice(ctx->device));
  const int chunk = 1 << 16;
  DevBuf<float> X, p, P;
  if (P.alloc((size_t)chunk * NOUT, ctx) || X.alloc((size_t)chunk * NIN, ctx) || p.alloc(NPARAM, ctx))
    return andr_fail(ctx, ANDR_ERR_ALLOC, "MLP buffers");
  hipStream_t st = ctx->stream;
  ANDR_HIP(ctx, hipMemcpyAsync(p.p, params, sizeof(float) * NPARAM, hipMemcpyHostToDevice, st));
  for (int64_t i0 = 0; i0 < npairs; i0 += chunk) {
    const int M = (int)std::min<int64_t>(chunk, npairs - i0);
    ANDR_HIP(ctx, hipMemcpyAsync(X.p, features + i0 * NIN, sizeof(float) * M * NIN, hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_mlp<false>, dim3(mlp_blocks(M)), dim3(256), 0, st, M, (const int *)nullptr, X.p,
                       (const int *)nullptr, p.p, P.p, (float *)nullptr, MlpAct{}, 1.f);
    ANDR_HIP(ctx, hipGetLastError());
    ANDR_HIP(ctx, hipMemcpyAsync(probs + i0 * NOUT, P.p, sizeof(float) * M * NOUT, hipMemcpyDeviceToHost, st));
    ANDR_HIP(ctx, hipStreamSynchronize(st));
  }
  return ANDR_OK;
}

extern "C" int andr_mlp_train(andr_ctx *ctx, int64_t npairs, const float *features, const int32_t *labels,
                              int32_t epochs, int32_t batch, float lr, uint64_t seed, float *params, float *loss_out) {
  if (!ctx || npairs <= 0 || npairs > (1 << 26) || !features || !labels || !params || epochs <= 0 || batch <= 0)
    return ctx ? andr_fail(ctx, ANDR_ERR_ARG, "andr_mlp_train arguments") : ANDR_ERR_ARG;
  ANDR_HIP(ctx, hipSetDevice(ctx->device));
  for (int64_t i = 0; i < npairs; ++i)
    if (labels[i] < 0 || labels[i] >= NOUT) return andr_fail(ctx, ANDR_ERR_ARG, "label out of range");
  const int N = (int)npairs, B = std::min<int>(batch, N);
  const int steps = N / B, samples = (steps + 15) / 16;  // the loss of every 16th minibatch of an epoch is kept
  MlpWork w;
  DevBuf<float> X, p, m, v, loss;
  DevBuf<int> L, idx;
  if (w.alloc(ctx, B) || X.call_alloc((size_t)N * NIN, ctx) || p.alloc(NPARAM, ctx) || m.alloc(NPARAM, ctx) ||
      v.alloc(NPARAM, ctx) || loss.call_alloc((size_t)(samples + 1) * B, ctx) || L.call_alloc(N, ctx) ||
      idx.call_alloc(N, ctx))
    return andr_fail(ctx, ANDR_ERR_ALLOC, "MLP training buffers");
  hipStream_t st = ctx->stream;
  ANDR_HIP(ctx, hipMemcpyAsync(X.p, features, sizeof(float) * (size_t)N * NIN, hipMemcpyHostToDevice, st));
  ANDR_HIP(ctx, hipMemcpyAsync(L.p, labels, sizeof(int) * N, hipMemcpyHostToDevice, st));
  ANDR_HIP(ctx, hipMemcpyAsync(p.p, params, sizeof(float) * NPARAM, hipMemcpyHostToDevice, st));
  ANDR_HIP(ctx, hipMemsetAsync(m.p, 0, sizeof(float) * NPARAM, st));
  ANDR_HIP(ctx, hipMemsetAsync(v.p, 0, sizeof(float) * NPARAM, st));
  std::mt19937_64 rng(seed);
  std::vector<int> perm(N);
  std::vector<float> hl((size_t)samples * B);
  int64_t t = 0;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  for (int ep = 0; ep < epochs; ++ep) {
    std::iota(perm.begin(), perm.end(), 0);
    std::shuffle(perm.begin(), perm.end(), rng);
    ANDR_HIP(ctx, hipMemcpyAsync(idx.p, perm.data(), sizeof(int) * N, hipMemcpyHostToDevice, st));
    for (int b = 0; b < steps; ++b) {
      ++t;
      const float c1 = 1.f - powf(b1, (float)t), c2 = 1.f - powf(b2, (float)t);
      float *bl = loss.p + (size_t)((b & 15) == 0 ? b / 16 : samples) * B;
      mlp_step(st, B, idx.p + (size_t)b * B, X.p, L.p, p.p, w, bl, nullptr,
               AdamStep{m.p, v.p, lr, b1, b2, eps, c1, c2});
    }
    ANDR_HIP(ctx, hipGetLastError());
    ANDR_HIP(ctx, hipMemcpyAsync(hl.data(), loss.p, sizeof(float) * hl.size(), hipMemcpyDeviceToHost, st));
    ANDR_HIP(ctx, hipStreamSynchronize(st));
    double lsum = 0.0;
    for (int b = 0; b < samples; ++b) {
      double s = 0.0;
      for (int i = 0; i < B; ++i) s += hl[(size_t)b * B + i];
      lsum += s / B;
    }
    if (loss_out) loss_out[ep] = (float)(lsum / std::max(1, samples));
  }
  ANDR_HIP(ctx, hipMemcpyAsync(params, p.p, sizeof(float) * NPARAM, hipMemcpyDeviceToHost, st));
  ANDR_HIP(ctx, hipStreamSynchronize(st));
  return ANDR_OK;
}

extern "C" int andr_set_quadrature_model(andr_ctx *ctx, const float *params, float confidence, double near_ratio,
                                         const int32_t *far_table) {
  if (!ctx || !params || !far_table || !(near_ratio > 0.0) || !(confidence >= 0.f && confidence <= 1.f))
    return ctx ? andr_fail(ctx, ANDR_ERR_ARG, "andr_set_quadrature_model arguments") : ANDR_ERR_ARG;
  for (int b = 0; b < ANDR_FAR_BINS; ++b)
    if (far_table[b] < 0 || far_table[b] > NCLS_DUN) return andr_fail(ctx, ANDR_ERR_ARG, "far_table class range");
  ANDR_HIP(ctx, hipSetDevice(ctx->device));
  std::vector<uint16_t> wb(NPARAM);
  for (int i = 0; i < NPARAM; ++i) {  // round to nearest even BF16
    uint32_t u;
    std::memcpy(&u, &params[i], 4);
    u += 0x7fffu + ((u >> 16) & 1u);
    wb[i] = (uint16_t)(u >> 16);
  }
  // packed operand tiles of the classifier after the tables (16-byte aligned)
  const size_t tiles_off = model_tiles_off();
  const size_t bytes = tiles_off + (size_t)CLS_NTILES * 64 * 4 * sizeof(uint16_t);
  std::vector<uint16_t> packed((size_t)CLS_NTILES * 64 * 4);
  for (int mt = 0; mt < 4; ++mt) {
    pack_tile(wb.data() + P_W1, NIN, NH, mt, 0, packed.data() + (size_t)(CLS_T_W1 + mt) * 256);
    pack_tile(wb.data() + P_W4, NH, NOUT, 0, mt, packed.data() + (size_t)(CLS_T_W4 + mt) * 256);
    for (int kt = 0; kt < 4; ++kt) {
      pack_tile(wb.data() + P_W2, NH, NH, mt, kt, packed.data() + (size_t)(CLS_T_W2 + 4 * mt + kt) * 256);
      pack_tile(wb.data() + P_W3, NH, NH, mt, kt, packed.data() + (size_t)(CLS_T_W3 + 4 * mt + kt) * 256);
    }
  }
  // the previous model is gone from here on: a learned call made after a failure below is refused
  ctx->has_model = false;
  if (ctx->d_model) (void)hipFree(ctx->d_model);
  ctx->d_model = nullptr;
  ANDR_HIP(ctx, hipMalloc(&ctx->d_model, bytes));
  char *base = (char *)ctx->d_model;
  float *fp = (float *)base;
  uint16_t *bp = (uint16_t *)(base + NPARAM * sizeof(float));
  int *far = (int *)(base + NPARAM * (sizeof(float) + sizeof(uint16_t)));
  int *npts = far + ANDR_FAR_BINS;
  int hn[8];
  for (int c = 0; c < NCLS_DUN; ++c) hn[c] = andr_rule(DUN_ID0 + c).npts;
  hn[NCLS_DUN] = 0;
  ANDR_HIP(ctx, hipMemcpy(fp, params, sizeof(float) * NPARAM, hipMemcpyHostToDevice));
  ANDR_HIP(ctx, hipMemcpy(bp, wb.data(), sizeof(uint16_t) * NPARAM, hipMemcpyHostToDevice));
  ANDR_HIP(ctx, hipMemcpy(far, far_table, sizeof(int) * ANDR_FAR_BINS, hipMemcpyHostToDevice));
  ANDR_HIP(ctx, hipMemcpy(npts, hn, sizeof(hn), hipMemcpyHostToDevice));
  ANDR_HIP(ctx, hipMemcpy(base + tiles_off, packed.data(), sizeof(uint16_t) * packed.size(), hipMemcpyHostToDevice));
  ctx->has_model = true;
  ctx->model_conf = confidence;
  ctx->model_near = near_ratio;
  return ANDR_OK;
}

int andr_launch_stokes_system_learned(andr_ctx *ctx, SysJob *h_jobs, const SysJob *d_jobs, const int2 *d_rowmap,
                                      int nrows, int njobs, bool summed, LearnedStats *stats) {
  if (!ctx->has_model) return andr_fail(ctx, ANDR_ERR_STATE, "no quadrature model");
  char *base = (char *)ctx->d_model;
  const float *fp = (const float *)base;
  const int *far = (const int *)(base + NPARAM * (sizeof(float) + sizeof(uint16_t)));
  const size_t tiles_off = model_tiles_off();
  const bf16x4 *tiles = (const bf16x4 *)(base + tiles_off);
  DevBuf<unsigned long long> st;
  if (st.alloc(3 * (size_t)njobs, ctx)) return andr_fail(ctx, ANDR_ERR_ALLOC, "stats");
  ANDR_HIP(ctx, hipMemsetAsync(st.p, 0, 3 * sizeof(unsigned long long) * njobs, ctx->stream));
  const int tok = andr_prof_begin(ctx, "classify_pairs", 0.0, 0.0);
  auto classify = [&](auto kernel, int blocks) {
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(CLS_THREADS), 0, ctx->stream, d_jobs, d_rowmap, nrows, tiles, fp, far,
                       ctx->model_near, ctx->model_conf, st.p);
  };
  if (nrows >= CLS_WAVE_ROWS) classify(k_classify<true>, (nrows + CLS_WAVES - 1) / CLS_WAVES);
  else classify(k_classify<false>, nrows);
  andr_prof_end(ctx, tok);
  ANDR_HIP(ctx, hipGetLastError());
  std::vector<unsigned long long> hs(3 * (size_t)njobs);
  ANDR_HIP(ctx, hipMemcpyAsync(hs.data(), st.p, sizeof(unsigned long long) * hs.size(), hipMemcpyDeviceToHost,
                               ctx->stream));
  ANDR_HIP(ctx, hipStreamSynchronize(ctx->stream));
  // fast-form system: the six symmetric FP32 blocks, 6 F^2 entries of 4 bytes
  double bytes = 0.0, points = 0.0, near = 0.0, cls_bytes = 0.0;
  for (int i = 0; i < njobs; ++i) {
    bytes += 6.0 * h_jobs[i].g.ne * (double)h_jobs[i].g.ne * 4.0;
    cls_bytes += h_jobs[i].g.ne * (double)h_jobs[i].g.ne;  // one class byte per pair
    near += (double)(hs[3 * (size_t)i + 1] + hs[3 * (size_t)i + 2]);
    points += (double)hs[3 * (size_t)i];
    if (stats) {
      stats[i].points = (int64_t)hs[3 * (size_t)i];
      stats[i].learned = (int64_t)hs[3 * (size_t)i + 1];
      stats[i].fallback = (int64_t)hs[3 * (size_t)i + 2];
    }
  }
  if (tok >= 0) {  // the classification's work is known once the counts are back
    // two network passes per near pair (Stokeslet and stresslet), 2 x (6*64 + 64*64 + 64*64 + 64*8)
    // flops each on the BF16 matrix cores; the class bytes written
    ProfRec &r = andr_prof(ctx).pending[tok];
    r.flops = near * 2.0 * ANDR_MLP_FLOPS_PER_PASS;
    r.bytes = cls_bytes;
  }
  return andr_launch_stokes_system(ctx, d_jobs, d_rowmap, nrows, true, true, bytes,
                                   points * (summed ? ANDR_FLOPS_PER_STOKES_EVAL_SUM : ANDR_FLOPS_PER_STOKES_EVAL),
                                   summed);
}

int andr_upload_rules_learned(andr_ctx *ctx, const double *tab, const float *tabf) {
  return andr_upload_rules_here(ctx, tab, tabf);
}
