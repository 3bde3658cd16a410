// Multi-RHS LSQR on a dense device matrix: the plain FP64 drop-in for src/lib_lsqr.f.
//
// Every right-hand side follows its own Paige-Saunders recurrence (lsqr_LSQR, src/lib_lsqr.f:470-1207,
// damp = 0, conlim = 1e8, nconv = 1), but the two products of an iteration -- A v and A^T u -- are
// formed for all right-hand sides in one pass over A, so the matrix is streamed twice per iteration
// for the whole block instead of twice per iteration per right-hand side. Several right-hand sides
// share vectors of ANDR_NB interleaved columns; a single one runs on plain vectors (WD = 1 below),
// since eight columns for one cost eight times the partial sums and vector traffic.
//
// The u and v vectors are kept unnormalised together with their norms (true u = U / beta, true
// v = V / alpha); the products fold the normalisation into their scale factors, which removes the
// separate scaling passes of the reference (dscal at :947, :974, :980).
//
// A single right-hand side of at most 8192 unknowns takes two launches an iteration and reads A once: k_lsqr_pass
// does the work of 1. and 2. below on rows that stay in registers (not where they are narrow and many, PASS_MIN_COLS).
// Otherwise
// an iteration is three launches. A small system (an A of the order of the 256 MB cache) spends its
// time in the gaps and the latency of small kernels, not in the products, so the recurrences' scalar
// work and the vector updates ride along in the products' own kernels:
//   1. k_lsqr_av: the partial products of A V over column segments;
//   2. k_lsqr_atu: U = sx .* (A V) + sy .* U for its rows from those partials (each column panel for
//      itself, the first one keeps it), then the partial products of A^T U over row splits. Its blocks
//      start with the scalars that end the previous iteration (norm of V, plane rotations, stopping
//      tests), block (0, 0) for good (state B);
//   3. k_lsqr_v: V = sx .* (A^T U) + sy .* V from those partials, with the update of X and W that the
//      previous iteration still owes; starts with the scalars after A V (state A).
// With more than LSQR_FUSE_SEG column segments every panel's own sum over them would cost more than a
// launch (per row WD * 8 bytes a segment in each column panel against 1 KB of A), and
// k_lsqr_u forms U once, as for CSR matrices and for several right-hand sides of a large A (fuse_u below).
// Measured per iteration with seven launches and eight columns throughout against this: 3120^2, 6
// right-hand sides 73 -> 41 us; 4881 x 2717, one 84 -> 44 us; 1587^2, one 57 -> 18 us; 4897^2 in FP32, one
// 132 -> 40 us.
//
// The host reads the states of every LSQR_POLL-th iteration from pinned memory one poll late, so that
// the device never waits for it; the iterations enqueued past the end return at once. Where there is no pinned
// memory to be had it copies state B and waits.
#include "andr_internal.h"
#include "andr_solve.h"
#include "andr_prof.h"

#include <cmath>
#include <algorithm>
#include <cstring>
#include <type_traits>
#include <vector>

namespace {

constexpr int NB = ANDR_NB;

__device__ inline double d2norm(double a, double b) {  // lsqr_d2norm (src/lib_lsqr.f:1236-1263)
  double scale = fabs(a) + fabs(b);
  if (scale == 0.0) return 0.0;
  double x = a / scale, y = b / scale;
  return scale * sqrt(x * x + y * y);
}

typedef double d2n __attribute__((ext_vector_type(2)));
typedef double d4v __attribute__((ext_vector_type(4)));

// Loads of the system matrix. A matrix that the 256 MB cache holds is read with ordinary loads (KEEP): what of it
// is left in an L2 from the product before, and the second half of a line that two rows share, are then hits.
// A larger one is streamed past them. Measured: one pass over 106 MB 21.6 us streamed, 18.8 kept, 20 MB 9.9 and
// 7.5, FP32 96 MB 25.8 and 20.5; A^T U of 78 MB 20.0 and 17.2, A V 15.5 and 13.5; but 512 MB 84 and 90, 1.15 GB 173
// and 188. Each system of a batch is judged by itself, although four are solved at a time: four of 69 MB take 36 ms
// streamed and 30 kept, of 118 MB 60 and 53, three of 189 MB 85 and 82; only four of 189 MB 103 and 104.5.
constexpr double KEEP_BYTES = 256e6;
template <bool KEEP, class P>
__device__ inline auto stream_load(P p) {
  if constexpr (KEEP) return *p;
  else return __builtin_nontemporal_load(p);
}
typedef float f4n __attribute__((ext_vector_type(4)));

// ---- scalar state ----------------------------------------------------------------------------
// State A holds the columns after A V (k_lsqr_v writes it), state B at the end of an iteration
// (k_lsqr_atu / k_lsqr_u write it): each kernel reads one and its first block writes the other, so
// no block reads what another one of the same launch writes.

// Column sums of the partials part[i][k], i < np, k < WD, by a block of BS threads, in two parts: a
// thread's share (loads only: eight in flight, as the partials come from another kernel's blocks and
// each round trip to them is most of a microsecond), then the sum over the block, which thread k < WD
// receives for column k. Every thread of the block calls them; red holds BS / 64 * WD doubles.
template <int WD, int BS>
__device__ inline double thread_parts(const double *__restrict__ part, int np) {
  const int k = threadIdx.x % WD;
  double s = 0.0;
  for (int i = threadIdx.x / WD; i < np; i += 8 * (BS / WD)) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int j = i + u * (BS / WD);
      v[u] = j < np ? part[(size_t)j * WD + k] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) s += v[u];
  }
  return s;
}
template <int WD, int BS>
__device__ inline double block_sum(double s, double *red) {
  const int t = threadIdx.x;
#pragma unroll
  for (int o = WD; o < 64; o <<= 1) s += __shfl_xor(s, o, 64);
  __syncthreads();  // red may still be read from the previous call
  if ((t & 63) < WD) red[(t >> 6) * WD + (t & 63)] = s;
  __syncthreads();
  double v = 0.0;
  if (t < WD)
#pragma unroll
    for (int w = 0; w < BS / 64; w += 4)
      v += (red[w * WD + t] + red[(w + 1) * WD + t]) + (red[(w + 2) * WD + t] + red[(w + 3) * WD + t]);
  return v;
}
template <int WD, int BS>
__device__ inline double block_sum_parts(const double *__restrict__ part, int np, double *red) {
  return block_sum<WD, BS>(thread_parts<WD, BS>(part, np), red);
}

// the end of an iteration from |V|^2 and |W|^2: alpha, the plane rotations and the convergence tests
// (src/lib_lsqr.f:1015-1152); before the first one the initial recurrence values (:952-1008), whose
// "update" W = V / alpha has t1 = t2 = 0
__device__ inline void lsqr_end(LsqrState &S, double sv, double sw) {
  if (!S.active) {
    S.upd = 0;
    return;
  }
  S.upd = 1;  // the update of this iteration still applies (src/lib_lsqr.f:1057-1062)
  if (S.itn == 0) {
    S.alpha = S.beta > 0.0 ? sqrt(sv) : 0.0;
    S.t1 = S.t2 = 0.0;
    S.inv_alpha = S.alpha > 0.0 ? 1.0 / S.alpha : 0.0;
    S.rhobar = S.alpha;
    S.phibar = S.beta;
    S.bnorm = S.beta;
    S.rnorm = S.beta;
    if (S.alpha * S.beta == 0.0) S.active = 0;  // exact solution x = 0 (istop 0)
    return;
  }
  S.anorm = d2norm(S.anorm, d2norm(S.alpha, S.beta));  // (src/lib_lsqr.f:1009-1014, damp = 0)
  if (S.beta > 0.0) S.alpha = sqrt(sv);
  const double alpha = S.alpha, beta = S.beta;
  const double wnorm = sqrt(sw);
  const double rhbar1 = S.rhobar;
  const double rho = d2norm(rhbar1, beta);
  const double cs = rhbar1 / rho, sn = beta / rho;
  const double theta = sn * alpha;
  S.rhobar = -cs * alpha;
  const double phi = cs * S.phibar;
  S.phibar = sn * S.phibar;
  const double tau = sn * phi;
  S.t1 = phi / rho;
  S.t2 = -theta / rho;
  const double dknorm = (1.0 / rho) * wnorm;
  S.dnorm = d2norm(S.dnorm, dknorm);
  const double delta = S.sn2 * rho, gambar = -S.cs2 * rho;
  const double rhs = phi - delta * S.z, zbar = rhs / gambar;
  S.xnorm = d2norm(S.xnorm1, zbar);
  const double gamma = d2norm(gambar, theta);
  S.cs2 = gambar / gamma;
  S.sn2 = theta / gamma;
  S.z = rhs / gamma;
  S.xnorm1 = d2norm(S.xnorm1, S.z);
  const double acond = S.anorm * S.dnorm;
  S.res2 = d2norm(S.res2, 0.0);
  S.rnorm = d2norm(S.res2, S.phibar);
  const double arnorm = alpha * fabs(tau);
  const double test1 = S.rnorm / S.bnorm;
  const double test2 = S.rnorm > 0.0 ? arnorm / (S.anorm * S.rnorm) : 0.0;
  const double test3 = 1.0 / acond;
  double tt1 = test1 / (1.0 + S.anorm * S.xnorm / S.bnorm);
  const double rtol = S.btol + S.atol * S.anorm * S.xnorm / S.bnorm;
  const double tt3 = 1.0 + test3, tt2 = 1.0 + test2;
  tt1 = 1.0 + tt1;
  int istop = 0;
  if (S.itn >= S.itnlim) istop = 5;
  if (tt3 <= 1.0) istop = 4;
  if (tt2 <= 1.0) istop = 2;
  if (tt1 <= 1.0) istop = 1;
  if (test3 <= S.ctol) istop = 4;
  if (test2 <= S.atol) istop = 2;
  if (test1 <= rtol) istop = 1;
  S.istop = istop;
  S.inv_alpha = alpha > 0.0 ? 1.0 / alpha : 1.0;
  if (istop != 0) S.active = 0;
}

// the scales of U = sx .* (A V) + sy .* U alone, which every block needs. A column that stops in this
// very iteration still gets them: its U and V are not used any more and stay finite.
__device__ inline void lsqr_u_scales(const LsqrState &S, double sv, double &sx, double &sy) {
  sx = sy = 0.0;
  if (!S.active) return;
  const double alpha = S.beta > 0.0 ? sqrt(sv) : (S.itn == 0 ? 0.0 : S.alpha);
  if (alpha != 0.0 && S.beta != 0.0) {  // (a NaN passes, as through the recurrences)
    sx = 1.0 / alpha;
    sy = -alpha / S.beta;
  }
}

// BiCGSTAB's column state
struct BicgState {
  double rho, alpha, omega, bnorm2, tol2, a;  // a: alpha of this iteration (0 for a column that stopped)
  int active, itn, status;  // status: 0 converged, 1 iteration limit, 2 breakdown
};

template <int WD, class State>
__device__ inline bool any_active(const State *st) {
  int a = 0;
#pragma unroll
  for (int k = 0; k < WD; ++k) a |= st[k].active;
  return a != 0;
}

// What the kernels of one solve share.
struct LsqrVecs {
  LsqrState *sa, *sb;
  const double *pn;             // A V: nseg x m x WD
  int nseg;
  const double *uin;            // U before
  double *uout;                 // U after
  double *partU;                // |U|^2 per block of the kernel that forms U
  const double *partV, *partW;  // |V|^2, |W|^2 per block of k_lsqr_v
  int npv;
  LsqrState *host;              // a copy of state B for the host (pinned memory), or null
};

// The scales of U for the kernel that forms it, from a thread's share of the |V|^2 partials:
// sc[0..WD-1] = sx, sc[WD..] = sy.
template <int WD, int BS>
__device__ inline void lsqr_u_prologue(const LsqrVecs &L, double svt, double *red, double *sc) {
  const double sv = block_sum<WD, BS>(svt, red);
  if (threadIdx.x < WD) {
    double sx, sy;
    lsqr_u_scales(L.sa[threadIdx.x], sv, sx, sy);
    sc[threadIdx.x] = sx;
    sc[WD + threadIdx.x] = sy;
  }
  __syncthreads();
}
// The end of the previous iteration, state A to state B, by a block of its own (the scalar chain of
// some forty dependent operations would hold up a block that has a share of the product); host: a copy
// for the host (pinned memory) or null.
template <int WD, int BS>
__device__ inline void lsqr_end_block(const LsqrVecs &L, double *red) {
  const double svt = thread_parts<WD, BS>(L.partV, L.npv), swt = thread_parts<WD, BS>(L.partW, L.npv);
  const double sv = block_sum<WD, BS>(svt, red), sw = block_sum<WD, BS>(swt, red);
  if (threadIdx.x < WD) {
    LsqrState S = L.sa[threadIdx.x];
    lsqr_end(S, sv, sw);
    L.sb[threadIdx.x] = S;
    if (L.host) L.host[threadIdx.x] = S;
  }
}

// ---- A V ---------------------------------------------------------------------------------------
// P[segment][row][k] = A X over the segment's columns, FP64 A on the matrix cores
// (v_mfma_f64_16x16x4f64), NB interleaved columns. A block owns 16 T rows over the column segment
// blockIdx.y, its eight waves an eighth of the segment's columns each (wcols, a multiple of 16); their
// sums meet in LDS, so that a small system fills the chip with one or two segments instead of a dozen
// partial results per row. Lane (g = lane / 16, c = lane % 16) feeds row c of tile t with columns
// 16 kb + 4 g + s (s = 0..3, one instruction each) and column c of B = X (right-hand side c; the
// upper half c >= NB is zero). The result D[g + 4 v][c] sits in register v of lane (g, c).
// The tiles are read in whole 128-byte row segments and redistributed to the matrix-core layout
// through LDS (rows padded to 18 doubles): the matrix-core lane pattern itself covers 16 half lines a
// load, measured 4.6-5.3 against 6.9 TB/s on a 30 GB matrix. Lane = row rr = lane / 8 of an 8-row half
// tile, columns 2 p, 2 p + 1. LINES: every row starts on a 128-byte line. Otherwise a segment that
// starts at a row's own column 16 kb lies across two lines, and every line is asked for twice (3841^2: 31.8 us
// against 22.4 for 3840^2, with 8- and with 16-byte loads); so the lines themselves are read and put
// side by side in LDS, where row c's block kb starts sh(c) columns into line kb: 26 us. The first and last full
// blocks of a wave's columns, whose lines may reach past the matrix, are then read in the lane pattern.
// The column split depends on the matrix shape only, and every row's sum runs over its columns in the
// same order for every T, so the tile count (chosen by size or by the autotuner) never changes a bit.
constexpr int AV_WAVES = 8;
constexpr int AV_MAXCOLS = 1024;  // columns per wave at most

// SEP: the waves' sums stay apart, P[segment * AV_WAVES + wave] (BiCGSTAB, whose iterates part from
// each other by far more than rounding when the sums of a product are formed in another order).
template <int T, bool LINES, bool SEP, bool KEEP>
__global__ __launch_bounds__(64 * AV_WAVES) void k_lsqr_av(const double *__restrict__ A, int64_t lda, int m, int n,
                                                           const double *__restrict__ X, int wcols,
                                                           double *__restrict__ P,
                                                           const std::conditional_t<SEP, BicgState, LsqrState> *__restrict__ st) {
  const bool act = !st || any_active<NB>(st);
  if (!LINES && !act) return;  // uniform over the grid
  typedef const double __attribute__((address_space(1))) *gdp;
  constexpr int LR = LINES ? 18 : 34;
  __shared__ __attribute__((aligned(16))) double lt[AV_WAVES][T][16 * LR];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int row0 = blockIdx.x * 16 * T;
  const int g = lane >> 4, c = lane & 15;
  const bool hi = c >= NB;
  const int k0 = (blockIdx.y * AV_WAVES + wid) * wcols, kend = min(n, k0 + wcols);
  gdp lrow[T][2];
  int sh[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uintptr_t r = (uintptr_t)(A + (size_t)min(row0 + 16 * t + 8 * h + (lane >> 3), m - 1) * lda);
      lrow[t][h] = (gdp)(LINES ? r : r & ~(uintptr_t)127) + 2 * (lane & 7);
    }
    sh[t] = LINES ? 0 : (int)((uintptr_t)(A + (size_t)min(row0 + 16 * t + c, m - 1) * lda) >> 3 & 15);
  }
  const gdp xb = (gdp)(X + (size_t)(4 * g) * NB + (c & (NB - 1)));
  d4v acc[T];
#pragma unroll
  for (int t = 0; t < T; ++t) acc[t] = d4v{0.0, 0.0, 0.0, 0.0};
  auto lines = [&](int j, double (&a)[T][4]) {
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const d2n u = stream_load<KEEP>((const d2n __attribute__((address_space(1))) *)(lrow[t][h] + 16 * j));
        a[t][2 * h] = u.x;
        a[t][2 * h + 1] = u.y;
      }
  };
  // raw operands of one 16-column block (its second line, if it has two)
  auto load = [&](int kb, double (&a)[T][4], double (&x)[4]) {
    lines(LINES ? kb : kb + 1, a);
#pragma unroll
    for (int s = 0; s < 4; ++s) x[s] = xb[(size_t)(16 * kb + s) * NB];
  };
  auto put = [&](int j, const double (&a)[T][4]) {
    const int rr = lane >> 3, p = (LINES ? 0 : 16 * (j & 1)) + 2 * (lane & 7);
#pragma unroll
    for (int t = 0; t < T; ++t) {
      double *l = lt[wid][t];
      *(d2n *)&l[rr * LR + p] = d2n{a[t][0], a[t][1]};
      *(d2n *)&l[(8 + rr) * LR + p] = d2n{a[t][2], a[t][3]};
    }
  };
  // row segments -> LDS -> matrix-core values (in place); the tiles are per wave
  auto stage = [&](int kb, double (&a)[T][4]) {
    put(LINES ? kb : kb + 1, a);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const double *l = &lt[wid][t][c * LR];
      if constexpr (LINES) {
        const d2n u = *(const d2n *)&l[4 * g], w = *(const d2n *)&l[4 * g + 2];
        a[t][0] = u.x;
        a[t][1] = u.y;
        a[t][2] = w.x;
        a[t][3] = w.y;
      } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) a[t][s] = l[(16 * (kb & 1) + sh[t] + 4 * g + s) & 31];
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  auto step = [&](const double (&a)[T][4], const double (&x)[4]) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const double b = hi ? 0.0 : x[s];
#pragma unroll
      for (int t = 0; t < T; ++t) acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t][s], b, acc[t], 0, 0, 0);
    }
  };
  // one block in the lane pattern of the products, masked at the matrix's last column
  auto direct = [&](int kb) {
    double a[T][4], x[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int col = 16 * kb + 4 * g + s;
      const bool in = col < kend;
      x[s] = in ? X[(size_t)col * NB + (c & (NB - 1))] : 0.0;
#pragma unroll
      for (int t = 0; t < T; ++t) a[t][s] = in ? A[(size_t)min(row0 + 16 * t + c, m - 1) * lda + col] : 0.0;
    }
    step(a, x);
  };
  int kb = k0 >> 4, kb_end = kend >> 4;
  const int kb_all = (kend + 15) >> 4;
  if (!LINES && kb < kb_end) {
    direct(kb++);
    --kb_end;
  }
  // full 16-column blocks, two register sets in turn: the operands of the next block are requested
  // before the products of the current one (the last prefetch re-reads the final block)
  if (kb < kb_end) {
    double a0[T][4], a1[T][4], x0[4], x1[4];
    if (!LINES) {
      lines(kb, a1);
      put(kb, a1);
    }
    load(kb, a0, x0);
    if (!act) return;  // uniform over the grid; the first loads are under way while the state arrives
    for (; kb + 1 < kb_end; kb += 2) {
      load(kb + 1, a1, x1);
      __builtin_amdgcn_sched_barrier(0);
      stage(kb, a0);
      step(a0, x0);
      __builtin_amdgcn_sched_barrier(0);
      load(min(kb + 2, kb_end - 1), a0, x0);
      __builtin_amdgcn_sched_barrier(0);
      stage(kb + 1, a1);
      step(a1, x1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (kb < kb_end) {  // odd count: a0 holds block kb
      stage(kb, a0);
      step(a0, x0);
      ++kb;
    }
  }
  if (!act) return;
  for (; kb < kb_all; ++kb) direct(kb);
  if (SEP) {
    if (k0 < n) {
      double *p = P + (size_t)(blockIdx.y * AV_WAVES + wid) * m * NB;
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int r = row0 + 16 * t + g + 4 * v;
          if (!hi && r < m) p[(size_t)r * NB + c] = acc[t][v];
        }
    }
    return;
  }
  // the waves' sums, wave by wave: red[w][row of the block][k] over the staging tiles (16 T x 8 doubles
  // of the 16 T x 18 of each wave)
  __syncthreads();
  double *red = &lt[0][0][0];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (!hi) red[(wid * 16 * T + 16 * t + g + 4 * v) * NB + c] = acc[t][v];
  __syncthreads();
  for (int e = threadIdx.x; e < 16 * T * NB; e += 64 * AV_WAVES) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < AV_WAVES; ++w) s += red[w * 16 * T * NB + e];
    if (row0 + e / NB < m) P[((size_t)blockIdx.y * m + row0) * NB + e] = s;
  }
}

// P[segment][row] = A x for one right-hand side: a wave owns eight rows over a column segment, 16 bytes
// per lane and row (1 KB of a row per load), two register sets in turn; bound by the matrix stream.
template <class ST, bool KEEP>
__global__ __launch_bounds__(256) void k_lsqr_av1(const ST *__restrict__ A, int64_t lda, int m, int n,
                                                  const double *__restrict__ x, int seglen, double *__restrict__ P,
                                                  const LsqrState *__restrict__ st) {
  if (!st->active) return;
  constexpr int CPL = 16 / sizeof(ST);  // columns per lane and load
  constexpr int STEP = 64 * CPL;
  typedef ST vec __attribute__((ext_vector_type(CPL)));
  typedef const vec __attribute__((address_space(1))) *gvp;
  const int lane = threadIdx.x & 63;
  const int row0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 8;
  if (row0 >= m) return;  // no barriers below
  const int k0 = blockIdx.y * seglen, kend = min(n, k0 + seglen);
  const ST *row[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) row[r] = A + (size_t)min(row0 + r, m - 1) * lda;
  double acc[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) acc[r] = 0.0;
  struct Set {
    vec a[8];
    double x[CPL];
  };
  auto load = [&](int k, Set &s) {
    const int j = k + CPL * lane;
#pragma unroll
    for (int r = 0; r < 8; ++r) s.a[r] = stream_load<KEEP>((gvp)(row[r] + j));
#pragma unroll
    for (int q = 0; q < CPL; ++q) s.x[q] = x[j + q];
  };
  auto step = [&](const Set &s) {
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
      for (int q = 0; q < CPL; ++q) acc[r] += (double)s.a[r][q] * s.x[q];
  };
  const int nfull = (kend - k0) / STEP;
  int k = k0;
  if (nfull > 0) {
    Set s0, s1;
    load(k, s0);
    int i = 0;
    for (; i + 1 < nfull; i += 2) {
      load(k + STEP, s1);
      __builtin_amdgcn_sched_barrier(0);
      step(s0);
      __builtin_amdgcn_sched_barrier(0);
      load(i + 2 < nfull ? k + 2 * STEP : k, s0);
      __builtin_amdgcn_sched_barrier(0);
      step(s1);
      __builtin_amdgcn_sched_barrier(0);
      k += 2 * STEP;
    }
    if (i < nfull) {
      step(s0);
      k += STEP;
    }
  }
  for (int j = k + lane; j < kend; j += 64) {  // the last columns of the segment
    const double xv = x[j];
#pragma unroll
    for (int r = 0; r < 8; ++r) acc[r] += (double)row[r][j] * xv;
  }
  // reduce-scatter over the lanes: lane l ends with the sum of row l / 8
#pragma unroll
  for (int half = 4; half >= 1; half >>= 1) {
    const bool up = (lane & (8 * half)) != 0;
#pragma unroll
    for (int i = 0; i < half; ++i) {
      const double keep = up ? acc[i + half] : acc[i];
      const double send = up ? acc[i] : acc[i + half];
      acc[i] = keep + __shfl_xor(send, 8 * half, 64);
    }
  }
  double s = acc[0];
  s += __shfl_xor(s, 4, 64);
  s += __shfl_xor(s, 2, 64);
  s += __shfl_xor(s, 1, 64);
  const int r = row0 + (lane >> 3);
  if ((lane & 7) == 0 && r < m) P[(size_t)blockIdx.y * m + r] = s;
}

// ---- A^T U -------------------------------------------------------------------------------------
// P[split][j][k] = sum over the split's rows of A[i][j] U[i][k]. A block owns CW columns over the rows
// of split blockIdx.y, its eight waves rw rows each; U of the block's rows sits in LDS (read as
// broadcasts) and the waves' sums meet there in a fixed order, which leaves an eighth of the partial
// results of a wave-wide split. FORM: U is formed here from the partials of A V (see the head of the
// file), by every column panel for its own use and by the first one (blockIdx.x = 0) for keeping.
// A lane holds the columns of one 16-byte load of a row and their sums; the first rows are requested before
// U is formed. Bound by the matrix stream; 3120^2 with 6 right-hand sides 22.6 -> 20.0 us, and an
// eighth of the partial results for k_lsqr_v (13.8 -> 4.8 us); 4881 x 2717 with one 24.3 -> 19.4 us.
// Where U is given a wave takes AT_CHUNK rows of it at a time into its own part of the LDS, the next ones under way, so
// that its rows may be many: the partial results of a large A, eight columns written and read again for every split,
// are then nothing beside it (61440^2: 5.84 ms with 32 rows a wave, 5.21 with 64, 4.88 with 128, 4.47 with 512, 6.76
// TB/s).
constexpr int AT_WAVES = 8, AT_MAXRW = 32, AT_MAXRW_GIVEN = 512, AT_CHUNK = 64;
constexpr int at_cols(size_t elem) { return 64 * 16 / (int)elem; }  // a 16-byte load per lane

template <class ST, int WD, bool FORM, bool KEEP>
__global__ __launch_bounds__(64 * AT_WAVES, 4) void k_lsqr_atu(const ST *__restrict__ A, int64_t lda, int m, int n, int rw,
                                                            LsqrVecs L, double *__restrict__ P) {
  constexpr int BS = 64 * AT_WAVES, CW = at_cols(sizeof(ST)), LV = CW / 64;  // columns per lane
  constexpr int RMAX = AT_WAVES * (FORM ? AT_MAXRW : AT_CHUNK);
  typedef ST vec __attribute__((ext_vector_type(LV)));
  typedef const vec __attribute__((address_space(1))) *gvp;
  __shared__ __attribute__((aligned(16))) double ul[RMAX * WD];
  __shared__ __attribute__((aligned(16))) double red[AT_WAVES / 2 * CW * WD];
  __shared__ double sc[2 * WD];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  if (FORM && blockIdx.y == gridDim.y - 1) {  // one block more for the scalars
    if (blockIdx.x == 0) lsqr_end_block<WD, BS>(L, red);
    return;
  }
  const int i0 = blockIdx.y * AT_WAVES * rw, nr = min(AT_WAVES * rw, m - i0);  // nr >= 1
  // the lane's columns j ..; past the end column 0 is loaded and nothing stored (a load that starts before
  // the end may reach into the row padding)
  const int j = blockIdx.x * CW + LV * lane, jc = j < n ? j : 0;
  const int r0 = wid * rw;  // the wave's rows within the block
  const int rn = max(0, min(rw, nr - r0));
  const ST *base = A + (size_t)i0 * lda;
  constexpr int UN = WD == 1 ? 8 : 4;  // rows per register set
  struct Set {
    vec a[UN];
  };
  auto load = [&](int r, Set &s) {
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const ST *row = base + (size_t)min(r0 + min(r + u, max(rn - 1, 0)), nr - 1) * lda;
      s.a[u] = stream_load<KEEP>((gvp)(row + jc));
    }
  };
  Set s0, s1;
  load(0, s0);  // the first rows are under way while U is formed
  __builtin_amdgcn_sched_barrier(0);
  if (FORM) {
    // everything the block reads before A goes out at once: the state, the norm partials, the sums
    // over the column segments and the old U
    constexpr int NE = RMAX * WD / BS > 0 ? RMAX * WD / BS : 1;  // values of U per thread
    const bool act = any_active<WD>(L.sa);
    const double svt = thread_parts<WD, BS>(L.partV, L.npv);
    double se[NE], ue[NE];
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const int e = tid + i * BS;
      se[i] = ue[i] = 0.0;
      if (e < nr * WD) {
        const size_t o = (size_t)i0 * WD + e;
        ue[i] = L.uin[o];
        for (int sg = 0; sg < L.nseg; ++sg) se[i] += L.pn[(size_t)sg * m * WD + o];
      }
    }
    if (!act) return;  // uniform over the grid
    lsqr_u_prologue<WD, BS>(L, svt, red, sc);
    const bool keep = blockIdx.x == 0;
    const int k = tid % WD;  // the same for all of a thread's values (BS % WD == 0)
    double y2 = 0.0;
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const int e = tid + i * BS;
      const double u = e < nr * WD ? sc[k] * se[i] + sc[WD + k] * ue[i] : 0.0;
      if (keep && e < nr * WD) L.uout[(size_t)i0 * WD + e] = u;
      y2 += u * u;
      if (e < RMAX * WD) ul[e] = u;
    }
    if (keep) {  // uniform over the block
      const double s = block_sum<WD, BS>(y2, red);
      if (tid < WD) L.partU[(size_t)blockIdx.y * WD + tid] = s;
    }
    __syncthreads();
  } else if (!any_active<WD>(L.sb)) {
    return;
  }
  double acc[LV][WD];
#pragma unroll
  for (int q = 0; q < LV; ++q)
#pragma unroll
    for (int k = 0; k < WD; ++k) acc[q][k] = 0.0;
  auto step = [&](int r, const Set &s) {  // r: the set's first row in the LDS
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      double uv[WD];
#pragma unroll
      for (int k = 0; k < WD; ++k) uv[k] = ul[(r + u) * WD + k];  // zero past the last row
#pragma unroll
      for (int q = 0; q < LV; ++q) {
        const double av = (double)s.a[u][q];
#pragma unroll
        for (int k = 0; k < WD; ++k) acc[q][k] += av * uv[k];
      }
      // (the U of all the rows at once would take the registers of half the waves in flight)
      if (WD > 1 && u % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    }
  };
  // two register sets in turn over rows first .. end - 1 (rw and AT_CHUNK are multiples of 2 UN); the last loads
  // repeat the last row
  auto rows = [&](int first, int end, int o) {  // row r of the wave is row o + r of the LDS
#pragma unroll 1
    for (int r = first; r < end; r += 2 * UN) {
      load(r + UN, s1);
      __builtin_amdgcn_sched_barrier(0);
      step(o + r, s0);
      __builtin_amdgcn_sched_barrier(0);
      load(r + 2 * UN, s0);
      __builtin_amdgcn_sched_barrier(0);
      step(o + r + UN, s1);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if constexpr (FORM) {
    rows(0, rn, r0);
  } else {
    static_assert(AT_CHUNK == 64, "WD values of a chunk of U per lane");
    double un[WD], *uw = ul + wid * AT_CHUNK * WD;
    const double *ug = L.uin + (size_t)(i0 + r0) * WD;
    auto given = [&](int r) {
#pragma unroll
      for (int k = 0; k < WD; ++k) {
        const int e = lane + 64 * k;
        un[k] = r + e / WD < rn ? ug[(size_t)r * WD + e] : 0.0;
      }
    };
    given(0);
#pragma unroll 1
    for (int r = 0; r < rn; r += AT_CHUNK) {
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();  // the last chunk is read
#pragma unroll
      for (int k = 0; k < WD; ++k) uw[lane + 64 * k] = un[k];
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
      given(r + AT_CHUNK);
      rows(r, min(r + AT_CHUNK, rn), wid * AT_CHUNK - r);
    }
  }
  // the waves' sums: (0 + 4) (1 + 5) (2 + 6) (3 + 7), then (0 + 2) (1 + 3), then (0 + 1)
#pragma unroll
  for (int half = AT_WAVES / 2; half >= 1; half >>= 1) {
    __syncthreads();
    if (wid >= half && wid < 2 * half) {
      double *d = red + (size_t)(wid - half) * CW * WD;
#pragma unroll
      for (int q = 0; q < LV; ++q)
#pragma unroll
        for (int k = 0; k < WD; ++k) d[(q * WD + k) * 64 + lane] = acc[q][k];
    }
    __syncthreads();
    if (wid < half) {
      const double *d = red + (size_t)wid * CW * WD;
#pragma unroll
      for (int q = 0; q < LV; ++q)
#pragma unroll
        for (int k = 0; k < WD; ++k) acc[q][k] += d[(q * WD + k) * 64 + lane];
    }
  }
  if (wid != 0) return;
#pragma unroll
  for (int q = 0; q < LV; ++q)
    if (j + q < n) {
      double *p = P + ((size_t)blockIdx.y * n + j + q) * WD;
#pragma unroll
      for (int k = 0; k < WD; ++k) p[k] = acc[q][k];
    }
}

// ---- both products of an iteration in one pass over A (one right-hand side) ----------------------
// A row gives u_i = sx (A_i v) + sy u_i and then takes u_i A_i into A^T u, whose normalisation comes later
// anyway: with a block owning whole rows (rpb of them, n <= 1024 PASS_CHUNKS PASS_LV columns over its 1024 threads)
// they stay in registers in between, and A is read once per iteration instead of twice. A thread holds CH
// pairs of columns of R rows in each of two register sets, its part of v and of A^T u. The rows' sums
// meet in LDS, one barrier per R rows: a wave adds across its halves and 16-lane rows with lane swaps, each wave
// then sums the sixteen waves' shares for itself. One block per CU, each with its part of A^T u for
// k_lsqr_v. A block's rows, and its XCD, are the same in every iteration. Bound by the matrix stream: 4881 x
// 2717 18.8 us where the two products took 20.3 and 19.4, 1587^2 7.5 (6.2 + 8.2), 4897^2 in FP32 20.5 (17.5 + 16.2).
// A set of eight rows takes a block some 2 us however narrow they are, as most of its threads have no columns; so
// fewer than PASS_MIN_COLS columns go this way only while a block has no more than two sets (m <= 4080), where the
// launch that it saves counts. Kernels of an iteration, one pass against two products: 128 columns, 4000 rows 13.3
// and 13.6 us, 6000 15.6 and 13.7, 64000 68 and 36, 200000 188 and 82; 32 columns 200000 185 and 47; 320 columns
// 64000 70 and 60; 384 70 and 65; 448 71 and 76; 512 86 and 107.
constexpr int PASS_BS = 1024, PASS_BLOCKS = 255, PASS_CHUNKS = 4, PASS_LV = 2, PASS_MIN_COLS = 400;
// rows of a register set: 128 bytes a thread in both
constexpr int pass_rows(size_t elem, int ch) { return (ch == 1 ? 8 : ch == 2 ? 4 : 2) * (elem == 4 && ch > 1 ? 2 : 1); }

// a over lanes i and i + 32 in the lower half, b's in the upper half
__device__ inline double swap_add32(double a, double b) {
  const uint64_t ua = __builtin_bit_cast(uint64_t, a), ub = __builtin_bit_cast(uint64_t, b);
  const auto l = __builtin_amdgcn_permlane32_swap((unsigned)ua, (unsigned)ub, false, false);
  const auto h = __builtin_amdgcn_permlane32_swap((unsigned)(ua >> 32), (unsigned)(ub >> 32), false, false);
  return __builtin_bit_cast(double, (uint64_t)h[0] << 32 | l[0]) + __builtin_bit_cast(double, (uint64_t)h[1] << 32 | l[1]);
}
// the same for neighbouring rows of 16 lanes: a in the even ones, b in the odd ones
__device__ inline double swap_add16(double a, double b) {
  const uint64_t ua = __builtin_bit_cast(uint64_t, a), ub = __builtin_bit_cast(uint64_t, b);
  const auto l = __builtin_amdgcn_permlane16_swap((unsigned)ua, (unsigned)ub, false, false);
  const auto h = __builtin_amdgcn_permlane16_swap((unsigned)(ua >> 32), (unsigned)(ub >> 32), false, false);
  return __builtin_bit_cast(double, (uint64_t)h[0] << 32 | l[0]) + __builtin_bit_cast(double, (uint64_t)h[1] << 32 | l[1]);
}
template <int CTRL>
__device__ inline double dpp_add(double a) {
  const uint64_t u = __builtin_bit_cast(uint64_t, a);
  const unsigned l = __builtin_amdgcn_mov_dpp((int)u, CTRL, 0xf, 0xf, true),
                 h = __builtin_amdgcn_mov_dpp((int)(u >> 32), CTRL, 0xf, 0xf, true);
  return a + __builtin_bit_cast(double, (uint64_t)h << 32 | l);
}
// the sum over each row of 16 lanes, in all of them (rotations by 8, 4, 2 and 1)
__device__ inline double row_sum16(double a) {
  return dpp_add<0x121>(dpp_add<0x122>(dpp_add<0x124>(dpp_add<0x128>(a))));
}
__device__ inline double read_lane(double a, int lane) {
  const uint64_t u = __builtin_bit_cast(uint64_t, a);
  const unsigned l = __builtin_amdgcn_readlane((int)u, lane), h = __builtin_amdgcn_readlane((int)(u >> 32), lane);
  return __builtin_bit_cast(double, (uint64_t)h << 32 | l);
}

template <class ST, int CH, bool KEEP>
__global__ __launch_bounds__(PASS_BS) void k_lsqr_pass(const ST *__restrict__ A, int64_t lda, int m, int n, int rpb,
                                                       const double *__restrict__ V, LsqrVecs L,
                                                       double *__restrict__ P) {
  constexpr int LV = PASS_LV, R = pass_rows(sizeof(ST), CH), RQ = (R + 3) / 4;
  typedef ST vec __attribute__((ext_vector_type(LV)));
  typedef const vec __attribute__((address_space(1))) *gvp;
  __shared__ double red[2][R][16], pre[PASS_BS / 64], sc[2];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, g = lane >> 4, w = lane & 15;
  if (blockIdx.x == gridDim.x - 1) {  // one block more for the scalars
    lsqr_end_block<1, PASS_BS>(L, pre);
    return;
  }
  const int i0 = blockIdx.x * rpb, nr = min(rpb, m - i0);  // nr >= 1
  const ST *base = A + (size_t)i0 * lda;
  // row of the R in this lane's row of 16 lanes (q = 0, 1): where the sums end up
  auto rof = [&](int q) { return R == 2 ? g >> 1 : g + 4 * q; };
  struct Set {
    vec a[R][CH];
    double u[RQ];  // the old U of the rows rof(q)
  };
  auto load = [&](int r, Set &s) {
#pragma unroll
    for (int rr = 0; rr < R; ++rr) {
      const ST *row = base + (size_t)min(r + rr, nr - 1) * lda;
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const int j = LV * (tid + PASS_BS * c);
        const gvp p = (gvp)(row + (c < CH - 1 || j < n ? j : 0));  // all pieces but the last are within the row
        s.a[rr][c] = stream_load<KEEP>(p);
      }
    }
#pragma unroll
    for (int q = 0; q < RQ; ++q) s.u[q] = L.uin[i0 + min(r + rof(q), nr - 1)];
  };
  Set s0, s1;
  load(0, s0);  // the first rows are under way while the scalars are formed
  const bool act = any_active<1>(L.sa);
  const double svt = thread_parts<1, PASS_BS>(L.partV, L.npv);
  double x[CH][LV], acc[CH][LV];
#pragma unroll
  for (int c = 0; c < CH; ++c)
#pragma unroll
    for (int q = 0; q < LV; ++q) {
      const int j = LV * (tid + PASS_BS * c) + q;
      x[c][q] = j < n ? V[j] : 0.0;
      acc[c][q] = 0.0;
    }
  __builtin_amdgcn_sched_barrier(0);
  if (!act) return;  // uniform over the grid
  lsqr_u_prologue<1, PASS_BS>(L, svt, pre, sc);
  const double sx = sc[0], sy = sc[1];
  double y2 = 0.0;
  auto dots = [&](const Set &s, int b) {
    double d[R];
#pragma unroll
    for (int rr = 0; rr < R; ++rr) {
      d[rr] = 0.0;
#pragma unroll
      for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int q = 0; q < LV; ++q) {
          double a = (double)s.a[rr][c][q];
          if (c == CH - 1 && LV * (tid + PASS_BS * c) + q >= n) a = 0.0;  // row padding, whatever it holds
          d[rr] += a * x[c][q];
        }
    }
#pragma unroll
    for (int q = 0; q < RQ; ++q) {
      double t;
      if constexpr (R == 2) {
        const double h = swap_add32(d[0], d[1]);
        t = swap_add16(h, h);
      } else {
        t = swap_add16(swap_add32(d[4 * q], d[4 * q + 2]), swap_add32(d[4 * q + 1], d[4 * q + 3]));
      }
      t = row_sum16(t);
      if (w == 0) red[b][rof(q)][wid] = t;
    }
  };
  auto update = [&](int r, const Set &s, int b) {
    double y[RQ];
#pragma unroll
    for (int q = 0; q < RQ; ++q) {
      const double t = row_sum16(red[b][rof(q)][w]);
      y[q] = r + rof(q) < nr ? sx * t + sy * s.u[q] : 0.0;
      if (wid == 0 && w == 0 && (R > 2 || (g & 1) == 0) && r + rof(q) < nr) {
        L.uout[i0 + r + rof(q)] = y[q];
        y2 += y[q] * y[q];
      }
    }
#pragma unroll
    for (int rr = 0; rr < R; ++rr) {
      const double yr = read_lane(y[rr / 4], R == 2 ? 32 * rr : 16 * (rr & 3));
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        vec a = s.a[rr][c];
        if (sizeof(ST) == 4) asm("" : "+v"(a));  // converted again: the FP64 values kept from dots() would spill
#pragma unroll
        for (int q = 0; q < LV; ++q) acc[c][q] += (double)a[q] * yr;
      }
    }
  };
  // (asking for both sets before the scalars and for each again as soon as it is used up: 21.9 against 21.5 us)
#pragma unroll 1
  for (int r = 0; r < nr; r += 2 * R) {
    load(r + R, s1);
    __builtin_amdgcn_sched_barrier(0);
    dots(s0, 0);
    __syncthreads();
    update(r, s0, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (r + R >= nr) break;  // uniform over the block
    load(r + 2 * R, s0);
    __builtin_amdgcn_sched_barrier(0);
    dots(s1, 1);
    __syncthreads();
    update(r + R, s1, 1);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int c = 0; c < CH; ++c)
#pragma unroll
    for (int q = 0; q < LV; ++q) {
      const int j = LV * (tid + PASS_BS * c) + q;
      if (j < n) P[(size_t)blockIdx.x * n + j] = acc[c][q];
    }
  if (wid == 0) {
    y2 += __shfl_xor(y2, 16, 64);
    y2 += __shfl_xor(y2, 32, 64);
    if (tid == 0) L.partU[blockIdx.x] = y2;
  }
}

// U formed on its own (many column segments, CSR): U = sx .* sum_s P[s] + sy .* U, |U|^2 per block.
template <int WD>
__global__ __launch_bounds__(256) void k_lsqr_u(int m, LsqrVecs L) {
  __shared__ double red[4 * WD];
  __shared__ double sc[2 * WD];
  if (blockIdx.x == gridDim.x - 1) {  // one block more for the scalars
    lsqr_end_block<WD, 256>(L, red);
    return;
  }
  const bool act = any_active<WD>(L.sa);
  const double svt = thread_parts<WD, 256>(L.partV, L.npv);
  const int t = blockIdx.x * 256 + threadIdx.x, k = t % WD;
  double s = 0.0, y2 = 0.0;
  if (t < m * WD)
    for (int sg = 0; sg < L.nseg; ++sg) s += L.pn[(size_t)sg * m * WD + t];
  if (!act) return;  // uniform over the grid
  lsqr_u_prologue<WD, 256>(L, svt, red, sc);
  if (t < m * WD) {
    const double u = sc[k] * s + sc[WD + k] * L.uin[t];
    L.uout[t] = u;
    y2 = u * u;
  }
  const double sum = block_sum<WD, 256>(y2, red);
  if (threadIdx.x < WD) L.partU[(size_t)blockIdx.x * WD + threadIdx.x] = sum;
}

// ---- V, X and W --------------------------------------------------------------------------------
// V = sx .* sum_s P[s] + sy .* V, with the update of X and W the previous iteration owes (it needs the
// old V): X += t1 W, W = V / alpha + t2 W; |V|^2 and |W|^2 per block. beta = |U| first. INIT: V = sum_s P[s] / beta, W = 0 before the first iteration.
// A block's 256 threads are 64 values (j, k) times four quarters of the splits; at most V_MAXBLOCKS
// blocks, so that the norms are few partials for the kernels that sum them.
// (After k_lsqr_pass, with its 255 splits: 16 values times sixteen shares.)
constexpr int V_MAXBLOCKS = 512;
constexpr int v_values(int shares) { return 256 / shares; }

template <int WD, bool INIT, int SHARES>
__global__ __launch_bounds__(256) void k_lsqr_v(int n, int nsplit, const double *__restrict__ P, LsqrState *sa,
                                                LsqrState *sb, const double *__restrict__ partU, int npu,
                                                double *__restrict__ V, double *__restrict__ X, double *__restrict__ W,
                                                double *__restrict__ partV, double *__restrict__ partW) {
  constexpr int NV = v_values(SHARES);
  __shared__ double red[4 * WD];
  __shared__ double sc[2 * WD], st[3 * WD];
  __shared__ int su[WD];
  __shared__ double part[SHARES][NV];
  const int tid = threadIdx.x;
  // k is the same in every turn of the loop below (NV % WD == 0, also times the grid)
  const int val = tid % NV, q = tid / NV, k = val % WD;
  struct Turn {
    double s, v, w, x;  // the quarter's share of the splits; the old V, W, X (first wave)
  };
  auto load = [&](int t, Turn &c) {
    c.s = c.v = c.w = c.x = 0.0;
    if (t >= n * WD) return;
    const double *p = P + t;
    const size_t stride = (size_t)n * WD;
    for (int sp = q; sp < nsplit; sp += 8 * SHARES) {
      double a[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) a[u] = sp + u * SHARES < nsplit ? p[(sp + u * SHARES) * stride] : 0.0;
#pragma unroll
      for (int u = 0; u < 8; ++u) c.s += a[u];
    }
    if (!INIT && q == 0) {
      c.v = V[t];
      c.w = W[t];
      c.x = X[t];
    }
  };
  // the first turn's loads go out with those of the scalars
  Turn cur;
  if (!INIT) {
    int any = 0;
#pragma unroll
    for (int c = 0; c < WD; ++c) any |= sb[c].active | sb[c].upd;
    const double uut = thread_parts<WD, 256>(partU, npu);
    load(blockIdx.x * NV + val, cur);
    if (!any) return;  // uniform over the grid; state A holds the stopped columns already
    const double uu = block_sum<WD, 256>(uut, red);
    if (tid < WD) {
      const LsqrState &S = sb[tid];
      const int active = S.active;
      const double beta = sqrt(uu), alpha = S.alpha;
      st[tid] = S.t1;
      st[WD + tid] = S.t2;
      st[2 * WD + tid] = S.inv_alpha;
      su[tid] = S.upd;
      sc[tid] = active && beta > 0.0 ? 1.0 / beta : 0.0;
      sc[WD + tid] = active ? (beta > 0.0 ? -beta / alpha : 1.0) : 0.0;  // beta = 0: V unchanged
      if (blockIdx.x == gridDim.x - 1) {
        sa[tid] = S;
        if (active) {
          sa[tid].itn += 1;
          sa[tid].beta = beta;
        }
      }
    }
  } else {
    load(blockIdx.x * NV + val, cur);
    if (tid < WD) sc[tid] = sb[tid].active && sb[tid].beta > 0.0 ? 1.0 / sb[tid].beta : 0.0;
  }
  double v2 = 0.0, w2 = 0.0;
  for (int t0 = blockIdx.x * NV; t0 < n * WD; t0 += gridDim.x * NV) {  // uniform over the block
    const int t = t0 + val;
    __syncthreads();  // the scalars are there; the sums of the previous turn are read
    part[q][val] = cur.s;
    __syncthreads();
    const double vold = cur.v, wold = cur.w, xold = cur.x;
    if (t0 + gridDim.x * NV < n * WD) load(t + gridDim.x * NV, cur);
    if (q == 0 && t < n * WD) {  // the first share's lanes hold the turn's values
      double s = 0.0;
#pragma unroll
      for (int h = 0; h < SHARES; h += 4)
        s += (part[h][val] + part[h + 1][val]) + (part[h + 2][val] + part[h + 3][val]);
      if (INIT) {
        const double v = sc[k] * s;
        V[t] = v;
        W[t] = 0.0;
        X[t] = 0.0;
        v2 += v * v;
      } else {
        double w = wold;
        if (su[k]) {
          X[t] = xold + st[k] * wold;
          w = vold * st[2 * WD + k] + st[WD + k] * wold;
          W[t] = w;
        }
        const double v = sc[k] * s + sc[WD + k] * vold;
        V[t] = v;
        v2 += v * v;
        w2 += w * w;
      }
    }
  }
  if (tid >= 64) return;  // the first wave's first NV lanes hold the sums, the others zeros
#pragma unroll
  for (int o = WD; o < 64; o <<= 1) {
    v2 += __shfl_xor(v2, o, 64);
    w2 += __shfl_xor(w2, o, 64);
  }
  if (tid < WD) {
    partV[(size_t)blockIdx.x * WD + tid] = v2;
    partW[(size_t)blockIdx.x * WD + tid] = w2;
  }
}

// ---- start, polls and finish -------------------------------------------------------------------
// column k of the interleaved X0 (stride NB) as the solve's own start vector, and x_s = x0 / q
template <int WD>
__global__ void k_lsqr_x0(int n, const double *__restrict__ X0, const double *__restrict__ q, double *__restrict__ Xs) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * WD) return;
  const int j = t / WD, k = t % WD;
  const double x = X0[(size_t)j * NB + k];
  Xs[t] = q ? x / q[j] : x;
}

// U = B - sum_s P[s] (P = A x_s); |U|^2 and |B|^2 per block
template <int WD>
__global__ __launch_bounds__(256) void k_lsqr_u0(int m, int nseg, const double *__restrict__ P,
                                                 const double *__restrict__ B, double *__restrict__ U,
                                                 double *__restrict__ partU, double *__restrict__ partB) {
  __shared__ double red[2][4 * WD];
  const int t = blockIdx.x * 256 + threadIdx.x, k = t % WD;
  double u2 = 0.0, b2 = 0.0;
  if (t < m * WD) {
    const double b = B[(size_t)(t / WD) * NB + k];
    double s = 0.0;
    for (int sg = 0; sg < nseg; ++sg) s += P[(size_t)sg * m * WD + t];
    const double u = b - s;
    U[t] = u;
    u2 = u * u;
    b2 = b * b;
  }
#pragma unroll
  for (int o = WD; o < 64; o <<= 1) {
    u2 += __shfl_xor(u2, o, 64);
    b2 += __shfl_xor(b2, o, 64);
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane < WD) {
    red[0][wid * WD + lane] = u2;
    red[1][wid * WD + lane] = b2;
  }
  __syncthreads();
  if (threadIdx.x < WD) {
    const int c = threadIdx.x;
    partU[(size_t)blockIdx.x * WD + c] = (red[0][c] + red[0][WD + c]) + (red[0][2 * WD + c] + red[0][3 * WD + c]);
    partB[(size_t)blockIdx.x * WD + c] = (red[1][c] + red[1][WD + c]) + (red[1][2 * WD + c] + red[1][3 * WD + c]);
  }
}

// beta = ||U||, btol = eps ||b|| / ||r0|| (src/lib_lsqr.f:84-100); both states
template <int WD>
__global__ __launch_bounds__(256) void k_lsqr_start(LsqrState *sa, LsqrState *sb, const double *partU,
                                                    const double *partB, int np, double eps, int nrhs, int itnlim) {
  __shared__ double red[4 * WD];
  const double sr = block_sum_parts<WD, 256>(partU, np, red);
  const double sn = block_sum_parts<WD, 256>(partB, np, red);
  const int k = threadIdx.x;
  if (k >= WD) return;
  LsqrState S = {};
  const double nrm_r = sqrt(sr);
  const double nrm_b = sqrt(sn);
  S.atol = eps;
  S.btol = eps * nrm_b / nrm_r;
  S.ctol = 1.0 / 1.0e8;
  S.cs2 = -1.0;
  S.beta = nrm_r;
  S.active = k < nrhs ? 1 : 0;
  S.itnlim = itnlim;
  sa[k] = S;
  sb[k] = S;
}

// the state at the end of the last iteration of all (the limit): what the next one's end block would write
template <int WD>
__global__ __launch_bounds__(256) void k_lsqr_poll(LsqrVecs L) {
  __shared__ double red[4 * WD];
  lsqr_end_block<WD, 256>(L, red);
}

// x = q .* (x + the owed update) + x0, into the interleaved X
template <int WD>
__global__ void k_lsqr_finish(int n, const double *__restrict__ q, const double *__restrict__ Xl,
                              const double *__restrict__ W, const LsqrState *__restrict__ sb, double *__restrict__ X) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * WD) return;
  const int j = t / WD, k = t % WD;
  const double x = Xl[t] + (sb[k].upd ? sb[k].t1 * W[t] : 0.0);
  double *px = X + (size_t)j * NB + k;
  *px = (q ? q[j] * x : x) + *px;
}

// ---- sparse products (CSR) -----------------------------------------------------------------------
// y = A x, 0-based row pointers and columns: eight lanes per row take its entries in turn, their sums
// meet in a fixed order. For one right-hand side (the Fortran seam has one).
__global__ __launch_bounds__(256) void k_csr_mv(int rows, const int64_t *__restrict__ ia, const int32_t *__restrict__ ja,
                                                const double *__restrict__ va, const double *__restrict__ x,
                                                double *__restrict__ y, const LsqrState *__restrict__ st) {
  if (!st->active) return;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int r = t >> 3, l = t & 7;
  double acc = 0.0;
  if (r < rows)
    for (int64_t p = ia[r] + l; p < ia[r + 1]; p += 8) acc += va[p] * x[ja[p]];
  acc += __shfl_xor(acc, 1, 64);
  acc += __shfl_xor(acc, 2, 64);
  acc += __shfl_xor(acc, 4, 64);
  if (r < rows && l == 0) y[r] = acc;
}

// ---- column scaling (lsqr_precon) ------------------------------------------------------------
template <class ST>
__global__ __launch_bounds__(256) void k_colsq(const ST *__restrict__ A, int64_t lda, int m, int n, int rows_per_split,
                                               double *__restrict__ P) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  const int s = blockIdx.y;
  if (j >= n) return;
  const int i0 = s * rows_per_split, i1 = min(m, i0 + rows_per_split);
  double acc = 0.0;
  for (int i = i0; i < i1; ++i) {
    const double a = (double)A[(size_t)i * lda + j];
    acc += a * a;
  }
  P[(size_t)s * n + j] = acc;
}

__global__ void k_colq(int n, int nsplit, const double *__restrict__ P, double *__restrict__ q) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  double s = 0.0;
  for (int sp = 0; sp < nsplit; ++sp) s += P[(size_t)sp * n + j];
  q[j] = 1.0 / sqrt(s);
}

template <class ST>
__global__ __launch_bounds__(256) void k_colmul(ST *__restrict__ A, int64_t lda, int m, int n, const double *__restrict__ q) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const double qj = q[j];
  for (int i = blockIdx.y; i < m; i += gridDim.y) A[(size_t)i * lda + j] = (ST)((double)A[(size_t)i * lda + j] * qj);
}

int splits_for(int m, int n) {
  const int panels = (n + 255) / 256;
  int s = (2048 + panels - 1) / panels;  // aim at >= 2048 workgroups
  s = std::max(1, std::min(s, (m + 63) / 64));
  return s;
}

}  // namespace

int andr_colscale(andr_ctx *ctx, void *A, bool fp32, int64_t lda, int m, int n, double *q) {
  const int ns = splits_for(m, n);
  const int rps = (m + ns - 1) / ns;
  DevBuf<double> P;
  if (P.alloc((size_t)ns * n, ctx)) return andr_fail(ctx, ANDR_ERR_ALLOC, "column scaling scratch");
  dim3 g1((n + 255) / 256, ns);
  if (fp32)
    hipLaunchKernelGGL(k_colsq<float>, g1, dim3(256), 0, ctx->stream, (const float *)A, lda, m, n, rps, P.p);
  else
    hipLaunchKernelGGL(k_colsq<double>, g1, dim3(256), 0, ctx->stream, (const double *)A, lda, m, n, rps, P.p);
  hipLaunchKernelGGL(k_colq, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, n, ns, P.p, q);
  dim3 g2((n + 255) / 256, std::min(m, 256));
  if (fp32)
    hipLaunchKernelGGL(k_colmul<float>, g2, dim3(256), 0, ctx->stream, (float *)A, lda, m, n, q);
  else
    hipLaunchKernelGGL(k_colmul<double>, g2, dim3(256), 0, ctx->stream, (double *)A, lda, m, n, q);
  ANDR_HIP(ctx, hipGetLastError());
  ANDR_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return ANDR_OK;
}

namespace {

constexpr int LSQR_POLL = 8;  // iterations between reads of the convergence state

// More column segments than this and U is formed by a kernel of its own: in k_lsqr_atu every panel of
// columns sums them again, WD * 8 bytes a row and segment (L2) against 1 KB of A.
constexpr int LSQR_FUSE_SEG = 2, LSQR_FUSE_SEG1 = 16;

// Whether k_lsqr_atu forms U. With several right-hand sides and an A beyond the 256 MB cache the panels' own sums
// and the short splits that they need cost more than k_lsqr_u's launch: three plain tensors of bodies of 2420 elements
// (422 MB) 200 ms formed in the product, 177 apart; of 5120 (1.9 GB) 1170 and 1002; but of 1620 (189 MB) 79 and 82,
// and below eight panels (200000 x 200) 199 and 209 us an iteration.
constexpr int LSQR_FUSE_PANELS = 8;
bool fuse_u(int m, int n, int64_t lda, bool fp32, int wd, int nseg, int panels) {
  if (nseg > (wd == 1 ? LSQR_FUSE_SEG1 : LSQR_FUSE_SEG)) return false;
  return wd == 1 || panels < LSQR_FUSE_PANELS || (double)m * lda * (fp32 ? 4 : 8) <= KEEP_BYTES;
}

// How A X splits its columns, a function of the shape alone (so that the tile count never changes the
// sums): nseg column segments of AV_WAVES * wcols columns. Two segments while there are fewer than 128
// 64-row tiles, else one wave per SIMD or less would be in flight; no more than AV_MAXCOLS columns per wave.
struct AvShape {
  int nseg, wcols;
};
AvShape av_shape(int m, int n) {
  AvShape s;
  s.nseg = std::max((n + AV_WAVES * AV_MAXCOLS - 1) / (AV_WAVES * AV_MAXCOLS), m < 8192 && n >= 512 ? 2 : 1);
  s.wcols = ((n + AV_WAVES * s.nseg - 1) / (AV_WAVES * s.nseg) + 15) / 16 * 16;
  s.nseg = (n + AV_WAVES * s.wcols - 1) / (AV_WAVES * s.wcols);
  return s;
}
// 16-row tiles per block where the autotuner does not choose: two while four leave the chip short of
// blocks (3120^2: 18.1 us with four, 15.8 with two)
int av_tiles(int m, int nseg) { return (m + 63) / 64 * nseg < 512 ? 2 : 4; }

// A X into the segment partials P (FP64, NB interleaved columns)
template <int T, bool SEP>
void launch_av_t(hipStream_t st, const double *A, int64_t lda, int m, int n, const double *X, AvShape sh, double *P,
                 const std::conditional_t<SEP, BicgState, LsqrState> *s) {
  const dim3 grid((m + 16 * T - 1) / (16 * T), sh.nseg), blk(64 * AV_WAVES);
  const bool lines = lda % 16 == 0 && (uintptr_t)A % 128 == 0;
  if constexpr (T > 4)
    if (!lines) return launch_av_t<4, SEP>(st, A, lda, m, n, X, sh, P, s);  // two lines of eight tiles do not fit the LDS
  auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, blk, 0, st, A, lda, m, n, X, sh.wcols, P, s); };
  const bool keep = (double)m * lda * sizeof(double) <= KEEP_BYTES;
  if (lines && keep) go(k_lsqr_av<T, true, SEP, true>);
  else if (lines) go(k_lsqr_av<T, true, SEP, false>);
  else if constexpr (T <= 4) {
    if (keep) go(k_lsqr_av<T, false, SEP, true>);
    else go(k_lsqr_av<T, false, SEP, false>);
  }
}
template <bool SEP>
void launch_av(hipStream_t st, int tiles, const double *A, int64_t lda, int m, int n, const double *X, AvShape sh,
               double *P, const std::conditional_t<SEP, BicgState, LsqrState> *s) {
  if (tiles == 2) launch_av_t<2, SEP>(st, A, lda, m, n, X, sh, P, s);
  else if (SEP || tiles == 4) launch_av_t<4, SEP>(st, A, lda, m, n, X, sh, P, s);
  else if constexpr (!SEP) launch_av_t<8, false>(st, A, lda, m, n, X, sh, P, s);
}

// One LSQR solve, advanced in blocks of iterations on a stream of its own (several solves of a batch
// then overlap on the device); the profiling tokens are taken only on the context's stream.
struct LsqrRun {
  andr_ctx *ctx = nullptr;
  hipStream_t st = nullptr;
  const void *A = nullptr;
  bool fp32 = false;
  int64_t lda = 0;
  int m = 0, n = 0, nrhs = 0, wd = NB, itnlim = 0, it = 0;  // wd: columns of the vectors, 1 or NB
  const double *q = nullptr;
  double *X = nullptr;
  bool done = false;
  AvShape av{1, 16};  // A X: column segments (one right-hand side: of av.wcols columns)
  int tilesN = 4;     // A X: 16-row tiles per block (autotuned)
  int rw = 8, splits = 1;  // A^T U: rows per wave, row splits
  int blocksV = 0, partsU = 0;
  bool fuse = false;  // U is formed in the A^T U kernel
  int rpb = 0, blocksP = 0, chunks = 0;  // both products in one pass: rows per block and blocks (0: not so)
  int cur = 0;        // U of the last iteration is U[cur]
  // sparse mode: A and A^T in CSR (0-based, device); A is then unused
  const int64_t *cia = nullptr, *tia = nullptr;
  const int32_t *cja = nullptr, *tja = nullptr;
  const double *cva = nullptr, *tva = nullptr;
  int64_t nnz = 0;
  DevBuf<double> U[2], V, W, Xl, Xs, P, PN, partU, partB, partV, partW;
  DevBuf<LsqrState> S;  // state A, state B
  LsqrState hs[NB];
  LsqrState *slot = nullptr;  // two polls' states, pinned host memory of the context (null: none to be had)
  hipEvent_t ev[2] = {nullptr, nullptr};
  int polls = 0, read = 0;  // polls enqueued and read
  double abytes = 0, vbytes = 0, aflops = 0;

  LsqrRun() = default;
  LsqrRun(const LsqrRun &) = delete;
  LsqrRun &operator=(const LsqrRun &) = delete;
  ~LsqrRun() {
    if (ctx) (void)hipStreamSynchronize(st);  // nothing in flight writes the slot or the workspaces any more
    if (slot) andr_pinned_release(ctx, slot);
    for (auto e : ev)
      if (e) (void)hipEventDestroy(e);
  }
  int tok(const char *name, double bytes) { return tok(name, bytes, aflops); }
  int tok(const char *name, double bytes, double flops) {
    return st == ctx->stream ? andr_prof_begin(ctx, name, bytes, flops) : -1;
  }
  LsqrState *sa() const { return S.p; }
  LsqrState *sb() const { return S.p + NB; }

  // Autotuner of the FP64 product: on the first large system of a (log2 m, log2 n) bucket, time the
  // product with 2, 4 and 8 tiles per block on the actual matrix (its output goes to the segment
  // partials only) and keep the fastest for the bucket. The choice does not change results.
  int tune_tiles() {
    const std::pair<int, int> key{ilog2c(m), ilog2c(n)};
    auto it = ctx->tune_gemv_n.find(key);
    if (it != ctx->tune_gemv_n.end()) {
      tilesN = it->second.first;
      return ANDR_OK;
    }
    ANDR_HIP(ctx, hipDeviceSynchronize());  // time the candidates alone on the device
    hipEvent_t e0, e1;
    ANDR_HIP(ctx, hipEventCreate(&e0));
    ANDR_HIP(ctx, hipEventCreate(&e1));
    int best = 4;
    float best_ms = 1e30f;
    for (int tiles : {2, 4, 8}) {
      auto launch = [&]() { launch_av<false>(st, tiles, (const double *)A, lda, m, n, Xs.p, av, PN.p, nullptr); };
      launch();  // warm-up
      float ms = 1e30f;
      for (int rep = 0; rep < 2; ++rep) {
        (void)hipEventRecord(e0, st);
        launch();
        (void)hipEventRecord(e1, st);
        (void)hipEventSynchronize(e1);
        float t = 0.f;
        (void)hipEventElapsedTime(&t, e0, e1);
        ms = std::min(ms, t);
      }
      if (ms < best_ms) {
        best_ms = ms;
        best = tiles;
      }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    ANDR_HIP(ctx, hipGetLastError());
    ctx->tune_gemv_n[key] = {best, best_ms};
    tilesN = best;
    return ANDR_OK;
  }
  static int ilog2c(int v) {
    int b = 0;
    while ((1 << b) < v) ++b;
    return b;
  }

  LsqrVecs vecs() {
    return {sa(), sb(), PN.p, av.nseg, U[cur].p, U[cur ^ 1].p, partU.p, partV.p, partW.p, blocksV, nullptr};
  }
  // A Xin into the segment partials
  void gemv_n(const double *Xin) {
    const int t = tok("lsqr_gemv_n", abytes + vbytes + (double)av.nseg * m * wd * 8.0);
    if (cia) {
      hipLaunchKernelGGL(k_csr_mv, dim3((m + 31) / 32), dim3(256), 0, st, m, cia, cja, cva, Xin, PN.p, sb());
    } else if (wd == 1) {
      const dim3 grid((m + 31) / 32, av.nseg);
      const bool keep = (double)m * lda * (fp32 ? 4 : 8) <= KEEP_BYTES;
      auto go = [&](auto kernel, auto elem) {
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, (const decltype(elem) *)A, lda, m, n, Xin, av.wcols, PN.p, sb());
      };
      if (fp32 && keep) go(k_lsqr_av1<float, true>, 0.0f);
      else if (fp32) go(k_lsqr_av1<float, false>, 0.0f);
      else if (keep) go(k_lsqr_av1<double, true>, 0.0);
      else go(k_lsqr_av1<double, false>, 0.0);
    } else {
      launch_av<false>(st, tilesN, (const double *)A, lda, m, n, Xin, av, PN.p, sb());
    }
    andr_prof_end(ctx, t);
  }
  // A^T U into the split partials; form: U from the segment partials first (into U[cur ^ 1])
  void gemv_t(const LsqrVecs &L, bool form) {
    const int t = tok("lsqr_gemv_t", abytes + vbytes + (double)splits * n * wd * 8.0);
    const int cols = at_cols(fp32 ? 4 : 8);
    const dim3 grid((n + cols - 1) / cols, splits + (form ? 1 : 0)), blk(64 * AT_WAVES);
    if (cia) {
      hipLaunchKernelGGL(k_csr_mv, dim3((n + 31) / 32), dim3(256), 0, st, n, tia, tja, tva, L.uin, P.p, sb());
    } else {
      const bool keep = (double)m * lda * (fp32 ? 4 : 8) <= KEEP_BYTES;
      auto go = [&](auto kernel, auto elem) {
        hipLaunchKernelGGL(kernel, grid, blk, 0, st, (const decltype(elem) *)A, lda, m, n, rw, L, P.p);
      };
      auto pick = [&](auto wdc, auto elem) {
        typedef decltype(elem) E;
        constexpr int W = decltype(wdc)::value;
        if (form && keep) go(k_lsqr_atu<E, W, true, true>, elem);
        else if (form) go(k_lsqr_atu<E, W, true, false>, elem);
        else if (keep) go(k_lsqr_atu<E, W, false, true>, elem);
        else go(k_lsqr_atu<E, W, false, false>, elem);
      };
      if (wd != 1) pick(std::integral_constant<int, NB>{}, 0.0);
      else if (fp32) pick(std::integral_constant<int, 1>{}, 0.0f);
      else pick(std::integral_constant<int, 1>{}, 0.0);
    }
    andr_prof_end(ctx, t);
  }

  // workspace, initial state, x_s = x0 / q, U = b - A x_s, V = A^T U / beta
  int begin(andr_ctx *c, hipStream_t stream, const void *A_, bool fp32_, int64_t lda_, int m_, int n_,
            const double *q_, const double *B, double *X_, int nrhs_, int maxit, double eps) {
    ctx = c;
    st = stream;
    A = A_;
    fp32 = fp32_;
    lda = lda_;
    m = m_;
    n = n_;
    q = q_;
    X = X_;
    nrhs = nrhs_;
    if (nrhs < 1 || nrhs > NB) return andr_fail(ctx, ANDR_ERR_ARG, "nrhs must be 1..%d", NB);
    if (m < 1 || n < 1) return andr_fail(ctx, ANDR_ERR_ARG, "empty system");
    wd = nrhs == 1 ? 1 : NB;
    if ((fp32 || cia) && wd != 1) return andr_fail(ctx, ANDR_ERR_ARG, "FP32 and sparse systems take one right-hand side");
    if (!cia && (lda % (fp32 ? 4 : 2) || ((uintptr_t)A % 16)))
      return andr_fail(ctx, ANDR_ERR_ARG, "rows of the system matrix must start on 16-byte boundaries");
    if (cia) {
      av = {1, n};
    } else if (wd == 1) {
      // a wave per eight rows: segments (of whole 1 KB loads) while there are fewer than 2048 waves
      const int rowwaves = (m + 7) / 8;
      const int want = std::min(std::max(1, (2048 + rowwaves - 1) / rowwaves), std::max(1, n / 256));
      av.wcols = ((n + want - 1) / want + 255) / 256 * 256;
      av.nseg = (n + av.wcols - 1) / av.wcols;
    } else {
      av = av_shape(m, n);
    }
    const int cols = at_cols(fp32 ? 4 : 8), panels = (n + cols - 1) / cols;
    fuse = !cia && fuse_u(m, n, lda, fp32, wd, av.nseg, panels);
    // Rows per wave of A^T U: the fewest (16, the finest split that keeps two register sets busy) whose
    // blocks run at once, two on each CU; a second, nearly empty round of blocks costs more than the
    // longer waves (3120^2, 6 right-hand sides: 650 blocks of 16 rows a wave 25.2 us, 425 of 24 20.0).
    rw = 16;
    const int maxrw = fuse || wd == 1 ? AT_MAXRW : AT_MAXRW_GIVEN;
    while (rw < maxrw && panels * ((m + AT_WAVES * rw - 1) / (AT_WAVES * rw) + 1) > 512) rw += wd == 1 ? 16 : 8;
    splits = cia ? 1 : (m + AT_WAVES * rw - 1) / (AT_WAVES * rw);
    // one pass over A where a block's threads hold whole rows (4881 x 2717, with k_lsqr_v: 24 us an iteration, 44
    // with a kernel for each product) and narrow rows are few (PASS_MIN_COLS)
    chunks = (n + PASS_BS * PASS_LV - 1) / (PASS_BS * PASS_LV);
    if (wd == 1 && !cia && chunks <= PASS_CHUNKS) {
      const int R = pass_rows(fp32 ? 4 : 8, chunks);  // whole register sets: a shorter last one loads as much
      const int rows = ((m + PASS_BLOCKS - 1) / PASS_BLOCKS + R - 1) / R * R;
      if (n >= PASS_MIN_COLS || rows <= 2 * R) {
        rpb = rows;
        blocksP = (m + rpb - 1) / rpb;
      }
    }
    const int vv = v_values(blocksP ? 16 : 4);
    blocksV = std::min((n * wd + vv - 1) / vv, V_MAXBLOCKS);
    const int blocksM = (m * wd + 255) / 256;
    partsU = blocksP ? blocksP : (fuse ? splits : blocksM);
    if (U[0].alloc((size_t)m * wd, ctx) || U[1].alloc((size_t)m * wd, ctx) || V.alloc((size_t)n * wd, ctx) ||
        W.alloc((size_t)n * wd, ctx) || Xl.alloc((size_t)n * wd, ctx) || Xs.alloc((size_t)n * wd, ctx) ||
        P.alloc((size_t)std::max(splits, blocksP) * n * wd, ctx) || PN.alloc((size_t)av.nseg * m * wd, ctx) ||
        partU.alloc((size_t)std::max(partsU, blocksM) * wd, ctx) || partB.alloc((size_t)blocksM * wd, ctx) ||
        partV.alloc((size_t)blocksV * wd, ctx) || partW.alloc((size_t)blocksV * wd, ctx) || S.alloc(2 * NB, ctx))
      return andr_fail(ctx, ANDR_ERR_ALLOC, "LSQR workspace (m=%d n=%d)", m, n);
    static_assert(2 * NB * sizeof(LsqrState) <= ANDR_PINNED_SLOT, "two polls' states in a pinned slot");
    slot = (LsqrState *)andr_pinned_alloc(ctx);
    for (auto &e : ev) ANDR_HIP(ctx, hipEventCreateWithFlags(&e, hipEventDisableTiming));
    std::memset(hs, 0, sizeof(hs));
    itnlim = maxit > 0 ? maxit : 10 * (m + n + 50);
    abytes = cia ? (double)nnz * 12.0 + (double)(m + 1) * 8.0 : (double)m * n * (fp32 ? 4.0 : 8.0);
    vbytes = ((double)m + n) * wd * 8.0;
    aflops = 2.0 * m * n * nrhs;
    return wd == 1 ? start<1>(B, eps) : start<NB>(B, eps);
  }
  template <int WD>
  int start(const double *B, double eps) {
    const int blocksM = (m * WD + 255) / 256;
    hipLaunchKernelGGL(k_lsqr_x0<WD>, dim3((n * WD + 255) / 256), dim3(256), 0, st, n, X, q, Xs.p);
    if (wd == NB) {
      tilesN = ctx->autotune ? av_tiles(m, av.nseg) : ctx->gemv_n_tiles;
      if (ctx->autotune && (double)m * n * 8.0 >= 2.56e8) {
        const int rc = tune_tiles();
        if (rc) return rc;
      }
    }
    // the state first: the products look at it
    hipLaunchKernelGGL(k_lsqr_start<WD>, dim3(1), dim3(256), 0, st, sa(), sb(), partU.p, partB.p, 0, eps, nrhs, itnlim);
    gemv_n(Xs.p);
    hipLaunchKernelGGL(k_lsqr_u0<WD>, dim3(blocksM), dim3(256), 0, st, m, av.nseg, PN.p, B, U[0].p, partU.p, partB.p);
    hipLaunchKernelGGL(k_lsqr_start<WD>, dim3(1), dim3(256), 0, st, sa(), sb(), partU.p, partB.p, blocksM, eps, nrhs,
                       itnlim);
    cur = 0;
    gemv_t(vecs(), false);
    launch_v<WD, true>(splits, nullptr, 0);
    ANDR_HIP(ctx, hipGetLastError());
    return ANDR_OK;
  }

  // enqueues iterations up to the next multiple of LSQR_POLL (or the iteration limit); the last one leaves
  // the columns' states in pinned host memory; no host wait
  int advance() {
    if (it >= itnlim) return ANDR_OK;
    if (wd == 1) iterate<1>();
    else iterate<NB>();
    ANDR_HIP(ctx, hipGetLastError());
    ANDR_HIP(ctx, hipEventRecord(ev[polls % 2], st));
    ++polls;
    return ANDR_OK;
  }
  template <int WD, bool INIT>
  void launch_v(int parts, const double *pu, int npu) {
    if (WD == 1 && blocksP)
      hipLaunchKernelGGL((k_lsqr_v<WD, INIT, WD == 1 ? 16 : 4>), dim3(blocksV), dim3(256), 0, st, n, parts, P.p, sa(),
                         sb(), pu, npu, V.p, Xl.p, W.p, partV.p, partW.p);
    else
      hipLaunchKernelGGL((k_lsqr_v<WD, INIT, 4>), dim3(blocksV), dim3(256), 0, st, n, parts, P.p, sa(), sb(), pu, npu,
                         V.p, Xl.p, W.p, partV.p, partW.p);
  }
  template <class ST, int CH>
  void pass_ch(const LsqrVecs &L) {
    const dim3 grid(blocksP + 1), blk(PASS_BS);
    if ((double)m * lda * sizeof(ST) <= KEEP_BYTES)
      hipLaunchKernelGGL((k_lsqr_pass<ST, CH, true>), grid, blk, 0, st, (const ST *)A, lda, m, n, rpb, V.p, L, P.p);
    else
      hipLaunchKernelGGL((k_lsqr_pass<ST, CH, false>), grid, blk, 0, st, (const ST *)A, lda, m, n, rpb, V.p, L, P.p);
  }
  template <class ST>
  void pass_st(const LsqrVecs &L) {
    if (chunks == 1) pass_ch<ST, 1>(L);
    else if (chunks == 2) pass_ch<ST, 2>(L);
    else if (chunks == 3) pass_ch<ST, 3>(L);
    else pass_ch<ST, 4>(L);
  }
  void pass(const LsqrVecs &L) {
    const int t = tok("lsqr_pass", abytes + 2.0 * vbytes + (double)blocksP * n * 8.0, 2.0 * aflops);
    if (fp32) pass_st<float>(L);
    else pass_st<double>(L);
    andr_prof_end(ctx, t);
  }
  template <int WD>
  void iterate() {
    LsqrState *host = slot ? slot + (polls % 2) * NB : nullptr;
    bool last;
    do {
      LsqrVecs L = vecs();
      ++it;
      last = it % LSQR_POLL == 0 || it >= itnlim;
      if (last && it < itnlim) L.host = host;  // the state before this iteration, by the way
      if (WD == 1 && blocksP) {
        pass(L);
      } else {
        gemv_n(V.p);
        if (!fuse) {
          hipLaunchKernelGGL(k_lsqr_u<WD>, dim3((m * WD + 255) / 256 + 1), dim3(256), 0, st, m, L);
          L.uin = L.uout;
        }
        gemv_t(L, fuse);
      }
      launch_v<WD, false>(blocksP ? blocksP : splits, partU.p, partsU);
      cur ^= 1;
    } while (!last);
    if (it >= itnlim) {
      LsqrVecs L = vecs();
      L.host = host;
      hipLaunchKernelGGL(k_lsqr_poll<WD>, dim3(1), dim3(256), 0, st, L);
    }
  }

  // waits for the oldest poll that was not read yet; done when no column is active or the limit is
  // reached. The device meanwhile works on the iterations after it, which are no-ops (the kernels
  // return on a stopped state) when that poll turns out to be the last.
  int poll_state() {
    if (!slot) {  // state B of the last iteration enqueued; an update that k_lsqr_v has applied is still marked as owed
                  // there until the next iteration's end, or the limit's, clears it: finish() must not see it
      ANDR_HIP(ctx, hipMemcpyAsync(hs, sb(), sizeof(LsqrState) * wd, hipMemcpyDeviceToHost, st));
      ANDR_HIP(ctx, hipStreamSynchronize(st));
      bool any = false;
      for (int k = 0; k < nrhs; ++k) any = any || hs[k].active || hs[k].upd;
      done = !any || it >= itnlim;
      return ANDR_OK;
    }
    ANDR_HIP(ctx, hipEventSynchronize(ev[read % 2]));
    std::memcpy(hs, slot + (read % 2) * NB, sizeof(LsqrState) * wd);
    ++read;
    bool any = false;
    for (int k = 0; k < nrhs; ++k) any = any || hs[k].active;
    done = !any || (it >= itnlim && read == polls);
    return ANDR_OK;
  }
  // one round of a solve: iterations ahead of the poll that is waited for
  int round() {
    const int rc = advance();
    return rc ? rc : poll_state();
  }

  // x = q .* x + x0; iteration counts and stop codes are those of the last poll
  int finish(int *nit, int *istop) {
    if (wd == 1)
      hipLaunchKernelGGL(k_lsqr_finish<1>, dim3((n + 255) / 256), dim3(256), 0, st, n, q, Xl.p, W.p, sb(), X);
    else
      hipLaunchKernelGGL(k_lsqr_finish<NB>, dim3((n * NB + 255) / 256), dim3(256), 0, st, n, q, Xl.p, W.p, sb(), X);
    ANDR_HIP(ctx, hipGetLastError());
    ANDR_HIP(ctx, hipStreamSynchronize(st));
    for (int k = 0; k < nrhs; ++k) {
      if (nit) nit[k] = hs[k].itn;
      if (istop) istop[k] = hs[k].istop;
    }
    return ANDR_OK;
  }
};

}  // namespace

int andr_lsqr_device(andr_ctx *ctx, const void *A, bool fp32, int64_t lda, int m, int n, const double *q,
                     const double *B, double *X, int nrhs, int maxit, double eps, int *nit, int *istop) {
  LsqrRun R;
  int rc = R.begin(ctx, ctx->stream, A, fp32, lda, m, n, q, B, X, nrhs, maxit, eps);
  if (rc) return rc;
  if ((rc = R.advance())) return rc;
  while (!R.done)
    if ((rc = R.round())) return rc;
  return R.finish(nit, istop);
}

int andr_lsqr_device_csr(andr_ctx *ctx, int m, int n, int64_t nnz, const int64_t *ia, const int32_t *ja,
                         const double *a, const int64_t *tia, const int32_t *tja, const double *ta, const double *q,
                         const double *B, double *X, int nrhs, int maxit, double eps, int *nit, int *istop) {
  LsqrRun R;
  R.cia = ia;
  R.cja = ja;
  R.cva = a;
  R.tia = tia;
  R.tja = tja;
  R.tva = ta;
  R.nnz = nnz;
  int rc = R.begin(ctx, ctx->stream, nullptr, false, 0, m, n, q, B, X, nrhs, maxit, eps);
  if (rc) return rc;
  if ((rc = R.advance())) return rc;
  while (!R.done)
    if ((rc = R.round())) return rc;
  return R.finish(nit, istop);
}

int andr_lsqr_device_batch(andr_ctx *ctx, int count, const LsqrJob *jobs) {
  if (count <= 0) return ANDR_OK;
  if (count == 1 || andr_prof(ctx).on) {  // profiled: one after another, so that each event pair times one launch
    for (int i = 0; i < count; ++i) {
      const LsqrJob &J = jobs[i];
      const int rc =
          andr_lsqr_device(ctx, J.A, J.fp32, J.lda, J.m, J.n, J.q, J.B, J.X, J.nrhs, J.maxit, J.eps, J.nit, J.istop);
      if (rc) return rc;
    }
    return ANDR_OK;
  }
  ANDR_HIP(ctx, hipStreamSynchronize(ctx->stream));  // the systems are ready
  const int nst = std::min(count, LSQR_STREAMS);
  std::vector<hipStream_t> streams(nst, nullptr);
  int rc = ANDR_OK;
  for (int i = 0; i < nst && !rc; ++i)
    if (hipStreamCreateWithFlags(&streams[i], hipStreamNonBlocking) != hipSuccess)
      rc = andr_fail(ctx, ANDR_ERR_HIP, "stream creation for the LSQR batch");
  {
    std::vector<LsqrRun> runs(count);
    for (int i = 0; i < count && !rc; ++i) {
      const LsqrJob &J = jobs[i];
      rc = runs[i].begin(ctx, streams[i % nst], J.A, J.fp32, J.lda, J.m, J.n, J.q, J.B, J.X, J.nrhs, J.maxit, J.eps);
    }
    // all solves advance together, a block of iterations at a time, each on its stream
    for (auto &R : runs)
      if (!rc) rc = R.advance();
    for (bool left = !rc; left && !rc;) {
      left = false;
      for (auto &R : runs)
        if (!R.done && !rc) rc = R.advance();
      for (auto &R : runs)
        if (!R.done && !rc) {
          rc = R.poll_state();
          left = left || !R.done;
        }
    }
    for (int i = 0; i < count && !rc; ++i) rc = runs[i].finish(jobs[i].nit, jobs[i].istop);
    for (auto s : streams)
      if (s) (void)hipStreamSynchronize(s);  // the workspaces go back to the cache after this
  }
  for (auto s : streams)
    if (s) (void)hipStreamDestroy(s);
  return rc;
}

// ---- BiCGSTAB with a Jacobi preconditioner ---------------------------------------------------
// The Krylov alternative of the reference's LIS path for square systems (parLISslvSet
// "-i bicgstab -p jacobi -tol 1.0e-8 -maxiter 1000", src/mod_par.f90:288). LIS is not part of the
// reference's sources; the algorithm is the published preconditioned BiCGSTAB (van der Vorst 1992,
// in the form of Barrett et al., Templates, 1994, fig. 2.10): the preconditioner M = diag(A) acts
// on the search directions, the residual is the true one, and a column stops when
// ||r||_2 <= tol ||b||_2 (LIS's default criterion). NB columns advance together, each with its own
// scalars; the products are the matrix-core A X above.
namespace {

// An iteration is seven launches (the products two of them): vector kernels over n x NB elements, a thread
// each, that leave the dot products' partial sums p1 and p2, a pair of rows per block, and begin with the scalar
// step from the sums of the one before, done by every block alike; one block writes the new states to another
// array, as the others may still read the old one: S0 -> k_bicg_p -> S1 -> k_bicg_s -> S2 -> k_bicg_x -> S0.
// Latency of 121 blocks at n = 3841: 13 launches of 2.3 to 4.9 us beside the two products are now five of 4.3 to
// 4.6; the iterations enqueued past the end return at once. The sums keep the order of separate dot products:
// the iterates part from each other by far more than rounding where it changes.
__device__ inline void bicg_parts(double a, double b, double *__restrict__ p1, double *__restrict__ p2,
                                  double (*red)[4 * NB]) {
#pragma unroll
  for (int off = 8; off < 64; off <<= 1) {
    a += __shfl_xor(a, off, 64);
    b += __shfl_xor(b, off, 64);
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  __syncthreads();  // red may still be read
  if (lane < NB) {
    red[0][wid * NB + lane] = a;
    red[1][wid * NB + lane] = b;
  }
  __syncthreads();
  if (threadIdx.x < NB) {
    const int k = threadIdx.x;
    p1[(size_t)blockIdx.x * NB + k] = (red[0][k] + red[0][NB + k]) + (red[0][2 * NB + k] + red[0][3 * NB + k]);
    if (p2) p2[(size_t)blockIdx.x * NB + k] = (red[1][k] + red[1][NB + k]) + (red[1][2 * NB + k] + red[1][3 * NB + k]);
  }
}

// element t of A X from its segments' partial sums
__device__ inline double bicg_seg_sum(int64_t nb, int nseg, const double *__restrict__ P, int64_t t) {
  double s = 0.0;
  for (int s0 = 0; s0 < nseg; s0 += 8) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = P[(size_t)min(s0 + u, nseg - 1) * nb + t];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (s0 + u < nseg) s += v[u];
  }
  return s;
}

// Jacobi: dinv[j] = 1 / A[j][j] (1 where the diagonal is zero, as a Jacobi preconditioner leaves it)
__global__ void k_bicg_diag(const double *__restrict__ A, int64_t lda, int n, double *__restrict__ dinv) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const double d = A[(size_t)j * lda + j];
  dinv[j] = d != 0.0 ? 1.0 / d : 1.0;
}

// r = b - A x from the segments of A x; r_hat = r; p = v = 0; partials of b . b and r . r
__global__ __launch_bounds__(256) void k_bicg_init(int n, const double *__restrict__ B, int nseg,
                                                   const double *__restrict__ AX, double *__restrict__ R,
                                                   double *__restrict__ Rh, double *__restrict__ P,
                                                   double *__restrict__ V, double *__restrict__ pb,
                                                   double *__restrict__ pr) {
  __shared__ double red[2][4 * NB];
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  double bb = 0.0, rr = 0.0;
  if (t < n * NB) {
    const double b = B[t], r = b - bicg_seg_sum((int64_t)n * NB, nseg, AX, t);
    R[t] = r;
    Rh[t] = r;
    P[t] = 0.0;
    V[t] = 0.0;
    bb = b * b;
    rr = r * r;
  }
  bicg_parts(bb, rr, pb, pr, red);
}

// start: ||b||^2 and ||r0||^2; columns with r0 already small are done. rr, rho: r . r and r_hat . r (the same as
// r_hat = r) for the first iteration
__global__ void k_bicg_start(BicgState *st, const double *pb, const double *pr, int np, double tol, int nrhs,
                             double *rr, double *rho) {
  __shared__ double red[4 * NB];
  const double b2 = block_sum_parts<NB, 256>(pb, np, red);
  const double r2 = block_sum_parts<NB, 256>(pr, np, red);
  for (int i = threadIdx.x; i < np * NB; i += blockDim.x) rr[i] = rho[i] = pr[i];
  const int k = threadIdx.x;
  if (k >= NB) return;
  BicgState S;
  S.rho = S.alpha = S.omega = 1.0;
  S.a = 0.0;
  S.bnorm2 = b2;
  S.tol2 = tol * tol * b2;
  S.itn = 0;
  S.status = 0;
  S.active = k < nrhs && r2 > S.tol2 ? 1 : 0;
  st[k] = S;
}

// convergence: ||r||^2 <= tol^2 ||b||^2; omega = 0 (with r not small) is a breakdown. Done again with the same
// sum it changes nothing: the poll's kernel and the next iteration both begin with it.
__device__ inline void bicg_check(BicgState &S, double r2, int itnlim) {
  if (!S.active) return;
  if (r2 <= S.tol2) {
    S.active = 0;
    S.status = 0;
  } else if (S.omega == 0.0) {
    S.active = 0;
    S.status = 2;
  } else if (S.itn >= itnlim) {
    S.active = 0;
    S.status = 1;
  }
}
__global__ void k_bicg_check(BicgState *st, const double *rr, int np, int itnlim) {
  __shared__ double red[4 * NB];
  const double r2 = block_sum_parts<NB, 256>(rr, np, red);
  if (threadIdx.x < NB) bicg_check(st[threadIdx.x], r2, itnlim);
}

// rho_new = r_hat . r; beta = (rho_new / rho) (alpha / omega); p = r + beta (p - omega v); y = dinv .* p
__global__ __launch_bounds__(256) void k_bicg_p(int n, int np, const double *__restrict__ rr,
                                                const double *__restrict__ rhop, const double *__restrict__ R,
                                                const double *__restrict__ V, double *__restrict__ P,
                                                double *__restrict__ Yv, const double *__restrict__ dinv,
                                                const BicgState *__restrict__ s0, BicgState *__restrict__ s1,
                                                int itnlim) {
  __shared__ double red[4 * NB], sc[2][NB];
  __shared__ int act[NB];
  const int t = blockIdx.x * blockDim.x + threadIdx.x, tt = min(t, n * NB - 1);
  const double r = R[tt], p0 = P[tt], v = V[tt], d = dinv[tt >> 3];
  const double ps = thread_parts<NB, 256>(rr, np), qs = thread_parts<NB, 256>(rhop, np);
  const double r2 = block_sum<NB, 256>(ps, red);
  const double rho = block_sum<NB, 256>(qs, red);
  if (threadIdx.x < NB) {
    const int k = threadIdx.x;
    BicgState S = s0[k];
    bicg_check(S, r2, itnlim);
    double beta = 0.0;
    if (S.active && rho == 0.0) {  // breakdown: r_hat orthogonal to r
      S.active = 0;
      S.status = 2;
    } else if (S.active) {
      S.itn += 1;
      beta = S.itn == 1 ? 0.0 : (rho / S.rho) * (S.alpha / S.omega);
      S.rho = rho;
    }
    sc[0][k] = beta;
    sc[1][k] = S.omega;
    act[k] = S.active;
    if (blockIdx.x == gridDim.x - 1) s1[k] = S;
  }
  __syncthreads();
  if (t >= n * NB) return;
  const int k = t & 7;
  if (!act[k]) {
    Yv[t] = 0.0;
    return;
  }
  const double p = r + sc[0][k] * (p0 - sc[1][k] * v);
  P[t] = p;
  Yv[t] = d * p;
}

// v = A y from its segments; partials of r_hat . v
__global__ __launch_bounds__(256) void k_bicg_v(int n, int nseg, const double *__restrict__ AY,
                                                const double *__restrict__ Rh, double *__restrict__ V,
                                                double *__restrict__ p1, const BicgState *__restrict__ st) {
  __shared__ double red[2][4 * NB];
  if (!any_active<NB>(st)) return;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  double a = 0.0;
  if (t < n * NB) {
    const double v = bicg_seg_sum((int64_t)n * NB, nseg, AY, t);
    V[t] = v;
    a = Rh[t] * v;
  }
  bicg_parts(a, 0.0, p1, nullptr, red);
}

// alpha = rho / (r_hat . v); s = r - alpha v (into R); z = dinv .* s
__global__ __launch_bounds__(256) void k_bicg_s(int n, int np, const double *__restrict__ p1, double *__restrict__ R,
                                                const double *__restrict__ V, double *__restrict__ Z,
                                                const double *__restrict__ dinv, const BicgState *__restrict__ s1,
                                                BicgState *__restrict__ s2) {
  __shared__ double red[4 * NB], sc[NB];
  const bool any = any_active<NB>(s1);
  if (!any && blockIdx.x != gridDim.x - 1) return;
  const int t = blockIdx.x * blockDim.x + threadIdx.x, tt = min(t, n * NB - 1);
  const double r = R[tt], v = V[tt], d = dinv[tt >> 3];
  const double rv = block_sum_parts<NB, 256>(p1, np, red);
  if (threadIdx.x < NB) {
    const int k = threadIdx.x;
    BicgState S = s1[k];
    S.a = 0.0;
    if (S.active && rv == 0.0) {
      S.active = 0;
      S.status = 2;
    } else if (S.active) {
      S.alpha = S.a = S.rho / rv;
    }
    sc[k] = S.a;
    if (blockIdx.x == gridDim.x - 1) s2[k] = S;
  }
  __syncthreads();
  if (!any || t >= n * NB) return;
  const double s = r - sc[t & 7] * v;
  R[t] = s;
  Z[t] = d * s;
}

// t = A z from its segments; partials of t . s and t . t
__global__ __launch_bounds__(256) void k_bicg_t(int n, int nseg, const double *__restrict__ AZ,
                                                const double *__restrict__ R, double *__restrict__ Tv,
                                                double *__restrict__ p1, double *__restrict__ p2,
                                                const BicgState *__restrict__ st) {
  __shared__ double red[2][4 * NB];
  if (!any_active<NB>(st)) return;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  double a = 0.0, b = 0.0;
  if (t < n * NB) {
    const double v = bicg_seg_sum((int64_t)n * NB, nseg, AZ, t);
    Tv[t] = v;
    a = v * R[t];
    b = v * v;
  }
  bicg_parts(a, b, p1, p2, red);
}

// omega = (t . s) / (t . t); x += alpha y; x += omega z; r = s - omega t; partials of r . r and r_hat . r
__global__ __launch_bounds__(256) void k_bicg_x(int n, int np, const double *__restrict__ p1,
                                                const double *__restrict__ p2, double *__restrict__ X,
                                                const double *__restrict__ Yv, const double *__restrict__ Z,
                                                double *__restrict__ R, const double *__restrict__ Tv,
                                                const double *__restrict__ Rh, double *__restrict__ rr,
                                                double *__restrict__ rho, const BicgState *__restrict__ s2,
                                                BicgState *__restrict__ s0) {
  __shared__ double red[2][4 * NB], sc[2][NB];
  const bool any = any_active<NB>(s2);
  const int t = blockIdx.x * blockDim.x + threadIdx.x, tt = min(t, n * NB - 1);
  const double x0 = X[tt], y = Yv[tt], z = Z[tt], s = R[tt], v = Tv[tt], h = Rh[tt];
  const double as = thread_parts<NB, 256>(p1, np), bs = thread_parts<NB, 256>(p2, np);
  const double ts = block_sum<NB, 256>(as, red[0]);
  const double tp = block_sum<NB, 256>(bs, red[0]);
  if (threadIdx.x < NB) {
    const int k = threadIdx.x;
    BicgState S = s2[k];
    double om = 0.0;
    if (S.active && tp != 0.0) S.omega = om = ts / tp;
    sc[0][k] = S.a;
    sc[1][k] = om;
    if (blockIdx.x == gridDim.x - 1) s0[k] = S;
  }
  __syncthreads();
  double a = 0.0, b = 0.0;
  if (t < n * NB) {
    const double al = sc[0][t & 7], w = sc[1][t & 7];
    double x = x0;
    x += al * y;
    x += w * z;
    const double r = s - w * v;
    if (any) {
      X[t] = x;
      R[t] = r;
    }
    a = r * r;
    b = h * r;
  }
  if (any) bicg_parts(a, b, rr, rho, red);
}

}  // namespace

namespace {
// the shape of the BiCGSTAB product A X: column segments and the partial sums they leave (a function
// of n only, so that the workspace size is known before the call)
struct BicgLayout {
  int seglen, nseg, blocksM;
};
BicgLayout bicg_layout(int n) {
  BicgLayout L;
  L.seglen = AV_MAXCOLS;
  const int64_t rw = (n + 63) / 64;
  if (rw * ((n + AV_MAXCOLS - 1) / AV_MAXCOLS) < 2048) L.seglen = (int)std::max<int64_t>(256, ((int64_t)n * rw / 2048 + 15) / 16 * 16);
  L.nseg = (n + L.seglen - 1) / L.seglen;
  L.blocksM = (n * NB + 255) / 256;
  return L;
}
// doubles of each workspace array, in the order they are carved from a caller's region
void bicg_sizes(int n, size_t sz[12]) {
  const BicgLayout L = bicg_layout(n);
  for (int i = 0; i < 7; ++i) sz[i] = (size_t)n * NB;  // r, r_hat, p, v, y, z, t
  sz[7] = n;                                           // dinv
  sz[8] = (size_t)L.blocksM * NB;                      // p1
  sz[9] = (size_t)L.blocksM * NB;                      // p2
  sz[10] = 3 * ((sizeof(BicgState) * NB + 7) / 8);     // per-column states S0, S1, S2
  // A X segment partials; from the end of an iteration to its next product, those of r . r and r_hat . r
  sz[11] = std::max((size_t)L.nseg * n, 2 * (size_t)L.blocksM) * NB;
}
}  // namespace

size_t andr_bicgstab_ws_bytes(int n) {
  size_t sz[12], tot = 0;
  bicg_sizes(n, sz);
  for (size_t v : sz) tot += (v + 31) / 32 * 32;  // every array on a 256-byte boundary
  return tot * sizeof(double);
}

int andr_bicgstab_device(andr_ctx *ctx, const double *A, int64_t lda, int n, const double *B, double *X, int nrhs,
                         int maxit, double tol, int *nit, int *status, double *ws, size_t ws_bytes) {
  if (nrhs < 1 || nrhs > NB) return andr_fail(ctx, ANDR_ERR_ARG, "nrhs must be 1..%d", NB);
  if (n < 1) return andr_fail(ctx, ANDR_ERR_ARG, "empty system");
  hipStream_t st = ctx->stream;
  const BicgLayout L = bicg_layout(n);
  const int tiles = av_tiles(n, (L.nseg + AV_WAVES - 1) / AV_WAVES);
  const int nb = L.blocksM;
  // workspace: the context's memory cache, or carved from the caller's region (no allocation)
  constexpr int NW = 12;
  DevBuf<double> own[NW];
  double *w[NW];
  size_t sz[NW];
  bicg_sizes(n, sz);
  if (ws) {
    if (ws_bytes < andr_bicgstab_ws_bytes(n))
      return andr_fail(ctx, ANDR_ERR_ARG, "BiCGSTAB workspace of %zu bytes, %zu needed (n=%d)", ws_bytes,
                       andr_bicgstab_ws_bytes(n), n);
    double *cur = ws;
    for (int i = 0; i < NW; ++i) {
      w[i] = cur;
      cur += (sz[i] + 31) / 32 * 32;
    }
  } else {
    for (int i = 0; i < NW; ++i) {
      if (own[i].alloc(sz[i], ctx)) return andr_fail(ctx, ANDR_ERR_ALLOC, "BiCGSTAB workspace (n=%d)", n);
      w[i] = own[i].p;
    }
  }
  double *Rr = w[0], *Rh = w[1], *P = w[2], *V = w[3], *Yv = w[4], *Z = w[5], *Tt = w[6], *dinv = w[7], *p1 = w[8],
         *p2 = w[9], *pn = w[11];
  BicgState *S = (BicgState *)w[10], *S1 = S + NB, *S2 = S + 2 * NB;
  double *rr = pn, *rho = pn + (size_t)nb * NB;
  const int gb = nb;
  auto product = [&](const double *in, const BicgState *s) {  // no profiling records with a caller's workspace
    const int t = ws ? -1 : andr_prof_begin(ctx, "lsqr_gemv_n", (double)n * n * 8.0 + (2.0 + L.nseg) * n * NB * 8.0, 2.0 * n * n * nrhs);
    launch_av<true>(st, tiles, A, lda, n, n, in, {(L.nseg + AV_WAVES - 1) / AV_WAVES, L.seglen}, pn, s);
    andr_prof_end(ctx, t);
  };
  hipLaunchKernelGGL(k_bicg_diag, dim3((n + 255) / 256), dim3(256), 0, st, A, lda, n, dinv);
  product(X, nullptr);  // A x0
  hipLaunchKernelGGL(k_bicg_init, dim3(gb), dim3(256), 0, st, n, B, L.nseg, pn, Rr, Rh, P, V, p1, p2);
  hipLaunchKernelGGL(k_bicg_start, dim3(1), dim3(256), 0, st, S, p1, p2, nb, tol, nrhs, rr, rho);
  const int itnlim = maxit > 0 ? maxit : 1000;
  BicgState hs[NB];
  for (int it = 0; it < itnlim;) {
    for (int inner = 0; inner < 8 && it < itnlim; ++inner, ++it) {
      hipLaunchKernelGGL(k_bicg_p, dim3(gb), dim3(256), 0, st, n, nb, rr, rho, Rr, V, P, Yv, dinv, S, S1, itnlim);
      product(Yv, S1);
      hipLaunchKernelGGL(k_bicg_v, dim3(gb), dim3(256), 0, st, n, L.nseg, pn, Rh, V, p1, S1);
      hipLaunchKernelGGL(k_bicg_s, dim3(gb), dim3(256), 0, st, n, nb, p1, Rr, V, Z, dinv, S1, S2);
      product(Z, S2);
      hipLaunchKernelGGL(k_bicg_t, dim3(gb), dim3(256), 0, st, n, L.nseg, pn, Rr, Tt, p1, p2, S2);
      hipLaunchKernelGGL(k_bicg_x, dim3(gb), dim3(256), 0, st, n, nb, p1, p2, X, Yv, Z, Rr, Tt, Rh, rr, rho, S2, S);
    }
    hipLaunchKernelGGL(k_bicg_check, dim3(1), dim3(256), 0, st, S, rr, nb, itnlim);
    ANDR_HIP(ctx, hipGetLastError());
    ANDR_HIP(ctx, hipMemcpyAsync(hs, S, sizeof(hs), hipMemcpyDeviceToHost, st));
    ANDR_HIP(ctx, hipStreamSynchronize(st));
    bool any = false;
    for (int k = 0; k < nrhs; ++k) any = any || hs[k].active;
    if (!any) break;
  }
  ANDR_HIP(ctx, hipMemcpyAsync(hs, S, sizeof(hs), hipMemcpyDeviceToHost, st));
  ANDR_HIP(ctx, hipStreamSynchronize(st));
  for (int k = 0; k < nrhs; ++k) {
    if (nit) nit[k] = hs[k].itn;
    if (status) status[k] = hs[k].active ? 1 : hs[k].status;
  }
  return ANDR_OK;
}
