// Multigrid-preconditioned CG on the GPU.
//
// Replaces HYPRE PCG + BoomerAMG (ProjectionP.f90:95-116, 267-299).  The
// outer CG, its dot products and the residual are FP64; the V-cycle runs in
// T = float (mixed) or double (FP64).  CG scalars stay in device memory: the
// host only polls a convergence flag the finalize kernel writes into pinned
// host memory, one iteration behind.
//
// The search direction p and the iterate x are not carried through the
// iterations.  With p_k = z_k - m_k + beta_k p_{k-1} the CG needs p only in
// q = A p (a recurrence of its own, q_k = A (z_k - m_k) + beta_k q_{k-1}), in
// (p, q), which equals (z - m, q) because beta makes the new direction
// A-orthogonal to the last one, and in x, which is a combination of the z_k.
// So the preconditioned residuals are kept (kZRing of them) and x is formed
// from them in one pass at the end.
//
// Multigrid: cell-centred coarsening by 2, piecewise-constant transfers
// (restriction = sum over children, prolongation = injection), coarse face
// coefficients = scale * sum of the fine face coefficients they cover (the
// Galerkin product for these transfers, scaled), red-black Gauss-Seidel
// (pre: red,black; post: black,red -- a symmetric V-cycle).  The last levels,
// of up to about 4096 cells, run in one single-workgroup kernel.
//
// Grid kernels run one cell per thread on 64x4 workgroups whose order is
// remapped so that each XCD owns a contiguous slab (stencil halos stay in one
// L2); reductions store one partial per workgroup and a one-workgroup
// finalize kernel folds them in a fixed order.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "sp_device.h"
#include "sp_geom.h"
#include "sp_internal.h"
#include "sp_smooth_cell.h"
#include "sp_smooth_fused.h"

namespace sp {
namespace {

template <typename T>
struct LevelView {
  int nx, ny, nz;
  const T *cx, *cy, *cz, *e;
  T* x;
  T* b;
  const uint8_t* act;  // active mask (level 0 only), else nullptr
};

template <typename T>
__device__ inline T diag_of(const LevelView<T>& L, int i, int j, int k, int64_t n) {
  const int64_t sy = L.nx, sz = (int64_t)L.nx * L.ny;
  T d = i > 0 ? L.cx[n - 1] : T(0);
  d = d + (j > 0 ? L.cy[n - sy] : T(0));
  d = d + (k > 0 ? L.cz[n - sz] : T(0));
  d = d + L.cx[n];
  d = d + L.cy[n];
  d = d + L.cz[n];
  if (L.e) d = d + L.e[n];
  return d;
}

// sum_nb c_f x_nb
template <typename T>
__device__ inline T offdiag_sum(const LevelView<T>& L, int i, int j, int k, int64_t n) {
  const int64_t sy = L.nx, sz = (int64_t)L.nx * L.ny;
  T s = T(0);
  if (i > 0) s += L.cx[n - 1] * L.x[n - 1];
  if (j > 0) s += L.cy[n - sy] * L.x[n - sy];
  if (k > 0) s += L.cz[n - sz] * L.x[n - sz];
  if (i < L.nx - 1) s += L.cx[n] * L.x[n + 1];
  if (j < L.ny - 1) s += L.cy[n] * L.x[n + sy];
  if (k < L.nz - 1) s += L.cz[n] * L.x[n + sz];
  return s;
}

// One colour of Gauss-Seidel; one thread per cell pair along i (the pair
// holds one cell of each colour).  zero_init: x starts at 0 (the other colour
// is written as 0).  FINE only distinguishes the finest level in profiles.
template <typename T, bool FINE>
__global__ void __launch_bounds__(256) k_gs(LevelView<T> L, int color, int zero_init, T omega,
                                            const Scalars* S) {
  if (S->done) return;
  const int nxh = (L.nx + 1) >> 1;
  const Cell3 q = cell_of(nxh, L.ny, L.nz);
  if (!q.in) return;
  const int j = q.b, k = q.c;
  const int par = (j + k + color) & 1;
  const int i = 2 * q.a + par;
  const int64_t row = (int64_t)L.nx * (j + (int64_t)L.ny * k);
  if (zero_init) {
    const int io = 2 * q.a + (par ^ 1);
    if (io < L.nx) L.x[row + io] = T(0);
  }
  if (i >= L.nx) return;
  const int64_t n = row + i;
  const T d = diag_of(L, i, j, k, n);
  if (!(d > T(0))) {
    if (zero_init) L.x[n] = T(0);
    return;
  }
  T s = L.b[n];
  if (!zero_init) s += offdiag_sum(L, i, j, k, n);
  // FP32 multiplies by the hardware reciprocal; over-relaxed by omega
  const T v = sizeof(T) == 4 ? s * smoother_rcp(d) : s / d;
  const T x0 = zero_init ? T(0) : L.x[n];
  L.x[n] = x0 + omega * (v - x0);
}

// One step of the Chebyshev semi-iteration for D^-1 A (Saad, Iterative
// Methods for Sparse Linear Systems, 2nd ed., Algorithm 12.1):
//   d <- c1 d + c2 D^-1 (b - A x_in),  x_out = x_in + d
// (c1 unused on the first step; x_in == nullptr stands for x_in = 0).
// x_out is another buffer than x_in: every lane reads its neighbours' x_in.
template <typename T, bool FINE>
__global__ void __launch_bounds__(256) k_cheb(LevelView<T> L, const T* __restrict__ xin,
                                              T* __restrict__ xout, T* __restrict__ dv, T c1,
                                              T c2, int first, const Scalars* S) {
  if (S->done) return;
  const Cell3 q = cell_of(L.nx, L.ny, L.nz);
  if (!q.in) return;
  const int i = q.a, j = q.b, k = q.c;
  const int64_t n = i + (int64_t)L.nx * (j + (int64_t)L.ny * k);
  const T d = diag_of(L, i, j, k, n);
  if (!(d > T(0))) {
    xout[n] = T(0);
    dv[n] = T(0);
    return;
  }
  T r = L.b[n];
  T x0 = T(0);
  if (xin) {
    LevelView<T> V = L;
    V.x = const_cast<T*>(xin);
    x0 = xin[n];
    r = r - (d * x0 - offdiag_sum(V, i, j, k, n));
  }
  const T z = sizeof(T) == 4 ? r * smoother_rcp(d) : r / d;
  const T dn = first ? c2 * z : c1 * dv[n] + c2 * z;
  dv[n] = dn;
  xout[n] = x0 + dn;
}

// Coarse b = sum over children of the fine residual.
template <typename T, bool FINE>
__global__ void __launch_bounds__(256) k_resid_restrict(LevelView<T> F, LevelView<T> C,
                                                        const Scalars* S) {
  if (S->done) return;
  const Cell3 q = cell_of(C.nx, C.ny, C.nz);
  if (!q.in) return;
  T s = T(0);
#pragma unroll
  for (int cc = 0; cc < 2; ++cc)
#pragma unroll
    for (int bb = 0; bb < 2; ++bb)
#pragma unroll
      for (int aa = 0; aa < 2; ++aa) {
        const int fi = 2 * q.a + aa, fj = 2 * q.b + bb, fk = 2 * q.c + cc;
        if (fi >= F.nx || fj >= F.ny || fk >= F.nz) continue;
        const int64_t m = fi + (int64_t)F.nx * (fj + (int64_t)F.ny * fk);
        const T d = diag_of(F, fi, fj, fk, m);
        if (d > T(0)) s += F.b[m] - (d * F.x[m] - offdiag_sum(F, fi, fj, fk, m));
      }
  C.b[q.a + (int64_t)C.nx * (q.b + (int64_t)C.ny * q.c)] = s;
}

template <typename T, bool FINE>
__global__ void __launch_bounds__(256) k_prolong(LevelView<T> F, LevelView<T> C, const Scalars* S) {
  if (S->done) return;
  const Cell3 q = cell_of(F.nx, F.ny, F.nz);
  if (!q.in) return;
  const int64_t m = q.a + (int64_t)F.nx * (q.b + (int64_t)F.ny * q.c);
  const bool act = F.act ? F.act[m] != 0 : diag_of(F, q.a, q.b, q.c, m) > T(0);
  if (act) F.x[m] += C.x[(q.a >> 1) + (int64_t)C.nx * ((q.b >> 1) + (int64_t)C.ny * (q.c >> 1))];
}

// ---- single-workgroup V-cycle over the small levels ----

// The last levels of the V-cycle in one workgroup.  Every cell belongs to one
// thread for the whole launch: couplings, b and 1/d in registers, x in LDS
// (one array per level with a border of zeros, so a neighbour read needs no
// test).  Threads own i pairs, one red and one black cell: two pairs per
// thread on the first level, one on one of the others.  All levels are loaded
// at once.
//
// The time is a chain of about forty barrier-separated steps on one CU, so
// what counts is the instructions and LDS accesses of a step.  With the
// couplings in LDS too, cell indices formed in every step and the level table
// read from global memory two levels (8^3 and 4^3) took 22 us a cycle, and a
// 16^3 level was better off in legs of 9 us (FP32) each; here the three levels
// take 21 us in FP32 and 29 in FP64 (event times, 5 us of them the launch).
//
// BIG = 4: a coarsest level alone with four pairs per thread, for one that two
// do not hold (a hierarchy cut short, a grid too thin to coarsen).  In FP32
// the couplings of four still fit the registers (FP64 spills with two).  It
// beats one launch per half-sweep over the whole chip, and keeps the mean out
// of a singular system's coarse solve, up to the last size it holds (whole
// solves: 40 x 40 x 3 7.25 -> 5.29 ms, 50 x 50 x 2 6.81 -> 5.05, one level of
// 18^3 3.34 -> 2.96, of 20^3 3.65 -> 3.41, of 24 x 24 x 14 3.82 -> 3.55).
constexpr int kTailThreads = 1024, kTailLevels = 8;

template <typename T>
struct TailArgs {
  int n;  // levels
  int pre, post, coarse_sweeps, singular;
  T omega[kTailLevels];  // over-relaxation of the Gauss-Seidel updates
  int nx[kTailLevels], ny[kTailLevels], nz[kTailLevels];
  int first[kTailLevels];           // first thread of a level (levels 1 and up)
  int xo[kTailLevels], ro[kTailLevels];  // LDS offsets: x with its border, residual
  const T *cx[kTailLevels], *cy[kTailLevels], *cz[kTailLevels], *e[kTailLevels];
  const T* b;
  T* x;
};

template <typename T>
int64_t tail_pairs(const Level<T>& L) { return (int64_t)((L.nx + 1) / 2) * L.ny * L.nz; }
// Threads that a level's pairs take, in whole waves.
inline int tail_threads(int nx, int ny, int nz) { return ((nx + 1) / 2 * ny * nz + 63) / 64 * 64; }

// n / d for n and d below 2^23: the float estimate is within 1 of the quotient.
__device__ inline unsigned small_div(unsigned n, unsigned d) {
  unsigned q = (unsigned)((float)n * __builtin_amdgcn_rcpf((float)d));
  if (q * d > n) --q;
  else if ((q + 1) * d <= n) ++q;
  return q;
}

// Cells 2a and 2a + 1 of one row; [0] the red one (i + j + k even), [1] the
// black one.  The second cell of a pair cut by an odd nx has 1/d = 0 and lies
// on the LDS border, where it writes 0.
template <typename T, bool HAS_E>
struct TailPair {
  T cw[2], ce[2], cs[2], cn[2], cb[2], ct[2], b[2], rd[2];
  T d[HAS_E ? 2 : 1];  // the diagonal, only where the couplings do not add up to it
  int at[2];           // x in LDS
  int m;               // cell index of cell 2a in the level
  int up;              // x of the parent cell in LDS
  bool any, hi, odd;   // the pair, its second cell exist; red is the second cell

  __device__ inline T diag(int q) const {
    if (HAS_E) return d[HAS_E ? q : 0];
    T v = cw[q] + cs[q];
    v = v + cb[q];
    v = v + ce[q];
    v = v + cn[q];
    return v + ct[q];
  }
  // cell index of q, and whether the cell exists
  __device__ inline int cell(int q) const { return m + ((q == 0) == odd ? 1 : 0); }
  __device__ inline bool exists(int q) const { return any && (hi || (q == 0) != odd); }
  // sum of the couplings times the neighbours' x
  __device__ inline T offdiag(int q, const T* xs, int py, int pz) const {
    const T* x = xs + at[q];
    T s = cw[q] * x[-1];
    s += ce[q] * x[1];
    s += cs[q] * x[-py];
    s += cn[q] * x[py];
    s += cb[q] * x[-pz];
    s += ct[q] * x[pz];
    return s;
  }
};

template <typename T, bool HAS_E>
__device__ inline void tail_load(TailPair<T, HAS_E>& P, const TailArgs<T>& A, int l, int t) {
  const int nx = A.nx[l], ny = A.ny[l], nz = A.nz[l], nxh = (nx + 1) >> 1;
  P.any = t < nxh * ny * nz;
  const unsigned tt = P.any ? (unsigned)t : 0u, jk = small_div(tt, nxh), a = tt - jk * nxh;
  const int k = (int)small_div(jk, ny), j = (int)jk - k * ny;
  const int py = nx + 2, pz = py * (ny + 2);
  P.odd = ((j + k) & 1) != 0;
  P.hi = 2 * (int)a + 1 < nx;
  P.m = 2 * (int)a + nx * (j + ny * k);
  // the parent: cell a of row j / 2, plane k / 2 of the next level
  if (l + 1 < A.n)
    P.up = A.xo[l + 1] + (int)a + 1 +
           (A.nx[l + 1] + 2) * ((j >> 1) + 1 + (A.ny[l + 1] + 2) * ((k >> 1) + 1));
  const T *cx = A.cx[l], *cy = A.cy[l], *cz = A.cz[l], *e = A.e[l];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int second = (q == 0) == P.odd ? 1 : 0, i = 2 * (int)a + second;
    const bool in = P.exists(q);
    P.at[q] = A.xo[l] + i + 1 + py * (j + 1) + pz * (k + 1);
    const int m = in ? P.m + second : P.m;  // a cell that exists
    const T cw = cx[i > 0 && in ? m - 1 : m], cs = cy[j > 0 ? m - nx : m],
            cb = cz[k > 0 ? m - nx * ny : m], ce = cx[m], cn = cy[m], ct = cz[m];
    const T b = l == 0 ? A.b[m] : T(0);
    // a cell that does not exist has no couplings
    P.cw[q] = in && i > 0 ? cw : T(0);
    P.cs[q] = in && j > 0 ? cs : T(0);
    P.cb[q] = in && k > 0 ? cb : T(0);
    P.ce[q] = in ? ce : T(0);
    P.cn[q] = in ? cn : T(0);
    P.ct[q] = in ? ct : T(0);
    P.b[q] = in ? b : T(0);
    // same order as the other kernels: W, S, B, E, N, T, then e
    T d = P.cw[q] + P.cs[q];
    d = d + P.cb[q];
    d = d + P.ce[q];
    d = d + P.cn[q];
    d = d + P.ct[q];
    if (HAS_E) {
      d = d + (in ? e[m] : T(0));
      P.d[HAS_E ? q : 0] = d;
    }
    P.rd[q] = d > T(0) ? T(1) / d : T(0);
  }
}

// The workgroup's state.  TOP: the first level (BIG pairs of every thread),
// otherwise level l (one pair of the threads with mine == l); the two are told
// apart at compile time so that the pairs stay in registers.
template <typename T, bool HAS_E, int BIG>
struct Tail {
  using Pair = TailPair<T, HAS_E>;
  const TailArgs<T>& A;
  T* xs;
  double (*red)[kTailThreads / 64];
  Pair big[BIG], small;
  int t, mine;

  template <bool TOP, typename F>
  __device__ __forceinline__ void own(int l, F f) {
    if constexpr (TOP) {
#pragma unroll
      for (int p = 0; p < BIG; ++p)
        if (big[p].any) f(big[p]);
    } else if (mine == l && small.any) {
      f(small);
    }
  }
  template <bool TOP, int Q>
  __device__ __forceinline__ void sweep(int l, bool zero = false) {
    const int py = A.nx[l] + 2, pz = py * (A.ny[l] + 2);
    const T om = A.omega[l];
    T* x = xs;
    own<TOP>(l, [=](Pair& P) __attribute__((always_inline)) {
      // 1/d = 0 keeps cells without couplings at 0
      if (zero) {
        x[P.at[Q]] = om * (P.b[Q] * P.rd[Q]);
      } else {
        const T x0 = x[P.at[Q]];
        x[P.at[Q]] = x0 + om * ((P.b[Q] + P.offdiag(Q, x, py, pz)) * P.rd[Q] - x0);
      }
    });
    __syncthreads();
  }
  // v -= mean of v over the cells with d > 0 (v: b or x of the last level)
  template <bool TOP, bool OF_X>
  __device__ __forceinline__ void project_mean(int l) {
    double s = 0.0, c = 0.0;
    T* x = xs;
    own<TOP>(l, [&](Pair& P) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < 2; ++q)
        if (P.rd[q] > T(0)) {
          s += (double)(OF_X ? x[P.at[q]] : P.b[q]);
          c += 1.0;
        }
    });
    s = wave_sum(s);
    c = wave_sum(c);
    if ((t & 63) == 0) { red[0][t >> 6] = s; red[1][t >> 6] = c; }
    __syncthreads();
    double ts = 0.0, tc = 0.0;
#pragma unroll
    for (int w = 0; w < kTailThreads / 64; ++w) { ts += red[0][w]; tc += red[1][w]; }
    const T mean = tc > 0 ? (T)(ts / tc) : T(0);
    own<TOP>(l, [=](Pair& P) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < 2; ++q)
        if (P.rd[q] > T(0)) {
          if (OF_X) x[P.at[q]] -= mean;
          else P.b[q] -= mean;
        }
    });
    __syncthreads();
  }
  // pre-smoothing of level l and coarse b = sum over the 2x2x2 children of
  // the fine residual
  template <bool TOP>
  __device__ __forceinline__ void down(int l) {
    sweep<TOP, 0>(l, true);
    sweep<TOP, 1>(l);
    for (int s = 1; s < A.pre; ++s) { sweep<TOP, 0>(l); sweep<TOP, 1>(l); }
    T* x = xs;
    T* r = xs + A.ro[l];
    const int nx = A.nx[l], ny = A.ny[l], nz = A.nz[l], py = nx + 2, pz = py * (ny + 2);
    // one value per pair, at the pair's first cell: its two cells are siblings
    own<TOP>(l, [=](Pair& P) __attribute__((always_inline)) {
      T v = T(0);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const T w = P.b[q] - (P.diag(q) * x[P.at[q]] - P.offdiag(q, x, py, pz));
        v += P.rd[q] > T(0) ? w : T(0);
      }
      r[P.m] = v;
    });
    __syncthreads();
    if (mine == l + 1 && small.any) {
      const int cnx = A.nx[l + 1], cny = A.ny[l + 1];
      // (i, j, k) of the pair's first cell; i is even
      const unsigned jk = small_div((unsigned)small.m, (unsigned)cnx);
      const int i = small.m - (int)jk * cnx, k = (int)small_div(jk, (unsigned)cny),
                j = (int)jk - k * cny;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int ci = i + ((q == 0) == small.odd ? 1 : 0);
        T s = T(0);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const int fj = 2 * j + (w & 1), fk = 2 * k + (w >> 1);
          const bool in = 2 * ci < nx && fj < ny && fk < nz;
          const T v = r[in ? 2 * ci + nx * (fj + ny * fk) : 0];
          s += in ? v : T(0);
        }
        small.b[q] = s;
      }
    }
  }
  template <bool TOP>
  __device__ __forceinline__ void coarsest(int l) {
    if (A.singular) project_mean<TOP, false>(l);
    sweep<TOP, 0>(l, true);
    sweep<TOP, 1>(l);
    for (int s = 1; s < A.coarse_sweeps; ++s) { sweep<TOP, 0>(l); sweep<TOP, 1>(l); }
    for (int s = 0; s < A.coarse_sweeps; ++s) { sweep<TOP, 1>(l); sweep<TOP, 0>(l); }
    if (A.singular) project_mean<TOP, true>(l);
  }
  // correction from level l + 1 and post-smoothing of level l
  template <bool TOP>
  __device__ __forceinline__ void up(int l) {
    T* x = xs;
    own<TOP>(l, [=](Pair& P) __attribute__((always_inline)) {
      const T v = x[P.up];
#pragma unroll
      for (int q = 0; q < 2; ++q)
        if (P.rd[q] > T(0)) x[P.at[q]] += v;
    });
    __syncthreads();
    for (int s = 0; s < A.post; ++s) { sweep<TOP, 1>(l); sweep<TOP, 0>(l); }
  }
};

template <typename T, bool HAS_E, int BIG>
__global__ void __launch_bounds__(kTailThreads) k_tail(TailArgs<T> A, const Scalars* S) {
  if (S->done) return;
  constexpr bool kAlone = BIG > 2;
  __shared__ double lds_raw[kTailLdsBytes / sizeof(double)];
  __shared__ double red[2][kTailThreads / 64];
  Tail<T, HAS_E, BIG> W{A, reinterpret_cast<T*>(lds_raw), red, {}, {}, (int)threadIdx.x, 0};
#pragma unroll
  for (int p = 0; p < BIG; ++p) tail_load(W.big[p], A, 0, W.t + p * kTailThreads);
  if constexpr (!kAlone) {
    for (int l = 1; l < A.n; ++l)
      if (W.t >= A.first[l]) W.mine = l;
    W.small.any = false;
    if (W.mine) tail_load(W.small, A, W.mine, W.t - A.first[W.mine]);
  }
  // the x arrays lie before the residuals
  for (int q = W.t; q < A.ro[0]; q += kTailThreads) W.xs[q] = T(0);
  __syncthreads();
  const int last = kAlone ? 0 : A.n - 1;
  if (last == 0) {
    W.template coarsest<true>(0);
  } else if constexpr (!kAlone) {
    W.template down<true>(0);
    for (int l = 1; l < last; ++l) W.template down<false>(l);
    W.template coarsest<false>(last);
    for (int l = last - 1; l > 0; --l) W.template up<false>(l);
    W.template up<true>(0);
  }
#pragma unroll
  for (int p = 0; p < BIG; ++p)
#pragma unroll
    for (int q = 0; q < 2; ++q)
      if (W.big[p].exists(q)) A.x[W.big[p].cell(q)] = W.xs[W.big[p].at[q]];
}

template <typename T>
__global__ void __launch_bounds__(256) k_coarsen(LevelView<T> F, LevelView<T> C, T* ccx, T* ccy,
                                                 T* ccz, T* ce, T scale) {
  const Cell3 q = cell_of(C.nx, C.ny, C.nz);
  if (!q.in) return;
  T sx = 0, sy = 0, sz = 0, se = 0;
  for (int cc = 0; cc < 2; ++cc)
    for (int bb = 0; bb < 2; ++bb)
      for (int aa = 0; aa < 2; ++aa) {
        const int fi = 2 * q.a + aa, fj = 2 * q.b + bb, fk = 2 * q.c + cc;
        if (fi >= F.nx || fj >= F.ny || fk >= F.nz) continue;
        const int64_t m = fi + (int64_t)F.nx * (fj + (int64_t)F.ny * fk);
        if (F.e) se += F.e[m];
        if (aa == 1) sx += F.cx[m];
        if (bb == 1) sy += F.cy[m];
        if (cc == 1) sz += F.cz[m];
      }
  const int64_t n = q.a + (int64_t)C.nx * (q.b + (int64_t)C.ny * q.c);
  ccx[n] = scale * sx;
  ccy[n] = scale * sy;
  ccz[n] = scale * sz;
  if (ce) ce[n] = scale * se;
}

// ---- outer CG (FP64) ----

struct CgArgs {
  int I, J, K;
  const double *cx, *cy, *cz, *e;
  const uint8_t* active;
  const float* dw;
  const double *dxp, *dyp, *dzp;
  const double* b;
  double *x, *r, *q;
  double* p;  // search direction at the last pass that formed x
  int slot;   // this iteration's entry in the history of z, beta, m and alpha
  double* z64;  // written by the Jacobi preconditioner only
  const float* z32;
  float* r32;
  Scalars* S;
  int32_t* hflag;  // pinned host flag (device view)
  double tol;
  RedSite site;
};

__device__ inline double zval(const CgArgs& A, int64_t n) {
  return A.z32 ? (double)A.z32[n] : A.z64[n];
}

__device__ inline double apply_row(const CgArgs& A, const double* v, int a, int b, int c,
                                   int64_t n) {
  // (A v)_n in difference form: sum of c_f (v_n - v_nb) plus the
  // diagonal-only terms.  Neighbouring values of an iterate with a large
  // level (a pressure fixed by a Dirichlet face) are close, so their
  // differences are exact and the result is accurate to the size of the
  // fluxes rather than to that of the level.
  const int64_t IJ = (int64_t)A.I * A.J;
  const double vn = v[n];
  double s = A.e ? A.e[n] * vn : 0.0;
  if (a > 0) s += A.cx[n - 1] * (vn - v[n - 1]);
  if (b > 0) s += A.cy[n - A.I] * (vn - v[n - A.I]);
  if (c > 0) s += A.cz[n - IJ] * (vn - v[n - IJ]);
  s += a < A.I - 1 ? A.cx[n] * (vn - v[n + 1]) : A.cx[n] * vn;
  s += b < A.J - 1 ? A.cy[n] * (vn - v[n + A.I]) : A.cy[n] * vn;
  s += c < A.K - 1 ? A.cz[n] * (vn - v[n + IJ]) : A.cz[n] * vn;
  return s;
}

// Residual of the refined pressure x + xd of a non-singular system:
// rt = b - A x - A xd on active cells, in difference form; max |rt|/V.
__global__ void __launch_bounds__(256) k_refine_residual(CgArgs A, const double* xd, double* rt) {
  const Col3 q = col_of(A.I, A.J, A.K);
  double v[1] = {0.0};
  if (q.in) {
    const int64_t IJ = (int64_t)A.I * A.J;
    const double dxy = A.dxp[q.a] * A.dyp[q.b];
    int64_t n = q.a + (int64_t)A.I * (q.b + (int64_t)A.J * q.c0);
    for (int c = q.c0; c < q.c1; ++c, n += IJ) {
      double rv = 0.0;
      if (A.active[n]) {
        rv = A.b[n] - apply_row(A, A.x, q.a, q.b, c, n);
        rv -= apply_row(A, xd, q.a, q.b, c, n);
        const double rr = fabs(rv) / (dxy * A.dzp[c]);
        v[0] = (rr > v[0] || rr != rr) ? rr : v[0];
      }
      rt[n] = rv;
    }
  }
  block_partials<kTileThreads, 1, 1u>(A.site, v);
}

__global__ void __launch_bounds__(kFinThreads) k_refine_residual_fin(CgArgs A, uint32_t nb) {
  double out[1];
  finalize_partials<kFinThreads, 1, 1u>(A.site, nb, out);
  if (flat_tid() == 0) A.S->npart[0] = out[0];
}

// y += x
__global__ void __launch_bounds__(256) k_refine_add(CgArgs A, const double* x, double* y) {
  const Col3 q = col_of(A.I, A.J, A.K);
  if (!q.in) return;
  const int64_t IJ = (int64_t)A.I * A.J;
  int64_t n = q.a + (int64_t)A.I * (q.b + (int64_t)A.J * q.c0);
  for (int c = q.c0; c < q.c1; ++c, n += IJ) y[n] += x[n];
}

// Jacobi preconditioner (SP_PRECOND_JACOBI): z = r / diagonal on active cells
__global__ void __launch_bounds__(256) k_cg_jacobi(CgArgs A) {
  if (A.S->done) return;
  const Col3 q = col_of(A.I, A.J, A.K);
  if (!q.in) return;
  const int64_t IJ = (int64_t)A.I * A.J;
  int64_t n = q.a + (int64_t)A.I * (q.b + (int64_t)A.J * q.c0);
  for (int c = q.c0; c < q.c1; ++c, n += IJ) {
    double d = q.a > 0 ? A.cx[n - 1] : 0.0;
    d = d + (q.b > 0 ? A.cy[n - A.I] : 0.0);
    d = d + (c > 0 ? A.cz[n - IJ] : 0.0);
    d = d + A.cx[n];
    d = d + A.cy[n];
    d = d + A.cz[n];
    if (A.e) d = d + A.e[n];
    A.z64[n] = (A.active[n] && d > 0.0) ? A.r[n] / d : 0.0;
  }
}

// r = b - mean(b) - A x  (x = 0, not read, when from_zero).  KC cells of a
// column per thread, the mask and b of all of them loaded first (cell
// index clamped into the column).
template <int KC>
__global__ void __launch_bounds__(256) k_cg_residual(CgArgs A, int from_zero) {
  const Col3 q = col_of<KC>(A.I, A.J, A.K);
  Scalars* S = A.S;
  const double bmean = S->bmean;
  double v[3] = {0.0, 0.0, 0.0};  // max |r|/V, non-finite, sum r
  if (q.in) {
    const int64_t IJ = (int64_t)A.I * A.J;
    const double dxy = A.dxp[q.a] * A.dyp[q.b];
    const int64_t n0 = q.a + (int64_t)A.I * (q.b + (int64_t)A.J * q.c0);
    bool act[KC];
    double bv[KC], dz[KC];
#pragma unroll
    for (int cc = 0; cc < KC; ++cc) {
      const int c = min(q.c0 + cc, q.c1 - 1);
      const int64_t n = n0 + IJ * (c - q.c0);
      act[cc] = A.active[n] != 0;
      bv[cc] = A.b[n];
      dz[cc] = A.dzp[c];
    }
#pragma unroll
    for (int cc = 0; cc < KC; ++cc) {
      const int c = q.c0 + cc;
      if (c >= q.c1) break;
      const int64_t n = n0 + IJ * cc;
      double rv = 0.0;
      if (act[cc]) {
        rv = bv[cc] - bmean;
        if (!from_zero) rv -= apply_row(A, A.x, q.a, q.b, c, n);
        const double rr = fabs(rv) / (dxy * dz[cc]);
        v[0] = (rr > v[0] || rr != rr) ? rr : v[0];
        if (!is_finite(rv)) v[1] = 1.0;
        v[2] += A.r32 ? (double)(float)rv : rv;
      }
      A.r[n] = rv;
      if (A.r32) A.r32[n] = (float)rv;
    }
  }
  block_partials<kTileThreads, 3, 3u>(A.site, v);
}
// cells per thread of k_cg_residual
constexpr int kResK = 4;

__global__ void __launch_bounds__(kFinThreads) k_cg_residual_fin(CgArgs A, uint32_t nb) {
  double out[3];
  finalize_partials<kFinThreads, 3, 3u>(A.site, nb, out);
  if (flat_tid() == 0) {
    Scalars* S = A.S;
    S->rmax = out[0];
    S->rsum = out[2];
    S->nhist = 0;
    S->nonfinite = S->nonfinite || out[1] > 0.0 || !is_finite(out[0]);
    S->done = (out[0] <= A.tol || S->nonfinite) ? 1 : 0;
    S->first = 1;
    S->alpha = 0.0;
    S->beta = 0.0;
    S->rz = 0.0;
    *A.hflag = S->done;
  }
}

// cells per thread of k_cg_spmv and k_cg_update on small grids
constexpr int kColShort = 4;

// The scalars of the new search direction p = (z - m) + beta p_old.
__device__ inline void set_direction(Scalars* S, int slot, double m, double rz, double beta) {
  S->zshift = m;
  S->beta = beta;
  S->rz = rz;
  S->first = 0;
  S->hist_m[slot] = m;
  S->hist_beta[slot] = beta;
  if (!is_finite(rz) || !is_finite(beta)) { S->nonfinite = 1; S->done = 1; }
}

// rz = (r, z), zq = (z, q);  beta = -alpha zq / rz_old: flexible CG, for the
// preconditioners without fused dot products (k_cg_dots2_fin).
// Singular systems: z is shifted by its diagonal-weighted mean m so the
// iterate keeps the pressure of the stiff (high-coefficient) phase near zero;
// (r, z-m) and (z-m, q) follow from the raw sums.
__global__ void __launch_bounds__(256) k_cg_dots(CgArgs A) {
  Scalars* S = A.S;
  if (S->done) return;
  const Col3 q = col_of(A.I, A.J, A.K);
  const bool first = S->first != 0;  // q is not written before the first product
  double v[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  if (q.in) {
    const int64_t IJ = (int64_t)A.I * A.J;
    int64_t n = q.a + (int64_t)A.I * (q.b + (int64_t)A.J * q.c0);
#pragma unroll 4
    for (int c = q.c0; c < q.c1; ++c, n += IJ) {
      if (A.active[n]) {
        const double z = zval(A, n), r = A.r[n], qq = first ? 0.0 : A.q[n];
        v[0] += r * z;
        v[1] += z * qq;
        v[2] += (double)A.dw[n] * z;
        v[3] += r;
        v[4] += qq;
      }
    }
  }
  block_partials<kTileThreads, 5, 0u>(A.site, v);
}

__global__ void __launch_bounds__(kFinThreads) k_cg_dots_fin(CgArgs A, uint32_t nb) {
  Scalars* S = A.S;
  if (S->done) return;
  double t[5];
  finalize_partials<kFinThreads, 5, 0u>(A.site, nb, t);
  if (flat_tid() == 0) {
    const double m = (S->singular && S->dsum > 0.0) ? t[2] / S->dsum : 0.0;
    const double rzm = t[0] - m * t[3], zqm = t[1] - m * t[4];
    set_direction(S, A.slot, m, rzm, S->first ? 0.0 : -S->alpha * zqm / S->rz);
  }
}

// Same as k_cg_dots_fin behind the fused V-cycle: (r,z) and (dw,z) from the
// finest post-smoother's partials, the sum of r from the update.  That V-cycle
// is a fixed symmetric operator up to its own rounding (pre: red, black,
// post: black, red, restriction the transpose of the prolongation), so z is
// orthogonal to the previous residual and beta = rz / rz_old needs no (z,q):
// the leg does not have to read q.  (Iteration counts with and without it
// agree to 2 in 180 on flat grids that need that many, and are equal below
// 100; k_cg_spmv_fin takes what rounding leaves of (z,q) into the step.)
__global__ void __launch_bounds__(kFinThreads) k_cg_dots2_fin(CgArgs A, uint32_t nb) {
  Scalars* S = A.S;
  if (S->done) return;
  double t[2];
  finalize_partials<kFinThreads, 2, 0u>(A.site, nb, t);
  if (flat_tid() == 0) {
    const double m = (S->singular && S->dsum > 0.0) ? t[1] / S->dsum : 0.0;
    const double rzm = t[0] - m * S->rsum;
    set_direction(S, A.slot, m, rzm, S->first ? 0.0 : rzm / S->rz);
  }
}

// The image of the search direction in one pass:
//   q = A (z - m) + beta q_old
// with (p, q) = (z - m, q) and (z - m, q_old) for alpha.  A 1 is the diagonal-only
// term e (the face couplings of a row sum to its diagonal minus e), so the
// stencil is applied to z, which is complete in memory.  Rows of inactive
// cells have no couplings and z = 0: q stays 0 there without a mask.  Each
// thread walks its column keeping z and the z-coupling of planes k-1 / k /
// k+1 in registers.
template <typename Z, int KC>
__global__ void __launch_bounds__(256) k_cg_spmv(CgArgs A, const Z* zv) {
  Scalars* S = A.S;
  if (S->done) return;
  const Col3 q = col_of<KC>(A.I, A.J, A.K);
  double v[2] = {0.0, 0.0};  // (z - m, q), (z - m, q_old)
  if (q.in) {
    const double beta = S->beta, m = S->zshift;
    const int64_t I = A.I, IJ = (int64_t)A.I * A.J;
    const int a = q.a, b = q.b;
    const int64_t dW = a > 0 ? 1 : 0, dE = a < A.I - 1 ? 1 : 0;
    const int64_t dS = b > 0 ? I : 0, dN = b < A.J - 1 ? I : 0;
    int64_t n = a + I * (b + (int64_t)A.J * q.c0);
    double zm = 0.0, czm = 0.0;
    if (q.c0 > 0) {
      zm = (double)zv[n - IJ];
      czm = A.cz[n - IJ];
    }
    double zc = (double)zv[n];
    for (int c = q.c0; c < q.c1; ++c, n += IJ) {
      const double zp = c < A.K - 1 ? (double)zv[n + IJ] : 0.0;
      const double cxm = a > 0 ? A.cx[n - dW] : 0.0;
      const double cym = b > 0 ? A.cy[n - dS] : 0.0;
      const double cx = A.cx[n], cy = A.cy[n], cz = A.cz[n];
      const double zw = (double)zv[n - dW], ze = (double)zv[n + dE];
      const double zs = (double)zv[n - dS], zn = (double)zv[n + dN];
      const double en = A.e ? A.e[n] : 0.0;
      const double qo = beta != 0.0 ? A.q[n] : 0.0;  // not written before the first product
      double d = cxm + cym;
      d = d + czm;
      d = d + cx;
      d = d + cy;
      d = d + cz;
      d = d + en;
      double az = d * zc;
      az -= cxm * zw;
      az -= cym * zs;
      az -= czm * zm;
      az -= cx * ze;
      az -= cy * zn;
      az -= cz * zp;
      const double qv = (az - m * en) + beta * qo;
      A.q[n] = qv;
      v[0] += (zc - m) * qv;
      v[1] += (zc - m) * qo;
      zm = zc;
      zc = zp;
      czm = cz;
    }
  }
  block_partials<kTileThreads, 2, 0u>(A.site, v);
}

__global__ void __launch_bounds__(kFinThreads) k_cg_spmv_fin(CgArgs A, uint32_t nb) {
  Scalars* S = A.S;
  if (S->done) return;
  double t[2];
  finalize_partials<kFinThreads, 2, 0u>(A.site, nb, t);
  if (flat_tid() == 0) {
    const double beta = S->beta;
    // (p, q) of p = (z - m) + beta p_old, also where beta has left p a little
    // short of A-orthogonal to p_old: alpha then still is the exact minimiser
    // along p (pq holds the last step's value, beta is 0 in the first)
    const double pq = t[0] + (beta != 0.0 ? beta * (t[1] + beta * S->pq) : 0.0);
    S->pq = pq;
    S->alpha = S->rz / pq;
    S->hist_alpha[A.slot] = S->alpha;
    S->nhist = A.slot + 1;
    if (!is_finite(S->alpha)) { S->nonfinite = 1; S->done = 1; }
  }
}

// r -= alpha q ; rmax = max |r|/V, and the sum of r as the V-cycle sees it
// (rounded to FP32 with an FP32 one): (r, z - m) is formed as (r, z) - m sum r,
// which is exact in m only with the sum of the very r of (r, z); z may sit on a
// shift m much larger than its variation.
template <int KC>
__global__ void __launch_bounds__(256) k_cg_update(CgArgs A) {
  Scalars* S = A.S;
  if (S->done) return;
  const Col3 q = col_of<KC>(A.I, A.J, A.K);
  const double alpha = S->alpha;
  double v[2] = {0.0, 0.0};  // max |r|/V, sum r
  if (q.in) {
    const int64_t IJ = (int64_t)A.I * A.J;
    const double dxy = A.dxp[q.a] * A.dyp[q.b];
    int64_t n = q.a + (int64_t)A.I * (q.b + (int64_t)A.J * q.c0);
#pragma unroll 4
    for (int c = q.c0; c < q.c1; ++c, n += IJ) {
      const double rv = A.r[n] - alpha * A.q[n];
      A.r[n] = rv;
      if (A.r32) A.r32[n] = (float)rv;
      const double rr = fabs(rv) / (dxy * A.dzp[c]);
      v[0] = (rr > v[0] || rr != rr) ? rr : v[0];  // a NaN sticks
      v[1] += A.r32 ? (double)(float)rv : rv;
    }
  }
  block_partials<kTileThreads, 2, 1u>(A.site, v);
}

// x from the kept z of the steps since the last such pass, one step after the
// other as a CG that carries p and x would form them:
//   p = (z_j - m_j) + beta_j p,   x += alpha_j p
// on active cells (0 elsewhere), from x = 0 when `assign`.  Fused
// multiply-adds in a fixed order, so x is the same to the last bit whatever
// number of z one pass covers: it does not depend on the memory there was for
// them.  m is taken off each z before the sum: in a two-phase system the stiff
// phase's z sits close to m, and its differences matter.  With `keep_p` (a
// full history in the middle of a solve) p is kept for the next pass.
// z, x and the mask are read and x is written once: 15 steps of an FP32
// V-cycle at 256^3 move 69 B a cell here, where carrying x and p through the
// iterations moved 32 B a cell in each of them.
template <typename Z>
struct ZHist {
  const Z* z[kZRing];
};
constexpr int kFlushCells = 4;  // cells per thread
template <typename Z>
__global__ void __launch_bounds__(256) k_cg_xflush(CgArgs A, ZHist<Z> H, int64_t N, int assign,
                                                   int keep_p) {
  const Scalars* S = A.S;
  const int nh = S->nhist;
  const int64_t n0 = (int64_t)blockIdx.x * (256 * kFlushCells) + threadIdx.x;
  double x[kFlushCells], p[kFlushCells];
  bool act[kFlushCells];
  // beta of a solve's first step is 0, and p is not written before
  const bool old = nh > 0 && S->hist_beta[0] != 0.0;
#pragma unroll
  for (int u = 0; u < kFlushCells; ++u) {
    const int64_t n = min(n0 + 256 * u, N - 1);
    act[u] = A.active[n] != 0;
    x[u] = assign ? 0.0 : A.x[n];
    p[u] = old ? A.p[n] : 0.0;
  }
#pragma unroll 4
  for (int j = 0; j < nh; ++j) {
    const double alpha = S->hist_alpha[j], beta = S->hist_beta[j], m = S->hist_m[j];
    const Z* z = H.z[j];
#pragma unroll
    for (int u = 0; u < kFlushCells; ++u) {
      p[u] = fma(beta, p[u], (double)z[min(n0 + 256 * u, N - 1)] - m);
      x[u] = fma(alpha, p[u], x[u]);
    }
  }
#pragma unroll
  for (int u = 0; u < kFlushCells; ++u) {
    const int64_t n = n0 + 256 * u;
    if (n >= N) break;
    A.x[n] = act[u] ? x[u] : 0.0;
    if (keep_p && nh > 0) A.p[n] = act[u] ? p[u] : 0.0;
  }
}
__global__ void k_cg_hist_reset(Scalars* S) { S->nhist = 0; }

__global__ void __launch_bounds__(kFinThreads) k_cg_update_fin(CgArgs A, uint32_t nb) {
  Scalars* S = A.S;
  if (S->done) return;
  double t[2];
  finalize_partials<kFinThreads, 2, 1u>(A.site, nb, t);
  if (flat_tid() == 0) {
    S->rmax = t[0];
    S->rsum = t[1];
    S->iter += 1;
    if (!is_finite(t[0])) S->nonfinite = 1;
    S->done = (t[0] <= A.tol || S->nonfinite) ? 1 : 0;
    *A.hflag = S->done;
  }
}

template <typename T>
LevelView<T> view_of(const Level<T>& L, const uint8_t* act = nullptr) {
  return LevelView<T>{L.nx, L.ny, L.nz, L.cx, L.cy, L.cz, L.e, L.x, L.b, act};
}

template <typename T>
double level_bytes(const Level<T>& L, double per_cell_words) {
  return (double)L.n * sizeof(T) * per_cell_words;
}

template <typename T>
void launch_gs(sp_ctx* c, const Level<T>& L, int color, int zero_init, bool fine) {
  const int nxh = (L.nx + 1) / 2;
  dim3 blk(64, 4, 1), grd = flat_grid(nxh, L.ny, L.nz);
  int slot;
  // algorithmic words per cell: b for one colour, the three face arrays,
  // x read (all) and written (one colour); a zero-init sweep writes all of x
  const double words = (zero_init ? 0.5 + 3.0 + 1.0 : 1.0 + 0.5 + 3.0 + 0.5) + (L.e ? 1.0 : 0.0);
  timer_begin(c, fine ? (zero_init ? "mg_gs0_fine" : "mg_gs_fine") : "mg_gs_coarse",
              level_bytes(L, words), &slot);
  if (fine)
    hipLaunchKernelGGL((k_gs<T, true>), grd, blk, 0, c->stream, view_of(L), color, zero_init,
                       (T)(fine ? c->prm.mg_omega : c->prm.mg_omega_coarse),
                       (const Scalars*)c->S);
  else
    hipLaunchKernelGGL((k_gs<T, false>), grd, blk, 0, c->stream, view_of(L), color, zero_init,
                       (T)(fine ? c->prm.mg_omega : c->prm.mg_omega_coarse),
                       (const Scalars*)c->S);
  timer_end(c, slot);
}

// m steps of the Chebyshev smoother on level L, from zero (pre) or from L.x
// (post); the result ends in L.x (L.xs is the other iterate buffer).
template <typename T>
void launch_cheb(sp_ctx* c, const Level<T>& L, int m, bool from_zero, bool fine) {
  constexpr double lmax = 2.0, lmin = lmax / 8.0;
  const double theta = 0.5 * (lmax + lmin), delta = 0.5 * (lmax - lmin), sigma = theta / delta;
  dim3 blk(64, 4, 1), grd = flat_grid(L.nx, L.ny, L.nz);
  const LevelView<T> V = view_of(L);
  // the last step writes L.x; a step never writes the buffer it reads
  T* buf[2] = {L.x, L.xs};
  int w = from_zero ? (m - 1) % 2 : 1;  // buffer of the first step's output
  const T* in = from_zero ? nullptr : L.x;
  double rho = 1.0 / sigma;
  int slot;
  for (int s = 0; s < m; ++s) {
    double c1 = 0.0, c2 = 1.0 / theta;
    if (s > 0) {
      const double rn = 1.0 / (2.0 * sigma - rho);
      c1 = rn * rho;
      c2 = 2.0 * rn / delta;
      rho = rn;
    }
    // words per cell: b and the three face arrays read, x in read (not on a
    // step from zero), d read after the first step, e read where present;
    // x out and d written
    const double words = 6.0 + (in ? 1.0 : 0.0) + (s > 0 ? 1.0 : 0.0) + (L.e ? 1.0 : 0.0);
    timer_begin(c, fine ? "mg_cheb_fine" : "mg_cheb_coarse", level_bytes(L, words), &slot);
    if (fine)
      hipLaunchKernelGGL((k_cheb<T, true>), grd, blk, 0, c->stream, V, in, buf[w], L.cd, (T)c1,
                         (T)c2, s == 0 ? 1 : 0, (const Scalars*)c->S);
    else
      hipLaunchKernelGGL((k_cheb<T, false>), grd, blk, 0, c->stream, V, in, buf[w], L.cd, (T)c1,
                         (T)c2, s == 0 ? 1 : 0, (const Scalars*)c->S);
    timer_end(c, slot);
    in = buf[w];
    w ^= 1;
  }
  if (in != L.x)  // post with an odd m: the result is in L.xs
    hipMemcpyAsync(L.x, in, sizeof(T) * (size_t)L.n, hipMemcpyDeviceToDevice, c->stream);
}

// Launch of a level's legs with tiles of Sh, per_cu workgroups on a CU at once.
template <typename Sh, typename T>
LegGrid leg_of(const sp_ctx* c, const Level<T>& L, int per_cu) {
  return leg_grid(L.nx, L.ny, L.nz, Sh::TX, Sh::TY, Sh::H,
                  (int64_t)std::max(1, c->num_cu) * per_cu);
}

// Small tiles for the levels below the finest of at most 32 x 32 columns:
// these have two 32 x 16 tiles, whose 10-step marches (2 planes + the 8-plane
// pipeline) run on 32 CUs.  Small tiles put a workgroup on every CU (32^3:
// 10.5 -> 7.8 us per leg); at 64 x 64 they measured slower than the large ones
// (13.0 against 11.7 us).
template <typename T>
bool small_legs(const Level<T>& L, bool fine) {
  return !fine && (int64_t)L.nx * L.ny <= 32 * 32;
}

// FP32: four cells per thread or one (four_cell_leg); one with a diagonal-only
// term.
template <int NU>
void plan_legs(const sp_ctx* c, Level<float>& L, bool fine) {
  using Four = FusedTile<float, false>;
  static_assert(Four::Q == 2 && 4 * Four::EP == kQEX && Four::EY == kQEY && Four::kPerCu == 1,
                "four_cell_leg weighs these tiles");
  L.four = !small_legs(L, fine) && !L.e &&
           four_cell_leg(L.nx, L.ny, L.nz, NU, std::max(1, c->num_cu));
  if (small_legs(L, fine)) L.leg = leg_of<CellShape<NU, kFEXs, kFEYs>>(c, L, 4);
  else if (L.four) L.leg = leg_of<FusedShape<NU, Four::Q, Four::EP, Four::EY>>(c, L, 1);
  else L.leg = leg_of<CellShape<NU, kFEX, kFEY>>(c, L, 1);
}
template <int NU, bool SMALL>
void plan_legs64(const sp_ctx* c, Level<double>& L) {
  using Tile = FusedTile<double, SMALL>;
  L.leg = leg_of<FusedShape<NU, Tile::Q, Tile::EP, Tile::EY>>(c, L, Tile::kPerCu);
}
template <int NU>
void plan_legs(const sp_ctx* c, Level<double>& L, bool) {
  if ((int64_t)L.nx * L.ny <= kSmallColumns) plan_legs64<NU, true>(c, L);
  else plan_legs64<NU, false>(c, L);
}

// One smoother leg.  KERNEL(MODE, FINE): the kernel of a form.
#define SP_LEG(KERNEL)                                                                         \
  do {                                                                                         \
    if (mode == 0) hipLaunchKernelGGL((KERNEL(0, false)), grd, blk, 0, c->stream, A, S);       \
    else if (fine) hipLaunchKernelGGL((KERNEL(1, true)), grd, blk, 0, c->stream, A, S);        \
    else hipLaunchKernelGGL((KERNEL(1, false)), grd, blk, 0, c->stream, A, S);                 \
  } while (0)

template <typename T, int NU, bool HAS_E, bool SMALL>
void launch_march(sp_ctx* c, const Level<T>& L, FusedArgs<T>& A, bool fine, int mode) {
  using Tile = FusedTile<T, SMALL>;
  constexpr int Q = Tile::Q, EP = Tile::EP, EY = Tile::EY;
  const dim3 grd(L.leg.gx, L.leg.gy, L.leg.gz), blk(EP * EY, 1, 1);
  const Scalars* S = c->S;
#define SP_K(MODE, FINE) k_smooth_fused<T, NU, Q, MODE, FINE, HAS_E, EP, EY>
  SP_LEG(SP_K);
#undef SP_K
}

template <int NU, bool HAS_E, int EX, int EY>
void launch_cell(sp_ctx* c, const Level<float>& L, FusedArgs<float>& A, bool fine, int mode) {
  const dim3 grd(L.leg.gx, L.leg.gy, L.leg.gz), blk(EX, EY, 1);
  const Scalars* S = c->S;
#define SP_K(MODE, FINE) k_smooth_cell<NU, MODE, FINE, HAS_E, EX, EY>
  SP_LEG(SP_K);
#undef SP_K
}
#undef SP_LEG

template <int NU>
void launch_leg(sp_ctx* c, const Level<float>& L, FusedArgs<float>& A, bool fine, int mode) {
  if (small_legs(L, fine)) {
    if (A.e) launch_cell<NU, true, kFEXs, kFEYs>(c, L, A, fine, mode);
    else launch_cell<NU, false, kFEXs, kFEYs>(c, L, A, fine, mode);
  } else if (L.four) {
    launch_march<float, NU, false, false>(c, L, A, fine, mode);
  } else {
    if (A.e) launch_cell<NU, true, kFEX, kFEY>(c, L, A, fine, mode);
    else launch_cell<NU, false, kFEX, kFEY>(c, L, A, fine, mode);
  }
}
template <int NU>
void launch_leg(sp_ctx* c, const Level<double>& L, FusedArgs<double>& A, bool fine, int mode) {
  if ((int64_t)L.nx * L.ny <= kSmallColumns) {
    if (A.e) launch_march<double, NU, true, true>(c, L, A, fine, mode);
    else launch_march<double, NU, false, true>(c, L, A, fine, mode);
  } else {
    if (A.e) launch_march<double, NU, true, false>(c, L, A, fine, mode);
    else launch_march<double, NU, false, false>(c, L, A, fine, mode);
  }
}

template <typename T, int NU>
void launch_fused(sp_ctx* c, Level<T>* lv, int l, int mode) {
  const Level<T>& L = lv[l];
  const Level<T>& C = lv[l + 1];
  FusedArgs<T> A{};
  A.nx = L.nx; A.ny = L.ny; A.nz = L.nz;
  A.cx = L.cx; A.cy = L.cy; A.cz = L.cz; A.e = L.e;
  A.b = L.b;
  A.cnx = C.nx; A.cny = C.ny;
  A.kchunk = L.leg.kchunk;
  A.omega = (T)(l == 0 ? c->prm.mg_omega : c->prm.mg_omega_coarse);
  if (mode == 0) { A.xout = L.xs; A.bc = C.b; }
  else { A.xin = L.xs; A.xc = C.x; A.xout = L.x; }
  if (mode == 1 && l == 0 && c->fuse_dots) {
    A.dots = 1;
    A.dsite = red_site(c, kSiteDots);
    c->dots_nb = (uint32_t)L.leg.gx * L.leg.gy * L.leg.gz;
  }
  const bool fine = l == 0;
  int slot;
  // algorithmic words per cell: pre b + 3 faces -> x (+ coarse b);
  // post x_pre + 3 faces + b -> x (+ coarse x)
  const double words = mode == 0 ? 5.0 + 0.125 : 6.0 + 0.125;
  timer_begin(c, fine ? (mode == 0 ? "mg_pre_fine" : "mg_post_fine")
                      : (mode == 0 ? "mg_pre_coarse" : "mg_post_coarse"),
              level_bytes(L, words + (L.e ? 1.0 : 0.0)), &slot);
  launch_leg<NU>(c, L, A, fine, mode);
  timer_end(c, slot);
}

// The V-cycle uses the temporally blocked smoother legs
bool fused_vcycle(const sp_ctx* c) {
  const int pre = std::max(1, c->prm.mg_pre), post = c->prm.mg_post;
  return pre == post && (pre == 1 || pre == 2) &&
         !(c->prm.flags & (SP_FLAG_UNFUSED_SMOOTHER | SP_FLAG_CHEBYSHEV));
}

template <typename T>
void vcycle(sp_ctx* c, Level<T>* lv) {
  const int L = c->levels, Lt = c->tail_level;
  // levels with a pre-smoothing leg and a restriction: those above the tail,
  // or every level but the coarsest when no level fits the tail
  const int Lp = Lt < L ? Lt : L - 1;
  const int pre = std::max(1, c->prm.mg_pre), post = c->prm.mg_post;
  const bool fused = fused_vcycle(c);
  const bool cheb = (c->prm.flags & SP_FLAG_CHEBYSHEV) != 0;
  dim3 blk(64, 4, 1);
  int slot;
  for (int l = 0; l < Lp; ++l) {
    const bool fine = l == 0;
    if (fused) {
      if (pre == 2) launch_fused<T, 2>(c, lv, l, 0);
      else launch_fused<T, 1>(c, lv, l, 0);
      continue;
    }
    if (cheb) {
      launch_cheb(c, lv[l], pre, true, fine);
    } else {
      launch_gs(c, lv[l], 0, 1, fine);
      launch_gs(c, lv[l], 1, 0, fine);
      for (int s = 1; s < pre; ++s) { launch_gs(c, lv[l], 0, 0, fine); launch_gs(c, lv[l], 1, 0, fine); }
    }
    dim3 grd = flat_grid(lv[l + 1].nx, lv[l + 1].ny, lv[l + 1].nz);
    timer_begin(c, fine ? "mg_restrict_fine" : "mg_restrict_coarse",
                level_bytes(lv[l], 5.0 + (lv[l].e ? 1.0 : 0.0)) + level_bytes(lv[l + 1], 1.0), &slot);
    if (fine)
      hipLaunchKernelGGL((k_resid_restrict<T, true>), grd, blk, 0, c->stream, view_of(lv[l]),
                         view_of(lv[l + 1]), (const Scalars*)c->S);
    else
      hipLaunchKernelGGL((k_resid_restrict<T, false>), grd, blk, 0, c->stream, view_of(lv[l]),
                         view_of(lv[l + 1]), (const Scalars*)c->S);
    timer_end(c, slot);
  }
  if (Lt >= L) {
    // the coarsest level does not fit the tail's LDS: the tail's coarsest
    // sweeps (red-black pairs from x = 0, then as many black-red pairs)
    // with the global-memory kernels
    const int Lc = L - 1;
    const bool fine = Lc == 0;
    const int cs = std::max(1, c->prm.mg_coarse_sweeps);
    launch_gs(c, lv[Lc], 0, 1, fine);
    launch_gs(c, lv[Lc], 1, 0, fine);
    for (int s = 1; s < cs; ++s) { launch_gs(c, lv[Lc], 0, 0, fine); launch_gs(c, lv[Lc], 1, 0, fine); }
    for (int s = 0; s < cs; ++s) { launch_gs(c, lv[Lc], 1, 0, fine); launch_gs(c, lv[Lc], 0, 0, fine); }
  } else {
    TailArgs<T> A{};
    A.n = L - Lt;
    A.pre = pre;
    A.post = post;
    A.coarse_sweeps = std::max(1, c->prm.mg_coarse_sweeps);
    A.singular = c->S_host->singular;
    A.b = lv[Lt].b;
    A.x = lv[Lt].x;
    int off = 0, thread = 0;
    for (int q = 0; q < A.n; ++q) {
      const Level<T>& G = lv[Lt + q];
      A.omega[q] = (T)(Lt + q == 0 ? c->prm.mg_omega : c->prm.mg_omega_coarse);
      A.nx[q] = G.nx; A.ny[q] = G.ny; A.nz[q] = G.nz;
      A.cx[q] = G.cx; A.cy[q] = G.cy; A.cz[q] = G.cz; A.e[q] = G.e;
      A.xo[q] = off;
      off += (G.nx + 2) * (G.ny + 2) * (G.nz + 2);
      A.first[q] = thread;
      if (q > 0) thread += tail_threads(G.nx, G.ny, G.nz);
    }
    for (int q = 0; q < A.n; ++q) {
      A.ro[q] = off;
      off += (int)lv[Lt + q].n;
    }
    timer_begin(c, "mg_tail", 0, &slot);
    auto launch = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(1), dim3(kTailThreads), 0, c->stream, A, (const Scalars*)c->S);
    };
    bool wide = false;
    if constexpr (sizeof(T) == 4) {
      wide = tail_pairs(lv[Lt]) > 2 * kTailThreads;
      if (wide) lv[Lt].e ? launch(k_tail<T, true, 4>) : launch(k_tail<T, false, 4>);
    }
    if (!wide) lv[Lt].e ? launch(k_tail<T, true, 2>) : launch(k_tail<T, false, 2>);
    timer_end(c, slot);
  }
  for (int l = Lp - 1; l >= 0; --l) {
    const bool fine = l == 0;
    if (fused) {
      if (pre == 2) launch_fused<T, 2>(c, lv, l, 1);
      else launch_fused<T, 1>(c, lv, l, 1);
      continue;
    }
    dim3 grd = flat_grid(lv[l].nx, lv[l].ny, lv[l].nz);
    const uint8_t* act = fine ? c->active : nullptr;
    timer_begin(c, fine ? "mg_prolong_fine" : "mg_prolong_coarse",
                fine ? level_bytes(lv[l], 2.0) + (double)lv[l].n + level_bytes(lv[l + 1], 1.0)
                     : level_bytes(lv[l], 5.0 + (lv[l].e ? 1.0 : 0.0)) + level_bytes(lv[l + 1], 1.0),
                &slot);
    if (fine)
      hipLaunchKernelGGL((k_prolong<T, true>), grd, blk, 0, c->stream, view_of(lv[l], act),
                         view_of(lv[l + 1]), (const Scalars*)c->S);
    else
      hipLaunchKernelGGL((k_prolong<T, false>), grd, blk, 0, c->stream, view_of(lv[l], act),
                         view_of(lv[l + 1]), (const Scalars*)c->S);
    timer_end(c, slot);
    if (cheb) {
      if (post > 0) launch_cheb(c, lv[l], post, false, fine);
    } else {
      for (int s = 0; s < post; ++s) { launch_gs(c, lv[l], 1, 0, fine); launch_gs(c, lv[l], 0, 0, fine); }
    }
  }
}

template <typename T>
sp_status setup_levels(sp_ctx* c, Level<T>* lv) {
  const int L = c->levels;
  dim3 blk(64, 4, 1);
  for (int l = 0; l < L; ++l) lv[l].e = c->has_e ? lv[l].e_store : nullptr;
  for (int l = 1; l < L; ++l) {
    Level<T>& C = lv[l];
    hipLaunchKernelGGL(k_coarsen<T>, flat_grid(C.nx, C.ny, C.nz), blk, 0, c->stream,
                       view_of(lv[l - 1]), view_of(C), C.cx, C.cy, C.cz, C.e,
                       (T)c->prm.mg_coarse_scale);
  }
  if (fused_vcycle(c)) {
    for (int l = 0; l < L; ++l) {
      if (c->prm.mg_pre == 2) plan_legs<2>(c, lv[l], l == 0);
      else plan_legs<1>(c, lv[l], l == 0);
    }
  }
  return SP_OK;
}

}  // namespace

// The first level of the tail kernel (c->tail_level): the levels from it on
// fit its threads (two pairs each on the first level, one on the others; four
// on a coarsest level alone in FP32) and LDS.  c->levels when not even the
// coarsest level does (a hierarchy cut short by mg_levels, or a large grid
// that cannot coarsen): the V-cycle then smooths the coarsest level in global
// memory.
template <typename T>
static int first_tail_level(const Level<T>* lv, int levels) {
  int best = levels;
  for (int l = levels - 1; l >= 0 && levels - l <= kTailLevels; --l) {
    int64_t lds = 0, threads = 0;
    for (int q = l; q < levels; ++q) {
      lds += (int64_t)sizeof(T) *
             ((int64_t)(lv[q].nx + 2) * (lv[q].ny + 2) * (lv[q].nz + 2) + lv[q].n);
      if (q > l && lv[q].n <= 4 * kTailThreads) threads += tail_threads(lv[q].nx, lv[q].ny, lv[q].nz);
    }
    const int big = sizeof(T) == 4 && l == levels - 1 ? 4 : 2;
    if (tail_pairs(lv[l]) > big * kTailThreads || threads > kTailThreads || lds > kTailLdsBytes)
      break;
    best = l;
  }
  return best;
}

void mg_tail_level(sp_ctx* c, bool fp32) {
  c->tail_level = fp32 ? first_tail_level(c->lf, c->levels) : first_tail_level(c->ld, c->levels);
}

sp_status mg_setup(sp_ctx* c) {
  if (c->prm.precond != SP_PRECOND_MG) return SP_OK;
  if (c->prm.precision == SP_PREC_MIXED) return setup_levels<float>(c, c->lf);
  return setup_levels<double>(c, c->ld);
}

// Solve A x = rhs - mean (singular) with the preconditioned
// CG until max |r_i| / V_i <= tol.  The operator arrays and c->S
// (bmean, singular) come from the assembly.  Writes x into c->x.
//   check_true: after convergence of the recursive residual, form the true
//               residual and restart from it (at most 3 times) if it is
//               above tol.  The forward projection instead measures the
//               divergence of the corrected field, which is the same
//               quantity, and resumes when needed.
//   resume:     continue from the current x (true residual, iteration count
//               kept) instead of starting from x = 0.
sp_status solve(sp_ctx* c, const double* rhs, double tol, sp_stats* st, bool check_true,
                bool resume) {
  const Dims& D = c->dm;
  const bool mixed = c->prm.precision == SP_PREC_MIXED;
  const bool mg = c->prm.precond == SP_PRECOND_MG;
  const dim3 blk(64, 4, 1);
  if (flat_blocks(D.I, D.J, D.K) > c->red_max_blocks)
    return fail(c, SP_ERR_INVALID_ARG, "grid too large for the reduction buffers");
  CgArgs A{};
  A.I = D.I; A.J = D.J; A.K = D.K;
  A.cx = c->cx; A.cy = c->cy; A.cz = c->cz; A.e = c->has_e ? c->ee : nullptr;
  A.active = c->active;
  A.dw = c->dw;
  A.dxp = c->dxp; A.dyp = c->dyp; A.dzp = c->dzp;
  A.b = rhs;
  A.x = c->x; A.r = c->r; A.q = c->q; A.p = c->p0;
  A.S = c->S;
  A.hflag = c->hflags_dev;
  A.tol = tol;
  if (mixed && mg) {
    A.r32 = c->r32;
  }
  int slot;
  const double NB = (double)D.N;
  const double eb = c->has_e ? 8.0 : 0.0;
  const double zb = (mixed && mg) ? 4.0 : 8.0;

  const uint32_t ncol = col_blocks(D.I, D.J, D.K);
  const dim3 cgrd = col_grid(D.I, D.J, D.K);
  // Cells per thread of k_cg_spmv and k_cg_update: kColK where that puts four
  // workgroups on every CU, kColShort below, where the 16 planes one after the
  // other are the time (event times of both kernels: 32^3 13.6 and 9.5 -> 7.6
  // and 6.9 us, 64^3 17.9 and 12.0 -> 8.7 and 7.5, 97 x 130 x 75 19.5 and 14.3
  // -> 13.2 and 10.7, 128^3 21.3 and 16.2 -> 19.7 and 14.4; at 160^3, beyond
  // the limit, 40.4 and 21.7 against 39.4 and 22.8 with four times the partial
  // sums).
  const bool shortcol = ncol < 4u * (uint32_t)std::max(1, c->num_cu);
  const uint32_t nshort = col_blocks_k<kColShort>(D.I, D.J, D.K);
  const dim3 sgrd = shortcol ? col_grid_k<kColShort>(D.I, D.J, D.K) : cgrd;
  const uint32_t nsp = shortcol ? nshort : ncol;
  auto launch_col = [&](auto kern, int site, const char* name, double bytes) {
    A.site = red_site(c, site);
    timer_begin(c, name, bytes, &slot);
    hipLaunchKernelGGL(kern, cgrd, blk, 0, c->stream, A);
    timer_end(c, slot);
  };
  auto finalize = [&](auto kern, int site, uint32_t nb) {
    A.site = red_site(c, site);
    timer_begin(c, "cg_finalize", 0, &slot);
    hipLaunchKernelGGL(kern, dim3(1), dim3(kFinThreads), 0, c->stream, A, nb);
    timer_end(c, slot);
  };
  // the ring stays this context's until the solve is over
  std::lock_guard<std::mutex> ring(c->zmutex);
  auto enqueue_residual = [&](int from_zero) {
    A.site = red_site(c, kSiteResidual);
    timer_begin(c, "cg_residual", NB * ((from_zero ? 8 + 1 : 8 * 5 + eb + 1) + 8 + (A.r32 ? 4 : 0)),
                &slot);
    hipLaunchKernelGGL(k_cg_residual<kResK>, col_grid_k<kResK>(D.I, D.J, D.K), blk, 0, c->stream,
                       A, from_zero);
    timer_end(c, slot);
    finalize(k_cg_residual_fin, kSiteResidual, col_blocks_k<kResK>(D.I, D.J, D.K));
  };
  // z of this step goes into its buffer of the ring
  auto precondition = [&]() {
    if (mixed && mg) {
      c->lf[0].x = static_cast<float*>(c->zring[A.slot]);
      A.z32 = c->lf[0].x;
    } else {
      A.z64 = static_cast<double*>(c->zring[A.slot]);
      if (mg) c->ld[0].x = A.z64;
    }
    if (mg) {
      if (mixed) vcycle<float>(c, c->lf);
      else vcycle<double>(c, c->ld);
    } else {
      launch_col(k_cg_jacobi, kSiteDots, "cg_jacobi", NB * (8 * 4 + eb + 1 + 8));
    }
  };

  hipError_t e;
  volatile int32_t* hflag = c->hflags;
  // the finest post-smoother forms the CG dot products when the V-cycle has
  // a fused leg on the finest level (a level above the tail, or above the
  // coarsest when no level fits the tail)
  const int legs = c->tail_level < c->levels ? c->tail_level : c->levels - 1;
  c->fuse_dots = mg && fused_vcycle(c) && legs > 0;
  c->dots_nb = 0;
  hipEvent_t evs[2];
  hipEventCreateWithFlags(&evs[0], hipEventDisableTiming);
  hipEventCreateWithFlags(&evs[1], hipEventDisableTiming);
  int it = 0;
  if (resume) {
    it = c->S_host->iter;
    hipError_t e0 = hipMemsetAsync(&c->S->done, 0, sizeof(int32_t), c->stream);
    if (e0 != hipSuccess) return hip_check(c, e0, "hipMemsetAsync");
    enqueue_residual(0);
  } else {
    enqueue_residual(1);
  }
  // x from the kept z (k_cg_xflush); `keep_p`: the solve goes on
  bool assign = !resume, carried = false;  // carried: p holds the last pass's direction
  auto form_x = [&](bool keep_p) {
    const dim3 grd((unsigned)((D.N + 256 * kFlushCells - 1) / (256 * kFlushCells)));
    // a full history's z, or what the device then says the last pass read
    timer_begin(c, "cg_xflush", NB * ((keep_p ? zb * c->zdepth + 8 : 0) + 1 + (assign ? 8 : 16) +
                                      (carried ? 8 : 0)), &slot);
    if (mixed && mg) {
      ZHist<float> H{};
      for (int j = 0; j < c->zdepth; ++j) H.z[j] = static_cast<const float*>(c->zring[j]);
      hipLaunchKernelGGL(k_cg_xflush<float>, grd, dim3(256), 0, c->stream, A, H, D.N,
                         assign ? 1 : 0, keep_p ? 1 : 0);
    } else {
      ZHist<double> H{};
      for (int j = 0; j < c->zdepth; ++j) H.z[j] = static_cast<const double*>(c->zring[j]);
      hipLaunchKernelGGL(k_cg_xflush<double>, grd, dim3(256), 0, c->stream, A, H, D.N,
                         assign ? 1 : 0, keep_p ? 1 : 0);
    }
    timer_end(c, slot);
    if (keep_p) hipLaunchKernelGGL(k_cg_hist_reset, dim3(1), dim3(1), 0, c->stream, c->S);
    assign = false;
    carried = keep_p;
  };
  int restarts = 0;
  const int max_iter = std::max(1, c->prm.max_iter);
  bool finished = false;
  while (!finished) {
    // one iteration in flight: enqueue iteration `it`, then wait for the
    // flag written at the end of iteration `it - 1`
    bool prev_pending = false;
    int cur = 0;
    A.slot = 0;
    while (it < max_iter) {
      if (A.slot == c->zdepth) {  // the ring is full and the solve goes on
        form_x(true);
        A.slot = 0;
      }
      precondition();
      if (c->fuse_dots) {
        finalize(k_cg_dots2_fin, kSiteDots, c->dots_nb);
      } else {
        launch_col(k_cg_dots, kSiteDots, "cg_dots", NB * (8 + zb + 8 + 4 + 1));
        finalize(k_cg_dots_fin, kSiteDots, ncol);
      }
      // z (stencil), q, three couplings, e -> q
      {
        A.site = red_site(c, kSiteSpmv);
        timer_begin(c, "cg_spmv", NB * (zb + 8 + 24 + eb + 8), &slot);
        const float* zf = A.z32;
        const double* zd = A.z64;
        if (zf && shortcol)
          hipLaunchKernelGGL((k_cg_spmv<float, kColShort>), sgrd, blk, 0, c->stream, A, zf);
        else if (zf)
          hipLaunchKernelGGL((k_cg_spmv<float, kColK>), sgrd, blk, 0, c->stream, A, zf);
        else if (shortcol)
          hipLaunchKernelGGL((k_cg_spmv<double, kColShort>), sgrd, blk, 0, c->stream, A, zd);
        else
          hipLaunchKernelGGL((k_cg_spmv<double, kColK>), sgrd, blk, 0, c->stream, A, zd);
        timer_end(c, slot);
      }
      finalize(k_cg_spmv_fin, kSiteSpmv, nsp);
      A.site = red_site(c, kSiteUpdate);
      timer_begin(c, "cg_update", NB * (8 * 2 + 8 + (A.r32 ? 4 : 0)), &slot);
      if (shortcol)
        hipLaunchKernelGGL(k_cg_update<kColShort>, sgrd, blk, 0, c->stream, A);
      else
        hipLaunchKernelGGL(k_cg_update<kColK>, sgrd, blk, 0, c->stream, A);
      timer_end(c, slot);
      finalize(k_cg_update_fin, kSiteUpdate, nsp);
      hipEventRecord(evs[cur], c->stream);
      ++it;
      ++A.slot;
      if (prev_pending) {
        e = hipEventSynchronize(evs[cur ^ 1]);
        if (e != hipSuccess) { hipEventDestroy(evs[0]); hipEventDestroy(evs[1]); return hip_check(c, e, "solve"); }
        if (*hflag) break;
      }
      prev_pending = true;
      cur ^= 1;
    }
    form_x(false);
    e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) { hipEventDestroy(evs[0]); hipEventDestroy(evs[1]); return hip_check(c, e, "solve"); }
    e = hipMemcpy(c->S_host, c->S, sizeof(Scalars), hipMemcpyDeviceToHost);
    if (e != hipSuccess) { hipEventDestroy(evs[0]); hipEventDestroy(evs[1]); return hip_check(c, e, "solve"); }
    timer_bytes(c, "cg_xflush", NB * zb * c->S_host->nhist);
    const int iters = c->S_host->iter;
    if (c->S_host->nonfinite || !check_true) break;
    // true residual of the final iterate
    hipMemsetAsync(&c->S->done, 0, sizeof(int32_t), c->stream);
    enqueue_residual(0);
    e = hipStreamSynchronize(c->stream);
    if (e == hipSuccess) e = hipMemcpy(c->S_host, c->S, sizeof(Scalars), hipMemcpyDeviceToHost);
    if (e != hipSuccess) { hipEventDestroy(evs[0]); hipEventDestroy(evs[1]); return hip_check(c, e, "solve"); }
    if (c->S_host->done || iters >= max_iter || restarts >= 3) {
      finished = true;
    } else {
      ++restarts;  // recursive residual drifted: restart from the true residual
      it = iters;
    }
  }
  hipEventDestroy(evs[0]);
  hipEventDestroy(evs[1]);
  if (st) {
    st->iterations = c->S_host->iter;
    st->converged = c->S_host->done && !c->S_host->nonfinite;
    st->residual_div = c->S_host->rmax;
    st->levels = mg ? c->levels : 1;
  }
  if (c->S_host->nonfinite) return fail(c, SP_ERR_NONFINITE, "non-finite value in the solve");
  return SP_OK;
}

// Iterative refinement of a non-singular system's pressure, kept as
// x + xd: the residual of x + xd in difference form, then, when it is above
// tol, a solve of A e = residual from e = 0 and xd += e.  The corrected
// velocity takes the differences of x and of xd separately, so it is not
// limited by the rounding of a pressure level that a Dirichlet face fixes.
// *rmax: max |residual|/V before the solve; *iters: its CG iterations.
sp_status refine(sp_ctx* c, double tol, double* rmax, int* iters) {
  const Dims& D = c->dm;
  CgArgs A{};
  A.I = D.I; A.J = D.J; A.K = D.K;
  A.cx = c->cx; A.cy = c->cy; A.cz = c->cz; A.e = c->has_e ? c->ee : nullptr;
  A.active = c->active;
  A.dxp = c->dxp; A.dyp = c->dyp; A.dzp = c->dzp;
  A.b = c->b;
  A.x = c->x;
  A.S = c->S;
  const dim3 blk(64, 4, 1);
  const dim3 cgrd = col_grid(D.I, D.J, D.K);
  const uint32_t ncol = col_blocks(D.I, D.J, D.K);
  hipError_t e;
  if (!c->xd_active) {
    e = hipMemsetAsync(c->xd, 0, sizeof(double) * D.N, c->stream);
    if (e != hipSuccess) return hip_check(c, e, "hipMemsetAsync(xd)");
    c->xd_active = true;
  }
  int slot;
  A.site = red_site(c, kSiteResidual);
  const double eb = c->has_e ? 8.0 : 0.0;
  timer_begin(c, "refine_residual", (double)D.N * (8 * 4 + 24 + eb + 1 + 8), &slot);
  hipLaunchKernelGGL(k_refine_residual, cgrd, blk, 0, c->stream, A, (const double*)c->xd, c->p1);
  hipLaunchKernelGGL(k_refine_residual_fin, dim3(1), dim3(kFinThreads), 0, c->stream, A, ncol);
  timer_end(c, slot);
  e = hipMemcpyAsync(c->S_host, c->S, sizeof(Scalars), hipMemcpyDeviceToHost, c->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  if (e != hipSuccess) return hip_check(c, e, "refine");
  *rmax = c->S_host->npart[0];
  *iters = 0;
  if (!(*rmax > tol)) return SP_OK;
  const int32_t iter_before = c->S_host->iter;  // the device count runs on across solves
  // solve A e = rt into the spare iterate, then xd += e
  std::swap(c->x, c->xe);
  sp_stats st{};
  sp_status s = solve(c, c->p1, tol, &st, false, false);
  std::swap(c->x, c->xe);
  if (s != SP_OK) return s;
  *iters = st.iterations - iter_before;
  timer_begin(c, "refine_add", (double)D.N * 24, &slot);
  hipLaunchKernelGGL(k_refine_add, cgrd, blk, 0, c->stream, A, (const double*)c->xe, c->xd);
  timer_end(c, slot);
  return SP_OK;
}

// x += xd (the refined pressure, rounded, for the adjoint's checkpoint).
sp_status fold_refinement(sp_ctx* c) {
  const Dims& D = c->dm;
  CgArgs A{};
  A.I = D.I; A.J = D.J; A.K = D.K;
  hipLaunchKernelGGL(k_refine_add, col_grid(D.I, D.J, D.K), dim3(64, 4, 1), 0, c->stream, A,
                     (const double*)c->xd, c->x);
  c->xd_active = false;
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? SP_OK : hip_check(c, e, "fold_refinement");
}

}  // namespace sp
