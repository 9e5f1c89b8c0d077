// Temporally blocked red-black Gauss-Seidel for one multigrid level.
//
// A workgroup of EP x EY threads owns a tile of (i,j) columns, 2*Q consecutive
// columns along i per thread, plus a halo of H = 2*NU columns on every side,
// and marches over a chunk of k planes.  The 2*NU half-sweeps are pipelined
// one plane apart: at step t the plane t is loaded, half-sweep s updates
// plane t-s+1 (pre) or t-s (post), so every array is streamed from HBM once
// per kernel instead of once per half-sweep.  Values along k live in
// per-thread register windows; the in-plane neighbours of a plane come from a
// ring of LDS planes written one step earlier (one barrier per step).  The
// halo shrinks by one column per half-sweep, so the tile's results are those
// of the plain sweep sequence:
//   pre  (MODE 0): x = 0; red, black, red, black ...; r = b - A x restricted
//                  (sum over 2x2x2 children) into the coarse right-hand side;
//                  x is written to xout.
//   post (MODE 1): x = xin + P xc (active cells); black, red, black, red ...;
//                  x is written to xout.
//
// In both modes the cell (i,j) is updated at step t exactly when i + j + t is
// even (half-sweep s touches plane t - s + 1 with colour s - 1, or plane
// t - s with colour s).  The cells of a thread are therefore named by the
// parity of i + j: pair m holds A_m (i + j even) and B_m; at even steps every
// thread updates its A cells, at odd steps its B cells.  A thread per cell
// would compute every half-sweep on both colours and throw half of them away;
// here every update is a wanted one, and which cells it takes is a
// compile-time choice.  The four in-plane neighbours of an A cell are B
// cells: along i the pair's own and that of the pair to the left (even rows)
// or to the right (odd rows), a register except at the thread's outer edge;
// along j the B cells of the same pair in the rows above and below.  LDS
// holds the A and the B cells of a plane apart, so a thread reads and writes
// its Q values of one colour as one vector.
//
// The march is unrolled by the window length W; with the chunk start t0 even
// and R = W, every register-window slot and LDS ring slot is a compile-time
// constant.
#pragma once

#include <hip/hip_runtime.h>

#include "sp_device.h"

namespace sp {

template <typename T>
struct FusedArgs {
  int nx, ny, nz;
  const T *cx, *cy, *cz, *e;
  const T* b;
  const T* xin;  // post: pre-smoothed x
  const T* xc;   // post: coarse correction
  T* xout;
  T* bc;         // pre: coarse right-hand side
  int cnx, cny;
  int kchunk;    // even
  T omega;       // over-relaxation: x += omega (x_gs - x)
  // finest post-smoother only: the CG dot products (r,z), (dw,z) of the z it
  // writes, as per-workgroup partials (r and the diagonal weight: the
  // right-hand side and diagonal the leg already holds)
  int dots;
  RedSite dsite;
};

// The extended tile of a leg (threads along i x rows) and pairs per thread.
//
// No unit is saturated at 256^3 (counters): 1.2 to 1.3 times the algorithmic
// bytes at 0.75 to 0.9 of the copy rate, the VALU a third busy; waits for loads
// and the barrier (about 40 % of a wave's cycles) and for issue (30 %) overlap
// only in part, for want of waves.
// FP32: four cells per thread with 16-byte loads (256 VGPRs, two waves per
// SIMD), a 64 x 16 interior whose rows are whole cache lines; measured at
// 256^3 with one cell per thread and a 32 x 16 interior 117 (pre) and 140 us
// (post), with a pair and 56 x 16 120 and 133 us, with this 105 and 116 us
// (floor at the card's copy rate: 70 and 84 us; all on one card).  FP64, whose
// windows do not fit the registers twice: a pair per thread, 32 x 16 interior
// (256^3: 272 and 274 -> 253 and 256 us).
//
// FP64 levels of at most 64 x 64 columns give too few large tiles to put one
// on every CU, and a march of few steps whose time is the latency of a step:
// 8 x 8 interior, two waves per workgroup (against one cell per thread, whole
// solves at 32^3 1642 -> 1257 us, 128^3 4175 -> 3542 us).
template <typename T, bool SMALL>
struct FusedTile {
  static constexpr bool kQuad = sizeof(T) == 4;
  static_assert(!(kQuad && SMALL), "FP32 levels of few columns take the one-cell leg");
  static constexpr int Q = kQuad ? 2 : 1;
  static constexpr int EP = SMALL ? 8 : (kQuad ? 18 : 20);
  static constexpr int EY = SMALL ? 16 : 24;
  static constexpr int kPerCu = SMALL ? 4 : 1;  // workgroups a CU holds at once (registers)
};
constexpr int64_t kSmallColumns = 64 * 64;

template <int NU, int Q, int EP, int EY>
struct FusedShape {
  static constexpr int H = 2 * NU;
  static constexpr int C = 2 * Q;                       // cells per thread
  static constexpr int HX = (H + C - 1) / C * C;        // halo along i, whole threads
  static constexpr int TX = C * EP - 2 * HX;            // interior columns along i
  static constexpr int TY = EY - 2 * H;
  static constexpr int W = H + 2;  // register window (planes)
  static constexpr int R = W;      // LDS ring (planes)
  static_assert(TX > 0 && TY > 0 && TY % 2 == 0 && H % 2 == 0,
                "the restriction pairs cells inside the tile interior");
};

// Barrier that orders LDS only: global loads issued for later planes stay in
// flight across it (the kernel's global stores are never read back inside
// the kernel).
__device__ inline void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// N consecutive elements.  Vec is aligned like one element, since the rows of
// a level start anywhere (global memory takes such loads whole); LVec is
// naturally aligned (LDS).
template <typename T, int N>
struct __attribute__((packed, aligned(sizeof(T)))) Vec {
  T v[N];
};
template <typename T, int N>
struct __attribute__((aligned(sizeof(T) * N))) LVec {
  T v[N];
};

// Element(s) at a 32-bit byte offset (every level array is below 4 GiB), so
// the loads use a scalar base plus one 32-bit vector offset.
template <typename V, typename T>
__device__ inline V at_off(const T* base, uint32_t byte_off) {
  return *reinterpret_cast<const V*>(reinterpret_cast<const char*>(base) + byte_off);
}
template <typename V, typename T>
__device__ inline void put_off(T* base, uint32_t byte_off, V v) {
  *reinterpret_cast<V*>(reinterpret_cast<char*>(base) + byte_off) = v;
}

template <typename T, int N>
__device__ inline void put_stream(T* base, uint32_t byte_off, const Vec<T, N>& v) {
  typedef T NV __attribute__((ext_vector_type(N), aligned(sizeof(T))));
  NV w;
#pragma unroll
  for (int c = 0; c < N; ++c) w[c] = v.v[c];
  __builtin_nontemporal_store(w, reinterpret_cast<NV*>(reinterpret_cast<char*>(base) + byte_off));
}

// 1/d of a smoother: FP32 uses the hardware reciprocal (1 ulp), which is
// ample for a preconditioner; FP64 divides.
__device__ inline float smoother_rcp(float d) { return __builtin_amdgcn_rcpf(d); }
__device__ inline double smoother_rcp(double d) { return 1.0 / d; }

// Raw loads of one plane.  The loads always target a valid address (the plane
// index is clamped, columns outside the domain read the first cells, cells
// past the end of a row read what follows) so their destination registers
// carry straight into the next pipeline step; validity is applied when the
// values are consumed.
template <typename T, int Q>
struct PlaneLoad {
  Vec<T, 2 * Q> b, cx, cy, cz, cym, e, xin;
  T cxm;
  Vec<T, Q> xc;
};

// Per-thread constants of the march.
template <int Q>
struct FusedCol {
  int tx, ty;
  bool odd;              // row parity: A is the second cell of each pair
  bool in[2 * Q];        // the thread's cells lie in the domain
  bool tile;             // the thread belongs to the tile interior
  uint32_t col;          // byte offset of the first cell in plane 0
  uint32_t plane;        // bytes per plane
  uint32_t dxm, dym;     // byte distance to the W / S face couplings
  uint32_t ccol;         // byte offset of the coarse column
  uint32_t cplane;       // bytes per coarse plane
};

template <typename T, int Q, int MODE, bool HAS_E>
__device__ inline void load_plane(PlaneLoad<T, Q>& L, const FusedArgs<T>& A, const FusedCol<Q>& C,
                                  int t) {
  using V = Vec<T, 2 * Q>;
  const int tc = t < 0 ? 0 : (t >= A.nz ? A.nz - 1 : t);
  const uint32_t n = C.col + C.plane * (uint32_t)tc;
  L.b = at_off<V>(A.b, n);
  L.cx = at_off<V>(A.cx, n);
  L.cy = at_off<V>(A.cy, n);
  L.cz = at_off<V>(A.cz, n);
  L.cxm = at_off<T>(A.cx, n + C.dxm);
  L.cym = at_off<V>(A.cy, n + C.dym);
  if (HAS_E) L.e = at_off<V>(A.e, n);
  if (MODE == 1) {
    L.xin = at_off<V>(A.xin, n);
    L.xc = at_off<Vec<T, Q>>(A.xc, C.ccol + C.cplane * (uint32_t)(tc >> 1));
  }
}

// Register windows along k; [2]: cells A and B, [Q]: pairs.  Logical plane o
// (0 = newest) of step u lives in physical slot (o + W - u % W) % W, so
// advancing one plane renames slots instead of moving registers (the march
// is unrolled by W).
template <typename T, int NU, int Q>
struct FusedState {
  static constexpr int H = 2 * NU, W = H + 2;
  T x[2][Q][W], b[2][Q][W], rd[2][Q][W], cz[2][Q][W];
  T cm[Q][W];                                  // coupling between a pair's cells
  T co[2][Q][W], cn[2][Q][W], cs[2][Q][W];     // outer, N and S couplings
  T d[2][Q][W];                                // diagonal, kept only with a diagonal-only term
  T racc[Q];
  double dacc[2];  // CG dot products (finest post-smoother)
};

// LDS planes: [ring slot][cell A / B][row][thread], with a border of zeros so
// every neighbour read is unconditional.
template <typename T, int Q, int EP, int EY>
using FusedLds = LVec<T, Q>[2][EY + 2][EP + 2];

// Diagonal of cell (c, m) of logical plane slot `o` (`ob`: the plane below).
template <typename T, int NU, int Q>
__device__ inline T fused_diag(const FusedState<T, NU, Q>& F, int c, int m, int o, int ob) {
  T d = F.co[c][m][o] + F.cm[m][o];
  d = d + F.cs[c][m][o];
  d = d + F.cn[c][m][o];
  d = d + F.cz[c][m][ob];
  d = d + F.cz[c][m][o];
  return d;
}

// base + the couplings of cell (c, *) of slot `o` times its neighbours; the
// thread's row and the rows above and below of the other colour come from LDS
template <typename T, int NU, int Q, int EP, int EY>
__device__ inline void fused_offdiag(const FusedState<T, NU, Q>& F, const FusedCol<Q>& C,
                                     const FusedLds<T, Q, EP, EY>& pl, int c, int o, int ob, int oa,
                                     T (&acc)[Q]) {
  const int lx = C.tx + 1, ly = C.ty + 1, n = 1 - c;
  // the outer neighbour lies to the left of A in even rows and of B in odd ones
  const bool right = C.odd == (c == 0);
  const T edge = pl[n][ly][right ? lx + 1 : lx - 1].v[0 + (Q > 1 ? (right ? 0 : Q - 1) : 0)];
  const LVec<T, Q> s = pl[n][ly - 1][lx], u = pl[n][ly + 1][lx];
#pragma unroll
  for (int m = 0; m < Q; ++m) {
    const T l = m > 0 ? F.x[n][m > 0 ? m - 1 : 0][o] : edge;
    const T r = m < Q - 1 ? F.x[n][m < Q - 1 ? m + 1 : m][o] : edge;
    acc[m] += F.co[c][m][o] * (Q == 1 ? edge : (right ? r : l));
    acc[m] += F.cs[c][m][o] * s.v[m];
    acc[m] += F.cn[c][m][o] * u.v[m];
    acc[m] += F.cm[m][o] * F.x[n][m][o];
    acc[m] += F.cz[c][m][ob] * F.x[c][m][ob];
    acc[m] += F.cz[c][m][o] * F.x[c][m][oa];
  }
}

// One pipeline step: plane t enters (from L), half-sweeps on the planes
// behind it, output/residual of plane t - H, restriction after the barrier.
// U = position of this step in the W-step unrolled march (t - t0 = U mod W).
template <typename T, int NU, int Q, int MODE, bool HAS_E, bool DOTS, int U, int EP, int EY>
__device__ inline void fused_step(FusedState<T, NU, Q>& F, const PlaneLoad<T, Q>& L,
                                  const FusedArgs<T>& A, const FusedCol<Q>& C,
                                  FusedLds<T, Q, EP, EY>* xs, LVec<T, Q> (*rs)[EY][EP], int t,
                                  int k0, int k1) {
  using Sh = FusedShape<NU, Q, EP, EY>;
  constexpr int H = Sh::H, W = Sh::W, R = Sh::R;
  static_assert(R == W && (W % 2) == 0, "ring slots are compile-time only for R == W, W even");
  auto S = [](int o) constexpr { return (o + W - U) % W; };        // register slot
  auto K = [](int o) constexpr { return ((U - o) % R + R) % R; };  // LDS ring slot
  const int lx = C.tx + 1, ly = C.ty + 1;
  const int q = t - H;
  const bool wr = q >= k0 && q < k1 && C.tile && C.in[0];

  // plane t enters; the couplings of cells outside the domain are arbitrary
  // finite values, and their 1/d = 0 keeps x = 0 there
  const bool vt = t >= 0 && t < A.nz;
#pragma unroll
  for (int m = 0; m < Q; ++m) {
    const T left = m > 0 ? L.cx.v[m > 0 ? 2 * m - 1 : 0] : L.cxm, right = L.cx.v[2 * m + 1];
    F.cm[m][S(0)] = L.cx.v[2 * m];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      auto pick = [&](const Vec<T, 2 * Q>& v) {
        return C.odd == (c == 0) ? v.v[2 * m + 1] : v.v[2 * m];
      };
      F.b[c][m][S(0)] = pick(L.b);
      F.cn[c][m][S(0)] = pick(L.cy);
      F.cs[c][m][S(0)] = pick(L.cym);
      const T cz = pick(L.cz);
      F.cz[c][m][S(0)] = t >= 0 ? cz : T(0);  // no coupling below plane 0
      F.co[c][m][S(0)] = C.odd == (c == 0) ? right : left;
      T d = fused_diag(F, c, m, S(0), S(1));
      if (HAS_E) {
        d = d + pick(L.e);
        F.d[c][m][S(0)] = d;
      }
      const bool in = C.odd == (c == 0) ? C.in[2 * m + 1] : C.in[2 * m];
      const bool dp = vt && in && d > T(0);
      F.rd[c][m][S(0)] = dp ? smoother_rcp(d) : T(0);
      F.x[c][m][S(0)] = MODE == 1 && dp ? pick(L.xin) + L.xc.v[m] : T(0);
    }
  }

  // the cells of this step's colour (t0 even, W even)
  constexpr int a = U & 1;
  LVec<T, Q> w[2];
#pragma unroll
  for (int m = 0; m < Q; ++m) {
    // first half-sweep of the pre leg, from x = 0
    if (MODE == 0) F.x[a][m][S(0)] = A.omega * (F.b[a][m][S(0)] * F.rd[a][m][S(0)]);
    w[0].v[m] = F.x[0][m][S(0)];
    w[1].v[m] = F.x[1][m][S(0)];
  }
  xs[K(0)][0][ly][lx] = w[0];
  xs[K(0)][1][ly][lx] = w[1];
#pragma unroll
  for (int s = MODE == 0 ? 2 : 1; s <= H; ++s) {
    const int o = MODE == 0 ? s - 1 : s;
    // planes outside [0, nz) have 1/d = 0 and stay 0, so no range test
    T acc[Q];
#pragma unroll
    for (int m = 0; m < Q; ++m) acc[m] = F.b[a][m][S(o)];
    fused_offdiag<T, NU, Q, EP, EY>(F, C, xs[K(o)], a, S(o), S(o + 1), S(o - 1), acc);
    LVec<T, Q> out;
#pragma unroll
    for (int m = 0; m < Q; ++m) {
      const T v = acc[m] * F.rd[a][m][S(o)];
      F.x[a][m][S(o)] += A.omega * (v - F.x[a][m][S(o)]);
      out.v[m] = F.x[a][m][S(o)];
    }
    xs[K(o)][a][ly][lx] = out;
  }

  if (wr) {
    Vec<T, 2 * Q> out;
#pragma unroll
    for (int m = 0; m < Q; ++m) {
      out.v[2 * m] = C.odd ? F.x[1][m][S(H)] : F.x[0][m][S(H)];
      out.v[2 * m + 1] = C.odd ? F.x[0][m][S(H)] : F.x[1][m][S(H)];
    }
    const uint32_t at = C.col + C.plane * (uint32_t)q;
    if (C.in[2 * Q - 1]) {
      // the pre leg's x is read again only after the coarser levels: written
      // past the caches it leaves them to the halos (256^3: 113 -> 105 us)
      if (MODE == 0 && Q > 1) put_stream(A.xout, at, out);
      else put_off(A.xout, at, out);
    } else {
#pragma unroll
      for (int c = 0; c < 2 * Q - 1; ++c)
        if (C.in[c]) put_off(A.xout, at + (uint32_t)(c * sizeof(T)), out.v[c]);
    }
  }
  LVec<T, Q> r;
  if (MODE == 0) {
#pragma unroll
    for (int m = 0; m < Q; ++m) r.v[m] = T(0);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      T acc[Q];
#pragma unroll
      for (int m = 0; m < Q; ++m)
        acc[m] = F.b[c][m][S(H)] -
                 (HAS_E ? F.d[c][m][S(H)] : fused_diag(F, c, m, S(H), S(H + 1))) * F.x[c][m][S(H)];
      fused_offdiag<T, NU, Q, EP, EY>(F, C, xs[K(H)], c, S(H), S(H + 1), S(H - 1), acc);
#pragma unroll
      for (int m = 0; m < Q; ++m) r.v[m] += F.rd[c][m][S(H)] > T(0) ? acc[m] : T(0);
    }
    rs[U & 1][C.ty][C.tx] = r;
  } else if (DOTS && A.dots && wr) {
    // (r, z) with the r the leg smooths with (the b window): in FP32 an rz
    // rounded at 1e-7 only perturbs the step length, and the x and r updates
    // stay consistent (both use the same alpha)
#pragma unroll
    for (int m = 0; m < Q; ++m)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const double z = (double)F.x[c][m][S(H)];
        const T d = HAS_E ? F.d[c][m][S(H)] : fused_diag(F, c, m, S(H), S(H + 1));
        F.dacc[0] += (double)F.b[c][m][S(H)] * z;
        F.dacc[1] += (double)d * z;
      }
  }
  lds_barrier();
  // a pair is a coarse cell's two children along i; the even row adds the odd
  // row's sum, then the two planes
  if (MODE == 0 && wr && !C.odd) {
    const LVec<T, Q> up = rs[U & 1][C.ty + 1][C.tx];
    constexpr bool first = (U & 1) == 0;  // q = t - H even
    Vec<T, Q> out;
#pragma unroll
    for (int m = 0; m < Q; ++m) {
      const T ps = r.v[m] + up.v[m];
      F.racc[m] = first ? ps : F.racc[m] + ps;
      out.v[m] = F.racc[m];
    }
    if (!first || q == A.nz - 1) {
      const uint32_t at = C.ccol + C.cplane * (uint32_t)(q >> 1);
      if (C.in[2 * Q - 2]) {
        put_off(A.bc, at, out);
      } else {
#pragma unroll
        for (int m = 0; m < Q - 1; ++m)
          if (C.in[2 * m]) put_off(A.bc, at + (uint32_t)(m * sizeof(T)), out.v[m]);
      }
    }
  }
}

// Planes of loads in flight: what the registers hold.
template <typename T>
constexpr int fused_pipe() {
  return sizeof(T) == 8 ? 1 : 2;
}

// Steps t + U, t + U + 1, ..., t + W - 1 of the march, each followed by the
// load of a later plane into the buffer it used (P planes of loads in flight;
// W is a multiple of P, so the buffer of every step is a compile-time
// choice).  CHECK: stop at t1 (the last, partial turn only).  Full turns
// carry no exit test, so the march loop has one back-edge whose in-flight
// loads are the same on every pass: an exit path per step would merge into
// the loop head with fewer loads in flight, and the compiler's wait counts
// there would drain the load pipeline on every turn.
template <typename T, int NU, int Q, int MODE, bool HAS_E, bool DOTS, bool CHECK, int P, int U,
          int EP, int EY>
__device__ inline void march_steps(FusedState<T, NU, Q>& F, PlaneLoad<T, Q> (&LB)[P],
                                   const FusedArgs<T>& A, const FusedCol<Q>& C,
                                   FusedLds<T, Q, EP, EY>* xs, LVec<T, Q> (*rs)[EY][EP], int t,
                                   int t1, int k0, int k1) {
  if constexpr (U < FusedState<T, NU, Q>::W) {
    if (CHECK && t + U >= t1) return;
    static_assert(FusedState<T, NU, Q>::W % P == 0, "load buffers must tile the window");
    PlaneLoad<T, Q>& L = LB[U % P];
    fused_step<T, NU, Q, MODE, HAS_E, DOTS, U, EP, EY>(F, L, A, C, xs, rs, t + U, k0, k1);
    load_plane<T, Q, MODE, HAS_E>(L, A, C, t + U + P);
    march_steps<T, NU, Q, MODE, HAS_E, DOTS, CHECK, P, U + 1, EP, EY>(F, LB, A, C, xs, rs, t, t1,
                                                                     k0, k1);
  }
}

template <typename T, int NU, int Q, int MODE, bool FINE, bool HAS_E, int EP, int EY>
__global__ void __launch_bounds__(EP * EY) k_smooth_fused(FusedArgs<T> A, const Scalars* S) {
  if (S->done) return;
  using Sh = FusedShape<NU, Q, EP, EY>;
  constexpr int H = Sh::H, HX = Sh::HX, TX = Sh::TX, TY = Sh::TY, W = Sh::W, R = Sh::R;
  __shared__ __attribute__((aligned(16))) FusedLds<T, Q, EP, EY> xs[R];
  __shared__ LVec<T, Q> rs[2][EY][EP];
  uint32_t bx, by, bz;
  xcd_block3(bx, by, bz);
  FusedCol<Q> C;
  C.tx = (int)(threadIdx.x % EP);
  C.ty = (int)(threadIdx.x / EP);
  const int i = (int)bx * TX - HX + Sh::C * C.tx, j = (int)by * TY - H + C.ty;
  const bool in_j = j >= 0 && j < A.ny;
  C.odd = (C.ty & 1) != 0;  // TY and H are even
#pragma unroll
  for (int c = 0; c < Sh::C; ++c) C.in[c] = in_j && i >= 0 && i + c < A.nx;
  C.tile = Sh::C * C.tx >= HX && Sh::C * C.tx < HX + TX && C.ty >= H && C.ty < H + TY;
  const uint32_t sz = (uint32_t)sizeof(T);
  C.col = C.in[0] ? (uint32_t)(i + A.nx * j) * sz : 0u;
  C.plane = (uint32_t)A.nx * (uint32_t)A.ny * sz;
  // W and S faces; at the domain's first column and row the couplings of the
  // row's last cell and of the last row, which are 0
  C.dxm = !C.in[0] ? 0u : (i > 0 ? 0u - sz : (uint32_t)(A.nx - 1) * sz);
  C.dym = !C.in[0] ? 0u : (j > 0 ? 0u - (uint32_t)A.nx * sz
                                 : (uint32_t)A.nx * (uint32_t)(A.ny - 1) * sz);
  C.ccol = C.in[0] ? (uint32_t)((i >> 1) + A.cnx * (j >> 1)) * sz : 0u;
  C.cplane = (uint32_t)A.cnx * (uint32_t)A.cny * sz;
  const int k0 = (int)bz * A.kchunk;
  const int k1 = min(k0 + A.kchunk, A.nz);

  FusedState<T, NU, Q> F;
#pragma unroll
  for (int m = 0; m < Q; ++m) {
    F.racc[m] = T(0);
#pragma unroll
    for (int o = 0; o < W; ++o) {
      F.cm[m][o] = T(0);
#pragma unroll
      for (int c = 0; c < 2; ++c)
        F.x[c][m][o] = F.b[c][m][o] = F.rd[c][m][o] = F.cz[c][m][o] = F.co[c][m][o] =
            F.cn[c][m][o] = F.cs[c][m][o] = F.d[c][m][o] = T(0);
    }
  }
  F.dacc[0] = F.dacc[1] = 0.0;
  constexpr int kLds = R * 2 * (EY + 2) * (EP + 2) * Q, kRs = 2 * EY * EP * Q;
  for (int q = (int)threadIdx.x; q < kLds; q += EP * EY) (&xs[0][0][0][0].v[0])[q] = T(0);
  for (int q = (int)threadIdx.x; q < kRs; q += EP * EY) (&rs[0][0][0].v[0])[q] = T(0);
  // cz of the plane below the first loaded one (bottom face of that plane):
  // logical plane 1 of the first step, physical slot 1
  {
    const int pb = k0 - H - 1;
    if (C.in[0] && pb >= 0 && pb < A.nz) {
      const Vec<T, 2 * Q> v = at_off<Vec<T, 2 * Q>>(A.cz, C.col + C.plane * (uint32_t)pb);
#pragma unroll
      for (int m = 0; m < Q; ++m) {
        F.cz[0][m][1] = C.odd ? v.v[2 * m + 1] : v.v[2 * m];
        F.cz[1][m][1] = C.odd ? v.v[2 * m] : v.v[2 * m + 1];
      }
    }
  }
  __syncthreads();

  // buffer u % P holds the planes of steps t0 + u (mod P)
  const int t0 = k0 - H, t1 = k1 + H;  // steps [t0, t1); t0 even
  constexpr bool DOTS = FINE && MODE == 1;
  constexpr int P = fused_pipe<T>();
  PlaneLoad<T, Q> LB[P];
#pragma unroll
  for (int u = 0; u < P; ++u) load_plane<T, Q, MODE, HAS_E>(LB[u], A, C, t0 + u);
  int t = t0;
  for (; t + W <= t1; t += W)
    march_steps<T, NU, Q, MODE, HAS_E, DOTS, false, P, 0, EP, EY>(F, LB, A, C, xs, rs, t, t1, k0,
                                                                 k1);
  if (t < t1)
    march_steps<T, NU, Q, MODE, HAS_E, DOTS, true, P, 0, EP, EY>(F, LB, A, C, xs, rs, t, t1, k0,
                                                                k1);
  if constexpr (DOTS) {
    // fixed order: thread sums through LDS, one wave adds them (the workgroup
    // is no whole number of waves)
    if (A.dots) {
      constexpr int NT = EP * EY;
      static_assert(sizeof(xs) >= 2 * NT * sizeof(double), "the sums reuse the planes");
      double* red = reinterpret_cast<double*>(&xs[0]);
      __syncthreads();
#pragma unroll
      for (int v = 0; v < 2; ++v) red[v * NT + (int)threadIdx.x] = F.dacc[v];
      __syncthreads();
      if (threadIdx.x < 64) {
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          double s = 0.0;
          for (int k = (int)threadIdx.x; k < NT; k += 64) s += red[v * NT + k];
          s = wave_sum(s);
          if (threadIdx.x == 0) A.dsite.part[(size_t)v * A.dsite.max_blocks + flat_block()] = s;
        }
      }
    }
  }
}

}  // namespace sp
