// The marching smoother leg with one cell per thread, for FP32 levels that
// the leg of sp_smooth_fused.h does not suit.
//
// Same march, tiles and results as there; a workgroup of EX x EY threads owns
// an interior of (EX - 2H) x (EY - 2H) columns, one per thread, every thread
// computes both colours' half-sweeps and keeps those of its own.  That wastes
// half of the arithmetic, but a step is a shorter chain and a thread holds
// one window of each array.  It is the better one
//   * where the large tiles do not shorten the march enough (small levels,
//     thin ones): a step is bound by its latency there (four_cell_leg);
//   * with a diagonal-only term, whose windows do not fit the registers two or
//     four times (160 x 96 x 96 with an outlet, whole solve: 2.88 ms against
//     3.16 with a pair and 3.96 with four, which spills).
// With the chunk start t0 even and R = W, every register-window slot and LDS
// ring slot is a compile-time constant.
#pragma once

#include <hip/hip_runtime.h>

#include "sp_smooth_fused.h"

namespace sp {

// Coarse levels too small in (i, j) to fill the chip with extended 40 x 24
// tiles march with 16 x 16 (an 8 x 8 interior at NU = 2): four waves per
// workgroup, several workgroups per CU.
constexpr int kFEXs = 16, kFEYs = 16;

template <int NU, int EX = kFEX, int EY = kFEY>
struct CellShape {
  static constexpr int H = 2 * NU;
  static constexpr int TX = EX - 2 * H;
  static constexpr int TY = EY - 2 * H;
  static constexpr int W = H + 2;  // register window (planes)
  static constexpr int R = W;      // LDS ring (planes)
  static_assert(TX > 0 && TY > 0 && TX % 2 == 0 && TY % 2 == 0,
                "the restriction pairs cells inside the tile interior");
};

// Raw loads of one plane.  The loads always target a valid address (the
// plane index is clamped, neighbours fall back to the cell itself) so their
// destination registers carry straight into the next pipeline step; validity
// is applied when the values are consumed.
struct CellLoad {
  float b, cx, cy, cz, cxm, cym, e, xin, xc;
  bool vt;
};

// Per-thread constants of the march.
struct CellCol {
  int i, j, tx, ty;
  bool in_ij, tile, vxm, vym;
  bool act_even;         // updated at even steps (i + j even)
  uint32_t col;          // byte offset of the (i, j) column in plane 0
  uint32_t plane;        // bytes per plane
  uint32_t dxm, dym;     // byte distance to the -x / -y neighbour (0 at the edge)
  uint32_t ccol;         // post: byte offset of the coarse column
  uint32_t cplane;       // post: bytes per coarse plane
};

template <int MODE, bool HAS_E>
__device__ inline void cell_load(CellLoad& L, const FusedArgs<float>& A, const CellCol& C, int t) {
  const int tc = t < 0 ? 0 : (t >= A.nz ? A.nz - 1 : t);
  const uint32_t n = C.col + C.plane * (uint32_t)tc;
  L.vt = C.in_ij && t >= 0 && t < A.nz;
  L.b = at_off<float>(A.b, n);
  L.cx = at_off<float>(A.cx, n);
  L.cy = at_off<float>(A.cy, n);
  L.cz = at_off<float>(A.cz, n);
  L.cxm = at_off<float>(A.cx, n - C.dxm);
  L.cym = at_off<float>(A.cy, n - C.dym);
  L.e = HAS_E ? at_off<float>(A.e, n) : 0.f;
  if (MODE == 1) {
    L.xin = at_off<float>(A.xin, n);
    L.xc = at_off<float>(A.xc, C.ccol + C.cplane * (uint32_t)(tc >> 1));
  } else {
    L.xin = 0.f;
    L.xc = 0.f;
  }
}

// Register windows along k.  Logical plane o (0 = newest) of step u lives in
// physical slot (o + W - u % W) % W, so advancing one plane renames slots
// instead of moving registers (the march is unrolled by W).
template <int NU, int MODE>
struct CellState {
  static constexpr int H = 2 * NU, W = H + 2;
  float xw[W], bw[W], dw[W], rdw[W], czw[W], cxw[W], cxmw[W], cyw[W], cymw[W];
  bool dpos[W];  // d > 0 of each plane, tested once when the plane enters
  float racc;
  double dacc[2];  // CG dot products (finest post-smoother)
};

// One pipeline step: plane t enters (from L), half-sweeps on the planes
// behind it, output/residual of plane t - H, restriction after the barrier.
// U = position of this step in the W-step unrolled march (t - t0 = U mod W).
template <int NU, int MODE, bool HAS_E, bool DOTS, int U, int EX, int EY>
__device__ inline void cell_step(CellState<NU, MODE>& F, const CellLoad& L,
                                  const FusedArgs<float>& A, const CellCol& C,
                                  float (*xs)[EY + 2][EX + 2], float (*rs)[EY][EX], int t,
                                  int k0, int k1) {
  using Sh = CellShape<NU, EX, EY>;
  constexpr int H = Sh::H, W = Sh::W, R = Sh::R;
  static_assert(R == W && (W % 2) == 0, "ring slots are compile-time only for R == W, W even");
  auto S = [](int o) constexpr { return (o + W - U) % W; };        // register slot
  auto Q = [](int o) constexpr { return ((U - o) % R + R) % R; };  // LDS ring slot
  const int tx = C.tx, ty = C.ty;
  // LDS planes carry a one-cell border of zeros: cell (tx, ty) is at
  // [ty + 1][tx + 1] and every neighbour read is unconditional
  const int lx = tx + 1, ly = ty + 1;

  const int q = t - H;
  const bool outq = q >= k0 && q < k1;
  const bool wr = outq && C.tile && C.in_ij;

  const float lb = L.vt ? L.b : 0.f, lcx = L.vt ? L.cx : 0.f, lcy = L.vt ? L.cy : 0.f;
  const float lcz = L.vt ? L.cz : 0.f, le = L.vt ? L.e : 0.f;
  const float lcxm = (L.vt && C.vxm) ? L.cxm : 0.f, lcym = (L.vt && C.vym) ? L.cym : 0.f;
  float d0 = lcxm;
  d0 = d0 + lcym;
  d0 = d0 + F.czw[S(1)];
  d0 = d0 + lcx;
  d0 = d0 + lcy;
  d0 = d0 + lcz;
  // the diagonal-only term; without one the sum stays as it is (adding +0
  // to a sum of non-negative couplings changes nothing)
  if (HAS_E) d0 = d0 + le;
  float x0 = 0.f;
  if (MODE == 1) x0 = d0 > 0.f ? L.xin + L.xc : 0.f;
  F.bw[S(0)] = lb; F.cxw[S(0)] = lcx; F.cxmw[S(0)] = lcxm; F.cyw[S(0)] = lcy;
  F.cymw[S(0)] = lcym; F.czw[S(0)] = lcz; F.dw[S(0)] = d0; F.xw[S(0)] = x0;
  F.dpos[S(0)] = d0 > 0.f;
  F.rdw[S(0)] = d0 > 0.f ? smoother_rcp(d0) : 0.f;
  xs[Q(0)][ly][lx] = x0;

  // cells of this thread's colour move this step (t0 even, W even)
  const bool act = (U & 1) ? !C.act_even : C.act_even;
#pragma unroll
  for (int s = 1; s <= H; ++s) {
    const int o = MODE == 0 ? s - 1 : s;
    // planes outside [0, nz) have d = 0 and stay 0, so no range test
    float v;
    if (MODE == 0 && s == 1) {
      v = F.bw[S(0)] * F.rdw[S(0)];
    } else {
      const float xW = xs[Q(o)][ly][lx - 1], xS = xs[Q(o)][ly - 1][lx];
      const float xE = xs[Q(o)][ly][lx + 1], xN = xs[Q(o)][ly + 1][lx];
      float acc = 0.f;
      acc += F.cxmw[S(o)] * xW;
      acc += F.cymw[S(o)] * xS;
      acc += F.czw[S(o + 1)] * F.xw[S(o + 1)];
      acc += F.cxw[S(o)] * xE;
      acc += F.cyw[S(o)] * xN;
      acc += F.czw[S(o)] * F.xw[S(o - 1)];
      v = (F.bw[S(o)] + acc) * F.rdw[S(o)];
    }
    v = F.xw[S(o)] + A.omega * (v - F.xw[S(o)]);
    // keep v in a register on every lane: a select whose operand is only
    // needed on some lanes would otherwise become an exec-masked branch
    __asm__ volatile("" : "+v"(v));
    const float xn = (act && F.dpos[S(o)]) ? v : F.xw[S(o)];
    F.xw[S(o)] = xn;
    xs[Q(o)][ly][lx] = xn;
  }

  if (MODE == 0) {
    float r = 0.f;
    if (wr && F.dpos[S(H)]) {
      const float xW = xs[Q(H)][ly][lx - 1], xS = xs[Q(H)][ly - 1][lx];
      const float xE = xs[Q(H)][ly][lx + 1], xN = xs[Q(H)][ly + 1][lx];
      float acc = 0.f;
      acc += F.cxmw[S(H)] * xW;
      acc += F.cymw[S(H)] * xS;
      acc += F.czw[S(H + 1)] * F.xw[S(H + 1)];
      acc += F.cxw[S(H)] * xE;
      acc += F.cyw[S(H)] * xN;
      acc += F.czw[S(H)] * F.xw[S(H - 1)];
      r = F.bw[S(H)] - (F.dw[S(H)] * F.xw[S(H)] - acc);
    }
    if (wr) put_off(A.xout, C.col + C.plane * (uint32_t)q, F.xw[S(H)]);
    // q = t0 + U - H (mod W) with t0 and H even: parity of q = parity of U
    if (q >= 0) rs[U & 1][ty][tx] = r;
  } else if (wr) {
    put_off(A.xout, C.col + C.plane * (uint32_t)q, F.xw[S(H)]);
    if (DOTS && A.dots) {
      const double z = (double)F.xw[S(H)];
      // (r, z) with the FP32 r the leg smooths with (the b window): an
      // rz rounded at 1e-7 only perturbs the step length, and the x and r
      // updates stay consistent (both use the same alpha)
      F.dacc[0] += (double)F.bw[S(H)] * z;
      F.dacc[1] += (double)F.dw[S(H)] * z;
    }
  }
  lds_barrier();
  if (MODE == 0 && wr && ((tx - H) & 1) == 0 && ((ty - H) & 1) == 0) {
    constexpr int sl = U & 1;
    float ps = rs[sl][ty][tx];
    ps += rs[sl][ty][tx + 1];
    ps += rs[sl][ty + 1][tx];
    ps += rs[sl][ty + 1][tx + 1];
    constexpr bool first = (U & 1) == 0;  // q even
    F.racc = first ? ps : F.racc + ps;
    if (!first || q == A.nz - 1) {
      // C.ccol: byte offset of the coarse column (i/2, j/2)
      put_off(A.bc, C.ccol + C.cplane * (uint32_t)(q >> 1), F.racc);
    }
  }
}

// Planes of loads in flight (six measured slower).  The window length W is a multiple of it,
// so the buffer of every step of the unrolled march is a compile-time choice.
template <int NU>
constexpr int cell_pipe() {
  return CellShape<NU>::W % 3 == 0 ? 3 : 2;
}

// Steps t + U, t + U + 1, ..., t + W - 1 of the march, each followed by the
// load of a later plane into the buffer it used.  CHECK: stop at t1 (the
// last, partial turn only).  Full turns carry no exit test, so the march loop
// has one back-edge whose in-flight loads are the same on every pass: an exit
// path per step would merge into the loop head with fewer loads in flight,
// and the compiler's wait counts there would drain the load pipeline on
// every turn.
template <int NU, int MODE, bool HAS_E, bool DOTS, bool CHECK, int U, int EX, int EY>
__device__ inline void cell_march(CellState<NU, MODE>& F, CellLoad (&LB)[cell_pipe<NU>()],
                                   const FusedArgs<float>& A, const CellCol& C,
                                   float (*xs)[EY + 2][EX + 2], float (*rs)[EY][EX], int t, int t1,
                                   int k0, int k1) {
  if constexpr (U < CellShape<NU>::W) {
    if (CHECK && t + U >= t1) return;
    constexpr int P = cell_pipe<NU>();
    static_assert(CellShape<NU>::W % P == 0, "load buffers must tile the window");
    CellLoad& L = LB[U % P];
    cell_step<NU, MODE, HAS_E, DOTS, U, EX, EY>(F, L, A, C, xs, rs, t + U, k0, k1);
    cell_load<MODE, HAS_E>(L, A, C, t + U + P);
    cell_march<NU, MODE, HAS_E, DOTS, CHECK, U + 1, EX, EY>(F, LB, A, C, xs, rs, t, t1, k0, k1);
  }
}

template <int NU, int MODE, bool FINE, bool HAS_E, int EX = kFEX, int EY = kFEY>
__global__ void __launch_bounds__(EX * EY) k_smooth_cell(FusedArgs<float> A, const Scalars* S) {
  if (S->done) return;
  using Sh = CellShape<NU, EX, EY>;
  constexpr int H = Sh::H, TX = Sh::TX, TY = Sh::TY, W = Sh::W, R = Sh::R;
  __shared__ float xs[R][EY + 2][EX + 2];
  __shared__ float rs[2][EY][EX];
  uint32_t bx, by, bz;
  xcd_block3(bx, by, bz);
  CellCol C;
  C.tx = threadIdx.x;
  C.ty = threadIdx.y;
  C.i = (int)bx * TX - H + C.tx;
  C.j = (int)by * TY - H + C.ty;
  C.in_ij = C.i >= 0 && C.i < A.nx && C.j >= 0 && C.j < A.ny;
  C.tile = C.tx >= H && C.tx < H + TX && C.ty >= H && C.ty < H + TY;
  C.vxm = C.i > 0;
  C.vym = C.j > 0;
  C.act_even = ((C.i + C.j) & 1) == 0;
  C.col = C.in_ij ? (uint32_t)(C.i + A.nx * C.j) * (uint32_t)sizeof(float) : 0u;
  C.plane = (uint32_t)A.nx * (uint32_t)A.ny * (uint32_t)sizeof(float);
  C.dxm = (C.in_ij && C.vxm) ? (uint32_t)sizeof(float) : 0u;
  C.dym = (C.in_ij && C.vym) ? (uint32_t)(A.nx * sizeof(float)) : 0u;
  C.ccol = C.in_ij ? (uint32_t)((C.i >> 1) + A.cnx * (C.j >> 1)) * (uint32_t)sizeof(float) : 0u;
  C.cplane = (uint32_t)A.cnx * (uint32_t)A.cny * (uint32_t)sizeof(float);
  const int k0 = (int)bz * A.kchunk;
  const int k1 = min(k0 + A.kchunk, A.nz);

  CellState<NU, MODE> F;
#pragma unroll
  for (int o = 0; o < W; ++o) {
    F.xw[o] = F.bw[o] = F.dw[o] = F.rdw[o] = F.czw[o] = F.cxw[o] = F.cxmw[o] = F.cyw[o] =
        F.cymw[o] = 0.f;
    F.dpos[o] = false;
  }
  F.racc = 0.f;
  F.dacc[0] = F.dacc[1] = 0.0;
  for (int q = C.ty * EX + C.tx; q < R * (EY + 2) * (EX + 2); q += EX * EY) (&xs[0][0][0])[q] = 0.f;
  for (int q = C.ty * EX + C.tx; q < 2 * EY * EX; q += EX * EY) (&rs[0][0][0])[q] = 0.f;
  // cz of the plane below the first loaded one (bottom face of that plane):
  // logical plane 1 of the first step, physical slot 1
  {
    const int pb = k0 - H - 1;
    if (C.in_ij && pb >= 0 && pb < A.nz)
      F.czw[1] = at_off<float>(A.cz, C.col + C.plane * (uint32_t)pb);
  }
  __syncthreads();

  // buffer u % P holds the planes of steps t0 + u (mod P)
  const int t0 = k0 - H, t1 = k1 + H;  // steps [t0, t1); t0 even
  constexpr int P = cell_pipe<NU>();
  constexpr bool DOTS = FINE && MODE == 1;
  CellLoad LB[P];
#pragma unroll
  for (int u = 0; u < P; ++u) cell_load<MODE, HAS_E>(LB[u], A, C, t0 + u);
  int t = t0;
  for (; t + W <= t1; t += W)
    cell_march<NU, MODE, HAS_E, DOTS, false, 0, EX, EY>(F, LB, A, C, xs, rs, t, t1, k0, k1);
  if (t < t1)
    cell_march<NU, MODE, HAS_E, DOTS, true, 0, EX, EY>(F, LB, A, C, xs, rs, t, t1, k0, k1);
  if constexpr (DOTS) {
    if (A.dots) block_partials<EX * EY, 2, 0u>(A.dsite, F.dacc);
  }
}

}  // namespace sp
