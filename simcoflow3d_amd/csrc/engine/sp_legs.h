// Launch shape of the marching smoother legs, and which of the two FP32 forms
// a level takes.  Host arithmetic only.
#pragma once

#include <cstdint>

namespace sp {

// Extended tiles (interior plus halo): one cell per thread (sp_smooth_cell.h),
// four cells per thread (sp_smooth_fused.h, FP32).
constexpr int kFEX = 40, kFEY = 24;
constexpr int kQEX = 72, kQEY = 24;

struct LegGrid {
  int gx, gy, gz, kchunk;
  int64_t cost;  // rounds of workgroups x planes a workgroup marches
};

// Tiles of tx x ty columns of an nx x ny x nz level, `slots` workgroups at a
// time.  k chunk: even (coarse cells never straddle chunks).  A workgroup
// marches kchunk + 2 halo planes one after the other, so pick the chunk that
// minimises rounds-of-workgroups x planes marched.
inline LegGrid leg_grid(int nx, int ny, int nz, int tx, int ty, int halo, int64_t slots) {
  LegGrid g{(nx + tx - 1) / tx, (ny + ty - 1) / ty, 0, 0, -1};
  const int64_t tiles = (int64_t)g.gx * g.gy;
  for (int kc = 2; kc <= ((nz + 1) & ~1); kc += 2) {
    const int64_t blocks = tiles * ((nz + kc - 1) / kc);
    const int64_t cost = ((blocks + slots - 1) / slots) * (kc + 2 * halo);
    if (g.cost < 0 || cost < g.cost) { g.cost = cost; g.kchunk = kc; }
  }
  g.gz = (nz + g.kchunk - 1) / g.kchunk;
  return g;
}

// Four cells per thread, or one (FP32, no diagonal-only term, one workgroup
// per CU in both forms).  A step of the large tile serves twice the columns in
// 1.2 to 1.5 times the small one's time, so the large tile is the better one
// when it marches fewer than 4/5 as many planes; with two sweeps only below
// 2/3, unless the rows do not start on 16 bytes: the one-cell leg's 40-wide
// tiles then straddle more lines, which costs it 8 to 10 %.
// Pre plus post leg, four cells against one, event times, two sweeps (cost
// ratio in parentheses): 256^3 (0.53) 0.89, 192^3 (0.50) 0.81, 1024 x 1024 x 8
// (0.50) 0.78, 128 x 128 x 512 (0.56) 0.94, 210^3 (0.62) 0.93, 128^3 (0.67)
// 1.03, 152^3 (0.70) 1.04, 132 x 124 x 40 (0.75) 1.10, 640 x 160 x 10 (0.78)
// 1.12, 256 x 256 x 8 (0.83) 1.20, 64^3 (1.0) 1.23; rows off 16 bytes: 126^3
// (0.67) 0.91, 99 x 101 x 103 (0.70) 0.95, 97 x 130 x 75 (0.70) 0.92,
// 113 x 113 x 60 (0.75) 1.01, 135 x 141 x 60 (0.80) 1.06; one sweep: 152^3
// (0.67) 0.94, 108 x 108 x 300 (0.77) 1.00, 132 x 124 x 40 (0.80) 1.02,
// 600 x 600 x 20 (0.88) 1.34.  Over 77 sizes and both sweeps the choice is
// 0.2 % off the faster form on average, a limit on the columns alone was 4 %.
inline bool four_cell_leg(int nx, int ny, int nz, int sweeps, int64_t slots) {
  const int h = 2 * sweeps, hx = (h + 3) / 4 * 4;
  const int64_t one = leg_grid(nx, ny, nz, kFEX - 2 * h, kFEY - 2 * h, h, slots).cost;
  const int64_t four = leg_grid(nx, ny, nz, kQEX - 2 * hx, kQEY - 2 * h, h, slots).cost;
  if (sweeps == 2 && nx % 4 == 0) return 3 * four < 2 * one;
  return 5 * four < 4 * one;
}

}  // namespace sp
