// The z and y passes of small grids as one: a workgroup transforms a whole
// plane of rows (z, then y, or back) and keeps it on the CU between the two, so
// the solve launches three kernels instead of five and reads and writes its
// arrays three times instead of five (ff_plane.hip).
#pragma once

#include "ff_kernels.hpp"

namespace ff {

// Line lengths with a plane phase compiled in: rows nz (M = nz/2 packed values)
// and columns ny, with the elements per thread of the passes' own kernels (the
// planner's defaults), so the results are theirs bit for bit.  The plan is used
// where the planner's agrees.  Rows of 160 and more would leave a plane of
// complex values no room in LDS; exchanging real and imaginary parts one after
// the other instead doubles the barriers, and was slower than the passes.  (These are
// the lengths that were measured, the batches' and other round ones; 54, 60, 75, 81, 90,
// 120 and 125 would fit and are not compiled in: every row length takes a kernel for each
// column length.)
struct PlaneLen {
  int n, ez, ey;  // nz or ny; elements per thread of the row (0: columns only) and of the column
};
constexpr PlaneLen kPlaneLens[] = {{32, 16, 8},  {36, 6, 6},   {40, 10, 20}, {48, 12, 12}, {50, 5, 10},  {64, 8, 8},
                                   {72, 6, 12},  {80, 20, 20}, {96, 12, 24}, {100, 10, 10}, {108, 6, 6}, {128, 8, 16},
                                   {160, 0, 20}};
constexpr int kNumPlaneLens = sizeof(kPlaneLens) / sizeof(kPlaneLens[0]);
constexpr int plane_index(int n) {
  for (int k = 0; k < kNumPlaneLens; ++k)
    if (kPlaneLens[k].n == n) return k;
  return -1;
}

constexpr int plane_row_pitch(int nz) { return (nz / 2 + 1) + ((nz / 2) >> 4) + 1; }

// LDS bytes of a plane.
constexpr size_t plane_lds(int nz, int ny, int f32) {
  const int rows = ny * plane_row_pitch(nz), cols = ny * (nz / 2 + 1) + ((ny - 1) >> kColPadShift) + 1;
  return (size_t)(rows > cols ? rows : cols) * (f32 ? 8 : 16);
}

// Threads of a plane's workgroup (0: none compiled in, or too large: more than
// 768 threads leave a lane 128 registers, too few for columns of 20 and 24
// values: 512x96x108 was 0.8 times as fast as its passes).
constexpr int plane_threads(int nz, int ny) {
  const int a = plane_index(nz), b = plane_index(ny);
  if (a < 0 || b < 0 || !kPlaneLens[a].ez) return 0;
  const int rows = ny * (nz / 2 / kPlaneLens[a].ez), cols = (nz / 2 + 1) * (ny / kPlaneLens[b].ey);
  const int t = ((rows > cols ? rows : cols) + 63) / 64 * 64;
  return t > (kPlaneLens[b].ey >= 20 ? 768 : 1024) || plane_lds(nz, ny, 0) > 160 * 1024 ? 0 : t;
}

// a.plane set: a.tw the row twiddles, a.tw2 the column ones, one workgroup per
// plane.
hipError_t plane_r2c(int f32, int in_f32, const Launch& l, const RowArgs& a);
hipError_t plane_c2r(int f32, int out_kind, int epi, const Launch& l, const RowArgs& a);

}  // namespace ff
