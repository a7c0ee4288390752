// step_plan.hpp -- which pass takes the steps of a box, and in what blocks: the
// rules of the D2Q9 passes (plane.hpp) and of the D3Q27 passes through LDS
// (march.hpp).  Plain C++ without HIP, so that the CPU tests can check them
// (tests/cpp/step_plan_test.cpp).
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

namespace m3lb {

// ---- several D2Q9 steps per launch ----
// Regions of the plane kernel and what moves in the box.
enum PlaneRegion { kPlaneSquare = 0, kPlaneWide = 1, kPlaneSmall = 2 };
enum PlaneNodes { kPlaneFluid = 0, kPlaneGeom = 1, kPlaneWalls = 2 };

struct RegionSize {
  int x, y;
};
constexpr RegionSize plane_region(int shape, int nodes) {
  return nodes == kPlaneWalls    ? RegionSize{32, 28}
         : shape == kPlaneSmall  ? RegionSize{24, 24}
         : shape == kPlaneWide   ? RegionSize{64, 32}
                                 : RegionSize{32, 32};
}

// With walls a corner sees two nodes further than a fluid node does.
constexpr int plane_margin(int steps, int nodes) { return steps + (nodes == kPlaneWalls ? 2 : 0); }

// Blocks of a pass of `steps` steps along each axis.
struct PlaneGrid {
  int ntx, nty;
};
inline PlaneGrid plane_grid(int sx, int sy, int steps, int shape, int nodes) {
  const RegionSize r = plane_region(shape, nodes);
  const int h = plane_margin(steps, nodes), cx = r.x - 2 * h, cy = r.y - 2 * h;
  return {(sx + cx - 1) / cx, (sy + cy - 1) / cy};
}

struct PlaneBox {
  int sx, sy;      // padded extents
  int nodes;       // PlaneNodes
  int elem_bytes;  // per stored population
  bool e2m13;
  uint64_t bytes;  // of the population array
  int cus;
  int nwall;       // regularised wall nodes, and whether corners are among them
  bool corners;
  bool force;
};

// Cells that a pass computes per node of the box and step: the margins, and what of
// the regions' cores the box leaves empty.
inline double plane_work(const PlaneBox& b, int steps, int shape) {
  const PlaneGrid g = plane_grid(b.sx, b.sy, steps, shape, b.nodes);
  const RegionSize r = plane_region(shape, b.nodes);
  return double(g.ntx) * g.nty * r.x * r.y / (double(b.sx) * b.sy);
}

// Planes of more than four rounds of blocks (fewer: a one-launch step is bound by its
// launch; 20000 x 4 FP64, 3.3 rounds, 1.46 times its speed), a few rows or columns
// wide: a region then holds little of the box.  The one-launch step has lanes idle too in rows shorter
// than a wave, so the work counts in proportion there.  Speed against one launch
// per step, CM, work in brackets, 200,000 and 262,144 nodes long: 8-byte rows (4 steps)
// 2 high (21) 0.46, 4 (11) 0.75-0.93, 8 (5.3) 0.99-1.24, 10 (4.3) 1.14-1.35, 18 (2.4) 1.3-
// 1.8, columns of any width (1.7 or less) 1.5-2.6; 4-byte (6 steps) rows 2 high
// 0.89, 4 (9.8) 0.81-0.96, 6 (6.6) 1.17, 8 (4.9) 1.33-1.5, columns up to 22 wide 0.8-0.97,
// 26 1.04, 30 1.18, 44 2.2; FP16 rows 1 high 0.49, 2 (20) 0.6-0.93, 8 (4.9) 0.96-1.28, 24
// (3.3) 0.89, 14 (2.8) 1.11-1.35, columns 60 wide (3.2) 0.71, 44 (1.6) 1.23; E2M13 rows 2
// high 0.71, 8 0.95, 14 1.04.  Two steps bring less: 8-byte rows 10 high (3.7) 0.89-0.96,
// 14 (2.6) 1.01-1.08; 4-byte rows 4 high (8.5) 0.68-0.87, 8 (4.3) 1.27, columns 36 wide 0.87-
// 1.02, 44 1.5; FP16 rows 10 high (2.9) 0.93, 14 (2.1) 1.05.
inline bool plane_fits(const PlaneBox& b, int steps, int shape) {
  const bool two = steps == 2;
  const PlaneGrid g = plane_grid(b.sx, b.sy, steps, shape, b.nodes);
  if (int64_t(g.ntx) * g.nty <= (two ? 2 : 4) * b.cus) return true;
  const double most = b.elem_bytes == 8   ? (two ? 3.0 : 5.0)
                      : b.elem_bytes == 4 ? (two ? 4.3 : 6.6)
                                          : (two ? 2.2 : 2.9);
  if (b.elem_bytes == 4 && b.sx < (two ? 40 : 26)) return false;
  return plane_work(b, steps, shape) * std::min(1.0, b.sx / 64.0) <= most;
}

// us per step of a walled plane, one launch per step (two launches, with corners four) and
// in passes of more than one round of blocks, and so the sizes up to which the passes
// pay.  Within a round they always do.  Speed of the pass of 4 steps
// against one launch per step, CM; channels (two straight walls): 500^2 FP64 1.15, FP32
// 1.05, FP16 1.07, E2M13 0.87; 800^2 1.12, 0.81, 0.84, 0.70; 1600^2 0.85, 0.66, 0.44, 0.41;
// 20000 x 40 0.80, 0.59, 0.47, 0.48; cavities: 500^2 1.99, 2.13, 2.03, 1.78; 800^2 1.63, 1.40,
// 1.30, 1.13; 1100^2 1.26, 1.11, 0.93, 0.82; 2050^2 1.07, 0.69, 0.53, 0.46; 4100^2 FP64
// 1.21.  A Guo force costs the FP64 pass most (800^2 channel, BGK: 23.4 us against 19.2).
// The model names the faster way for 688 of 714 measured cases (five storage types, 16
// to 8000 nodes wide, 2 and 4 steps); the four others that it gives to the passes are
// at most 4% slower there.
inline double walled_one(const PlaneBox& b) {
  const bool beyond = b.bytes > (256u << 20);  // the last-level cache
  const double ps = b.elem_bytes == 8   ? (!beyond ? 21.3 : b.bytes > (512u << 20) ? 30.0 : 26.0)
                    : b.elem_bytes == 4 ? (beyond ? 15.5 : 10.8)
                    : b.e2m13           ? (beyond ? 8.7 : 7.6)
                                        : (beyond ? 8.3 : 7.2);
  const double start = b.elem_bytes == 8 ? 7.3 : b.elem_bytes == 4 ? 6.3 : 8.0;
  return start + (b.corners ? 11.5 : 0.0) + double(b.sx) * b.sy * ps * 1e-6;
}
inline double walled_pass(const PlaneBox& b, int steps) {
  const PlaneGrid g = plane_grid(b.sx, b.sy, steps, kPlaneSquare, kPlaneWalls);
  const double blocks = double(g.ntx) * g.nty;
  const bool two = steps == 2;
  const bool beyond = b.bytes > (256u << 20);
  const double round = b.elem_bytes == 8   ? (two ? (beyond ? 7.2 : 6.8) : b.force ? 10.4 : 8.8)
                       : b.elem_bytes == 4 ? (two ? 4.9 : 6.7)
                       : b.e2m13           ? (two ? 6.3 : 8.9)
                                           : (two ? 5.6 : 7.7);
  // a block with walls takes longer: its share, at 20 wall nodes a block
  const double walled = std::min(1.0, b.nwall / (20.0 * blocks));
  return (6.0 + std::ceil(blocks / b.cus) * (round + (two ? 2.5 : 3.4) * walled)) / steps;
}

struct PlanePlan {
  int steps = 0;  // of the next launch, even; 0: one launch per step
  int shape = 0, nodes = 0;
};

// Region and steps per launch.  While the blocks of a region fit the chip in
// one round, a launch lasts as long as one block: the most steps that still
// fit, in the smallest region (fewer nodes of margin per wave).  us per step,
// FP64 BGK / FP32 CM:
//   128^2  24 x 24 regions, 8 steps 1.17 / 1.05; 32 x 32, 8 1.34 / 1.21
//   192^2  24 x 24, 6 1.42 / 1.24;  32 x 32, 8 1.50 / 1.32
//   256^2  32 x 32, 8 1.67 / 1.41;  6 steps 1.80 / 1.56
//   320^2  32 x 32, 6 1.95 / 1.63;  8 steps (two rounds) 2.76 / 2.16
//   384^2  32 x 32, 4 2.41 / 2.09;  6 steps 2.98 / 2.47, 8 3.67 / 2.95
// with walls (cavity FP64 CM): 129^2 8 steps 3.7, 6 3.8, 4 4.5; 257^2 4.7, 5.6, 7.8.
// Larger planes are bound by traffic and by the work on margins: 4-byte and
// 2-byte populations take 64 x 32 regions and 6 steps (1024^2 FP32 7.9 us per
// step, 8.0 at 4 steps, 9.3 with 32 x 32 regions, 11.1 one launch per step;
// 4096^2 93, 96, 125 and 189), 8-byte ones 32 x 32 and 4 (1024^2 12.0 us, 12.2
// at 6, 13.5 with 64 x 32 regions, 23.6 one launch per step; 4096^2 169 and 426).
// left: the steps that are left for passes.  A pass of two steps has cores of
// 60 x 28 nodes in 64 x 32 regions: up to two rounds of such blocks the 32 x 32
// regions, with twice the blocks, keep more of the chip at work (speed against
// one launch per step, 64 x 32 / 32 x 32: 400x390 FP32 0.92 / 1.28, with geometry 0.66 /
// 1.16, 520x510 0.79 / 1.11, 700x690 0.98 / 1.18; 1024x1014 1.12 / 1.11, FP16 1.30 / 1.06),
// and E2M13 loses in either (520x510 0.97 / 0.99, with geometry 0.68 / 0.90, 700x690
// 0.86 / 0.94, 1024x1014 0.97 / 0.81).
inline PlanePlan plane_rule(const PlaneBox& b, int left) {
  PlanePlan p;
  p.nodes = b.nodes;
  const bool walls = b.nodes == kPlaneWalls;
  const int steps_shapes[5][2] = {{8, kPlaneSmall},  {6, kPlaneSmall}, {8, kPlaneSquare},
                                  {6, kPlaneSquare}, {4, kPlaneSquare}};
  for (const auto& c : steps_shapes) {
    if (walls && c[1] == kPlaneSmall) continue;
    const int steps = std::min(c[0], left & ~1);
    const PlaneGrid g = plane_grid(b.sx, b.sy, steps, c[1], b.nodes);
    if (int64_t(g.ntx) * g.nty > b.cus) continue;
    p.steps = steps;
    p.shape = c[1];
    return p;
  }
  p.shape = kPlaneSquare;
  if (walls || b.elem_bytes == 8) {
    p.steps = std::min(4, left & ~1);
  } else {
    p.shape = kPlaneWide;
    p.steps = std::min(6, left & ~1);
    if (p.steps == 2) {
      const PlaneGrid g = plane_grid(b.sx, b.sy, 2, kPlaneWide, b.nodes);
      if (int64_t(g.ntx) * g.nty <= 2 * b.cus) p.shape = kPlaneSquare;
      if (b.e2m13) p.steps = 0;
    }
    // 2-byte populations beyond the caches' reach of one XCD gain little (D2Q9
    // CM 2048^2, us per step: FP16 27.2 against 27.3, BF16 25.7 / 28.1, I16
    // 24.7 / 28.5), and E2M13 (32.0 / 30.6, its codec runs on the margins too)
    // and boxes with geometry (FP16 28.2 / 27.6, E2M13 34.0 / 29.4) lose
    if (b.elem_bytes == 2 && b.bytes > (32u << 20) && (b.e2m13 || b.nodes == kPlaneGeom))
      p.steps = 0;
  }
  if (walls ? walled_pass(b, p.steps) >= 0.97 * walled_one(b)
            : p.steps && !plane_fits(b, p.steps, p.shape))
    p.steps = 0;
  return p;
}

// ---- two D3Q27 steps per pass through LDS (march.hpp) ----
// Core of a block along x and y.
constexpr RegionSize march_core(int elem_bytes) {
  return elem_bytes == 8 ? RegionSize{32, 12} : RegionSize{64, 13};
}

struct MarchBox {
  int sx, sy, sz;  // padded extents
  int elem_bytes;
  int cus;
  bool geom;       // some node of the padded box is not Fluid
};

struct MarchPlan {
  bool on = false;
  int ntx = 0, nty = 0, nzc = 0;  // blocks along x, y and z
};

// The runs along z with the least rounds of blocks times planes of one (two planes
// and about half a plane's time of start are extra), none longer than `longest`.
inline double march_runs(const MarchBox& b, int longest, MarchPlan& p) {
  const int64_t cols = int64_t(p.ntx) * p.nty;
  const int first = (b.sz + longest - 1) / longest;
  // 4096 runs are 16 rounds of one column's blocks; a box of more planes than that
  // gains nothing from more, and is not to be searched plane by plane each call
  const int last = int(std::min<int64_t>(b.sz, int64_t(first) + 4095));
  double best = 0;
  for (int k = first; k <= last; ++k) {
    const double cost = double((cols * k + b.cus - 1) / b.cus) * ((b.sz + k - 1) / k + 2.5);
    if (k == first || cost < best) {
      best = cost;
      p.nzc = k;
    }
  }
  return best;
}

// on: the schedule keeps the chip's cells filled.  GLUPS against the pass of pair.hpp,
// 4-byte storage: 0.81 (192^3) 35.5 / 29.6, 0.65 (160^3) 28.3 / 28.9; 8-byte: 0.75
// (150x130x140) 16.1 / 13.0, 0.58 (74x172x118) 12.5 / 9.9.
//
// Blocks of long runs drift apart in z, and with them the lines and margins that
// neighbours share leave the caches before the neighbour comes: it shows where some
// blocks are slower than others (geometry), beyond 120 planes: 11 of 11 FP64 boxes with a
// halo at 0.79-1.02 of the speed of the pass of pair.hpp; with runs of up to 48
// planes 288x320x256 0.86 -> 1.09, 300x280x260 0.80 -> 1.04, 445x213x159 0.96 -> 1.10,
// 188x163x833 0.86 -> 1.03, 576x320x192 FP32 0.90 -> 1.08.  And where rows are no whole
// half lines and the last core of a row is short, in FP32 rows of up to 256 nodes,
// which the pass of pair.hpp takes in one tile: with runs of up to 16 planes 217x414x219 0.87 ->
// 1.01, 147x535x285 0.85 -> 1.08, 156x349x440 0.88 -> 1.06, 100x400x400 0.99 -> 1.10 (runs of
// up to 26 planes did not lose: 194x299x249 1.06, with 16 1.01).
inline MarchPlan march_rule(const MarchBox& b) {
  MarchPlan p;
  const RegionSize core = march_core(b.elem_bytes);
  p.ntx = (b.sx + core.x - 1) / core.x;
  p.nty = (b.sy + core.y - 1) / core.y;
  const double best = march_runs(b, b.sz, p);
  const double nodes = double(b.sx) * b.sy * b.sz;
  p.on = nodes / (best * b.cus * core.x * core.y) >= (b.elem_bytes == 8 ? 0.5 : 0.65);
  const int run = (b.sz + p.nzc - 1) / p.nzc;
  if (b.elem_bytes == 4 && b.sx <= 256 && b.sx % 16 != 0 && b.sx < 0.92 * core.x * p.ntx) {
    if (run > 26) march_runs(b, 16, p);
  } else if (b.geom && run > 120) {
    march_runs(b, 48, p);
  }
  return p;
}

}  // namespace m3lb
