// Host checks of step_plan.hpp.  Prints "ok".
#include "../../m3lb_amd/csrc/step_plan.hpp"

#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <string>

using namespace m3lb;

#define REQUIRE(x)                                \
  do {                                            \
    if (!(x)) {                                   \
      std::printf("line %d: %s\n", __LINE__, #x); \
      std::exit(1);                               \
    }                                             \
  } while (0)

namespace {
PlaneBox plane(int sx, int sy, int nodes, int elem_bytes, bool e2m13 = false) {
  PlaneBox b{};
  b.sx = sx;
  b.sy = sy;
  b.nodes = nodes;
  b.elem_bytes = elem_bytes;
  b.e2m13 = e2m13;
  b.bytes = uint64_t(sx) * uint64_t(sy) * 9 * uint64_t(elem_bytes);
  b.cus = 256;
  return b;
}

// Squares: the steps and regions the rule's measurements name.
void squares() {
  const struct {
    int n, elem_bytes, steps, shape;
  } want[] = {{128, 8, 8, kPlaneSmall},  {128, 4, 8, kPlaneSmall},  {192, 8, 6, kPlaneSmall},
              {256, 4, 8, kPlaneSquare}, {320, 8, 6, kPlaneSquare}, {384, 4, 4, kPlaneSquare},
              {1024, 8, 4, kPlaneSquare}, {1024, 4, 6, kPlaneWide}, {1024, 2, 6, kPlaneWide},
              {4096, 4, 6, kPlaneWide}};
  for (const auto& w : want) {
    const PlanePlan p = plane_rule(plane(w.n, w.n, kPlaneFluid, w.elem_bytes), 100);
    REQUIRE(p.steps == w.steps && p.shape == w.shape);
  }
  REQUIRE(plane_rule(plane(2048, 2048, kPlaneFluid, 2, true), 100).steps == 0);
  REQUIRE(plane_rule(plane(2050, 2050, kPlaneGeom, 2), 100).steps == 0);
  REQUIRE(plane_rule(plane(131, 131, kPlaneWalls, 8), 100).steps == 8);
}

// Every plan's cores cover the box, and its region holds a core and its margin.
void covers() {
  for (int nodes : {kPlaneFluid, kPlaneGeom, kPlaneWalls})
    for (int eb : {8, 4, 2})
      for (int sx : {1, 2, 7, 24, 65, 300, 1000, 70000})
        for (int sy : {1, 3, 16, 33, 250, 900}) {
          for (int left = 2; left <= 12; ++left) {
            const PlanePlan p = plane_rule(plane(sx, sy, nodes, eb), left);
            REQUIRE(p.steps % 2 == 0 && p.steps <= left);
            if (!p.steps) continue;
            const PlaneGrid g = plane_grid(sx, sy, p.steps, p.shape, nodes);
            const RegionSize r = plane_region(p.shape, nodes);
            const int h = plane_margin(p.steps, nodes);
            REQUIRE(p.shape != kPlaneWide || eb <= 4);  // no such kernel for 8-byte storage
            REQUIRE(nodes != kPlaneWalls || p.shape == kPlaneSquare);
            REQUIRE(g.ntx >= 1 && g.nty >= 1 && g.ntx <= sx && g.nty <= sy);
            REQUIRE((sx + g.ntx - 1) / g.ntx + 2 * h <= r.x);
            REQUIRE((sy + g.nty - 1) / g.nty + 2 * h <= r.y);
          }
        }
}

// Planes a few nodes thin and longer than one round of blocks: where a region holds
// too little of the box, one launch per step.
void thin() {
  const struct {
    int sx, sy, elem_bytes;
    bool on;
  } want[] = {{262144, 1, 8, false}, {262144, 4, 8, false}, {262144, 16, 8, true},
              {4, 262144, 8, true},  {262144, 1, 4, false}, {262144, 4, 4, false},
              {262144, 8, 4, true},  {4, 262144, 4, false}, {16, 262144, 4, false},
              {48, 262144, 4, true}, {262144, 1, 2, false}, {262144, 4, 2, false},
              {262144, 16, 2, true}, {60, 200000, 2, false}, {44, 200000, 2, true},
              {800000000, 1, 4, false},
              // few rounds: bound by launches
              {20000, 4, 8, true},   {2000, 8, 4, true},    {3, 5000, 2, true}};
  for (const auto& w : want) {
    const PlanePlan p = plane_rule(plane(w.sx, w.sy, kPlaneFluid, w.elem_bytes), 100);
    if ((p.steps > 0) != w.on) std::printf("%d x %d, %d bytes\n", w.sx, w.sy, w.elem_bytes);
    REQUIRE((p.steps > 0) == w.on);
  }
}

// Walled planes beyond one round of blocks, the measured faster way.
void walls() {
  const struct {
    int nx, ny;
    bool cavity;
    int elem_bytes;
    bool e2m13, on;
  } want[] = {{500, 500, false, 8, false, true},    {800, 800, false, 8, false, true},
              {1600, 1600, false, 8, false, false}, {20000, 40, false, 8, false, false},
              {500, 500, true, 8, false, true},     {1100, 1100, true, 8, false, true},
              {4100, 4100, true, 8, false, true},   {500, 500, false, 4, false, true},
              {800, 800, false, 4, false, false},   {1600, 1600, false, 4, false, false},
              {800, 800, true, 4, false, true},     {2050, 2050, true, 4, false, false},
              {800, 800, false, 2, false, false},   {800, 800, true, 2, false, true},
              {1100, 1100, true, 2, false, false},  {1600, 1600, true, 2, false, false},
              {500, 500, false, 2, true, false},    {600, 600, true, 2, true, true},
              {1100, 1100, true, 2, true, false},
              // within one round
              {33, 33, true, 2, true, true},        {129, 129, true, 4, false, true},
              {2000, 14, false, 2, true, true}};
  for (const auto& w : want) {
    PlaneBox b = plane(w.nx + (w.cavity ? 2 : 0), w.ny + 2, kPlaneWalls, w.elem_bytes, w.e2m13);
    b.nwall = 2 * w.nx + (w.cavity ? 2 * w.ny - 4 : 0);
    b.corners = w.cavity;
    const PlanePlan p = plane_rule(b, 100);
    if ((p.steps > 0) != w.on) std::printf("%d x %d, %d bytes\n", w.nx, w.ny, w.elem_bytes);
    REQUIRE((p.steps > 0) == w.on);
  }
}

// Passes of two steps: the region by the blocks it gives, and where one launch per
// step is faster.
void two_steps() {
  const struct {
    int n, nodes, elem_bytes;
    bool e2m13;
    int steps, shape;
  } want[] = {{400, kPlaneFluid, 4, false, 2, kPlaneSquare}, {400, kPlaneGeom, 2, false, 2, kPlaneSquare},
              {700, kPlaneGeom, 4, false, 2, kPlaneSquare},  {1024, kPlaneFluid, 4, false, 2, kPlaneWide},
              {1024, kPlaneGeom, 2, false, 2, kPlaneWide},   {400, kPlaneGeom, 2, true, 2, kPlaneSquare},
              {520, kPlaneGeom, 2, true, 0, 0},              {1024, kPlaneFluid, 2, true, 0, 0},
              {1024, kPlaneFluid, 8, false, 2, kPlaneSquare}, {100, kPlaneFluid, 8, false, 2, kPlaneSmall}};
  for (const auto& w : want) {
    for (int left : {2, 3}) {
      const PlanePlan p = plane_rule(plane(w.n, w.n, w.nodes, w.elem_bytes, w.e2m13), left);
      if (p.steps != w.steps) std::printf("%d^2, %d bytes, %d steps\n", w.n, w.elem_bytes, p.steps);
      REQUIRE(p.steps == w.steps && (!w.steps || p.shape == w.shape));
    }
  }
}

void march() {
  const struct {
    int sx, sy, sz, elem_bytes;
    bool on;
  } want[] = {{512, 512, 512, 4, true}, {192, 192, 192, 4, true},  {150, 97, 121, 4, false},
              {150, 130, 140, 8, true}, {300, 280, 260, 4, true}};
  for (const auto& w : want) {
    const MarchPlan p = march_rule({w.sx, w.sy, w.sz, w.elem_bytes, 256, false});
    const RegionSize core = march_core(w.elem_bytes);
    REQUIRE(p.on == w.on);
    REQUIRE(p.nzc >= 1 && p.nzc <= w.sz && p.ntx * core.x >= w.sx);
    REQUIRE((w.sy + p.nty - 1) / p.nty <= core.y);
  }
}
// Longest runs of planes: short where blocks drift apart.
void runs() {
  const struct {
    int sx, sy, sz, elem_bytes;
    bool geom;
    int longest;
  } want[] = {{288, 322, 256, 8, true, 48},   {288, 320, 256, 8, false, 256},
              {576, 322, 192, 4, true, 48},   {512, 512, 512, 4, false, 128},
              {217, 414, 219, 4, false, 16},  {100, 400, 400, 4, false, 16},
              {100, 402, 400, 4, true, 16},   {176, 419, 248, 4, false, 50},
              {192, 192, 192, 4, false, 192}, {256, 258, 256, 4, true, 120}};
  for (const auto& w : want) {
    const MarchPlan p = march_rule({w.sx, w.sy, w.sz, w.elem_bytes, 256, w.geom});
    const int run = (w.sz + p.nzc - 1) / p.nzc;
    if (run > w.longest) std::printf("%d x %d x %d: runs of %d\n", w.sx, w.sy, w.sz, run);
    REQUIRE(p.on && run <= w.longest);
    if (w.longest >= 50 && run <= 16) std::printf("%d x %d x %d: runs of %d\n", w.sx, w.sy, w.sz, run);
    if (w.longest >= 50) REQUIRE(run > 16);  // not shorter than it has to be
  }
}

// The rule runs at each step call: its cost does not grow with the box.
void long_boxes() {
  const auto t0 = std::chrono::steady_clock::now();
  int on = 0;
  for (int k = 0; k < 200; ++k) on += march_rule({4, 4, 10000000 + k, 4, 256, true}).on;
  const double s =
      std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  if (s > 1.0) std::printf("%.3f s for 200 calls\n", s);
  REQUIRE(on == 0 && s <= 1.0);
}
}  // namespace

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "squares") squares();
  else if (what == "covers") covers();
  else if (what == "thin") thin();
  else if (what == "walls") walls();
  else if (what == "two_steps") two_steps();
  else if (what == "march") march();
  else if (what == "runs") runs();
  else if (what == "long_boxes") long_boxes();
  else return 2;
  std::printf("ok\n");
  return 0;
}
