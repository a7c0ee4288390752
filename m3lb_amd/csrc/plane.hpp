// plane.hpp -- several D2Q9 esoteric-pull steps in one launch.
//
// A block owns a core of the plane and works on a region that is H nodes wider
// on every side.  It reads the region once, takes T steps in LDS, and writes
// the core's result to a second population array, so that memory is read and
// written once per T steps and T steps cost one launch.  The nodes of the
// margin are updated by every block whose region holds them (the same
// arithmetic on the same inputs, so the same bits); the margin shrinks by one
// node per step.
//
// The LDS image holds the population slots exactly as the array does
// (EsotericPull.hpp:12-17): at each parity a slot belongs to one node, which
// reads and writes it, so a step in LDS updates in place with one barrier.
// Step 0 reads its nodes' slots from the source array and leaves them, crossed,
// in LDS; the last step reads LDS and stores to the other array.  A node that
// does not move (Solid, Excluded, the halo) carries its slots across: it copies
// them into LDS at step 0 and from LDS to the other array at the last step.
// Slots that no fluid node touches at either parity are equal in both arrays
// from the start (the host copies the array once after every seeding or change
// of the flags).
//
// Regularised walls (straight walls and corners whose stencils lie on walls)
// are updated with the fluid nodes.  A corner's density is extrapolated from
// the closure densities of two nodes along an axis, so it sees two nodes
// further than a fluid node does: with walls the margin is T + 2.
#pragma once

#include "kernels.hpp"
#include "wrap.hpp"

namespace m3lb {

struct PlaneArgs {
  StepArgs a;
  void* out;      // the other population array
  int ntx, nty;   // blocks along x and y
  int core_x, more_x, core_y, more_y;  // sx / ntx, sx % ntx, sy / nty, sy % nty
  int steps;      // T, even
  int margin;     // H: T, with walls T + 2
  WallArgs w;     // WALLS only
};

// RX x RY nodes per region; NF threads take the fluid cells and, with walls, two
// more waves the straight wall cells and the corners.
template <int RX_, int RY_, int NF_, bool WAVES_ = false>
struct PlaneShape {
  static constexpr int RX = RX_, RY = RY_, NF = NF_, NW = WAVES_ ? 128 : 0, NT = NF + NW;
};

// What a block keeps of its wall cells, so that a step reads no tables: the
// velocity, code (bits 0..3), corner axis (4..7) and unknown directions (8..);
// for corners this step's extrapolated density and the gradient sums
// (d_x u, d_y v, d_x v + d_y u) of the finite-difference stress.  list: the
// wall cells, straight ones from the front, corners from the back.  A step's
// wall code is a long chain, bound by the rate at which one wave issues it (800
// instructions for a straight cell): one wave runs it for all straight cells of
// the region and another one for the corners, beside the waves of the fluid
// cells.  Cavity 129^2 FP64 CM, us per step: 18.4 one launch at a time; 9.3 with
// the wall cells updated with the rows (every wave then runs the chain for one
// or two lanes); 5.8 with waves that take fluid cells as well; 4.0 with waves of
// their own and the closure sums out of scratch memory; 3.7 with the corners'
// densities beside the other cells' work.
template <class R, int N, bool WALLS>
struct PlaneWalls {
  R u[3][N];
  R rho[N], grad[3][N];
  uint32_t info[N];
  uint16_t list[N];
  int straight, corners;
};
template <class R, int N>
struct PlaneWalls<R, N, false> {};

template <class K, int P>
__device__ __forceinline__ void lds_load(const typename K::T* s, int np, int c, int rx,
                                         const float* inv, typename K::R* f) {
  using C = typename K::C;
  constexpr int Q = K::Q;
  f[0] = C::dec(s[c], inv[0]);
  sfor<(Q - 1) / 2>([&](auto Pr) {
    constexpr int i = 2 * Pr + 1;
    const int nb = c + cvel<Q>(i, 1) * rx + cvel<Q>(i, 0);
    constexpr int l = P == 0 ? i : i + 1, r = P == 0 ? i + 1 : i;
    f[i] = C::dec(s[l * np + c], inv[l]);
    f[i + 1] = C::dec(s[r * np + nb], inv[r]);
  });
}

template <class K, int P>
__device__ __forceinline__ void lds_store(typename K::T* s, int np, int c, int rx,
                                          const float* sc, const typename K::R* f) {
  using C = typename K::C;
  constexpr int Q = K::Q;
  s[c] = C::enc(f[0], sc[0]);
  sfor<(Q - 1) / 2>([&](auto Pr) {
    constexpr int i = 2 * Pr + 1;
    const int nb = c + cvel<Q>(i, 1) * rx + cvel<Q>(i, 0);
    constexpr int l = P == 0 ? i : i + 1, r = P == 0 ? i + 1 : i;
    s[r * np + nb] = C::enc(f[i], sc[r]);
    s[l * np + c] = C::enc(f[i + 1], sc[l]);
  });
}

// A wall node's incoming set rebuilt (k_walls without the neighbour reads):
// rw is a corner's density, grad its gradient sums.
template <class K>
__device__ __forceinline__ void plane_wall(typename K::R* f, const WallArgs& w, uint32_t info,
                                           const typename K::R* uw, typename K::R rw,
                                           const typename K::R* grad,
                                           const Params<typename K::R>& p) {
  using R = typename K::R;
  constexpr int Q = K::Q;
  const int code = int(info & 15u);
  if constexpr (K::SHIFTED) sfor<Q>([&](auto I) { f[int(I)] += weight<K>(int(I)); });
  R Fv[3] = {R(0), R(0), R(0)};
  if constexpr (K::FORCE) {
    if (w.force_bc) { Fv[0] = p.F[0]; Fv[1] = p.F[1]; Fv[2] = p.F[2]; }
  }
  if (code != kNrmCorner) {
    int nrm[3];
    normal_of(code, nrm);
    rw = bc_density<K>(f, nrm, uw);
  }
  if (w.fd_corners && code == kNrmCorner) {
    R Pi[6] = {R(0), R(0), R(0), R(0), R(0), R(0)};
    const R kf = -R(2) * (R(1) / R(3)) * rw / p.omega;
    Pi[0] = kf * grad[0];
    Pi[1] = kf * grad[1];
    Pi[3] = kf * R(0.5) * grad[2];
    bc_apply_with_stress<K>(f, rw, uw, Pi);
  } else {
    bc_apply<K>(f, rw, uw, info >> 8, Fv);
  }
  if constexpr (K::SHIFTED) sfor<Q>([&](auto I) { f[int(I)] -= weight<K>(int(I)); });
}

// GEOM: some node of the padded box is not Fluid.  WALLS (implies GEOM):
// regularised walls.  The first step is an even one (parity 0), T is even.
template <class K, class S, bool GEOM, bool WALLS>
__global__ void __launch_bounds__(S::NT) k_plane(PlaneArgs pa) {
  using R = typename K::R;
  using T = typename K::T;
  using C = typename K::C;
  constexpr int Q = K::Q, RX = S::RX, RY = S::RY, NP = RX * RY;
  constexpr int kPerThread = NP / S::NF;
  static_assert(NP % S::NF == 0 && S::NF % 64 == 0, "whole rounds of threads and waves");
  static_assert(!WALLS || S::NW == 128, "walls have two waves of their own");
  __shared__ T s[Q * NP];
  __shared__ PlaneWalls<R, NP, WALLS> pw;
  const StepArgs& a = pa.a;
  const Dom& d = a.d;
  const int H = pa.margin;
  const unsigned tile = tile_of(blockIdx.x, gridDim.x, a.remap);
  const int ity = int(tile / unsigned(pa.ntx)), itx = int(tile - unsigned(ity) * unsigned(pa.ntx));
  // cores of core_x or core_x + 1 nodes, the first more_x of them the larger
  const int X0 = itx * pa.core_x + min(itx, pa.more_x), X1 = X0 + pa.core_x + (itx < pa.more_x);
  const int Y0 = ity * pa.core_y + min(ity, pa.more_y), Y1 = Y0 + pa.core_y + (ity < pa.more_y);
  const Params<R> p = params_of<K>(a);
  const T* A = static_cast<const T*>(a.f);
  T* B = static_cast<T*>(pa.out);
  if constexpr (WALLS) {
    if (threadIdx.x == 0) pw.straight = pw.corners = 0;
    __syncthreads();
  }

  // Padded coordinates of region cell c; false outside the box.
  auto cell_xy = [&](int c, int& X, int& Y) -> bool {
    X = X0 - H + c % RX;
    Y = Y0 - H + c / RX;
    if (X < 0 || X >= d.sx) {
      if (!d.px) return false;
      X = wrapped(X, d.sx);
    }
    if (Y < 0 || Y >= d.sy) {
      if (!d.py) return false;
      Y = wrapped(Y, d.sy);
    }
    return true;
  };
  // Whether cell c lies within `k` nodes of the core.
  auto within = [&](int c, int k) -> bool {
    const int x = c % RX - H, y = c / RX - H;
    return x >= -k && x < X1 - X0 + k && y >= -k && y < Y1 - Y0 + k;
  };
  auto inside = [&](int X, int Y) -> bool {
    return (d.px || (X >= 0 && X < d.sx)) && (d.py || (Y >= 0 && Y < d.sy));
  };
  // density of the corner at cell c from the incoming sets of the two nodes
  // along its axis (k_wall_density and k_corner_density)
  auto corner_rho = [&](uint32_t info, auto&& closure) -> R {
    const int e = int(info >> 4 & 15u);
    if (e == 0) return R(1);
    const int ax = (e - 1) >> 1, sg = (e & 1) ? 1 : -1;
    const R r1 = closure(sg, ax), r2 = closure(2 * sg, ax);
    return R(2) * r1 - r2;
  };
  auto density_of = [&](R* f, int code, const R* u) -> R {
    if constexpr (K::SHIFTED) sfor<Q>([&](auto I) { f[int(I)] += weight<K>(int(I)); });
    int nrm[3];
    normal_of(code, nrm);
    return bc_density<K>(f, nrm, u);
  };

  // ---- step 0: source array to LDS ----
  const bool fluid_wave = S::NW == 0 || int(threadIdx.x) < S::NF;
  uint32_t moves = 0;  // bit j: this thread's j-th cell is fluid
#pragma unroll 1
  for (int j = 0; fluid_wave && j < kPerThread; ++j) {
    const int c = int(threadIdx.x) + j * S::NF;
    int X, Y;
    if (!within(c, H - 1) || !cell_xy(c, X, Y)) continue;
    const int n = Y * d.sx + X, x = X - d.hx, y = Y - d.hy;
    const Offs o = offsets(d, x, y, 0);
    R f[Q];
    if constexpr (!GEOM) {
      load_node<K, 0, false>(A, a.stride, unsigned(n), o, a.inv_scale, f);
    } else {
      // the flag and the node's slots are read together; a node that does
      // not move leaves its slots in LDS as they are
      const uint8_t fl = a.flags[n];
      T raw[Q];
      raw[0] = A[unsigned(n)];
      sfor<(Q - 1) / 2>([&](auto Pr) {
        constexpr int i = 2 * Pr + 1;
        raw[i] = A[uint64_t(i) * a.stride + unsigned(n)];
        // a halo node's slot outside the box: any value, nothing reads it
        const int m = inside(X + cvel<Q>(i, 0), Y + cvel<Q>(i, 1)) ? n + nb_off<Q, i>(o) : n;
        raw[i + 1] = A[uint64_t(i + 1) * a.stride + unsigned(m)];
      });
      if (WALLS && fl == M3LB_REGWALL) {
        if constexpr (WALLS) {
          const int code = pa.w.bc_nrm[n];
          R uw[3];
          wall_velocity<K>(pa.w.wtab, pa.w.bc_tag, pa.w.wall_un, pa.w.un_scale, d.np, unsigned(n), uw);
          for (int k = 0; k < 3; ++k) pw.u[k][c] = uw[k];
          pw.info[c] = uint32_t(code) | uint32_t(pa.w.bc_ext[n]) << 4 | pa.w.bc_unk[n] << 8;
          if (code == kNrmCorner) {
            pw.list[NP - 1 - atomicAdd(&pw.corners, 1)] = uint16_t(c);
            R grad[3][3];
            corner_gradient<K>(d, x, y, 0, uw,
                               [&](int, int cx, int cy, int cz, R out[3]) {
                                 table_velocity<K>(pa.w.wtab, pa.w.bc_tag,
                                                   interior_id(d, cx, cy, cz), out);
                               },
                               grad);
            pw.grad[0][c] = grad[0][0];
            pw.grad[1][c] = grad[1][1];
            pw.grad[2][c] = grad[0][1] + grad[1][0];
            pw.rho[c] = corner_rho(pw.info[c], [&](int steps, int ax) -> R {
              const int xm = x + (ax == 0 ? steps : 0), ym = y + (ax == 0 ? 0 : steps);
              const unsigned m = interior_id(d, xm, ym, 0);
              R g[Q], u[3];
              load_node<K, 0, false>(A, a.stride, m, offsets(d, xm, ym, 0), a.inv_scale, g);
              wall_velocity<K>(pa.w.wtab, pa.w.bc_tag, pa.w.wall_un, pa.w.un_scale, d.np, m, u);
              return density_of(g, pa.w.bc_nrm[m], u);
            });
          }
          if (code != kNrmCorner) pw.list[atomicAdd(&pw.straight, 1)] = uint16_t(c);
        }
        continue;  // updated below, from the list
      }
      if (fl != M3LB_FLUID) {
        s[c] = raw[0];
        sfor<(Q - 1) / 2>([&](auto Pr) {
          constexpr int i = 2 * Pr + 1;
          s[i * NP + c] = raw[i];
          s[(i + 1) * NP + c + cvel<Q>(i, 1) * RX + cvel<Q>(i, 0)] = raw[i + 1];
        });
        continue;
      }
      sfor<Q>([&](auto I) { f[int(I)] = C::dec(raw[int(I)], a.inv_scale[int(I)]); });
    }
    moves |= 1u << j;
    (void)collide_fused<K>(f, p);
    lds_store<K, 0>(s, NP, c, RX, a.scale, f);
  }
  __syncthreads();
  int nstraight = 0, ncorner = 0;
  const int wall_lane = int(threadIdx.x) - S::NF;  // negative in the fluid waves
  if constexpr (WALLS) {
    nstraight = pw.straight;
    ncorner = pw.corners;
  }
  // The wall cells within k of the core at step t: one copy of the code for
  // every step (parity and ends at run time; with a copy for each the kernel
  // outgrows the instruction cache).  Opposite directions share their scale.
  auto wall_cells = [&](int t, int k) {
    if constexpr (WALLS) {
      if (fluid_wave) return;
      const int pp = t & 1;
      const bool corner = wall_lane >= 64;
#pragma unroll 1
      for (int w = wall_lane & 63; w < (corner ? ncorner : nstraight); w += 64) {
        const int c = pw.list[corner ? NP - 1 - w : w];
        if (!within(c, k)) continue;
        R f[Q];
        int X, Y;
        (void)cell_xy(c, X, Y);
        const unsigned n = unsigned(Y * d.sx + X);
        const Offs o = offsets(d, X - d.hx, Y - d.hy, 0);
        if (t == 0) {
          load_node<K, 0, false>(A, a.stride, n, o, a.inv_scale, f);
        } else {
          f[0] = C::dec(s[c], a.inv_scale[0]);
          sfor<(Q - 1) / 2>([&](auto Pr) {
            constexpr int i = 2 * Pr + 1;
            f[i] = C::dec(s[(i + pp) * NP + c], a.inv_scale[i]);
            f[i + 1] = C::dec(s[(i + 1 - pp) * NP + c + cvel<Q>(i, 1) * RX + cvel<Q>(i, 0)],
                              a.inv_scale[i]);
          });
        }
        const R uw[3] = {pw.u[0][c], pw.u[1][c], pw.u[2][c]};
        const R grad[3] = {pw.grad[0][c], pw.grad[1][c], pw.grad[2][c]};
        plane_wall<K>(f, pa.w, pw.info[c], uw, corner ? pw.rho[c] : R(0), grad, p);
        (void)collide_fused<K>(f, p);
        if (t == pa.steps - 1) {
          store_node<K, 1, false>(B, a.stride, n, o, a.scale, f);
        } else {
          s[c] = C::enc(f[0], a.scale[0]);
          sfor<(Q - 1) / 2>([&](auto Pr) {
            constexpr int i = 2 * Pr + 1;
            s[(i + 1 - pp) * NP + c + cvel<Q>(i, 1) * RX + cvel<Q>(i, 0)] = C::enc(f[i], a.scale[i]);
            s[(i + pp) * NP + c] = C::enc(f[i + 1], a.scale[i]);
          });
        }
      }
    }
  };

  // corners first: their stencils read slots that other nodes update.  Two
  // lanes take the two closure densities of a corner's stencil.  Up to 32
  // corners are read before the barrier and worked on after it, beside the
  // straight and the fluid cells.
  auto corners = [&](int t, int k) {
    if constexpr (WALLS) {
      if (ncorner == 0) return;
      const int pp = t & 1;
      R g[Q];
      int c = 0, cm = 0, e = 0;
      auto read = [&](int v) {  // every lane of the wave stays for the exchange below
        c = pw.list[NP - 1 - (v < ncorner ? v : 0)];
        e = int(pw.info[c] >> 4 & 15u);
        const int reach = ((e & 1) ? 1 : -1) * (1 + (wall_lane & 1));
        cm = c + (e == 0 ? 0 : reach * ((e - 1) >> 1 == 0 ? 1 : RX));
        // beyond the region: a corner that no core node sees in T steps
        if (cm < RX + 1 || cm >= NP - RX - 1) cm = c;
        g[0] = C::dec(s[cm], a.inv_scale[0]);
        sfor<(Q - 1) / 2>([&](auto Pr) {
          constexpr int i = 2 * Pr + 1;
          g[i] = C::dec(s[(i + pp) * NP + cm], a.inv_scale[i]);
          g[i + 1] = C::dec(s[(i + 1 - pp) * NP + cm + cvel<Q>(i, 1) * RX + cvel<Q>(i, 0)],
                            a.inv_scale[i]);
        });
      };
      auto finish = [&](int v) {
        const R u[3] = {pw.u[0][cm], pw.u[1][cm], pw.u[2][cm]};
        const R r1 = density_of(g, int(pw.info[cm] & 15u), u);
        const R r2 = __shfl_xor(r1, 1);
        if (!(wall_lane & 1) && v < ncorner && within(c, k)) {
          const R rho = e != 0 ? R(2) * r1 - r2 : R(1);
          pw.rho[c] = rho;
          if (t == pa.steps - 1) {
            int X, Y;
            (void)cell_xy(c, X, Y);
            static_cast<R*>(pa.w.bc_rho)[Y * d.sx + X] = rho;
          }
        }
      };
      const bool mine = wall_lane >= 64;
      const int v = (wall_lane & 63) >> 1;
      if (mine) {
        read(v);
        if (ncorner > 32) {
          finish(v);
#pragma unroll 1
          for (int v0 = 32; v0 < ncorner; v0 += 32) {
            read(v0 + v);
            finish(v0 + v);
          }
        }
      }
      __syncthreads();
      if (mine && ncorner <= 32) {
        finish(v);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // read by this wave's lanes
        __builtin_amdgcn_wave_barrier();
      }
    }
  };
  auto fluid_cells = [&](auto PP, int k) {
#pragma unroll 1
    for (int j = 0; j < kPerThread; ++j) {
      const int c = int(threadIdx.x) + j * S::NF;
      if (!(moves >> j & 1u) || !within(c, k)) continue;
      R f[Q];
      lds_load<K, int(PP)>(s, NP, c, RX, a.inv_scale, f);
      (void)collide_fused<K>(f, p);
      lds_store<K, int(PP)>(s, NP, c, RX, a.scale, f);
    }
  };
  if constexpr (WALLS) {
    wall_cells(0, H - 1);
    __syncthreads();
#pragma unroll 1
    for (int t = 1; t < pa.steps; ++t) {
      const bool last = t == pa.steps - 1;
      const int k = last ? 0 : H - 1 - t;
      corners(t, k);
      wall_cells(t, k);
      if (last) break;
      if (t & 1) fluid_cells(std::integral_constant<int, 1>{}, k);
      else fluid_cells(std::integral_constant<int, 0>{}, k);
      __syncthreads();
    }
  } else {
#pragma unroll 1
    for (int t = 1; t + 1 < pa.steps; t += 2) {
      fluid_cells(std::integral_constant<int, 1>{}, H - 1 - t);
      __syncthreads();
      fluid_cells(std::integral_constant<int, 0>{}, H - 2 - t);
      __syncthreads();
    }
  }

  // ---- last step: LDS to the other array ----
  auto put = [&](int c, const R* f) {
    int X, Y;
    (void)cell_xy(c, X, Y);
    store_node<K, 1, false>(B, a.stride, unsigned(Y * d.sx + X),
                            offsets(d, X - d.hx, Y - d.hy, 0), a.scale, f);
  };
#pragma unroll 1
  for (int j = 0; fluid_wave && j < kPerThread; ++j) {
    const int c = int(threadIdx.x) + j * S::NF;
    if (!within(c, 0)) continue;
    if (moves >> j & 1u) {
      R f[Q];
      lds_load<K, 1>(s, NP, c, RX, a.inv_scale, f);
      (void)collide_fused<K>(f, p);
      put(c, f);
    } else if constexpr (GEOM) {
      // a node that does not move: its slots as they are, but for those whose
      // owner at even steps lies outside the box (no node inside writes them:
      // LDS does not hold them, both arrays do)
      int X, Y;
      (void)cell_xy(c, X, Y);
      const int n = Y * d.sx + X;
      if (WALLS && a.flags[n] == M3LB_REGWALL) continue;
      const Offs o = offsets(d, X - d.hx, Y - d.hy, 0);
      B[unsigned(n)] = s[c];
      sfor<(Q - 1) / 2>([&](auto Pr) {
        constexpr int i = 2 * Pr + 1;
        constexpr int cx = cvel<Q>(i, 0), cy = cvel<Q>(i, 1);
        if (inside(X - cx, Y - cy)) B[uint64_t(i + 1) * a.stride + unsigned(n)] = s[(i + 1) * NP + c];
        if (inside(X + cx, Y + cy))
          B[uint64_t(i) * a.stride + unsigned(n + nb_off<Q, i>(o))] = s[i * NP + c + cy * RX + cx];
      });
    }
  }
}

}  // namespace m3lb
