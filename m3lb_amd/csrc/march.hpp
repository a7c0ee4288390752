// march.hpp -- two D3Q27 esoteric-pull steps in one pass, through LDS.
//
// A block owns a column of the box: a core of W x CY nodes in x and y and a run of
// z planes.  It marches along z.  For each plane it takes step t on the core and
// a margin around it (A), keeps what A sends out in LDS, and takes step t+1 on
// the plane before (B), whose inputs are then complete.  B is stored to a second
// population array, so that memory is read and written once for two steps.  The
// margin is taken by each block that needs it, with the same arithmetic on the
// same inputs, so the bits are those of two launches.
//
// LDS holds, by direction d, the value A sends from a cell along c_d: of the last
// plane for c_z = 0 and -1, of the last two for c_z = +1 (B of plane z takes c_z = +1
// from A(z-1), 0 from A(z), -1 from A(z+1)): 36 values per cell.  B reads its
// c_z = +1 and 0 inputs into registers before A overwrites them.  A CU holds one
// block, so the block hides its own latency: the next plane's slots are requested
// before this plane's arithmetic (512^3 FP32 CM 35.2 GLUPS; 32.7 with the request
// between A and B).
//
// What bounds it: cache lines.  A row of a region that starts beside a line reads
// and writes parts of lines that the neighbouring block needs too, and a line
// written in parts by two blocks costs most: cores of 48 nodes (1.5 lines) ran at
// 18.0 GLUPS, 32 at 25.8, 64 at 27.8.  So a core is whole lines wide, wide rather
// than high, and a slot is stored by the block whose core holds its place: B runs
// on one more column on each side and stores from there only what falls into the
// core, whole lines again (27.8 -> 32.7).
//
// Against the two-step pass of pair.hpp in the same runs, D3Q27 CM, GLUPS: FP32
// 512^3 31.6-32.1 -> 35.2, 384^3 29.7 -> 35.7, 256^3 31.0 -> 34-36, 192^3 29.6 ->
// 35.5, 300x280x260 25.9 -> 33.4; FP64 512^3 16.1 -> 17.5, 256^3 15.5 -> 16.5,
// 150x130x140 13.0 -> 16.1.
//
// With Solid nodes and a halo (a 512x256x256 channel of 200 spheres, 100 steps with
// readouts): 130 ms with the pass of pair.hpp, 129.7 while each remote slot's
// address was tested against the box, 122.5 with the offsets set once per block.
//
// A node that does not move (Solid, Excluded, the halo) leaves its slots as they
// are, which is to send each population back along its opposite direction; B
// stores them where the sender lies in the box.  Slots that no node of the box
// writes hold the same values in both arrays (the host copies the array once after
// every seeding or change of the flags).
#pragma once

#include "kernels.hpp"
#include "wrap.hpp"

namespace m3lb {

struct MarchArgs {
  StepArgs a;
  void* out;                           // the other population array
  int ntx, nty, nzc;   // blocks along x, y and z
  int core_y, more_y;  // sy / nty, sy % nty
  int run_z, more_z;   // sz / nzc, sz % nzc
};

// Region of a block: a core of W x CY nodes, two more columns on each side in x
// and a row on each side in y; one cell per thread, 36 values per cell in LDS.
template <class T>
struct MarchShape {
  static constexpr int W = sizeof(T) == 4 ? 64 : 32, CY = sizeof(T) == 4 ? 13 : 12;
  static constexpr int RX = W + 4, RY = CY + 2, NP = RX * RY, NT = sizeof(T) == 4 ? 1024 : 512;
  static_assert(NP <= NT && 36 * NP * sizeof(T) <= 160 * 1024, "a cell per thread, in LDS");
};

// Place of direction d among those of its c_z.
template <int d>
__host__ __device__ constexpr int march_rank() {
  int r = 0;
  for (int j = 0; j < d; ++j) r += cvel<27>(j, 2) == cvel<27>(d, 2);
  return r;
}

// Barrier for LDS alone: loads and stores of the population arrays stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// GEOM: some node of the padded box is not Fluid.  The first step is an even one.
template <class K, bool GEOM>
__global__ void __launch_bounds__(MarchShape<typename K::T>::NT) k_march(MarchArgs ma) {
  using R = typename K::R;
  using T = typename K::T;
  using C = typename K::C;
  using S = MarchShape<T>;
  constexpr int Q = K::Q, RX = S::RX, NP = S::NP;
  __shared__ T s[36 * NP];
  const StepArgs& a = ma.a;
  const Dom& d = a.d;
  const unsigned tile = tile_of(blockIdx.x, gridDim.x, a.remap);
  const unsigned plane = unsigned(ma.ntx) * unsigned(ma.nty);
  const int izc = int(tile / plane), xy = int(tile - unsigned(izc) * plane);
  const int ity = int(unsigned(xy) / unsigned(ma.ntx)), itx = xy - ity * ma.ntx;
  const int X0 = itx * S::W, nx = min(S::W, d.sx - X0);
  const int Y0 = ity * ma.core_y + min(ity, ma.more_y), ny = ma.core_y + (ity < ma.more_y);
  const int Z0 = izc * ma.run_z + min(izc, ma.more_z), Z1 = Z0 + ma.run_z + (izc < ma.more_z);
  const Params<R> p = params_of<K>(a);
  const T* A = static_cast<const T*>(a.f);
  T* B = static_cast<T*>(ma.out);

  const int c = int(threadIdx.x), cx = c % RX, cy = c / RX;
  // B runs on the core and a column on each side, and stores the slots whose place
  // along x lies in the core
  const bool core = cx >= 1 && cx <= nx + 2 && cy >= 1 && cy <= ny;
  const bool own = cx >= 2 && cx < nx + 2;                                       // its own place
  const bool own_r = cx >= 1 && cx < nx + 1, own_l = cx >= 3 && cx < nx + 3;  // x + 1, x - 1
  bool in = c < NP && cx <= nx + 3 && cy <= ny + 1;  // takes part in A
  int X = X0 - 2 + cx, Y = Y0 - 1 + cy;
  if (d.px) X = wrapped(X, d.sx);
  auto wrap = [](int& v, int n, bool per) -> bool {  // v in -1 .. n, false: outside
    if (v >= 0 && v < n) return true;
    v = v < 0 ? v + n : v - n;
    return per;
  };
  in = in && wrap(X, d.sx, d.px) && wrap(Y, d.sy, d.py);
  if (!in) X = Y = 0;
  Offs o = offsets(d, X - d.hx, Y - d.hy, 0);
  if constexpr (GEOM) {
    // a halo node's slots outside the box: any in it, nothing reads the value
    if (!d.px && X == 0) o.xm = 0;
    if (!d.px && X == d.sx - 1) o.xp = 0;
    if (!d.py && Y == 0) o.ym = 0;
    if (!d.py && Y == d.sy - 1) o.yp = 0;
  }
  const int sxy = d.sx * d.sy;
  const unsigned nxy = unsigned(Y * d.sx + X);
  auto plane_of = [&](int z, int& Z) -> bool {  // padded plane z, offsets along z
    Z = z;
    if (!wrap(Z, d.sz, d.pz)) return false;
    o.zm = Z != 0 ? -sxy : d.pz ? (d.nz - 1) * sxy : 0;
    o.zp = Z != d.sz - 1 ? sxy : d.pz ? -(d.nz - 1) * sxy : 0;
    return true;
  };
  auto inside = [&](int x, int y, int z) -> bool {
    return (d.px || (x >= 0 && x < d.sx)) && (d.py || (y >= 0 && y < d.sy)) &&
           (d.pz || (z >= 0 && z < d.sz));
  };

  // The slots of a node of plane z at an even step, requested ahead of their use.
  T raw[Q];
  bool fluid = false;
  auto request = [&](int z) {
    int Z;
    const bool ok = plane_of(z, Z);
    uint64_t stride = a.stride;
    asm volatile("" : "+s"(stride));  // 27 bases formed again, not held
    if (!ok || !in) return;
    const unsigned n = nxy + unsigned(Z * sxy);
    if constexpr (GEOM) fluid = a.flags[n] == M3LB_FLUID;
    raw[0] = ld<false>(A, n);
    sfor<(Q - 1) / 2>([&](auto Pr) {
      constexpr int i = 2 * Pr + 1;
      raw[i] = ld<false>(qbase(A, stride, i), n);
      raw[i + 1] = ld<false>(qbase(A, stride, i + 1), unsigned(int(n) + nb_off<Q, i>(o)));
    });
  };

  bool was_fluid = false;  // of this cell in the plane before
  request(Z0 - 1);
#pragma unroll 1
  for (int z = Z0 - 1; z <= Z1; ++z) {
    const bool step_b = z > Z0;  // B of plane z - 1
    T* up = s + (18 + (z & 1) * 9) * NP;  // c_z = +1 of plane z, and of plane z - 2 so far
    int Z;
    const bool ok = plane_of(z, Z);
    // A: what the node sends out, by direction
    R g[Q];
    const bool moves = !GEOM || fluid;
    if (!moves) {
      g[0] = C::dec(raw[0], 0.0f);
      sfor<(Q - 1) / 2>([&](auto Pr) {
        constexpr int i = 2 * Pr + 1;
        g[i] = C::dec(raw[i + 1], 0.0f);
        g[i + 1] = C::dec(raw[i], 0.0f);
      });
    } else {
      sfor<Q>([&](auto I) { g[int(I)] = C::dec(raw[int(I)], 0.0f); });
    }
    if (z < Z1) request(z + 1);
    if (moves && in) (void)collide_fused<K>(g, p);
    // B's inputs that A of this plane overwrites
    R f[Q];
    if (step_b && core) {
      sfor<Q>([&](auto I) {
        constexpr int i = I, cz = cvel<Q>(i, 2);
        const int from = c - cvel<Q>(i, 1) * RX - cvel<Q>(i, 0);
        if constexpr (cz == 1) f[i] = C::dec(up[march_rank<i>() * NP + from], 0.0f);
        if constexpr (cz == 0) f[i] = C::dec(s[march_rank<i>() * NP + from], 0.0f);
      });
    }
    lds_barrier();
    if (in && ok) {
      sfor<Q>([&](auto I) {
        constexpr int i = I, cz = cvel<Q>(i, 2), r = march_rank<i>() * NP;
        const T v = C::enc(g[i], 0.0f);
        if constexpr (cz == 1) up[r + c] = v;
        else if constexpr (cz == 0) s[r + c] = v;
        else s[9 * NP + r + c] = v;
      });
    }
    lds_barrier();
    const bool b_fluid = was_fluid;
    was_fluid = moves;
    if (!step_b || !core || !in) continue;
    // B
    sfor<Q>([&](auto I) {
      constexpr int i = I;
      if constexpr (cvel<Q>(i, 2) == -1)
        f[i] = C::dec(s[9 * NP + march_rank<i>() * NP + c - cvel<Q>(i, 1) * RX - cvel<Q>(i, 0)], 0.0f);
    });
    int Zb;
    (void)plane_of(z - 1, Zb);
    const unsigned n = nxy + unsigned(Zb * sxy);
    uint64_t stride = a.stride;
    asm volatile("" : "+s"(stride) : "v"(f[0]));
    if (!GEOM || b_fluid) {
      (void)collide_fused<K>(f, p);
      // the slots in three groups by their place along x
      auto put = [&](int q, unsigned m, R v) {
        st<false>(const_cast<T*>(qbase(B, stride, q)), m, C::enc(v, 0.0f));
      };
      auto put_remote = [&](auto EX) {
        sfor<(Q - 1) / 2>([&](auto Pr) {
          constexpr int i = 2 * Pr + 1;
          if constexpr (cvel<Q>(i, 0) == int(EX)) put(i, unsigned(int(n) + nb_off<Q, i>(o)), f[i]);
        });
      };
      if (own) {
        put(0, n, f[0]);
        sfor<(Q - 1) / 2>([&](auto Pr) { put(2 * Pr + 2, n, f[2 * Pr + 2]); });
        put_remote(std::integral_constant<int, 0>{});
      }
      if (own_r) put_remote(std::integral_constant<int, 1>{});
      if (own_l) put_remote(std::integral_constant<int, -1>{});
    } else {
      if (own) B[n] = C::enc(f[0], 0.0f);
      sfor<(Q - 1) / 2>([&](auto Pr) {
        constexpr int i = 2 * Pr + 1;
        constexpr int ex = cvel<Q>(i, 0), ey = cvel<Q>(i, 1), ez = cvel<Q>(i, 2);
        const bool at = ex == 0 ? own : ex == 1 ? own_r : own_l;
        if (own && inside(X - ex, Y - ey, Zb - ez))
          B[uint64_t(i + 1) * stride + n] = C::enc(f[i], 0.0f);
        if (at && inside(X + ex, Y + ey, Zb + ez))
          B[uint64_t(i) * stride + unsigned(int(n) + nb_off<Q, i>(o))] = C::enc(f[i + 1], 0.0f);
      });
    }
  }
}

}  // namespace m3lb
