// Work-group to node mapping of the flow kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "flow.hpp"

namespace corefl {
namespace tiles {

// XCD-aware tile order.  Workgroups are dispatched round-robin over the 8 XCDs, each with its own L2.
// A 1-D launch of 8*P workgroups is remapped so that the workgroups landing on one XCD take a contiguous
// run of tiles: along the plane (consecutive rows, the i and j stencils) or, for the z sweep, along k, so that
// the nodes of a stencil are read by workgroups sharing an L2.  The map b -> (b % 8) * P + b / 8 is a
// bijection on [0, 8P).
// Within a plane, a workgroup of 256 threads takes 256 consecutive nodes of the launch's nx x ny nodes in row-major
// order (i fastest), so that only the last workgroup of a plane has idle lanes whatever nx is: a 64-wide tiling of
// 257 nodes leaves a fifth wave per row with one active lane, a quarter more waves than nodes need.
struct TileGrid {
  int gx, gy, gz; // workgroups per plane (gy = 1), and planes (or plane groups) along k
  int fast;       // 0: plane chunk then k (each XCD takes a contiguous run), 2: k fastest
  int z0;         // first k tile (a launch over a slab of planes)
  int nx, ny;     // nodes of a plane covered by the launch
};

struct Tile {
  int z;    // plane (or plane group) index
  int i, j; // this thread's node, before the kernel's own offsets
};

// A launch over the nx x ny nodes of gz planes (or plane groups) starting at z0.
inline TileGrid plane_grid(int nx, int ny, int gz, int fast, int z0) {
  return TileGrid{(nx * ny + 255) / 256, 1, gz, fast, z0, nx, ny};
}

__device__ __forceinline__ bool xcd_tile(const TileGrid &t, unsigned block, Tile &out) {
  const unsigned total = (unsigned)t.gx * t.gz;
  const unsigned per = (total + 7) / 8;
  const unsigned n = (block % 8) * per + block / 8;
  if (n >= total) return false;
  unsigned x;
  if (t.fast == 2) {
    out.z = n % t.gz;
    x = n / t.gz;
  } else {
    x = n % t.gx;
    out.z = n / t.gx;
  }
  out.z += t.z0;
  const unsigned p = x * 256u + threadIdx.y * 64u + threadIdx.x, nx = t.nx;
  out.j = (int)(p / nx);
  out.i = (int)(p - (unsigned)out.j * nx);
  return out.j < t.ny;
}

inline unsigned tile_blocks(const TileGrid &t) {
  const unsigned total = (unsigned)t.gx * t.gz;
  return 8 * ((total + 7) / 8);
}

// The three directions of an interface kernel in one launch: work-groups [0, end[0]) take the x interfaces,
// [end[0], end[1]) the y and [end[1], end[2]) the z ones.  Each count is a multiple of 8, so a direction's tiles keep
// their XCDs.  Direction by direction a small block leaves most of the chip idle three times over (129 work-groups for
// each direction of a 33^3 block) and a large one pays three partly filled last rounds.  One launch takes 13 us on 33^3
// nodes (7.5 us a direction before) and 601 us on 129^3 (3 x 237).
struct SweepGrid {
  TileGrid t[3];
  unsigned end[3];
};

inline unsigned sweep_blocks(SweepGrid &g) {
  unsigned n = 0;
  for (int d = 0; d < 3; ++d) g.end[d] = n += g.t[d].gz > 0 ? tile_blocks(g.t[d]) : 0;
  return n;
}

// Calls f(direction, tile grid, work-group within it) with the direction as a compile-time constant.
template<class F> __device__ __forceinline__ void sweep(const SweepGrid &g, F &&f) {
  const unsigned n = blockIdx.x;
  if (n < g.end[0]) f(std::integral_constant<int, 0>{}, g.t[0], n);
  else if (n < g.end[1]) f(std::integral_constant<int, 1>{}, g.t[1], n - g.end[0]);
  else f(std::integral_constant<int, 2>{}, g.t[2], n - g.end[1]);
}

// The direction as a (uniform) value instead, for kernels whose directions differ in strides alone: one copy of the code.
template<class F> __device__ __forceinline__ void sweep_value(const SweepGrid &g, F &&f) {
  const unsigned n = blockIdx.x;
  const int dir = n < g.end[0] ? 0 : (n < g.end[1] ? 1 : 2);
  f(dir, g.t[dir], n - (dir == 0 ? 0u : g.end[dir - 1]));
}

// Interface fluxes along DIR go to this array.
__device__ __forceinline__ double *flux_array(const DevBlock &b, int dir) { return dir == 0 ? b.fx : (dir == 1 ? b.fy : b.fz); }

} // namespace tiles
} // namespace corefl
