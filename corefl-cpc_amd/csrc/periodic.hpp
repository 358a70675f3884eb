// Periodic sides of a block in one launch.
//
// The reference treats periodic faces one after another (apply_periodic, BoundCond.cu:3033-3083; periodic_exchange,
// DataCommunication.cu:628-683): each averages the coincident nodes of the two opposite sides and copies the layers
// inside one side into the ghosts beyond the other.  Nodes where two or three periodic sides meet are averaged once
// per direction, and the copies of an earlier direction are taken before the averages of a later one, so the faces
// cannot simply run side by side.  But the nodes that coincide form closed orbits (2 nodes on a side, 4 on an edge,
// 8 in a corner), every ghost copy reads one node, and both stay inside the orbit: one thread per orbit (and component,
// where components are independent) walks the directions in order and does what the face launches did, with the same
// operands in the same order.
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "flow.hpp"

namespace corefl {

// Orbits with something to do: those within ngg layers of a periodic side.  Along a periodic direction the nodes
// 0 .. ext-2 stand for their orbits (ext-1 coincides with 0); `shell` of them lie on or near the sides (all of them in
// a thin block), `core` do not.  Items: shell x any x any, then core x shell x any, then core x core x shell.
struct PeriodicPlan {
  int active[3];          // direction d has its two sides periodic, over their whole area
  unsigned shell[3], core[3];
  unsigned n[3], total;   // items of the three groups
  bool valid;             // false: some periodic face is partial or unpaired; the faces then run one by one
};

// Plan of the block's periodic faces (type 8), in boundary-file order: each direction's two sides must follow one
// another, directions ascending, every face covering its side.
inline PeriodicPlan periodic_plan(const DevBlock &b, const std::vector<DevFace> &faces) {
  PeriodicPlan p{};
  const int ext[3] = {b.mx, b.my, b.mz};
  std::vector<const DevFace *> f;
  for (const auto &q : faces)
    if (q.type == 8) f.push_back(&q);
  if (f.empty() || f.size() % 2) return p;
  int last = -1;
  for (size_t q = 0; q < f.size(); q += 2) {
    const int d = f[q]->face;
    if (d <= last || f[q + 1]->face != d || f[q]->direction != -f[q + 1]->direction || ext[d] < b.g + 2) return p;
    for (int e = 0; e < 2; ++e)
      for (int c = 0; c < 3; ++c)
        if (c != d && (f[q + e]->start[c] != 0 || f[q + e]->end[c] != ext[c] - 1)) return p;
    last = d;
    p.active[d] = 1;
  }
  double total = 0;
  for (int d = 0; d < 3; ++d) {
    const unsigned reps = p.active[d] ? ext[d] - 1 : ext[d];
    p.shell[d] = !p.active[d] ? 0u : (reps < 2u * b.g + 1 ? reps : 2u * b.g + 1);
    p.core[d] = reps - p.shell[d];
  }
  const unsigned r1 = p.shell[1] + p.core[1], r2 = p.shell[2] + p.core[2];
  total = (double)p.shell[0] * r1 * r2 + (double)p.core[0] * p.shell[1] * r2 + (double)p.core[0] * p.core[1] * p.shell[2];
  if (total >= 3e8) return p; // items times components in 32 bits
  p.n[0] = p.shell[0] * r1 * r2;
  p.n[1] = p.core[0] * p.shell[1] * r2;
  p.n[2] = p.core[0] * p.core[1] * p.shell[2];
  p.total = p.n[0] + p.n[1] + p.n[2];
  p.valid = p.total > 0;
  return p;
}

// Representative node of an item.
__device__ __forceinline__ bool periodic_item(const PeriodicPlan &p, int g, unsigned item, int (&c)[3]) {
  if (item >= p.total) return false;
  // shell index -> node: 0 .. g, then the g nodes before the far side (in a thin block simply all of them)
  auto shell = [&](int d, unsigned s) { return (int)(s <= (unsigned)g || !p.core[d] ? s : s + p.core[d]); };
  auto core = [&](int d, unsigned t) { return (int)t + (p.shell[d] ? g + 1 : 0); };
  const unsigned r1 = p.shell[1] + p.core[1];
  if (item < p.n[0]) {
    c[0] = shell(0, item % p.shell[0]);
    const unsigned q = item / p.shell[0];
    c[1] = (int)(q % r1);
    c[2] = (int)(q / r1);
  } else if ((item -= p.n[0]) < p.n[1]) {
    c[0] = core(0, item % p.core[0]);
    const unsigned q = item / p.core[0];
    c[1] = shell(1, q % p.shell[1]);
    c[2] = (int)(q / p.shell[1]);
  } else {
    item -= p.n[1];
    c[0] = core(0, item % p.core[0]);
    const unsigned q = item / p.core[0];
    c[1] = core(1, q % p.core[1]);
    c[2] = shell(2, q / p.core[1]);
  }
  return true;
}

// One orbit of N components: op.load(node, v) reads a node's components, op.store(node, v) writes those of an averaged
// node or a ghost.  All images (at most 8) are read before anything is written and averaged in registers: walking the
// directions through memory instead, a dependent round trip for every average and copy, took 25 us (air) and 60 us
// (viscous fluxes) on a 33^3 block.
template<int N, class Op>
__device__ __forceinline__ void periodic_orbit(const DevBlock &b, const PeriodicPlan &p, const int (&c)[3], const Op &op) {
  const int ext[3] = {b.mx, b.my, b.mz};
  const long st[3] = {1, b.d2, b.d1};
  long far[3];
  unsigned images = 0; // directions along which the orbit has two images
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    far[d] = (ext[d] - 1) * st[d];
    if (p.active[d] && c[d] == 0) images |= 1u << d;
  }
  const long base = (long)(c[2] + b.g) * b.d1 + (long)(c[1] + b.g) * b.d2 + (c[0] + b.g);
  auto node = [&](unsigned q) { return base + ((q & 1u) ? far[0] : 0) + ((q & 2u) ? far[1] : 0) + ((q & 4u) ? far[2] : 0); };
  double v[8][N];
#pragma unroll
  for (unsigned q = 0; q < 8; ++q)
    if (!(q & ~images)) op.load(node(q), v[q]);
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    if (!p.active[d]) continue;
    if (c[d] == 0) {
#pragma unroll
      for (unsigned q = 0; q < 8; ++q) {
        if ((q >> d & 1u) || (q & ~images)) continue;
#pragma unroll
        for (int l = 0; l < N; ++l) v[q][l] = v[q | 1u << d][l] = 0.5 * (v[q][l] + v[q | 1u << d][l]);
      }
    } else {
      // a node inside the near side is the ghost beyond the far one, and the other way round
#pragma unroll
      for (unsigned q = 0; q < 8; ++q) {
        if ((q >> d & 1u) || (q & ~images)) continue;
        if (c[d] <= b.g) op.store(node(q) + far[d], v[q]);
        if (c[d] >= ext[d] - 1 - b.g) op.store(node(q) - far[d], v[q]);
      }
    }
  }
  if (images)
#pragma unroll
    for (unsigned q = 0; q < 8; ++q)
      if (!(q & ~images)) op.store(node(q), v[q]);
}

// The nodes the orbits write, each once: for every periodic direction the ghosts beyond its two sides and the sides
// themselves, without the side nodes an earlier direction has already.  Items: direction 0's, then 1's, then 2's.
__device__ __forceinline__ bool periodic_written(const DevBlock &b, const PeriodicPlan &p, unsigned item, long &id) {
  const int ext[3] = {b.mx, b.my, b.mz};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    if (!p.active[d]) continue;
    const int e1 = d == 0 ? 1 : 0, e2 = d == 2 ? 1 : 2;
    const unsigned layers = 2u * (b.g + 1), area = (unsigned)ext[e1] * ext[e2];
    if (item >= layers * area) {
      item -= layers * area;
      continue;
    }
    // along x a node's layers are neighbours in memory, along y and z the nodes of a layer are
    const unsigned layer = d == 0 ? item % layers : item / area, at = d == 0 ? item / layers : item % area;
    int c[3];
    c[d] = layer <= (unsigned)b.g ? (int)layer - b.g : ext[d] - 1 + (int)layer - (b.g + 1);
    c[e1] = (int)(at % ext[e1]);
    c[e2] = (int)(at / ext[e1]);
    if (c[d] == 0 || c[d] == ext[d] - 1)
#pragma unroll
      for (int e = 0; e < d; ++e)
        if (p.active[e] && (c[e] == 0 || c[e] == ext[e] - 1)) return false;
    id = (long)(c[2] + b.g) * b.d1 + (long)(c[1] + b.g) * b.d2 + (c[0] + b.g);
    return true;
  }
  return false;
}

inline unsigned periodic_written_items(const DevBlock &b, const PeriodicPlan &p) {
  const int ext[3] = {b.mx, b.my, b.mz};
  unsigned n = 0;
  for (int d = 0; d < 3; ++d)
    if (p.active[d]) n += 2u * (b.g + 1) * ext[d == 0 ? 1 : 0] * ext[d == 2 ? 1 : 2];
  return n;
}

// Faces whose fills read and write nothing in common (outflow), in one launch: items first[q] .. first[q+1]-1 belong
// to face q, one per face node and ghost layer.
constexpr int kMaxFacesPerLaunch = 8;
struct FaceBatch {
  int n;
  DevFace f[kMaxFacesPerLaunch];
  unsigned first[kMaxFacesPerLaunch + 1];
};

inline std::vector<FaceBatch> face_batches(const DevBlock &b, const std::vector<DevFace> &faces, int type) {
  std::vector<FaceBatch> out;
  for (const auto &f : faces) {
    if (f.type != type) continue;
    const long items = (long)(f.end[0] - f.start[0] + 1) * (f.end[1] - f.start[1] + 1) * (f.end[2] - f.start[2] + 1) * b.g;
    if (out.empty() || out.back().n == kMaxFacesPerLaunch || (long)out.back().first[out.back().n] + items > 2147483647L)
      out.push_back(FaceBatch{});
    FaceBatch &B = out.back();
    B.f[B.n] = f;
    B.first[B.n + 1] = B.first[B.n] + (unsigned)items;
    ++B.n;
  }
  return out;
}

// Face node and ghost layer of item r of face f (on i faces the ghost layers of a node are contiguous in memory, so
// the layer varies fastest across lanes there; on j and k faces the face nodes do).
__device__ __forceinline__ void face_node_layer(const DevFace &f, int ghosts, unsigned r, int (&c)[3], int &g) {
  const unsigned n0 = f.end[0] - f.start[0] + 1, n1 = f.end[1] - f.start[1] + 1, n2 = f.end[2] - f.start[2] + 1;
  unsigned pt;
  if (f.face == 0) {
    g = (int)(r % (unsigned)ghosts) + 1;
    pt = r / (unsigned)ghosts;
  } else {
    const unsigned npt = n0 * n1 * n2;
    g = (int)(r / npt) + 1;
    pt = r % npt;
  }
  c[0] = f.start[0] + (int)(pt % n0);
  c[1] = f.start[1] + (int)((pt / n0) % n1);
  c[2] = f.start[2] + (int)(pt / (n0 * n1));
}

// The node an outflow item copies and the ghost node it fills.
__device__ __forceinline__ bool face_batch_item(const DevBlock &b, const FaceBatch &B, long &node, long &ghost) {
  const unsigned item = blockIdx.x * 256u + threadIdx.x;
  if (item >= B.first[B.n]) return false;
  int q = 0;
  while (item >= B.first[q + 1]) ++q;
  const DevFace &f = B.f[q];
  int c[3], g;
  face_node_layer(f, b.g, item - B.first[q], c, g);
  const long st = f.face == 0 ? 1 : (f.face == 1 ? b.d2 : b.d1);
  node = (long)(c[2] + b.g) * b.d1 + (long)(c[1] + b.g) * b.d2 + (c[0] + b.g);
  ghost = node + (long)(g * f.direction) * st;
  return true;
}

} // namespace corefl
