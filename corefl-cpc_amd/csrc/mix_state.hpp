// Conservative variables and acoustic speed of one mixture node from its primitive state, shared by the mixture
// flow, boundary and repair kernels: compute_cv_from_bv_1_point<Mixture> + compute_total_energy
// (FieldOperation.cuh:16-84) and the acoustic speed of update_physical_properties<Mixture>
// (FieldOperation.cuh:86-120).
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

#include "chem_device.hpp"
#include "flow.hpp"
#include "flow_mix.hpp"

namespace corefl {
namespace mixdev {

constexpr int NS = 9;

// cv and the acoustic speed of node id from its primitive state v = rho, u, v, w, p, T and mass fractions y.
__device__ inline void store_cons(const DevBlock &b, const MixArrays &x, long id, const double *v, const double *y) {
  const long sz = b.sz;
  const ChemMech &m = *x.mech;
  double h[NS], cp[NS];
  chemdev::h_cp<NS>(m, v[5], h, cp);
  double E = 0.5 * (v[1] * v[1] + v[2] * v[2] + v[3] * v[3]), imw = 0, cpt = 0;
#pragma unroll
  for (int l = 0; l < NS; ++l) {
    E += h[l] * y[l];
    imw += y[l] * m.imw[l];
    cpt += y[l] * cp[l];
    b.cv[id + (5 + l) * sz] = v[0] * y[l];
  }
  b.cv[id] = v[0];
  b.cv[id + sz] = v[0] * v[1];
  b.cv[id + 2 * sz] = v[0] * v[2];
  b.cv[id + 3 * sz] = v[0] * v[3];
  b.cv[id + 4 * sz] = E * v[0] - v[4];
  const double R = chemdev::kRu * imw;
  x.snd[id] = sqrt(cpt / (cpt - R) * R * v[5]);
}

__device__ inline void mix_cons(const DevBlock &b, const MixArrays &x, long id) {
  double v[6], y[NS];
#pragma unroll
  for (int l = 0; l < 6; ++l) v[l] = b.bv[id + l * b.sz];
#pragma unroll
  for (int l = 0; l < NS; ++l) y[l] = x.sv[id + l * b.sz];
  store_cons(b, x, id, v, y);
}

} // namespace mixdev
} // namespace corefl
