// Batched finite-rate chemistry of constant-volume cells on CDNA4: NASA-7 thermo, Arrhenius / third-body /
// Lindemann / Troe kinetics with Gibbs-energy reverse rates, the analytic d(omega)/d(rho Y) Jacobian, a
// partial-pivot LU, and the adaptive 4-stage Rosenbrock ROK4E with embedded error control.  FP64.
//
// Two launch shapes integrate a batch of cells over one chemistry sub-step:
//   * static: one thread per cell;
//   * queue: persistent waves that fetch cells from a global counter as lanes finish, one ballot and one
//     atomic per wave per fetch round, so a stiff cell holds only its own lane, not a whole fixed tile.
// Every cell stops after max_attempts step attempts (flagged), so each wave's loop ends.
#include "chem_kernels.hpp"

#include <cmath>

#include "chem_device.hpp"
#include "rok4e.hpp"

namespace corefl {

namespace {

using namespace chemdev;
using namespace rok4e;

using chemdev::lu;
using chemdev::lu_solve;

// Integration state of one cell.
template<int NS> struct Cell {
  double y[NS]; // rho Y
  double rho, E, T, time, h, err_last, dt;
  int steps, rejects, attempts;
};

// One ROK4E attempt (ConstVolumeReactor.cpp:173-476 with adaptive_time_step = 1): four stages over the third stage's
// source, and a last pass for the new temperature.  The stages are one loop around a single copy of the source, the
// temperature iteration and the solve: written out, the kernel is 113 KB of code, more than the 64 KB instruction cache
// of two CUs; rolled it is 57 KB.  An attempt of a wave takes 100 us, from 145 (2.1M igniting cells: 3.4 ms, from 4.9):
// 21700 vector instructions (28600), 680 scalar loads (2060) and no vector loads of coefficients.  It is bound by its one
// wave per SIMD: vector instructions are 38% of its cycles, scalar ones 25%, waits for loads 27%.  Two waves at 256
// registers keep 950 bytes a lane in scratch and take 4.9 ms.
template<int NS>
__device__ __forceinline__ void rok4e_attempt(const ChemMech *mp, Cell<NS> &s, double rtol, double atol) {
  const double dt = s.dt;
  double w[NS], J[NS * NS], k1[NS], k2[NS], k3[NS], ys[NS];
  int piv[NS];
  // The step ends the interval when it would leave less than 5% of itself (no sliver step, whose size
  // would otherwise become the proposal carried to the next sub-step).
  const double rem = dt - s.time;
  const double hs = s.h * kStretch >= rem ? rem : s.h;
  const double irho = 1.0 / s.rho; // products by 1/rho stand for the reference's divisions
#pragma unroll
  for (int l = 0; l < NS; ++l) k1[l] = k2[l] = k3[l] = 0;
  double Ts = s.T, err = 0;
#pragma unroll 1
  for (int st = 0; st < 5; ++st) {
    const ChemMech &m = opaque(mp);
    if (st != 3) { // the fourth stage takes the third's source
      if (st < 4)
#pragma unroll
        for (int l = 0; l < NS; ++l) ys[l] = stage_state(st, s.y[l], hs, k1[l], k2[l]);
      // st 4: ys is the new state, and an accepted step gets its temperature from the old one
      if (st > 0 && (st < 4 || err <= 1)) {
        double yk[NS];
#pragma unroll
        for (int l = 0; l < NS; ++l) yk[l] = ys[l] * irho;
        Ts = update_t<NS>(m, st == 4 ? s.T : Ts, yk, s.E);
      }
      if (st == 4) break;
      source<NS, true>(m, Ts, ys, w, J, nullptr, 1e-30, st == 0);
      if (st == 0) {
#pragma unroll
        for (int q = 0; q < NS * NS; ++q) J[q] = -hs * G * J[q];
#pragma unroll
        for (int l = 0; l < NS; ++l) J[l * NS + l] += 1.0;
        lu<NS>(J, piv);
      }
    }
    double k[NS];
#pragma unroll
    for (int l = 0; l < NS; ++l) k[l] = w[l] + stage_sum(st, k1[l], k2[l], k3[l]);
    lu_solve<NS>(J, piv, k);
#pragma unroll
    for (int l = 0; l < NS; ++l) k[l] -= stage_sum(st, k1[l], k2[l], k3[l]);
    if (st == 0) {
#pragma unroll
      for (int l = 0; l < NS; ++l) k1[l] = k[l];
    } else if (st == 1) {
#pragma unroll
      for (int l = 0; l < NS; ++l) k2[l] = k[l];
    } else if (st == 2) {
#pragma unroll
      for (int l = 0; l < NS; ++l) k3[l] = k[l];
    } else {
      double d2[NS];
#pragma unroll
      for (int l = 0; l < NS; ++l) {
        ys[l] = new_state(s.y[l], hs, k1[l], k2[l], k[l]);
        const double dy = error_term(ys[l], hs, k1[l], k2[l], k3[l], k[l], rtol, atol);
        d2[l] = dy * dy;
      }
      err = sqrt(species_sum<NS>(d2) / NS);
    }
  }
  double hstar = hs;
  if (s.steps > 0) hstar *= step_factor(s.err_last, err);
  else if (!(err <= 1)) hstar *= 0.2; // a NaN first-step error also cuts the step (the reference would repeat it)
  // a step cut short by the end of the interval does not shrink the proposal
  if (err <= 1 && hs < s.h) hstar = fmax(hstar, s.h);
  s.h = hstar;
  ++s.attempts;
  if (err <= 1) {
#pragma unroll
    for (int l = 0; l < NS; ++l) s.y[l] = ys[l];
    s.time += hs;
    s.err_last = fmax(err, 1e-30); // an exactly zero error would stall the PI controller (0^0.1 = 0)
    s.T = Ts;
    ++s.steps;
  } else {
    ++s.rejects;
  }
}

template<int NS> __device__ __forceinline__ void load_cell(const ChemBatch &b, int c, double dt, Cell<NS> &s) {
#pragma unroll
  for (int l = 0; l < NS; ++l) s.y[l] = b.rhoY[(long)l * b.n + c];
  dt = cell_dt(b, c, dt);
  s.dt = dt;
  s.rho = b.rho[c];
  s.E = b.e[c];
  s.T = b.T[c];
  s.h = b.h[c] > 0 ? fmin(b.h[c], dt) : dt;
  s.time = 0;
  s.err_last = 0;
  s.steps = s.rejects = s.attempts = 0;
}

template<int NS> __device__ __forceinline__ void store_cell(const ChemBatch &b, int c, const Cell<NS> &s, bool ok) {
#pragma unroll
  for (int l = 0; l < NS; ++l) b.rhoY[(long)l * b.n + c] = s.y[l];
  b.T[c] = s.T;
  b.h[c] = s.h;
  b.steps[c] = ok ? s.steps : -1;
  b.rejects[c] = s.rejects;
}

// Work item w of a launch: cell w, or cell list[w] of a device-side list of *n_list cells.
__device__ __forceinline__ int work_count(const ChemBatch &b) { return b.list ? *b.n_list : b.n; }
__device__ __forceinline__ int work_cell(const ChemBatch &b, int w) { return b.list ? b.list[w] : w; }

template<int NS>
__global__ __launch_bounds__(256) void k_chem_static(const ChemMech *__restrict__ mp, ChemBatch b, double dt,
                                                     double rtol, double atol, int max_attempts) {
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= work_count(b)) return;
  const int c = work_cell(b, w);
  Cell<NS> s;
  load_cell<NS>(b, c, dt, s);
  while (s.time < s.dt && s.attempts < max_attempts) rok4e_attempt<NS>(mp, s, rtol, atol);
  store_cell<NS>(b, c, s, s.time >= s.dt);
}

// Integration state of a cell that used up its attempt budget, for the cooperative kernel to resume.
template<int NS> __device__ __forceinline__ void store_partial(const ChemBatch &b, int c, const Cell<NS> &s) {
#pragma unroll
  for (int l = 0; l < NS; ++l) b.rhoY[(long)l * b.n + c] = s.y[l];
  b.T[c] = s.T;
  b.h[c] = s.h;
  b.steps[c] = s.steps;
  b.rejects[c] = s.rejects;
  b.tcur[c] = s.time;
  b.elast[c] = s.err_last;
}

// budget > 0: a cell still unfinished after `budget` attempts is handed over (appended to b.defer) once fewer than 3/16
// of the launch's lanes hold a cell.  An attempt of every cell takes 100 us here whatever their number up to one per
// lane (65536 lanes), and in the cooperative kernel 60 us for every 8192 cells, so the lines cross near 13000 cells;
// below, its shorter attempt counts.  When that is reached depends on how waves are scheduled; a cell's bits do not, since
// both kernels round alike.  (200003 igniting cells, 19.8 attempts on average and 122 at most: 9.7 ms, 17.7 in this kernel
// alone and 16.6 in the cooperative one.)
template<int NS>
__global__ __launch_bounds__(256) void k_chem_queue(const ChemMech *__restrict__ mp, ChemBatch b, double dt,
                                                    double rtol, double atol, int max_attempts, int *counter,
                                                    int budget) {
  const int lane = __lane_id();
  const int n_work = work_count(b);
  Cell<NS> s;
  int cell = -1;
  bool exhausted = false;
  while (true) {
    const bool need = cell < 0 && !exhausted;
    const unsigned long long mask = __ballot(need);
    if (mask) {
      const int leader = __ffsll((long long)mask) - 1;
      int base = 0;
      if (lane == leader) base = atomicAdd(counter, __popcll(mask));
      base = __shfl(base, leader, 64);
      if (need) {
        const int got = base + __popcll(mask & ((1ull << lane) - 1));
        if (got < n_work) {
          cell = work_cell(b, got);
          load_cell<NS>(b, cell, dt, s);
        } else {
          exhausted = true;
        }
      }
    }
    if (__ballot(cell >= 0) == 0) break;
    bool defer = false;
    if (cell >= 0) {
      rok4e_attempt<NS>(mp, s, rtol, atol);
      if (s.time >= s.dt || s.attempts >= max_attempts) {
        store_cell<NS>(b, cell, s, s.time >= s.dt);
        cell = -1;
      } else {
        defer = budget > 0 && s.attempts >= budget;
      }
    }
    unsigned long long dm = __ballot(defer);
    if (dm) {
      // every lane that found the queue empty has counted once more, so the lanes at work are the others
      int fetched = 0;
      if (lane == 0) fetched = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const long lanes = (long)gridDim.x * blockDim.x, idle = (long)__shfl(fetched, 0, 64) - n_work;
      if (idle < 0 || 16 * (lanes - idle) > 3 * lanes) defer = false;
      dm = __ballot(defer);
    }
    if (dm) {
      const int leader = __ffsll((long long)dm) - 1;
      int base = 0;
      if (lane == leader) base = atomicAdd(b.n_defer, __popcll(dm));
      base = __shfl(base, leader, 64);
      if (defer) {
        b.defer[base + __popcll(dm & ((1ull << lane) - 1))] = cell;
        store_partial<NS>(b, cell, s);
        cell = -1;
      }
    }
  }
}

template<int NS>
__global__ __launch_bounds__(256) void k_chem_omega(const ChemMech *__restrict__ mp, ChemBatch b, double *omega) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= b.n) return;
  double y[NS], w[NS];
#pragma unroll
  for (int l = 0; l < NS; ++l) y[l] = b.rhoY[(long)l * b.n + c];
  source<NS, false>(*mp, b.T[c], y, w, nullptr);
#pragma unroll
  for (int l = 0; l < NS; ++l) omega[(long)l * b.n + c] = w[l];
}

template<int NS>
__global__ __launch_bounds__(256) void k_chem_temperature(const ChemMech *__restrict__ mp, ChemBatch b) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= b.n) return;
  double yk[NS];
  const double irho = 1.0 / b.rho[c];
#pragma unroll
  for (int l = 0; l < NS; ++l) yk[l] = b.rhoY[(long)l * b.n + c] * irho;
  b.T[c] = update_t<NS>(*mp, b.T[c], yk, b.e[c]);
}

template<int NS> __global__ __launch_bounds__(256) void k_chem_energy(const ChemMech *__restrict__ mp, ChemBatch b) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= b.n) return;
  const ChemMech &m = *mp;
  double h[NS], cp[NS];
  const double t = b.T[c], irho = 1.0 / b.rho[c];
  h_cp<NS>(m, t, h, cp);
  double e = 0, imw = 0;
#pragma unroll
  for (int l = 0; l < NS; ++l) {
    const double y = b.rhoY[(long)l * b.n + c] * irho;
    e = fma(h[l], y, e);
    imw = fma(y, m.imw[l], imw);
  }
  b.e[c] = fma(-kRu * imw, t, e);
}

// One launch for all counters of a sub-step (they were three, of 4.9 us each).
__global__ void k_zero_counters(int *counter, int *n_defer) {
  counter[0] = counter[1] = 0;
  if (n_defer) *n_defer = 0;
}

} // namespace

hipError_t launch_chem_energy(const ChemMech *mech_dev, int ns, const ChemBatch &b, hipStream_t s) {
  if (ns != 9) return hipErrorNotSupported;
  if (b.n == 0) return hipSuccess;
  k_chem_energy<9><<<(b.n + 255) / 256, 256, 0, s>>>(mech_dev, b);
  return hipGetLastError();
}

hipError_t launch_chem_integrate(const ChemMech *mech_dev, int ns, const ChemBatch &b, double dt, double rtol,
                                 double atol, int max_attempts, const ChemLaunch &cfg, int *counter,
                                 hipStream_t s) {
  if (ns != 9) return hipErrorNotSupported;
  if (b.n == 0) return hipSuccess;
  if (cfg.queue == 2) {
    k_zero_counters<<<1, 1, 0, s>>>(counter, nullptr);
    return launch_chem_coop(mech_dev, ns, b, dt, rtol, atol, max_attempts, cfg.threads, cfg.blocks, false, counter, s);
  }
  if (cfg.queue == 3) {
    if (cfg.budget < 1) return hipErrorInvalidValue;
    k_zero_counters<<<1, 1, 0, s>>>(counter, b.n_defer);
    k_chem_queue<9><<<cfg.blocks, cfg.threads, 0, s>>>(mech_dev, b, dt, rtol, atol, max_attempts, counter,
                                                       cfg.budget);
    ChemBatch d = b;
    d.list = b.defer;
    d.n_list = b.n_defer;
    return launch_chem_coop(mech_dev, ns, d, dt, rtol, atol, max_attempts, 256, cfg.blocks, true, counter + 1, s);
  }
  if (cfg.queue) {
    k_zero_counters<<<1, 1, 0, s>>>(counter, nullptr);
    k_chem_queue<9><<<cfg.blocks, cfg.threads, 0, s>>>(mech_dev, b, dt, rtol, atol, max_attempts, counter, 0);
  } else {
    k_chem_static<9><<<(b.n + cfg.threads - 1) / cfg.threads, cfg.threads, 0, s>>>(mech_dev, b, dt, rtol, atol,
                                                                                  max_attempts);
  }
  return hipGetLastError();
}

hipError_t launch_chem_omega(const ChemMech *mech_dev, int ns, const ChemBatch &b, double *omega, hipStream_t s) {
  if (ns != 9) return hipErrorNotSupported;
  if (b.n == 0) return hipSuccess;
  k_chem_omega<9><<<(b.n + 255) / 256, 256, 0, s>>>(mech_dev, b, omega);
  return hipGetLastError();
}

hipError_t launch_chem_temperature(const ChemMech *mech_dev, int ns, const ChemBatch &b, hipStream_t s) {
  if (ns != 9) return hipErrorNotSupported;
  if (b.n == 0) return hipSuccess;
  k_chem_temperature<9><<<(b.n + 255) / 256, 256, 0, s>>>(mech_dev, b);
  return hipGetLastError();
}

} // namespace corefl
