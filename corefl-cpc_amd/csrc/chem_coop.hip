// Cooperative batched chemistry: one cell per 16-lane row of a wavefront (four cells per wave), for the cells
// whose long chains of ROK4E attempts set the latency of a sub-step.
//
// The one-lane kernels keep a cell's whole state (the 9 x 9 iteration matrix, four stage vectors, the
// mechanism's working arrays) in one lane: about 500 registers, one wave per SIMD, and every instruction of
// an attempt issued one after another.  Here lane a of a row owns species a (its partial density, stage
// values and row a of the matrix) and reactions a, a + 16, ...: the reaction rates of a source evaluation
// are computed side by side, each species row accumulates its production terms and Jacobian row, and the LU
// factorisation and the solves run row-parallel.  Values are exchanged within the row by DPP broadcasts
// (row_newbcast, a constant source lane), by ds_bpermute for a data-dependent pivot row, and through a
// small per-row LDS area for the rates and concentrations that the reaction lanes read at per-lane indices.
//
// The chain of one cell is latency: what counts is how long one instruction waits for the one before it.  So the
// mechanism lives in LDS, laid out so that a lane finds its reaction's or species' values at its own index (read from
// memory through per-lane and scalar loads, an attempt spent most of its 57 us on them); production terms are dense
// sums over the reactions, since a lane has nothing better to do; fall-off reactions share the last pass of 16, so that
// the other passes skip their exponentials; the temperature iteration runs on the mixture's own fit; rows are exchanged
// only where some cell pivots; and the four stages are one loop, so that the code stays in the instruction cache.
// An attempt of a wave takes 25 us alone on its SIMD and 37 us with a second one: the three sources 16, of which the
// Jacobian 2.5, the factorisation 2, the solves 2.3, the temperatures 3.5.
//
// The operations are those of the one-lane attempt (chem_kernels.hip), each sum in the same order, so that a cell gets the
// same bits wherever it is integrated and whenever it is handed over.
#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "chem_device.hpp"
#include "chem_kernels.hpp"
#include "rok4e.hpp"

namespace corefl {

namespace {

using namespace chemdev;
using namespace rok4e;

constexpr int RW = 16; // lanes per cell (one DPP row)

// value of lane K of this lane's 16-lane row (DPP row_newbcast)
template<int K> __device__ __forceinline__ double row_bcast_c(double x) {
  int2 v = __builtin_bit_cast(int2, x);
  v.x = __builtin_amdgcn_update_dpp(0, v.x, 0x150 + K, 0xF, 0xF, false);
  v.y = __builtin_amdgcn_update_dpp(0, v.y, 0x150 + K, 0xF, 0xF, false);
  return __builtin_bit_cast(double, v);
}

// f(std::integral_constant<int, I>) for I = B .. E-1, unrolled at compile time: every DPP control operand
// is then a constant (a loop of broadcasts would be unrolled only after the compiler's size estimate of it)
template<int B, int E, class F> __device__ __forceinline__ void static_for(F &&f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// Orders the LDS traffic of one wavefront: stores before this point are seen by loads after it.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int kPad = 16; // species index of an unused place on a reaction's side: concentration 1, g 0

// The mechanism in LDS.  Species tables [field][species]; the tables of the rates [field][place], places in the order of
// ChemMech::by_cost; the stoichiometry [reaction][species], since production is summed in the mechanism's order.
struct MechLds {
  double lo[7][kMaxSpec], hi[7][kMaxSpec];
  double t_low[kMaxSpec], t_mid[kMaxSpec], t_high[kMaxSpec];
  double ln_t_low[kMaxSpec], ln_t_high[kMaxSpec], inv_t_low[kMaxSpec], inv_t_high[kMaxSpec];
  double mw[kMaxSpec], imw[kMaxSpec];
  double A[kMaxReac], b[kMaxReac], Ea[kMaxReac], A2[kMaxReac], b2[kMaxReac], Ea2[kMaxReac], troe[4][kMaxReac];
  double tb[kMaxSpec][kMaxReac];
  double dnu[kMaxReac][kMaxSpec], nf[kMaxReac][kMaxSpec], nb[kMaxReac][kMaxSpec];
  int type[kMaxReac], rev[kMaxReac], iorder[kMaxReac], order[kMaxReac]; // order: the reaction of a place
  unsigned fsp[kMaxReac], bsp[kMaxReac];
  unsigned long long fnu[kMaxReac], bnu[kMaxReac];
};

__device__ __forceinline__ void stage_mechanism(const ChemMech &m, MechLds &S) {
  for (int i = threadIdx.x; i < kMaxSpec; i += blockDim.x) {
#pragma unroll
    for (int q = 0; q < 7; ++q) {
      S.lo[q][i] = m.lo[i][q];
      S.hi[q][i] = m.hi[i][q];
    }
    S.t_low[i] = m.t_low[i];
    S.t_mid[i] = m.t_mid[i];
    S.t_high[i] = m.t_high[i];
    S.ln_t_low[i] = m.ln_t_low[i];
    S.ln_t_high[i] = m.ln_t_high[i];
    S.inv_t_low[i] = m.inv_t_low[i];
    S.inv_t_high[i] = m.inv_t_high[i];
    S.mw[i] = m.mw[i];
    S.imw[i] = m.imw[i];
  }
  for (int p = threadIdx.x; p < m.nr; p += blockDim.x) {
    const int r = m.by_cost[p];
    const ReacRecord q = m.rec[r];
    S.A[p] = q.A;
    S.b[p] = q.b;
    S.Ea[p] = q.Ea;
    S.A2[p] = q.A2;
    S.b2[p] = q.b2;
    S.Ea2[p] = q.Ea2;
#pragma unroll
    for (int k = 0; k < 4; ++k) S.troe[k][p] = q.troe[k];
    S.order[p] = r;
    S.type[p] = q.type;
    S.rev[p] = q.rev;
    S.iorder[p] = q.iorder;
    unsigned f = q.fsp, b = q.bsp;
    for (int k = q.n_sides & 255; k < kMaxSide; ++k) f |= (unsigned)kPad << 8 * k;
    for (int k = q.n_sides >> 8; k < kMaxSide; ++k) b |= (unsigned)kPad << 8 * k;
    S.fsp[p] = f;
    S.bsp[p] = b;
    S.fnu[p] = q.fnu; // coefficient 0 in unused places
    S.bnu[p] = q.bnu;
  }
  for (int q = threadIdx.x; q < m.nr * kMaxSpec; q += blockDim.x) {
    const int p = q / kMaxSpec, n = q % kMaxSpec;
    S.dnu[p][n] = m.dnu[p][n];
    S.nf[p][n] = m.nf[p][n];
    S.nb[p][n] = m.nb[p][n];
    S.tb[n][p] = m.tb[m.by_cost[p]][n];
  }
}

// Per-row exchange area: concentrations and g/RT written by the species lanes, rates of progress written by
// the reaction lanes (q1 the net one where no Jacobian is formed).
struct RowLds {
  double c[kMaxSpec + 1], g[kMaxSpec + 1];
  double q1[kMaxReac], q2[kMaxReac];
};

// Sum over the row's 16 lanes, the same bits in all of them (each rotation adds two values that both lanes hold).
template<int N> __device__ __forceinline__ double row_rotate(double x) {
  int2 v = __builtin_bit_cast(int2, x);
  v.x = __builtin_amdgcn_update_dpp(0, v.x, 0x120 + N, 0xF, 0xF, false);
  v.y = __builtin_amdgcn_update_dpp(0, v.y, 0x120 + N, 0xF, 0xF, false);
  return __builtin_bit_cast(double, v);
}
__device__ __forceinline__ double row_sum(double x) {
  x += row_rotate<8>(x);
  x += row_rotate<4>(x);
  x += row_rotate<2>(x);
  x += row_rotate<1>(x);
  return x;
}

// g_a / (R T) of species a (the one-lane gibbs, one species).
__device__ __forceinline__ double own_gibbs(const MechLds &S, int a, double t, double lnT, double iT) {
  const bool below = t < S.t_low[a], above = t > S.t_high[a];
  const double tt = below ? S.t_low[a] : (above ? S.t_high[a] : t);
  const bool use_lo = below || (!above && t < S.t_mid[a]);
  double c[7];
#pragma unroll
  for (int q = 0; q < 7; ++q) c[q] = use_lo ? S.lo[q][a] : S.hi[q][a];
  const double lt = below ? S.ln_t_low[a] : (above ? S.ln_t_high[a] : lnT);
  const double itt = below ? S.inv_t_low[a] : (above ? S.inv_t_high[a] : iT);
  return gibbs_fit(c, tt, lt, itt);
}

// Newton temperature at fixed E (the one-lane update_t): yk = this lane's mass fraction (0 beyond NS).  The mixture's
// enthalpy and heat capacity are those of its summed coefficients where all species share their fit range, else the sums
// of the species' own.
template<int NS>
__device__ __forceinline__ double row_update_t(const ChemMech &m, const MechLds &S, RowLds &X, int a, int gl, double t, double yk,
                                               double E) {
  const double R = kRu * row_sum(yk * S.imw[a]), yr = yk * (kRu * S.imw[a]);
  double err = 1e+6, C[6];
  int side = -1;
  X.c[gl] = yr; // free between two sources
  wave_sync();
#pragma unroll 1
  for (int it = 0; it < 100 && err > 1e-8; ++it) {
    double h, cp;
    if (m.common_range) {
      const int now = t < m.ct_mid ? 0 : 1;
      if (now != side) { // all lanes of a row alike
        // lane q sums coefficient q over the species in their order, as the one-lane iteration does
        const int q = gl < 6 ? gl : 5;
        const double *c = now ? S.hi[q] : S.lo[q];
        double d = 0;
#pragma unroll
        for (int l = 0; l < NS; ++l) d = fma(X.c[l], c[l], d);
        static_for<0, 6>([&](auto Q) { C[decltype(Q)::value] = row_bcast_c<decltype(Q)::value>(d); });
        side = now;
      }
      h_cp_fit(C, 1.0, t, fmin(fmax(t, m.ct_low), m.ct_high), h, cp);
    } else {
      const double lo = S.t_low[a], hi = S.t_high[a], tt = t < lo ? lo : (t > hi ? hi : t);
      const bool use_lo = t < lo || (!(t > hi) && t < S.t_mid[a]);
      double c[6];
#pragma unroll
      for (int q = 0; q < 6; ++q) c[q] = use_lo ? S.lo[q][a] : S.hi[q][a];
      h_cp_fit(c, yr, t, tt, h, cp);
      h = row_sum(h);
      cp = row_sum(cp);
    }
    const double t1 = t - (fma(-R, t, h) - E) / (cp - R);
    err = fabs(1 - t1 / t);
    t = t1;
  }
  wave_sync();
  return t;
}

// Rates of progress of the reaction in place r at the row's state (the reaction body of the one-lane source).  (Two
// places at a time, their exponentials formed together without branches, take as long.)
__device__ __forceinline__ void reaction_rates(const ChemMech &m, const MechLds &S, const RowLds &X, int r, int ns, double t,
                                               double lnT, double iT, double &q1o, double &q2o) {
  const int ty = S.type[r], rev = S.rev[r], order = S.iorder[r];
  const unsigned fsp = S.fsp[r], bsp = S.bsp[r];
  const unsigned long long fnu = S.fnu[r], bnu = S.bnu[r];
  const double A2 = S.A2[r], b2 = S.b2[r], Ea2 = S.Ea2[r];
  // both sides at once: the sum of nu g and the product of c^nu
  double dg = 0, q1 = 1.0, q2 = ty != 0 ? 1.0 : 0.0;
  auto side = [&](unsigned sp, unsigned long long nu, int most, double sign, double &q) {
    for (int s = 0; s < most; ++s) {
      const int l = sp >> 8 * s & 255u, n = (short)(nu >> 16 * s & 65535u);
      const double x = X.c[l];
      dg = fma(X.g[l], sign * n, dg);
      if (n == 1) q *= x;
      else q *= int_pow(x, n);
    }
  };
  side(fsp, fnu, m.max_f, -1.0, q1);
  side(bsp, bnu, m.max_b, 1.0, q2);
  double cc = 0;
  if (ty >= 4)
    for (int l = 0; l < ns; ++l) cc = fma(X.c[l], S.tb[l][r], cc);
  const double kf = forward_rate(ty, S.A[r], S.b[r], S.Ea[r], A2, b2, Ea2, t, lnT, iT, cc, [&](int k) { return S.troe[k][r]; });
  double kb = 0;
  if (ty != 0 && rev == 1) {
    kb = arrhenius(lnT, iT, A2, b2, Ea2);
    if (ty == 4) kb *= cc;
  }
  if (m.need_gibbs && ty != 0 && ty != 2) kb = gibbs_reverse(kf, dg, order, kPatm / kRu * 1e-3 * iT, kRu / kPatm * 1e+3 * t);
  q1o = q1 * kf;
  q2o = q2 * kb;
}

// Chemical source of the row's cell, lane a omega_a; with jac (uniform) also row a of the Jacobian.  ya is this lane's
// rho Y.
template<int NS>
__device__ __forceinline__ double row_source(const ChemMech &m, const MechLds &S, RowLds &X, int a, int gl, double t, double ya,
                                             bool jac, double (&Jrow)[NS]) {
  const double lnT = log(t), iT = 1.0 / t;
  X.c[gl] = ya * S.imw[a] * 1e-3;
  X.g[gl] = m.need_gibbs ? own_gibbs(S, a, t, lnT, iT) : 0.0;
  wave_sync();
  const int nr = m.nr;
#pragma unroll 1
  for (int r0 = 0; r0 < nr; r0 += RW) {
    const int r = r0 + gl;
    if (r < nr) {
      double q1, q2;
      reaction_rates(m, S, X, r, NS, t, lnT, iT, q1, q2);
      const int o = S.order[r];
      X.q1[o] = jac ? q1 : q1 - q2;
      X.q2[o] = q2;
    }
  }
  wave_sync();
  const double scale = 1e+3 * S.mw[a];
  double w = 0;
  if (!jac && m.both_sides) { // a species' two coefficients one after the other, as the one-lane source adds them
    for (int r = 0; r < nr; ++r) w = fma(S.nb[r][a], X.q1[r], fma(-S.nf[r][a], X.q1[r], w));
  } else if (!jac) {
#pragma unroll 8
    for (int r = 0; r < nr; ++r) w = fma(S.dnu[r][a], X.q1[r], w);
  } else {
    // column n of a reaction's term is lane n's, and goes round the row
#pragma unroll
    for (int n = 0; n < NS; ++n) Jrow[n] = 0;
#pragma unroll 2
    for (int r = 0; r < nr; ++r) {
      const double q1 = X.q1[r], q2 = X.q2[r], dn = S.dnu[r][a];
      const double nf = S.nf[r][a], nb = S.nb[r][a], qn = q1 - q2, v = fma(nf, q1, -(nb * q2));
      w = fma(nb, qn, fma(-nf, qn, w));
      static_for<0, NS>([&](auto N) {
        constexpr int n = decltype(N)::value;
        Jrow[n] = fma(dn, row_bcast_c<n>(v), Jrow[n]);
      });
    }
    const double inv = ya > 1e-30 ? 1.0 / ya : 0.0;
    static_for<0, NS>([&](auto N) {
      constexpr int n = decltype(N)::value;
      Jrow[n] = Jrow[n] * row_bcast_c<n>(inv) * scale;
    });
  }
  wave_sync(); // the exchange area is rewritten by the next evaluation
  return w * scale;
}

// Row-parallel LU with partial pivoting of the matrix whose row a is held by lane a.  Leaves L (unit, below
// the diagonal), U above it and the reciprocal pivots on it, as the one-lane lu; returns the lane whose value
// row a of a permuted right-hand side takes.
template<int NS> __device__ __forceinline__ int row_lu(double *row, int a) {
  int piv[NS];
  static_for<0, NS>([&](auto K) {
    constexpr int k = decltype(K)::value;
    double col[NS];
    static_for<k, NS>([&](auto R) { col[decltype(R)::value] = row_bcast_c<decltype(R)::value>(row[k]); });
    int ik = k;
    double amax = 0;
#pragma unroll
    for (int r = k; r < NS; ++r) {
      const double v = fabs(col[r]);
      if (r == k) {
        amax = v;
      } else if (v > amax) {
        amax = v;
        ik = r;
      }
    }
    piv[k] = ik;
    double prow[NS];
    if (__any(ik != k)) {
#pragma unroll
      for (int t = 0; t < NS; ++t) {
        prow[t] = __shfl(row[t], ik, RW);
        const double krow = row_bcast_c<k>(row[t]);
        row[t] = a == k ? prow[t] : (a == ik ? krow : row[t]);
      }
    } else {
#pragma unroll
      for (int t = k; t < NS; ++t) prow[t] = row_bcast_c<k>(row[t]);
    }
    const double inv = 1.0 / prow[k];
    if (a > k) {
      const double l = row[k] * inv;
      row[k] = l;
#pragma unroll
      for (int t = k + 1; t < NS; ++t) row[t] = fma(-l, prow[t], row[t]);
    } else if (a == k) {
      row[k] = inv;
    }
  });
  // the sequential exchanges b[r] <-> b[piv[r]] of the solve, traced back from position a
  int pos = a;
#pragma unroll
  for (int r = NS - 1; r >= 0; --r) {
    if (pos == r) pos = piv[r];
    else if (pos == piv[r]) pos = r;
  }
  return pos;
}

// Solve with the factors of row_lu: lane a holds b_a on entry and x_a on return.
template<int NS> __device__ __forceinline__ double row_solve(const double *row, int a, int src, double b) {
  b = __shfl(b, src, RW);
  static_for<0, NS - 1>([&](auto T) {
    constexpr int t = decltype(T)::value;
    const double bt = row_bcast_c<t>(b);
    const double nb = fma(-row[t], bt, b);
    b = a > t ? nb : b;
  });
  if (a == NS - 1) b *= row[NS - 1];
  double fin[NS];
  fin[NS - 1] = row_bcast_c<NS - 1>(b);
  static_for<0, NS - 1>([&](auto I) {
    constexpr int r = NS - 2 - decltype(I)::value;
    double v = b;
#pragma unroll
    for (int t = r + 1; t < NS; ++t) v = fma(-row[t], fin[t], v);
    v *= row[r];
    b = a == r ? v : b;
    fin[r] = row_bcast_c<r>(b);
  });
  return b;
}

// Integration state of the row's cell (replicated across the row, species values per lane).
struct RowCell {
  double y; // rho Y of this lane's species (0 beyond NS)
  double rho, E, T, time, h, err_last, dt;
  int steps, rejects, attempts;
};

// One ROK4E attempt of the row's cell: the one-lane rok4e_attempt, species-parallel.
template<int NS>
__device__ __forceinline__ void row_attempt(const ChemMech &m, const MechLds &S, RowLds &X, int a, int gl,
                                            RowCell &s, double rtol, double atol) {
  const bool own = gl < NS; // lanes beyond NS carry zeros
  const double dt = s.dt;
  double Jrow[NS];
  const double rem = dt - s.time;
  const double hs = s.h * kStretch >= rem ? rem : s.h;
  const double irho = 1.0 / s.rho;
  double k1 = 0, k2 = 0, k3 = 0, w = 0, ys = s.y, Ts = s.T, err = 0;
  int src = 0;
#pragma unroll 1
  for (int st = 0; st < 5; ++st) {
    if (st != 3) { // the fourth stage takes the third's source
      if (st < 4) ys = stage_state(st, s.y, hs, k1, k2);
      // st 4: ys is the new state, and an accepted step gets its temperature from the old one
      if (st > 0 && (st < 4 || err <= 1)) Ts = row_update_t<NS>(m, S, X, a, gl, st == 4 ? s.T : Ts, own ? ys * irho : 0.0, s.E);
      if (st == 4) break;
      w = row_source<NS>(m, S, X, a, gl, Ts, ys, st == 0, Jrow);
      if (st == 0) {
#pragma unroll
        for (int n = 0; n < NS; ++n) {
          const double j = -hs * G * Jrow[n];
          Jrow[n] = n == a ? j + 1.0 : j;
        }
        src = row_lu<NS>(Jrow, a);
      }
    }
    const double c = stage_sum(st, k1, k2, k3);
    const double k = row_solve<NS>(Jrow, a, src, w + c) - c;
    if (st == 0) k1 = k;
    else if (st == 1) k2 = k;
    else if (st == 2) k3 = k;
    else {
      ys = new_state(s.y, hs, k1, k2, k);
      const double dy = error_term(ys, hs, k1, k2, k3, k, rtol, atol);
      err = sqrt(row_sum(own ? dy * dy : 0.0) / NS);
    }
  }
  double hstar = hs;
  if (s.steps > 0) hstar *= step_factor(s.err_last, err);
  else if (!(err <= 1)) hstar *= 0.2;
  if (err <= 1 && hs < s.h) hstar = fmax(hstar, s.h);
  s.h = hstar;
  ++s.attempts;
  if (err <= 1) {
    s.y = own ? ys : 0.0;
    s.time += hs;
    s.err_last = fmax(err, 1e-30);
    s.T = Ts;
    ++s.steps;
  } else {
    ++s.rejects;
  }
}


__device__ __forceinline__ int work_count(const ChemBatch &b) { return b.list ? *b.n_list : b.n; }
__device__ __forceinline__ int work_cell(const ChemBatch &b, int w) { return b.list ? b.list[w] : w; }

template<int NS>
__global__ __launch_bounds__(256) void k_chem_coop(const ChemMech *__restrict__ mp, ChemBatch b, double dt,
                                                   double rtol, double atol, int max_attempts, int *counter,
                                                   int resume) {
  __shared__ MechLds S;
  __shared__ RowLds rows[256 / RW];
  const int n_work = work_count(b);
  // work-groups beyond one row per cell would find the queue empty
  if ((long)blockIdx.x * (blockDim.x / RW) >= n_work) return;
  const ChemMech &m = *mp;
  stage_mechanism(m, S);
  if (threadIdx.x < blockDim.x / RW) {
    rows[threadIdx.x].c[kPad] = 1.0;
    rows[threadIdx.x].g[kPad] = 0.0;
  }
  __syncthreads();
  const int lane = __lane_id();
  const int gl = lane & (RW - 1);
  const int a = gl < NS ? gl : 0; // species of this lane (lanes beyond NS mirror species 0 and carry zeros)
  RowLds &X = rows[threadIdx.x / RW];
  RowCell s;
  int cell = -1;
  bool exhausted = false;
  while (true) {
    // one atomic per wave per fetch round; lane 0 of each row that needs a cell takes one
    const bool need = gl == 0 && cell < 0 && !exhausted;
    const unsigned long long mask = __ballot(need);
    if (mask) {
      const int leader = __ffsll((long long)mask) - 1;
      int base = 0;
      if (lane == leader) base = atomicAdd(counter, __popcll(mask));
      base = __shfl(base, leader, 64);
      int got = need ? base + __popcll(mask & ((1ull << lane) - 1)) : 0;
      got = __shfl(got, 0, RW);
      const bool row_needs = __shfl((int)need, 0, RW) != 0;
      if (row_needs) {
        if (got < n_work) {
          cell = work_cell(b, got);
          const double dtc = cell_dt(b, cell, dt);
          s.y = gl < NS ? b.rhoY[(long)gl * b.n + cell] : 0.0;
          s.rho = b.rho[cell];
          s.E = b.e[cell];
          s.T = b.T[cell];
          s.dt = dtc;
          if (resume) {
            s.h = b.h[cell];
            s.time = b.tcur[cell];
            s.err_last = b.elast[cell];
            s.steps = b.steps[cell];
            s.rejects = b.rejects[cell];
          } else {
            s.h = b.h[cell] > 0 ? fmin(b.h[cell], dtc) : dtc;
            s.time = 0;
            s.err_last = 0;
            s.steps = s.rejects = 0;
          }
          s.attempts = s.steps + s.rejects;
        } else {
          exhausted = true;
        }
      }
    }
    if (__ballot(cell >= 0) == 0) break;
    if (cell >= 0) {
      if (s.time < s.dt && s.attempts < max_attempts) row_attempt<NS>(m, S, X, a, gl, s, rtol, atol);
      if (s.time >= s.dt || s.attempts >= max_attempts) {
        if (gl < NS) b.rhoY[(long)gl * b.n + cell] = s.y;
        if (gl == 0) {
          b.T[cell] = s.T;
          b.h[cell] = s.h;
          b.steps[cell] = s.time >= s.dt ? s.steps : -1;
          b.rejects[cell] = s.rejects;
        }
        cell = -1;
      }
    }
  }
}

} // namespace

hipError_t launch_chem_coop(const ChemMech *mech_dev, int ns, const ChemBatch &b, double dt, double rtol,
                            double atol, int max_attempts, int threads, int blocks, bool resume, int *counter,
                            hipStream_t s) {
  if (ns != 9) return hipErrorNotSupported;
  if (b.n == 0) return hipSuccess;
  if (threads != 64 && threads != 128 && threads != 256) return hipErrorInvalidValue;
  if (blocks < 1) return hipErrorInvalidValue;
  k_chem_coop<9><<<blocks, threads, 0, s>>>(mech_dev, b, dt, rtol, atol, max_attempts, counter, resume ? 1 : 0);
  return hipGetLastError();
}

} // namespace corefl
