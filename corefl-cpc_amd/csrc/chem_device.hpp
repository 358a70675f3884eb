// Device thermo and kinetics of one cell, shared by the chemistry and surrogate kernels: NASA-7 h, cp and
// g/RT, Arrhenius / third-body / Lindemann / Troe rates with Gibbs-energy reverse rates, the chemical source
// and its Jacobian, and the Newton temperature at fixed internal energy.  FP64.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

#include "chem.hpp"

namespace corefl {
namespace chemdev {

// The one-lane and the cooperative integrator hand cells to one another at moments that scheduling sets, so both have to
// give a cell the same bits: what they share is written once, here and in rok4e.hpp, with every fused multiply-add spelled
// out and every sum in one order, and the files of both are compiled without contraction (but for the differences
// x -= a b marked so, where a negation written out would be an instruction of its own).

constexpr double kRu = 8314.462618, kPatm = 101325.0;
// constant divisions of the polynomial fits as products (a few ulp from the divided form)
constexpr double kThird = 1.0 / 3.0, kSixth = 1.0 / 6.0, kTwelfth = 1.0 / 12.0;

// The mechanism behind a pointer the optimiser cannot see through: its loads stay where they are used.  Hoisted out of
// the loops around them, a mechanism's hundreds of uniform values overflow the scalar registers, and every use becomes a
// read from a vector register's lane.
__device__ __forceinline__ const ChemMech &opaque(const ChemMech *mp) {
  typedef const __attribute__((address_space(4))) ChemMech *ConstMech;
  ConstMech mc = (ConstMech)mp;
  asm volatile("" : "+s"(mc));
  return *(const ChemMech *)mc;
}

// Which fit coefficients a wavefront needs: the low ones where every active lane is below the middle of the common fit
// range, the high ones where every lane is above it, else each lane its own (a flame front, ranges that differ between
// species, NaN).  On one side the coefficients are uniform scalar loads; lane by lane they are 27 vector loads of 16
// bytes for the nine species, at 1 wave per SIMD a wait for each.
enum FitSide { kFitLow, kFitHigh, kFitMixed };
__device__ __forceinline__ FitSide fit_side(const ChemMech &m, double t) {
  if (!m.common_range) return kFitMixed;
  if (__all(t < m.ct_mid)) return kFitLow;
  if (__all(t >= m.ct_mid)) return kFitHigh;
  return kFitMixed;
}

// h_k and cp_k per unit mass (Thermo.cu:470-520): the fit at the temperature clamped to [t_low, t_high], continued
// linearly outside (inside, the term (t - tt) cp is an exact zero).
__device__ __forceinline__ void h_cp_fit(const double *c, double R, double t, double tt, double &h, double &cp) {
  // fused multiply-adds written out: the copies for uniform and for per-lane coefficients round alike
  const double cc = fma(tt, fma(tt, fma(tt, fma(tt, c[4], c[3]), c[2]), c[1]), c[0]);
  const double hh = fma(tt, fma(tt, fma(tt, fma(tt, fma(tt, 0.2 * c[4], 0.25 * c[3]), c[2] * kThird), 0.5 * c[1]), c[0]), c[5]);
  h = fma(cc, t - tt, hh) * R;
  cp = cc * R;
}

template<int NS> __device__ __forceinline__ void h_cp(const ChemMech &m, double t, double *h, double *cp) {
  const FitSide side = fit_side(m, t);
  if (side != kFitMixed) {
    const double(*c)[7] = side == kFitLow ? m.lo : m.hi;
    const double tt = fmin(fmax(t, m.ct_low), m.ct_high);
#pragma unroll
    for (int i = 0; i < NS; ++i) h_cp_fit(c[i], kRu * m.imw[i], t, tt, h[i], cp[i]);
    return;
  }
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    const double tt = t < m.t_low[i] ? m.t_low[i] : (t > m.t_high[i] ? m.t_high[i] : t);
    const bool low = t < m.t_low[i] || (!(t > m.t_high[i]) && t < m.t_mid[i]);
    h_cp_fit(low ? m.lo[i] : m.hi[i], kRu * m.imw[i], t, tt, h[i], cp[i]);
  }
}

// g_k / (R T), clamped to the fit range (Thermo.cu:574-598).  lnT = log(t): one logarithm serves every
// species whose fit range holds t; the logarithms of the range ends are tabulated.
__device__ __forceinline__ double gibbs_fit(const double *c, double tt, double lt, double itt) {
  const double p = fma(tt, fma(tt, fma(tt, c[4] * 0.05, c[3] * kTwelfth), c[2] * kSixth), 0.5 * c[1]);
  return fma(-tt, p, fma(c[0], 1.0 - lt, fma(c[5], itt, -c[6])));
}

template<int NS>
__device__ __forceinline__ void gibbs(const ChemMech &m, double t, double lnT, double iT, double *g) {
  const FitSide side = fit_side(m, t);
  if (side != kFitMixed) {
    const double(*c)[7] = side == kFitLow ? m.lo : m.hi;
    const bool below = t < m.ct_low, above = t > m.ct_high;
    const double tt = below ? m.ct_low : (above ? m.ct_high : t);
    const double lt = below ? m.c_ln_low : (above ? m.c_ln_high : lnT);
    const double itt = below ? m.c_inv_low : (above ? m.c_inv_high : iT);
#pragma unroll
    for (int i = 0; i < NS; ++i) g[i] = gibbs_fit(c[i], tt, lt, itt);
    return;
  }
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    const bool below = t < m.t_low[i], above = t > m.t_high[i];
    const double tt = below ? m.t_low[i] : (above ? m.t_high[i] : t);
    const double *c = below ? m.lo[i] : (above ? m.hi[i] : (t < m.t_mid[i] ? m.lo[i] : m.hi[i]));
    const double lt = below ? m.ln_t_low[i] : (above ? m.ln_t_high[i] : lnT);
    const double itt = below ? m.inv_t_low[i] : (above ? m.inv_t_high[i] : iT);
    g[i] = gibbs_fit(c, tt, lt, itt);
  }
}

// A T^b exp(-Ea/T) as A exp(b ln T - Ea/T): one exponential per rate instead of a power and an exponential
// (the same value up to rounding).
__device__ __forceinline__ double arrhenius(double lnT, double iT, double A, double b, double Ea) {
  return A * exp(fma(b, lnT, -(Ea * iT)));
}

// x^k for an integer k (reaction orders and stoichiometric coefficients are integers: the parser rejects
// others), by repeated products as the reference's integer branch does.
__device__ __forceinline__ double int_pow(double x, int k) {
  const int n = k < 0 ? -k : k;
  double r = 1.0;
  for (int q = 0; q < n; ++q) r *= x;
  return k < 0 ? 1.0 / r : r;
}

// N sums over the species as the cooperative kernel's 16 lanes form them: the two halves, then quarters, pairs and
// neighbours (the places beyond NS hold zeros there).  term(l, v) gives species l's terms; they are taken as they are
// added, so that few are alive at a time.
template<int NS, int N, class F> __device__ __forceinline__ void species_sums(F &&term, double (&sum)[N]) {
  static_assert(NS <= 16);
  auto eighth = [&](int i, double (&v)[N]) { // places i and i + 8
#pragma unroll
    for (int q = 0; q < N; ++q) v[q] = 0.0;
    if (i < NS) term(i, v);
    if (i + 8 < NS) {
      double x[N];
      term(i + 8, x);
#pragma unroll
      for (int q = 0; q < N; ++q) v[q] += x[q];
    }
  };
  auto quarter = [&](int i, double (&v)[N]) {
    double x[N];
    eighth(i, v);
    eighth(i + 4, x);
#pragma unroll
    for (int q = 0; q < N; ++q) v[q] += x[q];
  };
  auto half = [&](int i, double (&v)[N]) {
    double x[N];
    quarter(i, v);
    quarter(i + 2, x);
#pragma unroll
    for (int q = 0; q < N; ++q) v[q] += x[q];
  };
  double x[N];
  half(0, sum);
  half(1, x);
#pragma unroll
  for (int q = 0; q < N; ++q) sum[q] += x[q];
}
template<int NS> __device__ __forceinline__ double species_sum(const double *x) {
  double sum[1];
  species_sums<NS>([&](int l, double (&v)[1]) { v[0] = x[l]; }, sum);
  return sum[0];
}

// Forward rate constant of a reaction of type ty: cc its third-body concentration (types 4 and up), troe(k) its fall-off
// parameters.
template<class Troe>
__device__ __forceinline__ double forward_rate(int ty, double A, double b, double Ea, double A2, double b2, double Ea2, double t,
                                               double lnT, double iT, double cc, Troe &&troe) {
  double kf = arrhenius(lnT, iT, A, b, Ea);
  if (ty == 3) {
    kf += arrhenius(lnT, iT, A2, b2, Ea2);
  } else if (ty == 4) {
    kf *= cc;
  } else if (ty > 4) {
    const double klow = arrhenius(lnT, iT, A2, b2, Ea2), khigh = kf;
    if (khigh < 1e-25 && klow < 1e-25) {
      kf = 0;
    } else {
      const double pr = klow * cc / khigh;
      double F = 1.0;
      if (ty > 5) {
        const double a = troe(0);
        double fc = fma(1 - a, exp(-t / troe(1)), a * exp(-t / troe(2)));
        if (ty == 7) fc += exp(-troe(3) * iT);
        const double lfc = log10(fc);
        const double cq = fma(-0.67, lfc, -0.4), nq = fma(-1.27, lfc, 0.75);
        const double lpr = log10(pr);
        const double tmp = (lpr + cq) / fma(-0.14, lpr + cq, nq);
        F = exp(2.302585092994046 * lfc / fma(tmp, tmp, 1.0)); // 10^x
      }
      kf = khigh * pr / (1.0 + pr) * F;
    }
  }
  return kf;
}

// Reverse rate constant from the forward one: dg the sum of nu g / (R T) over the products less that over the reactants,
// tp and itp p_atm / (R T) in kmol/m^3 and its reciprocal; kf / (tp^order exp(-dg)), without dividing.
__device__ __forceinline__ double gibbs_reverse(double kf, double dg, int order, double tp, double itp) {
  return kf * exp(dg) * int_pow(order < 0 ? tp : itp, order < 0 ? -order : order);
}

// Chemical source omega [kg/(m^3 s)] of one cell (FiniteRateChem.cu:1466-1605).  With JAC, also the
// Jacobian d omega / d(rho Y) with the rates of progress frozen (ConstVolumeReactor.cpp:1168-1187); columns of
// species with rho Y at or below floor are zero (1e-30 in the reactor, 1e-25 in Wu's EPI, StrangSplitting.cu:164).
// jac = false (uniform) leaves J alone.  With WD, also the destruction rates.
// Stoichiometry is walked through each reaction's species lists (a few entries) rather than all species, the net rate
// of a reaction added once per species; the Jacobian keeps static indices (register-resident) and skips rows and
// columns through the reaction's species bit masks.
template<int NS, bool JAC, bool WD = false>
__device__ __forceinline__ void source(const ChemMech &m, double t, const double *rhoY, double *w, double *J,
                                       double *wd = nullptr, double floor = 1e-30, bool jac = JAC) {
  double c[NS], g[NS], net[NS], de[NS];
#pragma unroll
  for (int l = 0; l < NS; ++l) {
    c[l] = rhoY[l] * m.imw[l] * 1e-3;
    net[l] = 0;
    de[l] = 0;
  }
  if constexpr (JAC) {
    if (jac)
#pragma unroll
      for (int q = 0; q < NS * NS; ++q) J[q] = 0;
  }
  const double lnT = log(t), iT = 1.0 / t;
  // Equilibrium constants are needed unless every reversible reaction carries explicit REV parameters
  // (FiniteRateChem.cu:1519-1557); then they are applied to every reaction of type other than 0 and 2.
  if (m.need_gibbs) gibbs<NS>(m, t, lnT, iT, g);
  const double tp = kPatm / kRu * 1e-3 * iT, itp = kRu / kPatm * 1e+3 * t;
  for (int r = 0; r < m.nr; ++r) {
    const ReacRecord q = m.rec[r];
    const int ty = q.type;
    const int nfs = q.n_sides & 255, nbs = q.n_sides >> 8;
    auto sp = [](unsigned s, int k) { return (int)(s >> 8 * k & 255u); };
    auto nu = [](unsigned long long s, int k) { return (int)(short)(s >> 16 * k & 65535u); };
    double cc = 0;
    if (ty >= 4) {
      double tb[NS];
#pragma unroll
      for (int l = 0; l < NS; ++l) tb[l] = m.tb[r][l];
#pragma unroll
      for (int l = 0; l < NS; ++l) cc = fma(c[l], tb[l], cc);
    }
    const double kf = forward_rate(ty, q.A, q.b, q.Ea, q.A2, q.b2, q.Ea2, t, lnT, iT, cc, [&](int k) { return q.troe[k]; });
    double kb = 0;
    if (ty != 0 && q.rev == 1) {
      kb = arrhenius(lnT, iT, q.A2, q.b2, q.Ea2);
      if (ty == 4) kb *= cc;
    }
    if (m.need_gibbs && ty != 0 && ty != 2) {
      double dg = 0;
      for (int s = 0; s < nfs; ++s) dg = fma(g[sp(q.fsp, s)], -(double)nu(q.fnu, s), dg);
      for (int s = 0; s < nbs; ++s) dg = fma(g[sp(q.bsp, s)], (double)nu(q.bnu, s), dg);
      kb = gibbs_reverse(kf, dg, q.iorder, tp, itp);
    }
    double q1 = 1.0, q2 = ty != 0 ? 1.0 : 0.0;
    for (int s = 0; s < nfs; ++s) q1 *= int_pow(c[sp(q.fsp, s)], nu(q.fnu, s));
    if (ty != 0)
      for (int s = 0; s < nbs; ++s) q2 *= int_pow(c[sp(q.bsp, s)], nu(q.bnu, s));
    q1 *= kf;
    q2 *= kb;
    const double qn = q1 - q2;
    for (int s = 0; s < nfs; ++s) {
      const int l = sp(q.fsp, s);
      const double n = nu(q.fnu, s);
      net[l] = fma(-n, qn, net[l]);
      if constexpr (WD) de[l] += q1 * n;
    }
    for (int s = 0; s < nbs; ++s) {
      const int l = sp(q.bsp, s);
      const double n = nu(q.bnu, s);
      net[l] = fma(n, qn, net[l]);
      if constexpr (WD) de[l] += q2 * n;
    }
    if constexpr (JAC) {
      if (!jac) continue;
      // the rows of the stoichiometric tables whole, a few wide loads, instead of entry by entry behind the mask bits
      const unsigned um = q.umask, am = q.amask;
      double v[NS], dn[NS];
#pragma unroll
      for (int n = 0; n < NS; ++n) {
        v[n] = fma(m.nf[r][n], q1, -(m.nb[r][n] * q2));
        dn[n] = m.dnu[r][n];
      }
#pragma unroll
      for (int a = 0; a < NS; ++a) {
        if (!(am >> a & 1u)) continue;
#pragma unroll
        for (int n = 0; n < NS; ++n)
          if (um >> n & 1u) J[a * NS + n] = fma(dn[a], v[n], J[a * NS + n]);
      }
    }
  }
#pragma unroll
  for (int l = 0; l < NS; ++l) {
    w[l] = net[l] * (1e+3 * m.mw[l]);
    if constexpr (WD) wd[l] = de[l] * (1e+3 * m.mw[l]);
  }
  if constexpr (JAC) {
    if (!jac) return;
#pragma unroll
    for (int n = 0; n < NS; ++n) {
      const double inv = rhoY[n] > floor ? 1.0 / rhoY[n] : 0.0;
#pragma unroll
      for (int a = 0; a < NS; ++a) J[a * NS + n] = J[a * NS + n] * inv * (1e+3 * m.mw[a]);
    }
  }
}

// Doolittle LU with partial pivoting, row-major (ConstVolumeReactor.cpp:1231-1262), and its solve.
template<int NS> __device__ __forceinline__ void lu(double *a, int *piv) {
#pragma clang fp contract(fast)
#pragma unroll
  for (int k = 0; k < NS; ++k) {
    // first row of largest |a[r][k]|; the running maximum keeps every array index static, so the matrix
    // stays in registers
    int ik = k;
    double amax = 0;
#pragma unroll
    for (int r = k; r < NS; ++r) {
#pragma unroll
      for (int t = 0; t < k; ++t) a[r * NS + k] -= a[r * NS + t] * a[t * NS + k];
      const double v = fabs(a[r * NS + k]);
      if (r == k) {
        amax = v;
      } else if (v > amax) {
        amax = v;
        ik = r;
      }
    }
    piv[k] = ik;
    // row exchange through value selects: every index stays static and no branch is formed (a branch per
    // candidate row lets the optimiser merge them into stores through a chosen address, which sends the
    // whole matrix to scratch memory); skipped where no lane exchanges anything, as in all but the stiff cells
    if (__any(ik != k))
#pragma unroll
    for (int r = k + 1; r < NS; ++r) {
      const bool sw = r == ik;
#pragma unroll
      for (int t = 0; t < NS; ++t) {
        const double x = a[r * NS + t], y = a[k * NS + t];
        a[r * NS + t] = sw ? y : x;
        a[k * NS + t] = sw ? x : y;
      }
    }
#pragma unroll
    for (int p = k + 1; p < NS; ++p)
#pragma unroll
      for (int t = 0; t < k; ++t) a[k * NS + p] -= a[k * NS + t] * a[t * NS + p];
    const double inv = 1.0 / a[k * NS + k];
#pragma unroll
    for (int r = k + 1; r < NS; ++r) a[r * NS + k] *= inv;
    a[k * NS + k] = inv; // the solve multiplies by the reciprocal pivot
  }
}

template<int NS> __device__ __forceinline__ void lu_solve(const double *a, const int *piv, double *b) {
#pragma clang fp contract(fast)
#pragma unroll
  for (int r = 0; r < NS; ++r) {
    if (__any(piv[r] != r))
#pragma unroll
    for (int q = r + 1; q < NS; ++q) {
      const bool sw = piv[r] == q;
      const double x = b[q], y = b[r];
      b[q] = sw ? y : x;
      b[r] = sw ? x : y;
    }
  }
#pragma unroll
  for (int r = 1; r < NS; ++r)
#pragma unroll
    for (int t = 0; t < r; ++t) b[r] -= a[r * NS + t] * b[t];
  b[NS - 1] *= a[NS * NS - 1];
#pragma unroll
  for (int r = NS - 2; r >= 0; --r) {
#pragma unroll
    for (int t = r + 1; t < NS; ++t) b[r] -= a[r * NS + t] * b[t];
    b[r] *= a[r * NS + r];
  }
}

// Newton iteration T -> T - (h - R T - e) / (cp - R) for the mixture of mass fractions yk until the relative change is
// at most tol (at most `most` times).  With a common fit range the iteration runs on the mixture's own fit (54 products,
// again for a lane that crosses the middle of the range) instead of nine species fits per iteration.
template<int NS>
__device__ __forceinline__ double newton_t(const ChemMech &m, double t, const double *yk, double R, double E, double tol, int most) {
  double err = 1e+6;
  int it = 0;
  if (m.common_range) {
    double C[6];
    int side = -1; // 0: C holds the low fit, 1: the high one
#pragma unroll 1
    for (; it < most && err > tol; ++it) {
      const int now = t < m.ct_mid ? 0 : 1;
      if (__any(now != side)) {
        const bool fresh = now != side;
        auto mix = [&](const double(*c)[7]) {
          double D[6] = {};
#pragma unroll
          for (int l = 0; l < NS; ++l) {
            const double yr = yk[l] * (kRu * m.imw[l]);
#pragma unroll
            for (int q = 0; q < 6; ++q) D[q] = fma(yr, c[l][q], D[q]);
          }
#pragma unroll
          for (int q = 0; q < 6; ++q) C[q] = fresh ? D[q] : C[q];
        };
        if (__all(now == 0)) mix(m.lo);
        else if (__all(now == 1)) mix(m.hi);
        else mix(now ? m.hi : m.lo);
        side = now;
      }
      double h, cp;
      h_cp_fit(C, 1.0, t, fmin(fmax(t, m.ct_low), m.ct_high), h, cp);
      const double t1 = t - (fma(-R, t, h) - E) / (cp - R);
      err = fabs(1 - t1 / t);
      t = t1;
    }
    return t;
  }
#pragma unroll 1
  for (; it < most && err > tol; ++it) {
    double hc[2];
    species_sums<NS>([&](int l, double (&v)[2]) {
      const double lo = m.t_low[l], hi = m.t_high[l], tt = t < lo ? lo : (t > hi ? hi : t);
      const bool low = t < lo || (!(t > hi) && t < m.t_mid[l]);
      h_cp_fit(low ? m.lo[l] : m.hi[l], yk[l] * (kRu * m.imw[l]), t, tt, v[0], v[1]);
    }, hc);
    const double t1 = t - (fma(-R, t, hc[0]) - E) / (hc[1] - R);
    err = fabs(1 - t1 / t);
    t = t1;
  }
  return t;
}

// T at fixed specific internal energy E (ConstVolumeReactor.cpp:970-995).
template<int NS> __device__ __forceinline__ double update_t(const ChemMech &m, double t, const double *yk, double E) {
  double x[NS];
#pragma unroll
  for (int l = 0; l < NS; ++l) x[l] = yk[l] * m.imw[l];
  return newton_t<NS>(m, t, yk, kRu * species_sum<NS>(x), E, 1e-8, 100);
}

// The coefficients of (1 + r)^-power.
struct PowerSeries {
  double c[11];
  constexpr explicit PowerSeries(double power) : c{1.0} {
    for (int k = 1; k < 11; ++k) c[k] = c[k - 1] * (-power - (k - 1)) / k;
  }
};

// What the collision integrals of a node's pairs share: t bounded to the table's range, T^-0.15504 and what its
// argument's rounding left out.
struct OmegaNode {
  double t, p, pl;
};

__device__ __forceinline__ OmegaNode omega_node(const ChemMech &m, double t, double lt) {
  const double a = -kOmegaSlow * lt, p = exp(a);
  return {fmin(t, m.t_omega), p, p * __builtin_fma(-kOmegaSlow, lt, -a)};
}

// Collision integral of binary diffusion of the pair (a, b) (Transport.cu:188-190), T* = T k_B / eps_ab:
// 1.0548 T*^-0.15504 + (T* + 0.55909)^-2.1705.  The first power is the node's times the pair's constant, the second comes
// from the mechanism's table by the leading 16 bits of T* + 0.55909 and a series in |r| < 0.031, cut where its next term
// is 4e-17: 20 instructions against the 110 of one logarithm and two exponentials.  Largest error against the exact value 2.8e-16
// (3.4e-16 before) at T from 200 to 4000 K and eps / k_B from 10 to 600 K.
__device__ __forceinline__ double omega_d(const ChemMech &m, const OmegaNode &w, int a, int b) {
  const double kbe = m.kbe[a][b];
  const double x = __builtin_fma(w.t, kbe, kOmegaShift), xl = __builtin_fma(w.t, kbe, kOmegaShift - x);
  // 0x3FE0: 1/2; the bound holds the index where a well depth of zero or less makes x negative or NaN (the pair's omega_hi
  // or the series is NaN then, and so is the result)
  const unsigned n = min((unsigned)(__double2hiint(x) >> 16) - 0x3FE0u, (unsigned)kOmegaTable - 1u);
  const double s = m.omega_table[n][0], e = m.omega_table[n][1];
  const double r = __builtin_fma(xl, s, __builtin_fma(x, s, -1.0));
  constexpr PowerSeries series(kOmegaPower);
  double q = series.c[10];
#pragma unroll
  for (int k = 9; k > 0; --k) q = __builtin_fma(q, r, series.c[k]);
  const double fast = __builtin_fma(e * r, q, e);
  return __builtin_fma(w.p, m.omega_hi[a][b], __builtin_fma(w.p, m.omega_lo[a][b], __builtin_fma(w.pl, m.omega_hi[a][b], fast)));
}

// compute_transport_property (Transport.cu:43-150) at temperature t and mass fractions y (cp: species cp per
// unit mass at t): Chapman-Enskog species viscosities mixed by Wilke's rule; species conductivities from
// Eucken's relation with the rotational-relaxation correction of linear and nonlinear molecules, mixed with
// the 1.065 factor; mixture-averaged rho D_k from the binary coefficients.
template<int NS>
__device__ inline void transport(const ChemMech &m, double t, const double *y, const double *cp, double &mu,
                                 double &lambda, double *rhoD) {
  // The reference's formulas with their powers of the reduced temperatures T k_B / eps written as exponentials
  // of ln T + ln(k_B / eps) (one logarithm per node instead of one per power), 1/(x x) for x^-2, and products
  // with tabulated or once-computed reciprocals in place of divisions: equal to the direct form to a few ulps.
  constexpr double pi = 3.14159265358979323846, Ru = 8314.462618;
  double x[NS], vs[NS];
  double imw = 0;
#pragma unroll
  for (int l = 0; l < NS; ++l) imw += y[l] * m.imw[l];
  const double mwt = 1.0 / imw;
  const double st = sqrt(t), lt = log(t);
  OmegaNode w = omega_node(m, t, lt);
#pragma unroll
  for (int l = 0; l < NS; ++l) {
    x[l] = y[l] * mwt * m.imw[l];
    const double td = t * m.lj_inv[l], u = td + 0.5;
    vs[l] = m.vis_coeff[l] * st * (u * u) / (1.147 * exp(-0.145 * (lt + m.log_lj_inv[l])) * (u * u) + 1.0);
  }
  double isq[NS];
#pragma unroll
  for (int l = 0; l < NS; ++l) isq[l] = 1.0 / sqrt(vs[l]);
  mu = 0;
  lambda = 0;
#pragma unroll
  for (int a = 0; a < NS; ++a) {
    const double R = Ru * m.imw[a];
    double lam = 15 * 0.25 * vs[a] * R;
    const int geom = m.geometry[a];
    if (geom == 1 || geom == 2) {
      const bool linear = geom == 1;
      const double tri = 1 / (t * m.kbe[a][a]);
      const double q = sqrt(tri * pi) * pi;
      const double ft = 1 + 0.5 * q + (2 + 0.25 * pi * pi) * tri + q * tri;
      const double rd = m.bdc[a][a] * st / (omega_d(m, w, a, a) * R);
      const double ab = (2.5 * vs[a] - rd) * ft / (pi * m.zrot[a] * vs[a] + ((linear ? 10.0 / 3 : 5.0) * vs[a] + 2.0 * rd) * ft);
      lam += (linear ? -5 : -7.5) * ab * vs[a] * R + rd * cp[a] + rd * ((linear ? 2 : 3) * ab - 2.5) * R;
    }
    double den = 0;
    const double sa = sqrt(vs[a]);
#pragma unroll
    for (int b = 0; b < NS; ++b) {
      double phi = 1.0;
      if (a != b) {
        const double num = 1.0 + sa * isq[b] * m.wdw[a][b];
        phi = num * num * m.sqw[a][b];
      }
      den += phi * x[b];
    }
    mu += vs[a] * x[a] / den;
    lambda += lam * x[a] / (1.065 * den - 0.065 * x[a]);
    asm volatile("" : "+v"(w.t), "+v"(lambda));
  }
  constexpr double eps = 1e-12;
  double num[NS], dsum[NS];
  double sum = 0;
#pragma unroll
  for (int l = 0; l < NS; ++l) {
    num[l] = (x[l] + eps) * m.mw[l];
    sum += num[l];
    dsum[l] = 0;
  }
  // one species' pairs at a time: the table's entries of all pairs requested at once need more registers than there are
#pragma unroll
  for (int l = 0; l < NS; ++l) {
#pragma unroll
    for (int n = l + 1; n < NS; ++n) {
      const double inv = omega_d(m, w, l, n) * m.inv_bdc[l][n];
      dsum[l] += (x[n] + eps) * inv;
      dsum[n] += (x[l] + eps) * inv;
    }
    asm volatile("" : "+v"(w.t), "+v"(dsum[l]));
  }
  const double f = st / Ru; // sqrt(T)^3 of the binary coefficients over R T
#pragma unroll
  for (int l = 0; l < NS; ++l) rhoD[l] = (sum - num[l]) * f / dsum[l];
}

} // namespace chemdev
} // namespace corefl
