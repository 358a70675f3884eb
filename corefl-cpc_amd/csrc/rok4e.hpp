// Coefficients of the 4-stage Rosenbrock method ROK4E with its embedded error estimate (Define.h:28-43), in
// the scaled form both chemistry integrators use: stage vectors solve (I - h G J) k = f, the G_ij are divided
// by G, and E_i are the error weights.
#pragma once

namespace corefl {
namespace rok4e {

constexpr double G = 0.572816062482135;
constexpr double A21 = 0.432364435748567, A31 = -0.51421131687617, A32 = 1.38227114461736;
constexpr double G21 = -0.602765307997356 / G, G31 = -1.389195789724843 / G, G32 = 1.072950969011413 / G;
constexpr double G41 = 0.992356412977094 / G, G42 = -1.390032613873701 / G, G43 = -0.440875890223325 / G;
constexpr double B1 = 0.194335256262729, B2 = 0.483167813989227, B4 = 0.322496929748044;
constexpr double E1 = -0.217819895945721 - B1, E2 = 1.03130847478467 - B2, E3 = 0.186511421161047, E4 = -B4;

// By stage: the weights of k1, k2 in the stage's state, and of k1, k2, k3 in its right-hand side.
__constant__ const double kStageA[4][2] = {{0, 0}, {A21, 0}, {A31, A32}, {A31, A32}};
__constant__ const double kStageG[4][3] = {{0, 0, 0}, {G21, 0, 0}, {G31, G32, 0}, {G41, G42, G43}};

// A step whose size h satisfies kStretch h >= (time left in the interval) is taken to the interval's end.
constexpr double kStretch = 1.05;

// A stage's state, the sum of earlier stages in its right-hand side, the new state and one species' term of the error
// estimate, one rounding for both integrators.
__device__ __forceinline__ double stage_state(int st, double y, double hs, double k1, double k2) {
  return fma(hs, fma(kStageA[st][0], k1, kStageA[st][1] * k2), y);
}
__device__ __forceinline__ double stage_sum(int st, double k1, double k2, double k3) {
  return fma(kStageG[st][0], k1, fma(kStageG[st][1], k2, kStageG[st][2] * k3));
}
__device__ __forceinline__ double new_state(double y, double hs, double k1, double k2, double k4) {
  return fma(hs, fma(B1, k1, fma(B2, k2, B4 * k4)), y);
}
__device__ __forceinline__ double error_term(double y, double hs, double k1, double k2, double k3, double k4, double rtol, double atol) {
  return hs * fma(E1, k1, fma(E2, k2, fma(E3, k3, E4 * k4))) / fma(rtol, y, atol);
}

// The PI controller's step factor after the first step, 0.8 err_last^0.1 (err + 1e-20)^-0.175 in [0.2, 5], its two powers
// as one exponential of logarithms.
__device__ __forceinline__ double step_factor(double err_last, double err) {
  return fmin(5.0, fmax(0.2, 0.8 * exp(fma(0.1, log(err_last), -0.175 * log(err + 1e-20)))));
}

} // namespace rok4e
} // namespace corefl
