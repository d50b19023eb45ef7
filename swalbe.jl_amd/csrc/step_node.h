// step_node.h -- the per-node arithmetic of the D2Q9 step shared by the step
// kernels: the FP64 expressions in the reference's order (no contraction) and
// the FP32 disjoining pressure.
#pragma once

#include "swalbe_batch.h"

namespace swalbe {

// power_broad's products in its order for the usual pairs without a run-time
// loop (1 a = a is exact; the m factors are the first m of the n); mode 1, 2:
// the raw-array forms fast_93, fast_32.
template <typename T>
__device__ __forceinline__ T powlaw(T a, int n, int m, int mode) {
  if (mode == 1) {
    const T t = (a * a) * a;
    return ((t * t) * t) - t;
  }
  if (mode == 2) return ((a * a) * a) - (a * a);
  if (n == 9 && m == 3) {
    const T a3 = (a * a) * a;
    const T a6 = ((a3 * a) * a) * a;
    return (((a6 * a) * a) * a) - a3;
  }
  if (n == 3 && m == 2) {
    const T a2 = a * a;
    return a2 * a - a2;
  }
  T tn = T(1), tm = T(1);
  for (int i = 0; i < n; ++i) tn *= a;
  for (int i = 0; i < m; ++i) tm *= a;
  return tn - tm;
}

// 1 / d refined to the point where a quotient by d takes three more operations:
// the instruction sequence of an IEEE FP64 division (v_rcp_f64, two Newton
// steps, quotient, residual correction: Markstein, IBM J. Res. Dev. 34 (1990)
// 111) without the scaling by cases.  Instead both operands are taken 2^64 times
// as large (S), so that the residual a - d q is exact down to subnormal a and the
// quotient the correctly rounded a / d, the compiler's bits, wherever a and d lie
// below 2^950 and d above 2^-12 (a subnormal quotient that lies halfway between
// two excepted).  Velocities do become that small: ahead of a front they halve
// with about every node, and 3 in 100 subnormal quotients come out wrong without.
// Zero, infinite and NaN operands go through v_div_fixup as in the compiler's
// sequence; operands beyond 2^950 count as infinite.  Several quotients by one d
// share the first six operations.  S costs two operations for a d and one quotient
// (0 to 3 % of a step, 4 of a line's of 3e6 nodes); a numerator that is a parameter
// of the film does without.
template <bool S = true>
struct Recip {
  double d, r;
  __device__ __forceinline__ explicit Recip(double den) : d(S ? den * 0x1p64 : den) {
    double x = __builtin_amdgcn_rcp(d);
    x = __builtin_fma(__builtin_fma(-d, x, 1.0), x, x);
    r = __builtin_fma(__builtin_fma(-d, x, 1.0), x, x);
  }
  __device__ __forceinline__ double div(double num) const {
    const double a = S ? num * 0x1p64 : num, q = a * r;
    return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-d, q, a), r, q), d, a);
  }
};

// Equilibrium population k at a node (src/equilibrium.jl:71-114), plain values.
template <typename T>
__device__ __forceinline__ T feq_k(int k, T h, T u, T v, T usq, T c56g, T g0) {
  const T w1 = T(1.0 / 9.0), w5 = T(1.0 / 36.0);
  T a;
  switch (k) {
    case 0: return h * ((T(1) - c56g * h) - T(2.0 / 3.0) * usq);
    case 1: return w1 * h * (((g0 * h + T(3) * u) + T(4.5) * (u * u)) - T(1.5) * usq);
    case 2: return w1 * h * (((g0 * h + T(3) * v) + T(4.5) * (v * v)) - T(1.5) * usq);
    case 3: return w1 * h * (((g0 * h - T(3) * u) + T(4.5) * (u * u)) - T(1.5) * usq);
    case 4: return w1 * h * (((g0 * h - T(3) * v) + T(4.5) * (v * v)) - T(1.5) * usq);
    case 5: a = u + v; return w5 * h * (((g0 * h + T(3) * a) + T(4.5) * (a * a)) - T(1.5) * usq);
    case 6: a = v - u; return w5 * h * (((g0 * h + T(3) * a) + T(4.5) * (a * a)) - T(1.5) * usq);
    case 7: a = u + v; return w5 * h * (((g0 * h - T(3) * a) + T(4.5) * (a * a)) - T(1.5) * usq);
    default: a = u - v; return w5 * h * (((g0 * h + T(3) * a) + T(4.5) * (a * a)) - T(1.5) * usq);
  }
}

// The same for g = 0, whose terms add or subtract an exact zero there.
template <typename T>
__device__ __forceinline__ T feq_k0(int k, T h, T u, T v, T usq) {
  const T w1 = T(1.0 / 9.0), w5 = T(1.0 / 36.0);
  if (k == 0) return h * (T(1) - T(2.0 / 3.0) * usq);
  const T a = k == 1 || k == 3 ? u : k == 2 || k == 4 ? v : k == 5 || k == 7 ? u + v
            : k == 6 ? v - u : u - v;
  const T lin = k == 3 || k == 4 || k == 7 ? -(T(3) * a) : T(3) * a;
  return (k <= 4 ? w1 : w5) * h * ((lin + T(4.5) * (a * a)) - T(1.5) * usq);
}

template <typename T>
__device__ __forceinline__ T force_term(int k, T Fx, T Fy) {
  const T c3 = T(1.0 / 3.0), c24 = T(1.0 / 24.0);
  switch (k) {
    case 1: return c3 * Fx;
    case 2: return c3 * Fy;
    case 3: return -(c3 * Fx);
    case 4: return -(c3 * Fy);
    case 5: return c24 * (Fx + Fy);
    case 6: return c24 * (Fy - Fx);
    case 7: return -(c24 * (Fx + Fy));
    case 8: return c24 * (Fx - Fy);
    default: return T(0);
  }
}

__device__ __forceinline__ float powlaw_f(float a, int n, int m, int mode) {
  if (mode == 1) {
    const float t = (a * a) * a;
    return (t * t - 1.0f) * t;
  }
  if (mode == 2) return (a - 1.0f) * (a * a);
  float tn = 1.0f, tm = 1.0f;
  for (int i = 0; i < n; ++i) tn *= a;
  for (int i = 0; i < m; ++i) tm *= a;
  return tn - tm;
}

__device__ __forceinline__ double powlaw_d(double a, int n, int m, int mode) {
  if (mode == 1) {
    const double t = (a * a) * a;
    return (t * t - 1.0) * t;
  }
  if (mode == 2) return (a - 1.0) * (a * a);
  double tn = 1.0, tm = 1.0;
  for (int i = 0; i < n; ++i) tn *= a;
  for (int i = 0; i < m; ++i) tm *= a;
  return tn - tm;
}

// The disjoining part of the film pressure, -γ κ [a^n - a^m] with
// a = hmin / (h + hcrit), at a node of stored height deviation dh.  Where the
// film nears hmin (h < hguard) the term dominates the pressure and is
// evaluated in FP64 from the stored height with an IEEE division; elsewhere
// in FP32 with v_rcp_f32.  kap is κ (a θ field's value, or the film's).
__device__ __forceinline__ float disjoining_f(const F32K& K, float dh, float kap, bool kap_field) {
#pragma clang fp contract(fast)
  const float hh = K.href + dh;
  if (K.guard && hh < K.hguard) {
    const double hd = K.href_d + (double)dh;
    const double a = K.hmin_d / (hd + K.hcrit_d);
    const double kd = kap_field ? (double)kap : K.kap_d;
    return (float)(-K.gamma_d * (kd * powlaw_d(a, K.n, K.m, K.powmode)));
  }
  const float a = K.hmin * __builtin_amdgcn_rcpf(hh + K.hcrit);
  return -K.gamma * (kap * powlaw_f(a, K.n, K.m, K.powmode));
}

}  // namespace swalbe
