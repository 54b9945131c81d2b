// Roots of reduced monic cubics for the quadratic-epigraph projections: the
// general one (proj.hip) and the one-dimensional one of the fused lifting
// kernels (lift.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace opy {

// Real root of y^3 + a y + b = 0 by Cardano's formula (one real root) or the
// trigonometric form (three real roots; the largest is returned).
template <typename T>
__device__ inline T reduced_monic_cubic(T a, T b) {
  if (a == T(0)) return b == T(0) ? T(0) : cbrt(-b);
  if (b == T(0) && a > T(0)) return T(0);
  const T Q = a / T(3);
  const T R = -b / T(2);
  const T Q3 = Q * Q * Q;
  const T D = Q3 + R * R;
  if (D <= T(0)) {
    const T th = acos(R / sqrt(-Q3));
    return T(2) * sqrt(-Q) * cos(th / T(3));
  }
  T A = cbrt(fabs(R) + sqrt(D));
  if (R < T(0)) A = -A;
  return A - Q / A;
}

// y - f(y)/f'(y) for f = y^3 + a y - q
__device__ inline float cubic_step(float y, float a, float q) {
  const float y2 = y * y;
  return __builtin_fmaf(-__builtin_fmaf(y, y2 + a, -q), __builtin_amdgcn_rcpf(__builtin_fmaf(3.f, y2, a)), y);
}
__device__ inline double cubic_step(double y, double a, double q) {
  const double y2 = y * y;
  return y - __builtin_fma(y, y2 + a, -q) / __builtin_fma(3.0, y2, a);
}

// The positive root of y^3 + a y = q (q > 0) by Newton's method from y0 at or
// above it: f is convex there, so the iterates fall towards the root, and the
// last step's rounding is all that is left of the error (Cardano's formula
// subtracts two terms that can be close).  The upper bounds
// sqrt(max(-a, 0)) + q^(1/3) and, for a > 0, q / a keep the start within a factor
// of 1.52 of the root; the relative error then falls to 0.17, 0.028, 1e-3, 1e-6
// and 1e-12, so five steps are exact in FP32 (1.2e-7 at most over 2 million
// pairs) and six in FP64.
template <typename T>
__device__ inline T cubic_root(T a, T q, T y0) {
  const float af = (float)a, qf = (float)q;
  const float cb = __builtin_amdgcn_exp2f(__builtin_amdgcn_logf(qf) * (1.f / 3.f)) * 1.00001f;
  float u = cb + __builtin_amdgcn_sqrtf(__builtin_fmaxf(-af, 0.f)) * 1.00001f;
  if (af > 0.f) u = __builtin_fminf(u, qf * __builtin_amdgcn_rcpf(af) * 1.00001f);
  T y = (T)u < y0 ? (T)u : y0;
#pragma unroll
  for (int it = 0; it < (sizeof(T) == 4 ? 5 : 6); ++it) y = cubic_step(y, a, q);
  return y;
}

// (v, x2) projected onto {x2 >= 0.5*alph*v^2} (one-dimensional x1, no
// truncation): the optimality condition of the general projection for M = 1.  A
// point outside has its projection at |v|' <= |v|, the upper start.
template <typename T>
__device__ inline void quadepi_project1(T& v, T& x2, T alph) {
  const T n2 = v * v;
  if (n2 > T(0)) {
    if (T(0.5) * alph * n2 > x2) {
      const T xn = fabs(v);
      const T l = T(2) / (alph * alph);
      const T yn = cubic_root(l * (T(1) - x2 * alph), l * xn, xn);
      v = v < T(0) ? -yn : yn;
      x2 = T(0.5) * alph * yn * yn;
    }
  } else if (x2 < T(0)) {
    x2 = T(0);
  }
}

}  // namespace opy
