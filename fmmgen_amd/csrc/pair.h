// One source-target pair of an operator variant in closed form (the example's
// P2P, example/calculate.cpp:24-40, and its dipole and quadrupole forms).
#pragma once

#include "variant_decl.h"

namespace fmm {
namespace FMM_VARIANT_NS {

// 1/r from the hardware estimate y of x^(-1/2), x = r^2, corrected in FP64 by
// the series of (1 - e)^(-1/2), e = 1 - x y^2, which cubes the estimate's
// relative error.  No case of x is treated apart: x = 0 (coincident particles)
// and infinite x give NaN, subnormal x (y^2 overflows) gives NaN or infinity.
// The callers repeat a sum that has come out as not finite with the generated
// body, which also settles the sums that are infinite by right.
__device__ __forceinline__ double inv_norm(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x, y * y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

__device__ __forceinline__ bool not_finite(double v) { return !(fabs(v) < __builtin_huge_val()); }

// One charge pair in FP64: q/r and q r^-3 (dx, dy, dz).  19 instructions and the
// estimate, against 23 in the generated body (its select of zero and infinite
// x).  The products are taken in the generated body's order, (q y) y y: y^3 by
// itself leaves the range before q r^-3 does.
__device__ __forceinline__ void charge_pair(double dx, double dy, double dz, double q, double* acc) {
  const double x = fma(dx, dx, fma(dy, dy, dz * dz));
  double s3;
  if constexpr (OUT == 3) {
    const double y = __builtin_amdgcn_rsq(x);
    const double y2 = y * y;
    const double e = fma(-x, y2, 1.0);
    const double q3 = (q * y) * y2, t = q3 * e;
    s3 = fma(t * e, 1.875, fma(t, 1.5, q3));
  } else {
    const double r = inv_norm(x), s = q * r;
    acc[0] += s;
    s3 = s * (r * r);
  }
  if constexpr (OUT != 1) {
    constexpr int F0 = OUT == 4 ? 1 : 0;
    acc[F0] = fma(s3, dx, acc[F0]);
    acc[F0 + 1] = fma(s3, dy, acc[F0 + 1]);
    acc[F0 + 2] = fma(s3, dz, acc[F0 + 2]);
  }
}

// One dipole or quadrupole pair, with u = d / r, no power of 1/r beyond that of
// the result itself:
//   dipole      phi = -r^-2 S.u,              F = r^-3 (S - 3 (S.u) u)
//   quadrupole  phi = r^-3 (3 Q - T),         F = 3 r^-4 ((5 Q - T) u - v),
//               v = grad of u.S.u, Q = u.S.u = u.v / 2, T = trace S.
// No second and third derivatives one by one as in the generated bodies.  200000
// uniform particles, FP64 near field: dipoles 3.99 -> 1.66 ms, quadrupoles 7.18 ->
// 2.48 ms; 4096 targets x 2^18 sources: dipoles 2.73 -> 1.43 ms, quadrupoles 6.02
// -> 2.16 ms.
__device__ __forceinline__ void multipole_pair(double dx, double dy, double dz, const double* S, double* acc) {
  constexpr int F0 = OUT == 4 ? 1 : 0;
  const double r = inv_norm(fma(dx, dx, fma(dy, dy, dz * dz)));
  const double x = dx * r, y = dy * r, z = dz * r, r2 = r * r, r3 = r2 * r;
  if constexpr (SO == 1) {
    const double s = fma(S[0], x, fma(S[1], y, S[2] * z));
    if constexpr (OUT != 3) acc[0] = fma(-r2, s, acc[0]);
    if constexpr (OUT != 1) {
      const double t = -3.0 * s;
      acc[F0] = fma(r3, fma(t, x, S[0]), acc[F0]);
      acc[F0 + 1] = fma(r3, fma(t, y, S[1]), acc[F0 + 1]);
      acc[F0 + 2] = fma(r3, fma(t, z, S[2]), acc[F0 + 2]);
    }
  } else {
    const double vx = fma(S[0] + S[0], x, fma(S[1], y, S[2] * z));
    const double vy = fma(S[1], x, fma(S[3] + S[3], y, S[4] * z));
    const double vz = fma(S[2], x, fma(S[4], y, (S[5] + S[5]) * z));
    const double q = fma(x, vx, fma(y, vy, z * vz)), tr = S[0] + S[3] + S[5];
    if constexpr (OUT != 3) acc[0] = fma(r3, fma(1.5, q, -tr), acc[0]);
    if constexpr (OUT != 1) {
      const double a = 3.0 * (r3 * r), b = fma(2.5, q, -tr);
      acc[F0] = fma(a, fma(b, x, -vx), acc[F0]);
      acc[F0 + 1] = fma(a, fma(b, y, -vy), acc[F0 + 1]);
      acc[F0 + 2] = fma(a, fma(b, z, -vz), acc[F0 + 2]);
    }
  }
}

// The pair of the near field, the direct sum and the Barnes-Hut leaves.  FP32
// pairs take the generated body: charges have no shorter form, and the closed
// dipole form rounds otherwise (8e-8 of the field apart; 3.97 instead of 5.70 ms
// at 10^6 Plummer dipoles).
template <typename T>
__device__ __forceinline__ void source_pair(T dx, T dy, T dz, const T* S, T* acc) {
  if constexpr (sizeof(T) == 4) fmmgen_ops::P2P<T>(dx, dy, dz, S, acc);
  else if constexpr (SO == 0) charge_pair(dx, dy, dz, S[0], acc);
  else multipole_pair(dx, dy, dz, S, acc);
}

}  // namespace FMM_VARIANT_NS
}  // namespace fmm
