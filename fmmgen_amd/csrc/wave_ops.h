// Pieces of the kernels in which one wave applies one operator to operands in
// LDS: powers, shifts along an axis, the fence between a wave's own LDS writes
// and reads.
#pragma once

#include "m2l_gemm.h"
#include "variant_decl.h"

namespace fmm {
namespace FMM_VARIANT_NS {

// Orders a wave's LDS accesses before and after it (the hardware keeps them in
// order; other waves are not waited for).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int k = 32; k > 0; k >>= 1) v += __shfl_xor(v, k);
  return v;
}

// x^k / k!, y^k / k!, z^k / k! for k <= Q, [axis * (Q + 1) + k], one a lane.
template <int Q>
__device__ __forceinline__ void wave_powers(int lane, double x, double y, double z, double* sP) {
  static_assert(3 * (Q + 1) <= 64, "a lane a power");
  const int axis = lane / (Q + 1), k = lane - axis * (Q + 1);
  if (axis < 3) {
    const double v = axis == 0 ? x : axis == 1 ? y : z;
    double w = 1.0, f = 1.0;
    static_for<Q>([&](auto K) {
      w = K < k ? w * v : w;
      f = K < k ? f * (K + 1) : f;
    });
    sP[lane] = w / f;
  }
}

// One axis of a shift on graded slots of degree <= Q:
//   DOWN (M2M): b_n = sum_k p_k a_{n - k e},  else (L2L): b_n = sum_k p_k a_{n + k e}.
template <int Q, int AXIS, bool DOWN>
__device__ __forceinline__ void wave_shift(int lane, const double* a, double* b, const double* p) {
  for (int j = lane; j < nterms(Q); j += 64) {
    const MultiIdx n = slot_multi_rt(j);
    int d = n.x + n.y + n.z, s = n.y + n.z, at = j;
    const int kmax = DOWN ? (AXIS == 0 ? n.x : AXIS == 1 ? n.y : n.z) : Q - d;
    double v = a[at];
    for (int k = 1; k <= kmax; ++k) {
      if constexpr (DOWN) {  // degree d -> d - 1, n_y + n_z s -> s - 1 on the y and z axes
        at -= d * (d + 1) / 2 + (AXIS >= 1 ? s : 0) + (AXIS == 2 ? 1 : 0);
        --d;
        if constexpr (AXIS >= 1) --s;
      } else {
        ++d;
        if constexpr (AXIS >= 1) ++s;
        at += d * (d + 1) / 2 + (AXIS >= 1 ? s : 0) + (AXIS == 2 ? 1 : 0);
      }
      v = fma(p[k], a[at], v);
    }
    b[j] = v;
  }
}

// The whole shift: x from a to b, y back, z to b.
template <int Q, bool DOWN>
__device__ __forceinline__ void wave_shift3(int lane, double* a, double* b, const double* p) {
  wave_shift<Q, 0, DOWN>(lane, a, b, p);
  wave_lds_fence();
  wave_shift<Q, 1, DOWN>(lane, b, a, p + Q + 1);
  wave_lds_fence();
  wave_shift<Q, 2, DOWN>(lane, a, b, p + 2 * (Q + 1));
  wave_lds_fence();
}

}  // namespace FMM_VARIANT_NS
}  // namespace fmm
