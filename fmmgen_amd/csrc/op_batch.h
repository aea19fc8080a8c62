// One operator over a batch of independent inputs: one wave an item, its
// operands staged in LDS by coalesced loads, the lanes over output slots.  The
// operators are linear maps whose structure the kernels use:
//   M2L, M2P  the derivative block degree by degree (lanes over the slots of a
//             degree) on the slots with n_z <= 2, and sums over the multipole
//             folded onto n_z <= 1 (the harmonic layout of m2l_gemm.h: a third
//             of the full sum's terms at order 8);
//   M2M, L2L  shifts by x, then y, then z (O(p^4) terms instead of O(p^6));
//   P2M, L2P  products of three powers a lane.
// Batches of 20000, before and after (a call with its launches): M2L order 10
// 1869 -> 110 us, order 12 4352 -> 183, order 4 61 -> 52; M2P order 10 1941 -> 61;
// M2M order 12 260 -> 149; L2L order 12 1042 -> 110; L2P order 12 630 -> 40 (a
// thread or one busy lane an item, strided rows and, above order 8, one lane's
// derivative block before).  M2L at order 10 is bound by the chain of LDS steps of
// an item at four waves a SIMD: the columns of the high degrees dealt to more
// lanes (half the steps) gained 6%, not kept.
#pragma once

#include <algorithm>

#include "wave_ops.h"

namespace fmm {
namespace FMM_VARIANT_NS {

// D_(x,y,z) of degree d with n_z <= 2 in LDS: slot d_base(d) + 3 y + z, so that
// the slot of a sum of two multi-indices is the sum of their slots + 3 d d'.
__host__ __device__ constexpr int d_base(int d) { return 3 * (d * (d + 1) / 2); }

// Harmonic slot j (degree d, n_y, n_z <= 1) found at run time.
struct HarmIdx {
  int d, y, z;
};
__device__ __forceinline__ HarmIdx harm_rt(int j) {
  const int d = (int)sqrtf((float)j + 0.5f), r = j - d * d, a = (r + 1) >> 1;
  const int z = r == 0 ? 0 : (r + 1) & 1;
  return HarmIdx{d, a - z, z};
}

// Derivative block at (x, y, z) up to degree PD, by one wave: the recurrence of
// the generated block (n_z <= 1) on lanes 0 .. 31, D_{k+2z} = -D_{k+2x} -
// D_{k+2y} of the degree before on lanes 32 .. 63.
template <int PD>
__device__ __forceinline__ void wave_derivs(int lane, double x, double y, double z, double* sD) {
  static_assert(2 * PD + 1 <= 32, "a degree's harmonic slots fit half a wave");
  const double ir = fmmgen_rsqrt(x * x + y * y + z * z), ir2 = ir * ir;
  if (lane == 0) sD[0] = ir;
  const int a = (lane + 1) >> 1, nz = lane == 0 ? 0 : (lane + 1) & 1, ny = a - nz, e = lane - 32;
  static_for<PD + 1>([&](auto DC) {
    constexpr int d = DC + 1;
    wave_lds_fence();
    if (d <= PD && lane < 2 * d + 1) {
      constexpr double c1 = -(double)(2 * d - 1) / d, c2 = -(double)(d - 1) / d;
      const int nx = d - a, at = 3 * ny + nz;
      const double* D1 = sD + d_base(d - 1);
      double v = c1 * ((double)nx * x * (nx >= 1 ? D1[at] : 0.0) + (double)ny * y * (ny >= 1 ? D1[at - 3] : 0.0) +
                       (nz ? z * D1[at - 1] : 0.0));
      if constexpr (d >= 2) {
        const double* D2 = sD + d_base(d - 2);
        v += c2 * ((double)(nx * (nx - 1)) * (nx >= 2 ? D2[at] : 0.0) +
                   (double)(ny * (ny - 1)) * (ny >= 2 ? D2[at - 6] : 0.0));
      }
      sD[d_base(d) + at] = ir2 * v;
    }
    if (d >= 3 && e >= 0 && e <= d - 3) {  // n_z = 2 of degree d - 1
      double* D = sD + d_base(d - 1) + 3 * e;
      D[2] = -D[0] - D[6];
    }
  });
  wave_lds_fence();
}

// Term tables of the fold (harmonic slots of degree SO .. P) and of the unfold
// in LDS: source slot | weight << 16, terms off[j] .. off[j + 1] - 1 of slot j.
template <int P>
struct OpTerms {
  using H = HarmTables<P>;
  static constexpr int NL = Op<P>::LS;
  static constexpr int unfold_terms() {
    int t = 0;
    for (int n = 0; n < NL; ++n) t += slot_multi(n).z / 2 + 1;
    return t;
  }
  static constexpr int NF = H::NF, NU = unfold_terms(), HS = H::HS;
  short fold_off[HS + 1], unf_off[NL + 1];
  int fold[NF], unf[NU];
  __device__ void load(int tid, int nt) {
    constexpr H tab{};
    for (int i = tid; i <= HS; i += nt) fold_off[i] = tab.fold_off[i];
    for (int i = tid; i < NF; i += nt) fold[i] = tab.fold_src[i] | ((int)tab.fold_w[i] << 16);
    for (int i = tid; i <= NL; i += nt) unf_off[i] = tab.unf_off[i];
    for (int i = tid; i < NU; i += nt) unf[i] = tab.unf_src[i] | ((int)tab.unf_w[i] << 16);
  }
};

// Adds a wave's sums to the outputs: the potential, minus the gradient.
__device__ __forceinline__ void put(int lane, double* o, double phi, double fx, double fy, double fz) {
  constexpr int F0 = OUT == 4 ? 1 : 0;
  if constexpr (OUT != 3) {
    phi = wave_sum(phi);
    if (lane == 0) o[0] += phi;
  }
  if constexpr (OUT != 1) {
    fx = wave_sum(fx);
    fy = wave_sum(fy);
    fz = wave_sum(fz);
    if (lane < 3) o[F0 + lane] -= lane == 0 ? fx : lane == 1 ? fy : fz;
  }
}

constexpr int kOpWaves = 4;  // items a block, which share the term tables

template <int P, int OPID>
__global__ __launch_bounds__(64 * kOpWaves) void k_op_wave(int n, const double* __restrict__ xyz,
                                                           const double* __restrict__ in, int in_stride,
                                                           double* __restrict__ out, int out_stride) {
  constexpr int MS = Op<P>::MS, LS = Op<P>::LS, OFF = nterms(SO - 1), Q = P - SO, J0 = harm_size(SO - 1);
  constexpr int W = kOpWaves;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int first = blockIdx.x * W + w, step = gridDim.x * W;
  auto items = [&](auto&& f) {
    for (long long i = first; i < n; i += step)
      f(xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2], in + i * in_stride, out + i * out_stride);
  };
  if constexpr (OPID == kOpM2L || OPID == kOpM2P) {
    constexpr int PD = OPID == kOpM2P && OUT != 1 ? P + 1 : P;
    constexpr int NL = OPID == kOpM2L ? harm_size(Q) : 1;
    __shared__ OpTerms<P> terms;
    __shared__ double aD[W][d_base(PD + 1)], aM[W][MS], aMh[W][harm_size(P) - J0], aL[W][NL];
    terms.load(threadIdx.x, 64 * W);
    __syncthreads();
    double *sD = aD[w], *sM = aM[w], *sMh = aMh[w], *sL = aL[w];
    items([&](double x, double y, double z, const double* a, double* o) {
      for (int j = lane; j < MS; j += 64) sM[j] = a[j];
      wave_derivs<PD>(lane, x, y, z, sD);
      for (int j = J0 + lane; j < harm_size(P); j += 64) {
        double v = 0.0;
        for (int t = terms.fold_off[j]; t < terms.fold_off[j + 1]; ++t) {
          const int f = terms.fold[t];
          v = fma((double)(f >> 16), sM[(f & 0xffff) - OFF], v);
        }
        sMh[j - J0] = v;
      }
      wave_lds_fence();
      if constexpr (OPID == kOpM2L) {
        for (int j = lane; j < NL; j += 64) {
          const HarmIdx r = harm_rt(j);
          const double* Dr = sD + d_base(r.d) + 3 * r.y + r.z;
          double acc = 0.0;
          static_for<Q + 1>([&](auto MC) {
            constexpr int dm = SO + MC;
            asm volatile("" ::: "memory");  // the multipole is read here, not kept in registers over the rows
            if (r.d + dm <= P) {
              const double* Dc = Dr + d_base(dm) + 3 * dm * r.d;
              double v = 0.0;
              static_for<2 * dm + 1>([&](auto RC) {
                constexpr MultiIdx m = harm_multi(dm * dm + RC);
                v = fma(Dc[3 * m.y + m.z], sMh[dm * dm + RC - J0], v);
              });
              acc += v;
            }
          });
          sL[j] = acc;
        }
        wave_lds_fence();
        for (int j = lane; j < LS; j += 64) {
          double v = 0.0;
          for (int t = terms.unf_off[j]; t < terms.unf_off[j + 1]; ++t) {
            const int f = terms.unf[t];
            v = fma((double)(f >> 16), sL[f & 0xffff], v);
          }
          o[j] += v;
        }
      } else {
        double phi = 0.0, fx = 0.0, fy = 0.0, fz = 0.0;
        for (int j = J0 + lane; j < harm_size(P); j += 64) {
          const HarmIdx r = harm_rt(j);
          const double m = sMh[j - J0];
          if constexpr (OUT != 3) phi = fma(m, sD[d_base(r.d) + 3 * r.y + r.z], phi);
          if constexpr (OUT != 1) {
            const double* D = sD + d_base(r.d + 1) + 3 * r.y + r.z;
            fx = fma(m, D[0], fx);
            fy = fma(m, D[3], fy);
            fz = fma(m, D[1], fz);
          }
        }
        put(lane, o, phi, fx, fy, fz);
      }
      wave_lds_fence();  // read before the next item is staged
    });
  }
  if constexpr (OPID == kOpM2M || OPID == kOpL2L) {
    constexpr bool DOWN = OPID == kOpM2M;
    constexpr int N = DOWN ? P : Q, LO = DOWN ? OFF : 0;  // multipoles below the source order are zero
    __shared__ double aA[W][nterms(N)], aB[W][nterms(N)], aP[W][3 * (N + 1)];
    items([&](double x, double y, double z, const double* a, double* o) {
      for (int j = lane; j < nterms(N); j += 64) aA[w][j] = j >= LO ? a[j - LO] : 0.0;
      wave_powers<N>(lane, x, y, z, aP[w]);
      wave_lds_fence();
      wave_shift3<N, DOWN>(lane, aA[w], aB[w], aP[w]);
      for (int j = LO + lane; j < nterms(N); j += 64) o[j - LO] += aB[w][j];
      wave_lds_fence();
    });
  }
  if constexpr (OPID == kOpL2P) {
    __shared__ double aP[W][3 * (Q + 1)];
    const double *X = aP[w], *Y = X + Q + 1, *Z = Y + Q + 1;
    items([&](double x, double y, double z, const double* a, double* o) {
      wave_powers<Q>(lane, x, y, z, aP[w]);
      wave_lds_fence();
      double phi = 0.0, fx = 0.0, fy = 0.0, fz = 0.0;
      for (int j = lane; j < LS; j += 64) {
        const MultiIdx m = slot_multi_rt(j);
        const double v = a[j], px = X[m.x], py = Y[m.y], pz = Z[m.z];
        if constexpr (OUT != 3) phi = fma(v, px * py * pz, phi);
        if constexpr (OUT != 1) {
          if (m.x > 0) fx = fma(v, X[m.x - 1] * py * pz, fx);
          if (m.y > 0) fy = fma(v, px * Y[m.y - 1] * pz, fy);
          if (m.z > 0) fz = fma(v, px * py * Z[m.z - 1], fz);
        }
      }
      put(lane, o, phi, fx, fy, fz);
      wave_lds_fence();
    });
  }
  if constexpr (OPID == kOpP2M || OPID == kOpP2MS) {
    // P2M: the charge formula q (-x)^n / n! at every source order; P2MS: one
    // particle's multipole sum_s S_s x^(n-s) / (n-s)!, |s| = SO
    __shared__ double aP[W][3 * (P + 1)];
    const double *X = aP[w], *Y = X + P + 1, *Z = Y + P + 1;
    items([&](double x, double y, double z, const double* a, double* o) {
      if constexpr (OPID == kOpP2M) wave_powers<P>(lane, -x, -y, -z, aP[w]);
      else wave_powers<P>(lane, x, y, z, aP[w]);
      wave_lds_fence();
      for (int j = lane; j < MS; j += 64) {
        const MultiIdx m = slot_multi_rt(j + OFF);
        if constexpr (OPID == kOpP2M || SO == 0) {
          o[j] += a[0] * X[m.x] * Y[m.y] * Z[m.z];
        } else {
          double v = 0.0;
          static_for<SS>([&](auto S) {
            constexpr MultiIdx s = slot_multi(OFF + S);
            if (m.x >= s.x && m.y >= s.y && m.z >= s.z)
              v = fma(a[S], X[m.x - s.x] * Y[m.y - s.y] * Z[m.z - s.z], v);
          });
          o[j] += v;
        }
      }
      wave_lds_fence();
    });
  }
}

template <int P>
void op_batch_order(int op, int n, const double* xyz, const double* in, int is, double* out, int os,
                    hipStream_t st) {
  const int g = std::min(nblk(n, kOpWaves), 2048);  // blocks stride over larger batches
  switch (op) {
    case kOpP2M: k_op_wave<P, kOpP2M><<<g, 64 * kOpWaves, 0, st>>>(n, xyz, in, is, out, os); break;
    case kOpM2M: k_op_wave<P, kOpM2M><<<g, 64 * kOpWaves, 0, st>>>(n, xyz, in, is, out, os); break;
    case kOpM2L: k_op_wave<P, kOpM2L><<<g, 64 * kOpWaves, 0, st>>>(n, xyz, in, is, out, os); break;
    case kOpL2L: k_op_wave<P, kOpL2L><<<g, 64 * kOpWaves, 0, st>>>(n, xyz, in, is, out, os); break;
    case kOpL2P: k_op_wave<P, kOpL2P><<<g, 64 * kOpWaves, 0, st>>>(n, xyz, in, is, out, os); break;
    case kOpM2P: k_op_wave<P, kOpM2P><<<g, 64 * kOpWaves, 0, st>>>(n, xyz, in, is, out, os); break;
    case kOpP2MS: k_op_wave<P, kOpP2MS><<<g, 64 * kOpWaves, 0, st>>>(n, xyz, in, is, out, os); break;
    default: throw Error{kInvalidArgument, "operator has no order"};
  }
}

}  // namespace FMM_VARIANT_NS
}  // namespace fmm
