// Barnes-Hut walk of one operator variant (Tree::compute_field_bh,
// example/tree.cpp:273-293, and evaluate_M2P_and_P2P,
// example/calculate.cpp:266-314), FP64.  Every particle walks the tree from the
// root: below an internal cell each child c is opened when
// r_c > theta |x_i - centre_c| and applied by M2P at x_i - centre_c otherwise; a
// leaf adds P2P from its particles except i.
//
// M2P.  The potential of a cell is sum_n M_n D_n, D_n = d^n (1/R), and every D_n
// of degree l is a combination of the 2l + 1 irregular solid harmonics
//   I_l^m = (-d_z)^(l-m) (d_x + i d_y)^m (1/R),  m = 0 .. l.
// So each cell's multipole is rewritten once (k_bh_coef) as coefficients of
// R_l^m = Re I_l^m and J_l^m = Im I_l^m, for the potential and, with
//   d_z I_l^m = -I_{l+1}^m,  d_x I_l^m = (I_{l+1}^{m+1} - I_{l+1}^{m-1}) / 2,
//   d_y I_l^m = -i (I_{l+1}^{m+1} + I_{l+1}^{m-1}) / 2,
// for the field; the walk evaluates I_l^m for one m after the other by
//   I_{m+1}^{m+1} = -(2m+1) (x + i y) / R^2 I_m^m,
//   I_{l+1}^m = ((2l+1) z I_l^m - (l^2 - m^2) I_{l-1}^m) / R^2,
// with two complex values live.  13 FP64 instructions a pair (l, m) (about 680
// at order 8), against the whole derivative block of the generated body in
// registers: 2^20 uniform particles, order 8, 15.8 -> 7.5 ms; 2^20 blobs 22.6 ->
// 10.2 ms; 1000 particles 655 -> 162 us.
#pragma once

#include "pair.h"
#include "wave_ops.h"

namespace fmm {
namespace FMM_VARIANT_NS {

// Coefficient rows: for m = 0 .. L1 and l = max(m, SO) .. L1 in this order the
// potential's coefficients of R_l^m and J_l^m (l <= P) and, with a field, those
// of -d_x (R, J) and -d_y (R, J) (l > SO; J for m > 0 only); the z component's
// are the potential's of degree l - 1.  A row begins with the cell's centre and
// half-width and is padded to whole 64-byte lines, which the walk reads by scalar
// loads of a line each.
template <int P>
struct BHRow {
  static constexpr int L1 = OUT == 1 ? P : P + 1, HEAD = 4;
  static constexpr int first(int m) { return m > SO ? m : SO; }
  static constexpr int pot(int m, int l) { return l <= P ? (m > 0 ? 2 : 1) : 0; }
  static constexpr int grad(int m, int l) { return OUT != 1 && l > SO ? (m > 0 ? 4 : 2) : 0; }
  static constexpr int at(int m, int l) {
    int s = HEAD;
    for (int k = 0; k <= m; ++k)
      for (int j = first(k); j <= L1 && (k < m || j < l); ++j) s += pot(k, j) + grad(k, j);
    return s;
  }
  static constexpr int step(int m, int l) {
    int s = 0;
    for (int k = 0; k < m; ++k) s += L1 - first(k) + 1;
    return s + l - first(m);
  }
  static constexpr int NSTEP = step(L1, L1) + 1;
  static constexpr int SIZE = (at(L1, L1) + pot(L1, L1) + grad(L1, L1) + 7) / 8 * 8;
};

// Table of k_bh_coef: D_(a,b,c) with q = a + b is (-1)^c times
// sum_m w[q][b][m] R_l^m (b even) or J_l^m (b odd), l = q + c:
// (d_x)^a (d_y)^b = 2^-q (A + B)^a (-i)^b (A - B)^b with A = d_x + i d_y,
// B = d_x - i d_y, and A^s B^t (-d_z)^c (1/R) = (-1)^t I_l^(s-t).
// Dyadic fractions of at most 13 bits: exact in FP32.
template <int P>
struct BHTab {
  float w[P + 1][P + 1][P + 1];
  unsigned char step_m[BHRow<P>::NSTEP], step_l[BHRow<P>::NSTEP];
  short step_at[BHRow<P>::NSTEP];
  static constexpr long long binom(int n, int k) {
    if (k < 0 || k > n) return 0;
    long long c = 1;
    for (int i = 0; i < k; ++i) c = c * (n - i) / (i + 1);
    return c;
  }
  constexpr BHTab() : w{}, step_m{}, step_l{}, step_at{} {
    for (int q = 0; q <= P; ++q)
      for (int b = 0; b <= q; ++b)
        for (int m = q & 1; m <= q; m += 2) {
          const int a = q - b, s = (q + m) / 2, t = q - s;
          long long v = 0;
          for (int k = 0; k <= b; ++k) {
            const long long x = binom(a, s - k) * binom(b, k);
            v += ((b - k) & 1) ? -x : x;
          }
          if (t & 1) v = -v;
          if ((b / 2) & 1) v = -v;
          if (m > 0) v *= 2;
          w[q][b][m] = (float)v / (float)(1 << q);
        }
    for (int m = 0; m <= BHRow<P>::L1; ++m)
      for (int l = BHRow<P>::first(m); l <= BHRow<P>::L1; ++l) {
        step_m[BHRow<P>::step(m, l)] = (unsigned char)m;
        step_l[BHRow<P>::step(m, l)] = (unsigned char)l;
        step_at[BHRow<P>::step(m, l)] = (short)BHRow<P>::at(m, l);
      }
  }
};

// Coefficient rows of every cell from its graded multipole: one wave a cell
// (four a block), the cell's row and then the potential's coefficients in LDS.
// HBM-bound by the rows it writes (2^20 particles, order 8: 37449 cells, 86 MB,
// 95 us).
template <int P>
__global__ __launch_bounds__(256) void k_bh_coef(int nc, const double* __restrict__ M, const double* __restrict__ cx,
                                                 const double* __restrict__ cy, const double* __restrict__ cz,
                                                 const double* __restrict__ cr, double* __restrict__ Q) {
  using Row = BHRow<P>;
  static constexpr BHTab<P> tab{};
  constexpr int MS = Op<P>::MS, OFF = nterms(SO - 1), LD = P + 3, NA = (P + 2) * LD;
  __shared__ double s_m[4][MS];
  __shared__ double s_a[4][2][NA];  // [real, imaginary][l * LD + m], 0 outside SO <= l <= P, m <= l
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int cell = blockIdx.x * 4 + wv;
  if (cell < nc)
    for (int j = lane; j < MS; j += 64) s_m[wv][j] = M[(size_t)cell * MS + j];
  __syncthreads();
  for (int e = lane; e < 2 * NA; e += 64) {
    const int im = e >= NA, r = e - im * NA, l = r / LD, m = r - l * LD;
    double v = 0.0;
    if (l >= SO && l <= P && m <= l) {
      for (int q = m; q <= l; q += 2) {
        double u = 0.0;
        for (int b = im; b <= q; b += 2) u += (double)tab.w[q][b][m] * s_m[wv][multi_slot(q - b, b, l - q) - OFF];
        v += ((l - q) & 1) ? -u : u;
      }
    }
    s_a[wv][im][r] = v;
  }
  __syncthreads();
  if (cell >= nc) return;
  const double* ar = s_a[wv][0];
  const double* ai = s_a[wv][1];
  double* row = Q + (size_t)cell * Row::SIZE;
  if (lane < 4) row[lane] = lane == 0 ? cx[cell] : lane == 1 ? cy[cell] : lane == 2 ? cz[cell] : cr[cell];
  for (int s = lane; s < Row::NSTEP; s += 64) {
    const int m = tab.step_m[s], l = tab.step_l[s];
    double* o = row + tab.step_at[s];
    if (l <= P) {
      *o++ = ar[l * LD + m];
      if (m > 0) *o++ = ai[l * LD + m];
    }
    if (OUT != 1 && l > SO) {
      const int b = (l - 1) * LD;  // degree l - 1
      const double rp = ar[b + m + 1], ip = ai[b + m + 1];
      const double rm = m > 0 ? (m == 1 ? 2.0 : 1.0) * ar[b + m - 1] : 0.0, im = m > 0 ? ai[b + m - 1] : 0.0;
      *o++ = 0.5 * (rp - rm);
      if (m > 0) *o++ = 0.5 * (ip - im);
      *o++ = 0.5 * (ip + im);
      if (m > 0) *o++ = -0.5 * (rp + rm);
    }
  }
}

// M2P of one cell (coefficient row, the same for the whole wave) at
// (dx, dy, dz), into acc.
template <int I>
using Int = std::integral_constant<int, I>;
typedef double BHLine __attribute__((ext_vector_type(8)));
typedef double BHQuad __attribute__((ext_vector_type(4), aligned(8)));
template <int P>
__device__ __forceinline__ void bh_m2p(double dx, double dy, double dz, const BHLine* __restrict__ row, double* acc) {
  using Row = BHRow<P>;
  constexpr int L1 = Row::L1, F0 = OUT == 4 ? 1 : 0;
  const double r2 = dx * dx + dy * dy + dz * dz;
  const double ir = fmmgen_rsqrt(r2), ir2 = ir * ir;
  const double xs = -dx * ir2, ys = -dy * ir2, zs = dz * ir2;
  double phi = 0.0, fx = 0.0, fy = 0.0, fz = 0.0;
  double Rm = ir, Jm = 0.0;  // I_m^m
  static_for<L1 + 1>([&](auto MC) {
    constexpr int m = MC;
    double R = Rm, J = Jm, Rb = 0.0, Jb = 0.0;  // degree l, degree l - 1
    static_for<L1 + 1 - m>([&](auto LC) {
      constexpr int l = m + LC;
      if constexpr (l >= SO) {
        auto q = [&](auto I) { return row[I / 8][I % 8]; };
        constexpr int c = Row::at(m, l), g = c + Row::pot(m, l);
        if constexpr (OUT != 3 && l <= P) {
          phi = fma(q(Int<c>{}), R, phi);
          if constexpr (m > 0) phi = fma(q(Int<c + 1>{}), J, phi);
        }
        if constexpr (OUT != 1 && l > SO) {
          fx = fma(q(Int<g>{}), R, fx);
          fy = fma(q(Int<g + (m > 0 ? 2 : 1)>{}), R, fy);
          if constexpr (m > 0) {
            fx = fma(q(Int<g + 1>{}), J, fx);
            fy = fma(q(Int<g + 3>{}), J, fy);
          }
          if constexpr (l > m) {
            constexpr int z = Row::at(m, l - 1);
            fz = fma(q(Int<z>{}), R, fz);
            if constexpr (m > 0) fz = fma(q(Int<z + 1>{}), J, fz);
          }
        }
      }
      if constexpr (l < L1) {
        const double t = (double)(2 * l + 1) * zs;
        if constexpr (l == m) {
          Rb = R;
          R *= t;
          if constexpr (m > 0) {
            Jb = J;
            J *= t;
          }
        } else {
          const double u = (double)(l * l - m * m) * ir2;
          const double Rn = fma(t, R, -(u * Rb));
          Rb = R;
          R = Rn;
          if constexpr (m > 0) {
            const double Jn = fma(t, J, -(u * Jb));
            Jb = J;
            J = Jn;
          }
        }
      }
    });
    if constexpr (m < L1) {
      const double a = (double)(2 * m + 1) * xs, b = (double)(2 * m + 1) * ys;
      if constexpr (m == 0) {
        Jm = b * Rm;
        Rm = a * Rm;
      } else {
        const double n = fma(a, Rm, -(b * Jm));
        Jm = fma(a, Jm, b * Rm);
        Rm = n;
      }
    }
  });
  if constexpr (OUT != 3) acc[0] += phi;
  if constexpr (OUT != 1) {
    acc[F0] += fx;
    acc[F0 + 1] += fy;
    acc[F0 + 2] += fz;
  }
}

// A block takes one group of 64 consecutive sorted particles (one or two leaves
// mostly) and walks the union of its paths on a stack in LDS whose entries carry
// the lanes that reached the cell; a lane applies M2P only at the cells where its
// own walk stops, so each particle sums exactly the reference's terms.  The
// distance of the criterion is rounded as the reference's host code rounds it, so
// every decision matches.  With W > 1 (small sets) every wave walks the same
// group, the waves take its applied cells and its leaves in turn, and their sums
// are added in a fixed order.
//
// Bound by the latency of the coefficient rows at six waves a SIMD (2^20
// particles, order 8: 60% of the FP64 issue rate).  Rows read by loads of 32 and
// 16 bytes 9.8 ms, of whole lines 8.4, the cell's centre in the row's first line
// and four leaf particles a load 7.4, runs of 64 blocks an XCD instead of 16
// (neighbouring groups read the same rows from one L2) 7.2.  Blocks of 2 and 4
// waves that walk 2 and 4 groups in step, for the scalar cache's sake, halve its
// misses but wait for each other: 7.7 and 8.5; 8 waves a SIMD leave too few
// scalar registers for the loads in flight: 7.8.
constexpr int kBHStack = 256;  // a pop pushes at most 8: 7 per level + 1
constexpr int kBHRun = 64;

template <int P, int W>
__global__ __launch_bounds__(64 * W) void k_bh(int n, const int* __restrict__ first_child,
                                               const int* __restrict__ nchild, const int* __restrict__ pstart,
                                               const int* __restrict__ pcount, const double* __restrict__ px,
                                               const double* __restrict__ py, const double* __restrict__ pz,
                                               const double* __restrict__ pS, const int* __restrict__ perm,
                                               const BHLine* __restrict__ Q, double theta, double* __restrict__ F) {
  __shared__ int s_cell[kBHStack];
  __shared__ unsigned long long s_lanes[kBHStack];
  __shared__ double s_sum[W > 1 ? W - 1 : 1][OUT][64];
  const int lane = threadIdx.x & 63, wv = W == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int k8 = blockIdx.x >> 3;
  const int group = (k8 / kBHRun * 8 + (blockIdx.x & 7)) * kBHRun + k8 % kBHRun;
  if (group > (n - 1) / 64) return;
  const int s = group * 64 + lane;
  const bool valid = s < n;
  const double xi = valid ? px[s] : 0.0, yi = valid ? py[s] : 0.0, zi = valid ? pz[s] : 0.0;
  double acc[OUT];
#pragma unroll
  for (int k = 0; k < OUT; ++k) acc[k] = 0.0;
  const unsigned long long all = __ballot(valid);
  if (threadIdx.x == 0) {
    s_cell[0] = 0;
    s_lanes[0] = all;
  }
  int top = 1, turn = 0;  // uniform over the block
  __syncthreads();
  while (top > 0) {
    --top;
    const int p = __builtin_amdgcn_readfirstlane(s_cell[top]);
    const bool mine = (s_lanes[top] >> lane) & 1ull;
    const int nch = nchild[p];
    if (nch > 0) {
      __syncthreads();  // the entry is read before a push overwrites it
      const int fc = first_child[p];
      // children pushed last to first, so they are walked in octant order
      for (int k = nch - 1; k >= 0; --k) {
        const BHLine* row = Q + (size_t)(fc + k) * (BHRow<P>::SIZE / 8);
        const double dx = xi - row[0][0], dy = yi - row[0][1], dz = zi - row[0][2];
        const bool open = mine && row[0][3] > theta * norm3_rn(dx, dy, dz);
        const unsigned long long lanes = __ballot(open);
        if (__ballot(mine && !open) != 0ull && (W == 1 || turn++ % W == wv)) {
          if (mine && !open) bh_m2p<P>(dx, dy, dz, row, acc);
        }
        if (lanes != 0ull && top < kBHStack) {
          if (threadIdx.x == 0) {
            s_cell[top] = fc + k;
            s_lanes[top] = lanes;
          }
          ++top;
        }
      }
      __syncthreads();  // the pushed entries
    } else if ((W == 1 || turn++ % W == wv) && mine) {
      const int b = pstart[p], e = b + pcount[p];
      double part[OUT];
#pragma unroll
      for (int k = 0; k < OUT; ++k) part[k] = 0.0;
      int j = b;
      for (; j + 4 <= e; j += 4) {  // four sources by scalar loads of 32 bytes
        const BHQuad x4 = *reinterpret_cast<const BHQuad*>(px + j), y4 = *reinterpret_cast<const BHQuad*>(py + j),
                     z4 = *reinterpret_cast<const BHQuad*>(pz + j);
        double S[4 * SS];
#pragma unroll
        for (int k = 0; k < SS; ++k) {
          const BHQuad w = *reinterpret_cast<const BHQuad*>(pS + (size_t)j * SS + 4 * k);
#pragma unroll
          for (int i = 0; i < 4; ++i) S[4 * k + i] = w[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (j + i != s) source_pair<double>(xi - x4[i], yi - y4[i], zi - z4[i], S + i * SS, part);
      }
      for (; j < e; ++j)
        if (j != s) source_pair<double>(xi - px[j], yi - py[j], zi - pz[j], pS + (size_t)j * SS, part);
      bool bad = false;
#pragma unroll
      for (int k = 0; k < OUT; ++k) bad = bad || not_finite(part[k]);
      if (bad) {  // coincident particles above all: the generated body
#pragma unroll
        for (int k = 0; k < OUT; ++k) part[k] = 0.0;
        for (int j = b; j < e; ++j)
          if (j != s) fmmgen_ops::P2P<double>(xi - px[j], yi - py[j], zi - pz[j], pS + (size_t)j * SS, part);
      }
#pragma unroll
      for (int k = 0; k < OUT; ++k) acc[k] += part[k];
    }
  }
  if constexpr (W > 1) {
    if (wv > 0) {
#pragma unroll
      for (int k = 0; k < OUT; ++k) s_sum[wv - 1][k][lane] = acc[k];
    }
    __syncthreads();
    if (wv > 0) return;
#pragma unroll
    for (int v = 0; v < W - 1; ++v)
#pragma unroll
      for (int k = 0; k < OUT; ++k) acc[k] += s_sum[v][k][lane];
  }
  if (valid) {
    const size_t i = (size_t)perm[s];
#pragma unroll
    for (int k = 0; k < OUT; ++k) F[i * OUT + k] = acc[k];
  }
}

// Waves a group by the number of groups: more of them fill the chip and shorten
// the longest walk, and repeat the walk itself.  Blobs, order 8, 1 | 4 | 8 waves:
// 32000 particles (500 groups) 1380 | 635 | 585 us, 64000 1806 | 915 | 987 us,
// 256000 3.70 | 2.68 | 3.12 ms, 2^20 10.4 | 10.2 | 12.6 ms; order 4 at 256000 1.42 |
// 1.46 | 2.01 ms, at 2^20 4.5 | 5.5 | 8.1 ms.
constexpr int kBHFewGroups = 512, kBHSomeGroups = 6144;
template <int P>
void bh_order(Tree& t, double* F, hipStream_t st) {
  const int n = (int)t.n;
  FMM_CHECK(7 * t.depth + 1 <= kBHStack, kUnsupported, "tree too deep for the Barnes-Hut walk");
  if (n == 0) return;
  PhaseTimer pt(t, kTBH, st);
  t.Qbh.alloc((size_t)t.ncells * BHRow<P>::SIZE);
  k_bh_coef<P><<<nblk(t.ncells, 4), 256, 0, st>>>(t.ncells, t.M.get(), t.cx.get(), t.cy.get(), t.cz.get(), t.cr.get(),
                                                   t.Qbh.get());
  const int groups = nblk(n, 64);
  auto run = [&](auto kern, int w) {
    const int grid = nblk(groups, 8 * kBHRun) * 8 * kBHRun;
    kern<<<grid, 64 * w, 0, st>>>(n, t.first_child.get(), t.nchild.get(), t.pstart.get(), t.pcount.get(), t.px.get(),
                                  t.py.get(), t.pz.get(), t.pS.get(), t.perm.get(),
                                  reinterpret_cast<const BHLine*>(t.Qbh.get()), t.theta, F);
  };
  if (groups <= kBHFewGroups) run(k_bh<P, 8>, 8);
  else if (groups <= kBHSomeGroups) run(k_bh<P, 4>, 4);
  else run(k_bh<P, 1>, 1);
}

}  // namespace FMM_VARIANT_NS
}  // namespace fmm
