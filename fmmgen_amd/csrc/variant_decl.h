// Declarations shared by the base and per-order translation units of one
// operator variant.  Included after the generated device operator header
// (namespace fmmgen_ops, FMMGEN_* macros) with FMM_VARIANT_NS defined.
#pragma once

#include "evaluate.h"
#include "fmm_common.h"

namespace fmm {
namespace FMM_VARIANT_NS {

constexpr int SO = FMMGEN_SOURCEORDER;
constexpr int SS = FMMGEN_SOURCESIZE;
constexpr int OUT = FMMGEN_OUTPUTSIZE;
constexpr int PMIN = FMMGEN_MINORDER;
constexpr int PMAX = FMMGEN_MAXORDER;  // exclusive

inline int nblk(long long n, int bs) { return (int)((n + bs - 1) / bs); }

template <int P>
struct Op {
  static constexpr int MS = msize(P, SO);
  static constexpr int LS = lsize(P, SO);
};

// Per-order phases (defined in the per-order translation units).
template <int P>
void far_field_order(Tree& t, int mode, int mask, hipStream_t st);
template <int P>
void l2p_final_order(Tree& t, int mode, int mask, double* F, hipStream_t st);
template <int P>
void op_batch_order(int op, int n, const double* xyz, const double* in, int in_stride, double* out,
                    int out_stride, hipStream_t st);
template <int P>
void bh_order(Tree& t, double* F, hipStream_t st);
// M2L of the listed chunks at order Q on expansions stored at order ps.
template <int Q>
void m2l_class(Tree& t, int mode, const int* chunks, int nch, int ps, hipStream_t st);
// Whether the M2L of an evaluation runs in the harmonic layout (p: the order
// the expansions are stored at).  Automatic: charges in the mixed and learned
// modes always; otherwise where the shorter GEMM pays for the fold and unfold
// launches, which is everywhere but at few groups and low order, and, for dipoles
// and quadrupoles in the mixed modes, only where it rounds no worse.  Measured
// (full -> harmonic, one evaluation, theta 0.5, ncrit 64):
//   FP64 charges   2^22 blobs, order 10 147 -> 66.6 ms; 2^20 uniform, order 8
//                  11.2 -> 8.9 ms, order 2 6.73 -> 6.55 ms; 10^5 (156k groups)
//                  order 4 932 -> 910 us; 2000 (383 groups) order 4 275 -> 278
//                  us, order 6 318 -> 313 us
//   FP32 dipoles   10^6 Plummer, theta 0.4, order 6 18.5 -> 13.5 ms; 10^5
//                  order 4 927 -> 917 us; 2000 302 -> 311 us
// Far-field error of the harmonic over the full form against FP64, mean of 12
// sets (uniform, blobs, Plummer, mixed; theta 0.4 to 0.55):
//   FP32    dipoles order 2 1.00, orders 3 to 8 0.85 to 0.95; quadrupoles orders
//           3 to 5 0.79 to 0.93, 6 1.07, 7 and 8 0.90
//   BF16x3  dipoles 1.00 to 1.01 (up to 1.03), quadrupoles 1.08 to 1.10 (up to
//           1.17): a folded multipole is split as one value
constexpr int kHarmMinOrder = 6, kHarmMinGroups = 1 << 14, kHarmMinGroupsMixed = 1 << 17;
inline bool m2l_harmonic(const Tree& t, int mode, int p) {
  if (t.m2l_form == kM2LFull) return false;
  if (t.m2l_form == kM2LHarmonic) return true;
  if (mode != 0 && SO > 0)
    return mode == 1 && p >= 3 && !(SO == 2 && p == 6) && t.sched.ngroups >= kHarmMinGroupsMixed;
  if (mode != 0) return true;
  return p >= kHarmMinOrder || t.sched.ngroups >= kHarmMinGroups;
}

// Whether the FP64 M2L stores every chunk's sums and adds a tile's chunks in
// order, so that an evaluation repeats bit for bit, instead of adding them into L
// with atomics: the finer chunk list at the orders whose rows are one wave's.
inline bool m2l_parts(const Tree& t, int p) { return p < kM2LBalancedOrder && t.sched.nchunks64 > 0; }
// Whether the near field of an evaluation stores its sums by items.
inline bool near_rows(const Tree& t, int mode) { return mode == 0 && t.p2p_items(true).rows > 0; }

// Order-independent phases (defined in the base translation unit).
void near_field(Tree& t, int mode, hipStream_t st);

}  // namespace FMM_VARIANT_NS
}  // namespace fmm
