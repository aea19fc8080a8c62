// Per-order kernels of one operator variant: P2M, M2M, M2L, L2L and L2P
// with the generated operator bodies inlined.  The phase arithmetic follows
// example/calculate.cpp:135-250:
//   P2M  per leaf, the example's P2M through M2M (generated P2M_S_<p>),
//        x = leaf centre - particle
//   M2M  one level at a time, deepest first, x = parent - child
//   M2L  per target cell over its M2L sources, x = target - source
//   L2L  one level at a time, root first, x = child - parent
//   L2P  per particle, x = particle - leaf centre, added in FP64 to the
//        near-field sum and written in caller order.
#pragma once

#include "m2l_gemm.h"
#include "variant_decl.h"
#include "wave_ops.h"

namespace fmm {
namespace FMM_VARIANT_NS {

// Output proxy of a generated body that keeps slots [LO, HI) in registers.
// Inlined with constant slot indices, every output outside the chunk folds
// to dead code, so one instantiation per chunk computes only its slots.
template <typename T, int LO, int HI>
struct ChunkAcc {
  T v[HI - LO];
  struct Ref {
    T* p;
    __device__ __forceinline__ void operator+=(T x) {
      if (p) *p += x;
    }
  };
  __device__ __forceinline__ Ref operator[](int k) { return Ref{(k >= LO && k < HI) ? &v[k - LO] : nullptr}; }
};

constexpr int kChunk = FMMGEN_CHUNK;  // expansion slots per thread (one pruned generated body per chunk)

template <int NCH, typename F>
__device__ __forceinline__ void dispatch_chunk(int ch, F&& f) {
  static_for<NCH>([&](auto C) {
    if (ch == C) f(C);
  });
}

// P2M: the example's P2M through M2M (example/calculate.cpp:135-161),
// x = leaf centre - particle, one thread per (leaf, slot chunk).
template <int P>
__global__ __launch_bounds__(64) void k_p2m(int nleaves, const int* __restrict__ leaves, const int* __restrict__ pstart,
                      const int* __restrict__ pcount, const double* __restrict__ cx, const double* __restrict__ cy,
                      const double* __restrict__ cz, const double* __restrict__ px, const double* __restrict__ py,
                      const double* __restrict__ pz, const double* __restrict__ pS, double* __restrict__ M) {
  constexpr int MS = Op<P>::MS, NCH = (MS + kChunk - 1) / kChunk;
  const int li = blockIdx.x * blockDim.x + threadIdx.x;
  if (li >= nleaves) return;
  const int c = leaves[li];
  const double x0 = cx[c], y0 = cy[c], z0 = cz[c];
  const int b = pstart[c], e = b + pcount[c];
  dispatch_chunk<NCH>(blockIdx.y, [&](auto C) {
    constexpr int LO = C * kChunk, HI = (LO + kChunk < MS) ? LO + kChunk : MS;
    ChunkAcc<double, LO, HI> acc;
#pragma unroll
    for (int k = 0; k < HI - LO; ++k) acc.v[k] = 0.0;
    for (int j = b; j < e; ++j)
      fmmgen_ops::P2M_S_chunk<P, LO / kChunk, double>(x0 - px[j], y0 - py[j], z0 - pz[j], pS + (size_t)j * SS, acc);
    double* Mc = M + (size_t)c * MS;
#pragma unroll
    for (int k = 0; k < HI - LO; ++k) Mc[LO + k] = acc.v[k];
  });
}

// The same for charges with one wave a leaf: lanes own slots, and 32 particles
// at a time stage q and u^k / k! (k <= P) in LDS, M_n += q X Y Z.  A thread a
// (leaf, chunk) leaves most of the chip idle on small sets and loops each lane
// over its own leaf: 2000 particles, order 4 17.5 -> 5.5 us; 2^20, order 8 117 ->
// 82 us.  Bound by the three LDS reads a slot and particle.
template <int P>
__global__ __launch_bounds__(64) void k_p2m_leaf(int nleaves, const int* __restrict__ leaves, const int* __restrict__ pstart,
                      const int* __restrict__ pcount, const double* __restrict__ cx, const double* __restrict__ cy,
                      const double* __restrict__ cz, const double* __restrict__ px, const double* __restrict__ py,
                      const double* __restrict__ pz, const double* __restrict__ pS, double* __restrict__ M) {
  static_assert(SO == 0 || P < 0, "charges only");
  constexpr int MS = Op<P>::MS, NPL = (MS + 63) / 64, NB = 32, PW = (3 * (P + 1)) | 1;
  __shared__ double pw[NB * PW];  // particle k: q X[0..P], Y[0..P], Z[0..P]
  const int lane = threadIdx.x, c = leaves[blockIdx.x];
  const double x0 = cx[c], y0 = cy[c], z0 = cz[c];
  int ea[NPL], eb[NPL], ec[NPL];
  double acc[NPL];
#pragma unroll
  for (int i = 0; i < NPL; ++i) {
    const MultiIdx m = slot_multi_rt(min(lane + 64 * i, MS - 1));
    ea[i] = m.x;
    eb[i] = P + 1 + m.y;
    ec[i] = 2 * (P + 1) + m.z;
    acc[i] = 0.0;
  }
  const int b = pstart[c], e = b + pcount[c];
  for (int base = b; base < e; base += NB) {
    const int nk = min(NB, e - base);
    wave_lds_fence();  // previous particles consumed
    for (int t = lane; t < 3 * nk; t += 64) {  // one (particle, axis) a lane
      const int k = t / 3, d = t - 3 * k, j = base + k;
      const double u = d == 0 ? x0 - px[j] : d == 1 ? y0 - py[j] : z0 - pz[j];
      double v = d == 0 ? pS[j] : 1.0;
      double* o = pw + k * PW + d * (P + 1);
      o[0] = v;
      static_for<P>([&](auto K) {
        v *= u * (1.0 / (K + 1));
        o[K + 1] = v;
      });
    }
    wave_lds_fence();
    for (int k = 0; k < nk; ++k) {
      const double* w = pw + k * PW;
#pragma unroll
      for (int i = 0; i < NPL; ++i) acc[i] = fma(w[ea[i]] * w[eb[i]], w[ec[i]], acc[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < NPL; ++i)
    if (lane + 64 * i < MS) M[(size_t)c * MS + lane + 64 * i] = acc[i];
}

// M2M of the levels of few parents: a block a parent, a wave a child.  Each wave
// shifts its child's multipole along the three axes in LDS (at most P + 1 terms
// a slot and axis), and the block adds the children in order.  A thread a
// (parent, chunk) takes the children one after the other: 10^5 particles, order 4
// 8.5 -> 4.7 us a level; levels of up to 512 parents, order 8 29 -> 10 us.  On 4096
// parents of eight children its generated bodies, the chip full, are faster (37
// against 73 us); from order 10 on they are not (2^22 blobs, all levels 1.9 -> 1.2
// ms).
constexpr int kM2MWaveParents = 1024, kM2MWaveOrder = 10;
template <int P>
__global__ __launch_bounds__(512) void k_m2m_wave(int beg, const int* __restrict__ first_child, const int* __restrict__ nchild,
                      const double* __restrict__ cx, const double* __restrict__ cy, const double* __restrict__ cz,
                      double* __restrict__ M) {
  constexpr int MS = Op<P>::MS, NT = nterms(P), OFF = NT - MS;
  __shared__ double sA[8][NT], sB[8][NT], sP[8][3 * (P + 1)];
  const int p = beg + blockIdx.x, k = nchild[p];
  if (k == 0) return;  // uniform over the block
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (w < k) {
    const int c = first_child[p] + w;
    for (int j = lane; j < NT; j += 64) sA[w][j] = j >= OFF ? M[(size_t)c * MS + j - OFF] : 0.0;
    wave_powers<P>(lane, cx[p] - cx[c], cy[p] - cy[c], cz[p] - cz[c], sP[w]);
    wave_lds_fence();
    wave_shift3<P, true>(lane, sA[w], sB[w], sP[w]);
  }
  __syncthreads();
  for (int j = threadIdx.x; j < MS; j += 512) {
    double v = 0.0;
    for (int c = 0; c < k; ++c) v += sB[c][j + OFF];
    M[(size_t)p * MS + j] = v;
  }
}

// M2M (example/calculate.cpp:163-187), x = parent - child, one thread per
// (parent, slot chunk) of one level; children are summed in registers.
template <int P>
__global__ __launch_bounds__(64) void k_m2m(int beg, int end, const int* __restrict__ first_child, const int* __restrict__ nchild,
                      const double* __restrict__ cx, const double* __restrict__ cy, const double* __restrict__ cz,
                      double* __restrict__ M) {
  constexpr int MS = Op<P>::MS, NCH = (MS + kChunk - 1) / kChunk;
  const int p = beg + blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= end) return;
  const int k = nchild[p];
  if (k == 0) return;
  const int fc = first_child[p];
  dispatch_chunk<NCH>(blockIdx.y, [&](auto C) {
    constexpr int LO = C * kChunk, HI = (LO + kChunk < MS) ? LO + kChunk : MS;
    ChunkAcc<double, LO, HI> acc;
#pragma unroll
    for (int j = 0; j < HI - LO; ++j) acc.v[j] = 0.0;
    for (int c = fc; c < fc + k; ++c)
      fmmgen_ops::M2M_chunk<P, LO / kChunk, double>(cx[p] - cx[c], cy[p] - cy[c], cz[p] - cz[c],
                                   static_cast<const double*>(M + (size_t)c * MS), acc);
    double* Mp = M + (size_t)p * MS;
#pragma unroll
    for (int j = 0; j < HI - LO; ++j) Mp[LO + j] = acc.v[j];
  });
}

// D vector of every M2L key (the derivative block of the generated M2L
// operator, fmmgen/writer.py:168-182), FP64, or normalised by the target
// half-width (Dhat_k = D_k r^(|k|+1)) and rounded to FP32.
template <int P, typename T, bool SCALED>
__global__ void k_dtab(int nkeys, const double* __restrict__ key_dx, const double* __restrict__ key_r,
                       T* __restrict__ Dtab) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nkeys) return;
  constexpr int MS = Op<P>::MS;
  double D[MS];
  fmmgen_ops::Dgen_o<P, double>(key_dx[3 * k], key_dx[3 * k + 1], key_dx[3 * k + 2], D);
  if constexpr (SCALED) {
    const double r = key_r[k];
    double pw[P + 2];
    pw[0] = r;
#pragma unroll
    for (int d = 1; d <= P + 1; ++d) pw[d] = pw[d - 1] * r;
#pragma unroll
    for (int j = 0; j < MS; ++j) D[j] *= pw[slot_degree(j + M2LPlan<P, SO>::OFF)];
  }
#pragma unroll
  for (int j = 0; j < MS; ++j) Dtab[(size_t)k * MS + j] = (T)D[j];
}

template <int P, int W, int LAY = kGraded>
const unsigned* ensure_index_table(Tree& t, hipStream_t st) {
  static_assert(W == 2 || W == 4 || W == 8, "blocks of 2, 4 or 8 waves");
  M2LSchedule& S = t.sched;
  const int wi = W == 8 ? 1 : (W == 2 ? 2 : 0);
  if (!S.idx_ready[LAY][P][wi]) {
    static const std::vector<unsigned> tab = m2l_index_table<P, SO, W, LAY>();  // once per process
    S.idxtab[LAY][P][wi].alloc(tab.size());
    FMM_HIP(hipMemcpyAsync(S.idxtab[LAY][P][wi].get(), tab.data(), sizeof(unsigned) * tab.size(),
                           hipMemcpyHostToDevice, st));
    FMM_HIP(hipStreamSynchronize(st));  // evaluations on other streams may follow
    S.idx_ready[LAY][P][wi] = true;
  }
  return S.idxtab[LAY][P][wi].get();
}

// Harmonic-layout M2L around the GEMM: fold every cell's multipole (M,
// graded, stride ms) into Mh and clear Lh (rows of order PS; with `parts` the
// GEMM writes rows of its own instead), then, after the GEMM, store the unfolded
// rows into L (graded, stride ls).
template <int PS, typename T>
void harm_fold(Tree& t, const T* M, int ms, DevBuf<T>& Mh, DevBuf<T>& Lh, hipStream_t st, bool parts = false) {
  const int nc = t.ncells, hs = harm_msize(PS, SO), ls = parts ? 0 : harm_lsize(PS, SO);
  Mh.alloc((size_t)nc * hs);
  if (!parts) Lh.alloc((size_t)nc * ls);
  if (nc == 0) return;
  constexpr int per = 4 * kHarmCellsPerWave;
  k_harm_fold<PS, SO, T><<<(nc + per - 1) / per, 256, 0, st>>>(nc, M, ms, Mh.get(), hs, Lh.get(), ls);
}
template <int PS, typename T, bool PART = false>
void harm_unfold(Tree& t, const DevBuf<T>& Lh, T* L, int ls, hipStream_t st) {
  if (t.ncells == 0) return;
  constexpr int per = 4 * kHarmCellsPerWave;
  k_harm_unfold<PS - SO, T, PART><<<(t.ncells + per - 1) / per, 256, 0, st>>>(
      t.ncells, Lh.get(), harm_lsize(PS, SO), L, ls, t.sched.cell_slot.get(), t.sched.chunk64_first.get());
}

template <int P, int W, int LAY = kGraded>
const unsigned* ensure_index_table32(Tree& t, hipStream_t st) {
  M2LSchedule& S = t.sched;
  if (!S.idx32_ready[LAY][P]) {
    static const std::vector<unsigned> tab = m2l_index_table32<P, SO, W, LAY>();  // once per process
    S.idxtab32[LAY][P].alloc(tab.size());
    FMM_HIP(hipMemcpyAsync(S.idxtab32[LAY][P].get(), tab.data(), sizeof(unsigned) * tab.size(),
                           hipMemcpyHostToDevice, st));
    FMM_HIP(hipStreamSynchronize(st));  // evaluations on other streams may follow
    S.idx32_ready[LAY][P] = true;
  }
  return S.idxtab32[LAY][P].get();
}

// FP64 M2L of the given chunks; PART: the chunks' sums are stored and a tile's
// chunks added in order (m2l_parts).
template <int P, bool PART>
void m2l_plain_run(Tree& t, int n, const int* tile, const int* g0, const int* g1, hipStream_t st) {
  M2LSchedule& S = t.sched;
  const int grid = ((n + 7) / 8) * 8;
  auto run = [&](auto kern, int W, const unsigned* idx, int mstride, int lstride, const double* M, double* L) {
    kern<<<grid, 64 * W, 0, st>>>(n, grid, S.tile_cells.get(), tile, g0, g1, S.group_key.get(), S.group_src.get(),
                                  S.key_dlevel.get(), S.Dtab64.get(), idx, t.tile_order_ptr(), nullptr, Op<P>::MS,
                                  mstride, lstride, M, L);
  };
  if (m2l_harmonic(t, 0, P)) {
    constexpr int W = m2l_waves<P, SO, double, kHarmonic>(), HL = harm_lsize(P, SO);
    const unsigned* idx = ensure_index_table<P, W, kHarmonic>(t, st);
    harm_fold<P, double>(t, t.M.get(), Op<P>::MS, t.Mh64, t.Lh64, st, PART);
    if (PART) t.Lpart.alloc((size_t)n * kTile * HL);
    DevBuf<double>& Lh = PART ? t.Lpart : t.Lh64;
    run(k_m2l_gemm<P, SO, double, false, W, kHarmonic, PART>, W, idx, harm_msize(P, SO), HL, t.Mh64.get(), Lh.get());
    harm_unfold<P, double, PART>(t, Lh, t.L.get(), Op<P>::LS, st);
    return;
  }
  constexpr int W = m2l_waves<P, SO, double>(), LS = Op<P>::LS;
  const unsigned* idx = ensure_index_table<P, W>(t, st);
  if (PART) t.Lpart.alloc((size_t)n * kTile * LS);
  run(k_m2l_gemm<P, SO, double, false, W, kGraded, PART>, W, idx, Op<P>::MS, LS, t.M.get(),
      PART ? t.Lpart.get() : t.L.get());
  if (PART)
    k_chunk_sum<double><<<nblk((long long)t.ncells * LS, 256), 256, 0, st>>>(
        t.ncells, LS, S.cell_slot.get(), S.chunk64_first.get(), t.Lpart.get(), t.L.get());
}

template <int P>
void m2l_plain(Tree& t, hipStream_t st) {
  M2LSchedule& S = t.sched;
  if (S.ngroups == 0) return;
  S.Dtab64.alloc((size_t)S.nkeys * Op<P>::MS);
  k_dtab<P, double, false><<<nblk(S.nkeys, 64), 64, 0, st>>>(S.nkeys, S.key_dx.get(), S.key_r.get(), S.Dtab64.get());
  const bool fine = S.nchunks64 > 0;
  const int n = fine ? S.nchunks64 : S.nchunks;
  const int* tile = fine ? S.chunk64_tile.get() : S.chunk_tile.get();
  const int* g0 = fine ? S.chunk64_g0.get() : S.chunk_g0.get();
  const int* g1 = fine ? S.chunk64_g1.get() : S.chunk_g1.get();
  if constexpr (P < kM2LBalancedOrder) {
    if (m2l_parts(t, P)) {
      m2l_plain_run<P, true>(t, n, tile, g0, g1, st);
      return;
    }
  }
  m2l_plain_run<P, false>(t, n, tile, g0, g1, st);
}

// L2L (example/calculate.cpp:219-234), x = child - parent, one thread per
// (child, slot chunk) of one level.
template <int P>
__global__ __launch_bounds__(64) void k_l2l(int beg, int end, const int* __restrict__ parent, const double* __restrict__ cx,
                      const double* __restrict__ cy, const double* __restrict__ cz, double* __restrict__ L) {
  constexpr int LS = Op<P>::LS, NCH = (LS + kChunk - 1) / kChunk;
  const int c = beg + blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= end) return;
  const int p = parent[c];
  dispatch_chunk<NCH>(blockIdx.y, [&](auto C) {
    constexpr int LO = C * kChunk, HI = (LO + kChunk < LS) ? LO + kChunk : LS;
    ChunkAcc<double, LO, HI> acc;
#pragma unroll
    for (int j = 0; j < HI - LO; ++j) acc.v[j] = 0.0;
    fmmgen_ops::L2L_chunk<P, LO / kChunk, double>(cx[c] - cx[p], cy[c] - cy[p], cz[c] - cz[p],
                                 static_cast<const double*>(L + (size_t)p * LS), acc);
    double* Lc = L + (size_t)c * LS;
#pragma unroll
    for (int j = 0; j < HI - LO; ++j) Lc[LO + j] += acc.v[j];
  });
}

// The same with a wave a child, four children a block: the parent's expansion is
// shifted axis by axis in LDS.  From local order 8 on the generated bodies cost
// more than the loops' indices: 2^20 particles, order 8 264 -> 82 us over all
// levels, 2^22 blobs, order 10 1.13 -> 0.72 ms.  At local orders 5 to 7 the bodies
// are the faster ones (2^20, order 6 72 against 98 us).
constexpr int kL2LWaveOrder = 8;
template <int P>
__global__ __launch_bounds__(256) void k_l2l_wave(int beg, int end, const int* __restrict__ parent, const double* __restrict__ cx,
                      const double* __restrict__ cy, const double* __restrict__ cz, double* __restrict__ L) {
  constexpr int LS = Op<P>::LS, Q = P - SO;
  __shared__ double sA[4][LS], sB[4][LS], sP[4][3 * (Q + 1)];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, c = beg + blockIdx.x * 4 + w;
  if (c >= end) return;  // no barrier below
  const int p = parent[c];
  for (int j = lane; j < LS; j += 64) sA[w][j] = L[(size_t)p * LS + j];
  wave_powers<Q>(lane, cx[c] - cx[p], cy[c] - cy[p], cz[c] - cz[p], sP[w]);
  wave_lds_fence();
  wave_shift3<Q, false>(lane, sA[w], sB[w], sP[w]);
  double* Lc = L + (size_t)c * LS;
  for (int j = lane; j < LS; j += 64) Lc[j] += sB[w][j];
}

// Near plus far field.  Fnear: a row a particle, or with row_off a row a work
// item and target (the items of leaf c from row_off[c], pcount[c] rows each),
// added in the items' order.  (Rows instead of atomics into one output, for the
// sake of repeatable sums, with the M2L's by chunks: 2000 particles 54.0 -> 53.5 us
// an evaluation, 10^5 493 -> 484 us, 2^20 7.06 -> 7.00 ms.)
template <int P>
__global__ __launch_bounds__(64) void k_l2p_final(int n, const int* __restrict__ leaf_of, const int* __restrict__ perm,
                            const double* __restrict__ cx, const double* __restrict__ cy,
                            const double* __restrict__ cz, const double* __restrict__ px,
                            const double* __restrict__ py, const double* __restrict__ pz,
                            const double* __restrict__ L, const double* __restrict__ Fnear,
                            const long long* __restrict__ row_off, const int* __restrict__ pstart,
                            const int* __restrict__ pcount, int use_l2p, double* __restrict__ F) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  double acc[OUT];
  const int c = leaf_of[j];
#pragma unroll
  for (int k = 0; k < OUT; ++k) acc[k] = Fnear && !row_off ? Fnear[(size_t)j * OUT + k] : 0.0;
  if (Fnear && row_off) {
    const int nt = pcount[c], m = (int)((row_off[c + 1] - row_off[c]) / nt);  // items of the leaf
    const double* row = Fnear + (size_t)(row_off[c] + (j - pstart[c])) * OUT;
    constexpr int B = 4;  // rows in flight (past the last one: that one again, not added)
    for (int i = 0; i < m; i += B) {
      double x[B][OUT];
#pragma unroll
      for (int u = 0; u < B; ++u)
#pragma unroll
        for (int k = 0; k < OUT; ++k) x[u][k] = row[(size_t)min(i + u, m - 1) * nt * OUT + k];
#pragma unroll
      for (int u = 0; u < B; ++u)
        if (i + u < m) {
#pragma unroll
          for (int k = 0; k < OUT; ++k) acc[k] += x[u][k];
        }
    }
  }
  if (use_l2p) {
    fmmgen_ops::L2P_o<P, double>(px[j] - cx[c], py[j] - cy[c], pz[j] - cz[c], L + (size_t)c * Op<P>::LS, acc);
  }
  const int i = perm[j];
#pragma unroll
  for (int k = 0; k < OUT; ++k) F[(size_t)i * OUT + k] = acc[k];
}

}  // namespace FMM_VARIANT_NS
}  // namespace fmm

#include "bh.h"
#include "op_batch.h"
#include "variant_mixed.h"

namespace fmm {
namespace FMM_VARIANT_NS {

template <int P>
void m2l_mixed(Tree& t, int mode, hipStream_t st) {
  M2LSchedule& S = t.sched;
  if (S.ngroups == 0) return;
  S.Dtab32.alloc((size_t)S.nkeys * Op<P>::MS);
  k_dtab<P, float, true><<<nblk(S.nkeys, 64), 64, 0, st>>>(S.nkeys, S.key_dx.get(), S.key_r.get(), S.Dtab32.get());
  const bool harm = m2l_harmonic(t, mode, P);
  if (harm) harm_fold<P, float>(t, t.Mf.get(), Op<P>::MS, t.Mhf, t.Lhf, st);
  if (t.use_tile_order && t.m2l_classes) {  // learned order: one launch per tile-order class
    t.m2l_classes(t, mode, P, st);
  } else {
    m2l_class<P>(t, mode, nullptr, S.nchunks, P, st);
  }
  if (harm) harm_unfold<P, float>(t, t.Lhf, t.Lf.get(), Op<P>::LS, st);
}

// FP32 / BF16x3 M2L of the listed chunks (all when chunks == nullptr) at
// order Q, on expansions and D vectors stored at order ps (the layouts are
// prefixes: row strides of order ps).
template <int Q>
void m2l_class(Tree& t, int mode, const int* chunks, int nch, int ps, hipStream_t st) {
  M2LSchedule& S = t.sched;
  if (nch == 0) return;
  const int grid = ((nch + 7) / 8) * 8;
  const int ms = msize(ps, SO), ls = lsize(ps, SO);
  if (mode == 2) {  // BF16x3 split precision
    if (m2l_harmonic(t, mode, ps)) {
      constexpr int W32 = m2l_waves32<Q, SO, kHarmonic>();
      const unsigned* idx = ensure_index_table32<Q, W32, kHarmonic>(t, st);
      k_m2l_bf16x3<Q, SO, W32, kHarmonic><<<grid, 64 * W32, 0, st>>>(
          nch, grid, S.tile_cells.get(), S.chunk_tile.get(), S.chunk_g0.get(), S.chunk_g1.get(), S.group_key.get(),
          S.group_src.get(), S.key_dlevel.get(), S.Dtab32.get(), idx, t.tile_order_ptr(), chunks, ms,
          harm_msize(ps, SO), harm_lsize(ps, SO), t.Mhf.get(), t.Lhf.get());
      return;
    }
    constexpr int W32 = m2l_waves32<Q, SO>();
    const unsigned* idx = ensure_index_table32<Q, W32>(t, st);
    k_m2l_bf16x3<Q, SO, W32><<<grid, 64 * W32, 0, st>>>(nch, grid, S.tile_cells.get(), S.chunk_tile.get(), S.chunk_g0.get(),
                                             S.chunk_g1.get(), S.group_key.get(), S.group_src.get(),
                                             S.key_dlevel.get(), S.Dtab32.get(), idx, t.tile_order_ptr(), chunks,
                                             ms, ms, ls, t.Mf.get(), t.Lf.get());
    return;
  }
  if (m2l_harmonic(t, mode, ps)) {
    constexpr int W = m2l_waves<Q, SO, float, kHarmonic>();
    const unsigned* idx = ensure_index_table<Q, W, kHarmonic>(t, st);
    k_m2l_gemm<Q, SO, float, true, W, kHarmonic><<<grid, 64 * W, 0, st>>>(
        nch, grid, S.tile_cells.get(), S.chunk_tile.get(), S.chunk_g0.get(), S.chunk_g1.get(), S.group_key.get(),
        S.group_src.get(), S.key_dlevel.get(), S.Dtab32.get(), idx, t.tile_order_ptr(), chunks, ms,
        harm_msize(ps, SO), harm_lsize(ps, SO), t.Mhf.get(), t.Lhf.get());
    return;
  }
  constexpr int W = m2l_waves<Q, SO, float>();
  const unsigned* idx = ensure_index_table<Q, W>(t, st);
  k_m2l_gemm<Q, SO, float, true, W><<<grid, 64 * W, 0, st>>>(
      nch, grid, S.tile_cells.get(), S.chunk_tile.get(), S.chunk_g0.get(), S.chunk_g1.get(), S.group_key.get(),
      S.group_src.get(), S.key_dlevel.get(), S.Dtab32.get(), idx, t.tile_order_ptr(), chunks, ms, ms, ls,
      t.Mf.get(), t.Lf.get());
}

template <int P>
void far_field_order(Tree& t, int mode, int mask, hipStream_t st) {
  if (mode != 0) {
    far_field_mixed<P>(t, mode, mask, st);
    return;
  }
  const int nc = t.ncells;
  if (mask & kPhaseP2M) {
    PhaseTimer pt(t, kTP2M, st);
    auto run = [&](auto kern, dim3 grid) {
      kern<<<grid, 64, 0, st>>>(t.nleaves, t.leaves.get(), t.pstart.get(), t.pcount.get(), t.cx.get(), t.cy.get(),
                                t.cz.get(), t.px.get(), t.py.get(), t.pz.get(), t.pS.get(), t.M.get());
    };
    if constexpr (SO == 0) run(k_p2m_leaf<P>, t.nleaves);
    else run(k_p2m<P>, dim3(nblk(t.nleaves, 64), (Op<P>::MS + kChunk - 1) / kChunk));
  }
  if (mask & kPhaseM2M) {
    PhaseTimer pt(t, kTM2M, st);
    for (int l = t.depth - 2; l >= 0; --l) {
      const int b = t.level_off[l], e = t.level_off[l + 1];
      if (P >= kM2MWaveOrder || e - b <= kM2MWaveParents) {
        k_m2m_wave<P><<<e - b, 512, 0, st>>>(b, t.first_child.get(), t.nchild.get(), t.cx.get(), t.cy.get(),
                                             t.cz.get(), t.M.get());
        continue;
      }
      if constexpr (P < kM2MWaveOrder)
        k_m2m<P><<<dim3(nblk(e - b, 64), (Op<P>::MS + kChunk - 1) / kChunk), 64, 0, st>>>(
            b, e, t.first_child.get(), t.nchild.get(), t.cx.get(), t.cy.get(), t.cz.get(), t.M.get());
    }
  }
  if (mask & kPhaseM2L) {
    PhaseTimer pt(t, kTM2L, st);
    m2l_plain<P>(t, st);
  }
  if (mask & kPhaseL2L) {
    PhaseTimer pt(t, kTL2L, st);
    for (int l = 1; l < t.depth; ++l) {
      const int b = t.level_off[l], e = t.level_off[l + 1];
      if constexpr (P - SO >= kL2LWaveOrder)
        k_l2l_wave<P><<<nblk(e - b, 4), 256, 0, st>>>(b, e, t.parent.get(), t.cx.get(), t.cy.get(), t.cz.get(),
                                                      t.L.get());
      else
        k_l2l<P><<<dim3(nblk(e - b, 64), (Op<P>::LS + kChunk - 1) / kChunk), 64, 0, st>>>(
            b, e, t.parent.get(), t.cx.get(), t.cy.get(), t.cz.get(), t.L.get());
    }
  }
}

template <int P>
void l2p_final_order(Tree& t, int mode, int mask, double* F, hipStream_t st) {
  if (mode != 0) {
    l2p_mixed<P>(t, mask, F, st);
    return;
  }
  const int n = (int)t.n;
  PhaseTimer pt(t, kTL2P, st);
  const bool rows = near_rows(t, mode);
  k_l2p_final<P><<<nblk(n, 64), 64, 0, st>>>(n, t.leaf_of.get(), t.perm.get(), t.cx.get(), t.cy.get(),
                                               t.cz.get(), t.px.get(), t.py.get(), t.pz.get(), t.L.get(),
                                               !(mask & kPhaseP2P) ? nullptr : rows ? t.Fseg.get() : t.Fp2p.get(),
                                               rows ? t.p2p64.row_off.get() : nullptr, t.pstart.get(),
                                               t.pcount.get(), (mask & kPhaseL2P) ? 1 : 0, F);
}

}  // namespace FMM_VARIANT_NS
}  // namespace fmm

#define FMM_INSTANTIATE_ORDER(P)                                                                        \
  namespace fmm {                                                                                       \
  namespace FMM_VARIANT_NS {                                                                            \
  template void far_field_order<P>(Tree&, int, int, hipStream_t);                                       \
  template void l2p_final_order<P>(Tree&, int, int, double*, hipStream_t);                              \
  template void op_batch_order<P>(int, int, const double*, const double*, int, double*, int, hipStream_t); \
  template void bh_order<P>(Tree&, double*, hipStream_t);                                                 \
  template void m2l_class<P>(Tree&, int, const int*, int, int, hipStream_t);                         \
  }                                                                                                     \
  }
