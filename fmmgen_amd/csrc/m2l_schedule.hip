// M2L schedule: target tiles and (tile, offset) groups.
//
// The M2L list (example/calculate.cpp:190-206, one M2L(A - B, M_B, L_A) per
// pair) is regrouped so that the translation runs as small GEMMs:
//   * target cells that have M2L sources are cut into tiles of kTile cells
//     of one level, ordered by (octant, parent octant) class and then
//     canonically, so the cells of a tile share most relative offsets;
//   * a pair's key is (target level, source level, centre offset in units
//     of the finer half-width).  Centres sit on a dyadic lattice, so all
//     pairs of one key share one translation matrix T[n][m] = D_{n+m}
//     (up to the last-bit rounding of the FP64 centres);
//   * a group is (tile, key): at most one source per tile column (the
//     source of a target at a given key is unique), so the group is one
//     16-column operand of the tile's GEMM; the tile's group list is cut
//     into chunks (a block each) whose results add atomically, or are stored
//     and added in order (m2l_parts).
#include <cstring>

#include <rocprim/rocprim.hpp>

#include <algorithm>
#include <cmath>

#include "evaluate.h"
#include "fmm_common.h"

namespace fmm {

namespace {

inline int blocks(long long n, int bs) { return (int)((n + bs - 1) / bs); }

struct HasM2L {  // cells with M2L sources
  const int* off;
  __host__ __device__ int operator()(int c) const { return off[c + 1] > off[c] ? 1 : 0; }
};

// cnt[l] = cells with M2L sources before level l (rank: their exclusive scan)
__global__ void k_level_ranks(int depth, const int* __restrict__ level_off, const int* __restrict__ rank,
                              int* __restrict__ cnt) {
  const int l = blockIdx.x * blockDim.x + threadIdx.x;
  if (l <= depth) cnt[l] = rank[level_off[l]];
}

// Tile order of a level's targets: (octant, parent octant) class first,
// canonical order inside a class.  Away from the domain boundary, cells of
// one class see the same set of relative M2L offsets, so a tile of them
// fills its 16 columns for most offsets.  Cells without M2L work sort last.
// With a per-cell order hint (the learned order the cell is predicted to
// run at), cells of one class are further ordered by hint, so that a tile
// (which runs at the largest order of its cells) holds cells of one order.
__global__ void k_tile_keys(int nc, const int* __restrict__ off, const int* __restrict__ level,
                            const int* __restrict__ octant, const int* __restrict__ parent,
                            const int* __restrict__ hint, unsigned long long* __restrict__ key) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nc) return;
  const bool has = off[c + 1] > off[c];
  const unsigned cls = (unsigned)(octant[c] * 8 + octant[parent[c]]);
  const unsigned h = hint ? (unsigned)min(max(hint[c], 0), 15) : 0u;
  key[c] = has ? (((unsigned long long)level[c] << 42) | ((unsigned long long)cls << 36) |
                  ((unsigned long long)h << 32) | (unsigned)c)
               : (31ull << 42);
}

// Tiles of 16 in key order, starting anew on every level: level l holds sorted
// entries from cnt[l] and tiles from base[l].
__global__ void k_assign_tiles(int total, const unsigned long long* __restrict__ key_sorted,
                               const int* __restrict__ cnt, const int* __restrict__ base, int* __restrict__ slot,
                               int* __restrict__ tile_cells) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const unsigned long long k = key_sorted[i];
  const int c = (int)(k & 0xffffffffu), l = (int)(k >> 42);
  const int j = i - cnt[l], t = base[l] + j / kTile, col = j % kTile;
  slot[c] = t * kTile + col;
  tile_cells[t * kTile + col] = c;
}

// Per pair: key (target level, source level, quantised offset per axis, lb and
// qb bits a field) and the pair's target.  Offsets are integer multiples of the
// finer half-width, at most half in size; half < 2^(qb - 1).
__global__ void k_pair_key(long long m, const int* __restrict__ off, const int* __restrict__ src, int ncells,
                           const int* __restrict__ level, const double* __restrict__ cx,
                           const double* __restrict__ cy, const double* __restrict__ cz,
                           const double* __restrict__ cr, int lb, int qb, int half,
                           unsigned long long* __restrict__ key, int* __restrict__ tgt) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= m) return;
  // target of entry i by binary search in the CSR offsets
  int lo = 0, hi = ncells;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= i) lo = mid; else hi = mid;
  }
  const int A = lo, B = src[i];
  tgt[i] = A;
  const double rf = fmin(cr[A], cr[B]);
  const unsigned long long qx = (unsigned long long)(llrint((cx[A] - cx[B]) / rf) + half);
  const unsigned long long qy = (unsigned long long)(llrint((cy[A] - cy[B]) / rf) + half);
  const unsigned long long qz = (unsigned long long)(llrint((cz[A] - cz[B]) / rf) + half);
  unsigned long long k = (unsigned long long)level[A];
  k = (k << lb) | (unsigned)level[B];
  k = (k << qb) | qx;
  k = (k << qb) | qy;
  key[i] = (k << qb) | qz;
}

// flag[m] = 0: the scan's last entry is the number of runs
__global__ void k_run_flags64(long long m, const unsigned long long* __restrict__ k, int* __restrict__ flag) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i > m) return;
  flag[i] = i < m && (i == 0 || k[i] != k[i - 1]) ? 1 : 0;
}

// Key ids in pair order and one representative pair per key.
__global__ void k_key_ids(long long m, const int* __restrict__ flag, const int* __restrict__ pos,
                          const int* __restrict__ order, const int* __restrict__ tgt, const int* __restrict__ src,
                          const int* __restrict__ level, const double* __restrict__ cx,
                          const double* __restrict__ cy, const double* __restrict__ cz,
                          const double* __restrict__ cr, int* __restrict__ keyid, double* __restrict__ key_dx,
                          double* __restrict__ key_r, int* __restrict__ key_dlevel) {
  const long long j = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (j >= m) return;
  const int id = pos[j] + flag[j] - 1;  // inclusive rank
  const int i = order[j];
  keyid[i] = id;
  if (flag[j]) {
    const int A = tgt[i], B = src[i];
    key_dx[3 * id + 0] = cx[A] - cx[B];
    key_dx[3 * id + 1] = cy[A] - cy[B];
    key_dx[3 * id + 2] = cz[A] - cz[B];
    key_r[id] = cr[A];
    key_dlevel[id] = level[A] - level[B];
  }
}

__global__ void k_group_keys(long long m, int kb, const int* __restrict__ tgt, const int* __restrict__ keyid,
                             const int* __restrict__ slot, unsigned long long* __restrict__ comp) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i < m) comp[i] = ((unsigned long long)((unsigned)slot[tgt[i]] / kTile) << kb) | (unsigned)keyid[i];
}

// Groups and the first group of every tile (every tile has one: its cells all
// have M2L sources); tile_first[ntiles] = the number of groups.
__global__ void k_fill_groups(long long m, int kb, int ntiles, const unsigned long long* __restrict__ comp,
                              const int* __restrict__ order, const int* __restrict__ flag,
                              const int* __restrict__ pos, const int* __restrict__ tgt,
                              const int* __restrict__ src, const int* __restrict__ slot,
                              int* __restrict__ group_key, int* __restrict__ group_src,
                              int* __restrict__ tile_first) {
  const long long j = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (j >= m) return;
  const int g = pos[j] + flag[j] - 1;
  const int i = order[j];
  const unsigned long long c = comp[j];
  if (flag[j]) {
    group_key[g] = (int)(c & ((1ull << kb) - 1));
    const int t = (int)(c >> kb);
    if (j == 0 || (int)(comp[j - 1] >> kb) != t) tile_first[t] = g;
  }
  if (j == m - 1) tile_first[ntiles] = g + 1;
  group_src[(long long)g * kTile + (unsigned)slot[tgt[i]] % kTile] = src[i];
}

// Work items of a tile: its groups cut into equal runs of at most
// len; nch[ntiles] = 0, so that the scan's last entry is their number.
__global__ void k_chunk_count(int ntiles, int len, const int* __restrict__ goff, int* __restrict__ nch) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t <= ntiles) nch[t] = t < ntiles ? (goff[t + 1] - goff[t] + len - 1) / len : 0;
}
__global__ void k_chunk_fill(int ntiles, const int* __restrict__ goff, const int* __restrict__ nch,
                             const int* __restrict__ first, int* __restrict__ tile, int* __restrict__ g0,
                             int* __restrict__ g1) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntiles) return;
  const int G = goff[t + 1] - goff[t], n = nch[t];
  for (int k = 0; k < n; ++k) {
    const int c = first[t] + k;
    tile[c] = t;
    g0[c] = goff[t] + (int)((long long)G * k / n);
    g1[c] = goff[t] + (int)((long long)G * (k + 1) / n);
  }
}

template <typename T>
void scan_ex(Scratch& s, const T* in, T* out, long long n, hipStream_t st) {
  size_t bytes = 0;
  FMM_HIP(rocprim::exclusive_scan(nullptr, bytes, in, out, T(0), (size_t)n, rocprim::plus<T>(), st));
  void* tmp = s.get(bytes);
  FMM_HIP(rocprim::exclusive_scan(tmp, bytes, in, out, T(0), (size_t)n, rocprim::plus<T>(), st));
}

int read_int(const int* d, hipStream_t st) {
  int h = 0;
  FMM_HIP(hipMemcpyAsync(&h, d, sizeof(int), hipMemcpyDeviceToHost, st));
  FMM_HIP(hipStreamSynchronize(st));
  return h;
}

int bits_for(unsigned long long v) {  // bits that hold 0 .. v
  int b = 1;
  while (v >>= 1) ++b;
  return b;
}

// Pair indices in the order of their keys (stable), low `bits` bits.
void sort_order(Tree& t, const unsigned long long* key, unsigned long long* key_sorted, int* order, long long m,
                int bits, hipStream_t st) {
  const rocprim::counting_iterator<int> iota(0);
  size_t bytes = 0;
  FMM_HIP(rocprim::radix_sort_pairs(nullptr, bytes, key, key_sorted, iota, order, (size_t)m, 0, bits, st));
  void* tmp = t.scratch.get(bytes);
  FMM_HIP(rocprim::radix_sort_pairs(tmp, bytes, key, key_sorted, iota, order, (size_t)m, 0, bits, st));
}

}  // namespace

void build_m2l_schedule(Tree& t, hipStream_t st) {
  M2LSchedule& S = t.sched;
  S.tile_pairs_ready = false;  // statistics and maps of the previous tiles
  S.cell_tile_ready = false;
  const int nc = t.ncells;
  const long long m = t.n_m2l;
  FMM_CHECK(m < (1LL << 31), kOutOfMemory, "more than 2^31 M2L pairs");
  // tiles of every level
  DevBuf<int> rank, lvl;
  S.cell_slot.alloc(nc);
  FMM_HIP(hipMemsetAsync(S.cell_slot.get(), 0xff, sizeof(int) * nc, st));
  {
    const int D = t.depth;
    rank.alloc(nc + 1);
    lvl.alloc(3 * (D + 1));  // level offsets; ranks and first tiles of the levels
    int* const lcnt = lvl.get() + (D + 1);
    int* const lbase = lcnt + (D + 1);
    FMM_HIP(hipMemcpyAsync(lvl.get(), t.level_off.data(), sizeof(int) * (D + 1), hipMemcpyHostToDevice, st));
    auto has = rocprim::make_transform_iterator(rocprim::counting_iterator<int>(0), HasM2L{t.m2l_off.get()});
    size_t bytes = 0;
    FMM_HIP(rocprim::inclusive_scan(nullptr, bytes, has, rank.get() + 1, (size_t)nc, rocprim::plus<int>(), st));
    void* tmp = t.scratch.get(bytes);
    FMM_HIP(rocprim::inclusive_scan(tmp, bytes, has, rank.get() + 1, (size_t)nc, rocprim::plus<int>(), st));
    FMM_HIP(hipMemsetAsync(rank.get(), 0, sizeof(int), st));
    k_level_ranks<<<1, 64, 0, st>>>(D, lvl.get(), rank.get(), lcnt);
    std::vector<int> cnt(D + 1), base(D + 1, 0);
    FMM_HIP(hipMemcpyAsync(cnt.data(), lcnt, sizeof(int) * (D + 1), hipMemcpyDeviceToHost, st));
    FMM_HIP(hipStreamSynchronize(st));
    for (int l = 0; l < D; ++l) base[l + 1] = base[l] + (cnt[l + 1] - cnt[l] + kTile - 1) / kTile;
    S.ntiles = base[D];
    S.tile_cells.alloc((size_t)std::max(S.ntiles, 1) * kTile);
    S.tile_group_off.alloc(S.ntiles + 1);
    if (m == 0) {
      S.ngroups = S.nkeys = S.nchunks = S.nchunks64 = 0;
      FMM_HIP(hipMemsetAsync(S.tile_group_off.get(), 0, sizeof(int) * (S.ntiles + 1), st));
      FMM_HIP(hipStreamSynchronize(st));
      return;
    }
    FMM_HIP(hipMemsetAsync(S.tile_cells.get(), 0xff, sizeof(int) * S.ntiles * kTile, st));
    FMM_HIP(hipMemcpyAsync(lbase, base.data(), sizeof(int) * (D + 1), hipMemcpyHostToDevice, st));
    DevBuf<unsigned long long> k0, k1;
    k0.alloc(nc);
    k1.alloc(nc);
    k_tile_keys<<<blocks(nc, 256), 256, 0, st>>>(nc, t.m2l_off.get(), t.level.get(), t.octant.get(), t.parent.get(),
                                                 t.tile_hint_ptr(), k0.get());
    FMM_HIP(rocprim::radix_sort_keys(nullptr, bytes, k0.get(), k1.get(), (size_t)nc, 0, 47, st));
    tmp = t.scratch.get(bytes);
    FMM_HIP(rocprim::radix_sort_keys(tmp, bytes, k0.get(), k1.get(), (size_t)nc, 0, 47, st));
    k_assign_tiles<<<blocks(cnt[D], 256), 256, 0, st>>>(cnt[D], k1.get(), lcnt, lbase, S.cell_slot.get(),
                                                        S.tile_cells.get());
    FMM_HIP(hipStreamSynchronize(st));  // base, k0 and k1 end here
  }
  DevBuf<unsigned long long> key, key_sorted;
  DevBuf<int> tgt, order, fl, pos, keyid;
  key.alloc(m); key_sorted.alloc(m); tgt.alloc(m); order.alloc(m);
  fl.alloc(m + 1); pos.alloc(m + 1); keyid.alloc(m);
  // fields as wide as the largest offset needs: every 8 bits less are a pass
  // less of the sort over all pairs
  FMM_CHECK(t.m2l_maxq < (1 << 17), kUnsupported, "M2L offset beyond 2^17 half-widths (tree too deep)");
  const int qb = bits_for((unsigned long long)t.m2l_maxq) + 1, lb = bits_for((unsigned long long)t.depth);
  k_pair_key<<<blocks(m, 256), 256, 0, st>>>(m, t.m2l_off.get(), t.m2l_src.get(), nc, t.level.get(), t.cx.get(),
                                             t.cy.get(), t.cz.get(), t.cr.get(), lb, qb, t.m2l_maxq, key.get(),
                                             tgt.get());
  // distinct keys
  sort_order(t, key.get(), key_sorted.get(), order.get(), m, 2 * lb + 3 * qb, st);
  k_run_flags64<<<blocks(m + 1, 256), 256, 0, st>>>(m, key_sorted.get(), fl.get());
  scan_ex(t.scratch, fl.get(), pos.get(), m + 1, st);
  S.nkeys = read_int(pos.get() + m, st);
  S.key_dx.alloc(3 * (size_t)S.nkeys);
  S.key_r.alloc(S.nkeys);
  S.key_dlevel.alloc(S.nkeys);
  k_key_ids<<<blocks(m, 256), 256, 0, st>>>(m, fl.get(), pos.get(), order.get(), tgt.get(), t.m2l_src.get(),
                                            t.level.get(), t.cx.get(), t.cy.get(), t.cz.get(), t.cr.get(),
                                            keyid.get(), S.key_dx.get(), S.key_r.get(), S.key_dlevel.get());
  // groups = runs of (tile, key)
  const int kb = bits_for((unsigned long long)S.nkeys - 1);
  k_group_keys<<<blocks(m, 256), 256, 0, st>>>(m, kb, tgt.get(), keyid.get(), S.cell_slot.get(), key.get());
  sort_order(t, key.get(), key_sorted.get(), order.get(), m, kb + bits_for((unsigned long long)S.ntiles - 1), st);
  k_run_flags64<<<blocks(m + 1, 256), 256, 0, st>>>(m, key_sorted.get(), fl.get());
  scan_ex(t.scratch, fl.get(), pos.get(), m + 1, st);
  S.ngroups = read_int(pos.get() + m, st);
  S.group_key.alloc(S.ngroups);
  S.group_src.alloc((size_t)S.ngroups * kTile);
  FMM_HIP(hipMemsetAsync(S.group_src.get(), 0xff, sizeof(int) * (size_t)S.ngroups * kTile, st));
  k_fill_groups<<<blocks(m, 256), 256, 0, st>>>(m, kb, S.ntiles, key_sorted.get(), order.get(), fl.get(), pos.get(),
                                                tgt.get(), t.m2l_src.get(), S.cell_slot.get(), S.group_key.get(),
                                                S.group_src.get(), S.tile_group_off.get());
  // work items: runs of groups of one tile
  DevBuf<int> nch, first32;
  nch.alloc(S.ntiles + 1);
  auto cut = [&](int len, int& count, DevBuf<int>& first, DevBuf<int>& tile, DevBuf<int>& g0, DevBuf<int>& g1) {
    first.alloc(S.ntiles + 1);
    k_chunk_count<<<blocks(S.ntiles + 1, 256), 256, 0, st>>>(S.ntiles, len, S.tile_group_off.get(), nch.get());
    scan_ex(t.scratch, nch.get(), first.get(), S.ntiles + 1, st);
    count = read_int(first.get() + S.ntiles, st);
    tile.alloc(count);
    g0.alloc(count);
    g1.alloc(count);
    k_chunk_fill<<<blocks(S.ntiles, 256), 256, 0, st>>>(S.ntiles, S.tile_group_off.get(), nch.get(), first.get(),
                                                        tile.get(), g0.get(), g1.get());
  };
  cut(kGroupsPerChunk, S.nchunks, first32, S.chunk_tile, S.chunk_g0, S.chunk_g1);
  const int len = std::max(kGroupsPerChunkMin, S.ngroups / kChunkTarget);
  S.nchunks64 = 0;
  if (len < kGroupsPerChunk) cut(len, S.nchunks64, S.chunk64_first, S.chunk64_tile, S.chunk64_g0, S.chunk64_g1);
  FMM_HIP(hipStreamSynchronize(st));
}

}  // namespace fmm
