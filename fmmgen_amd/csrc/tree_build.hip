// Octree build and dual-traversal interaction lists on the GPU.
//
// Reproduces example/tree.cpp:130-233 (build_tree) and
// example/calculate.cpp:81-133 (interact_dehnen_lazy) bit for bit on the
// geometry, with a canonical cell numbering:
//   * root centre = the FP64 mean of example/tree.cpp:145-156, whose sum runs
//     in index order with one rounding per addition (evaluated in parallel,
//     bit for bit, see k_mean_steps), half-width = 1.001 x the
//     largest per-axis deviation (order-free max reduction);
//   * a cell splits iff it holds >= ncrit particles; only non-empty octants
//     become children; child centre = parent centre +- r/2 by the same FP64
//     operations as example/tree.cpp:95-98, octant bits x->1, y->2, z->4
//     from strict '>' compares (example/tree.cpp:193);
//   * the subdivision runs one level at a time: an octant histogram per
//     split cell, a scan that numbers the children (level-major, octant-path
//     order inside a level), and a per-particle 64-bit path key; one stable
//     radix sort of the keys puts every cell's particles in one contiguous
//     range with increasing caller index inside a leaf (the order the
//     reference leaf lists have);
//   * the dual traversal runs breadth first over a frontier of (target,
//     source) cell pairs with scan compaction.  Each pair takes the same
//     decision as the recursion (opening criterion R*theta > rmax_A +
//     rmax_B with correctly rounded FP64 and no contraction), so the M2L and
//     P2P lists are the reference's lists as multisets.
#pragma clang fp contract(off)

#include <cstring>

#include <rocprim/rocprim.hpp>

#include <algorithm>
#include <cmath>

#include "fmm_common.h"

namespace fmm {

namespace {

constexpr int kMaxSplitLevels = 21;  // 3 key bits per level in 63 bits

__device__ __forceinline__ double rmax_of(double r) { return sqrt_rn((3.0 * r) * r); }

// The mean of the positions with the reference's sequential FP64 sum
// s <- RN(s + x), bit for bit, without its chain of n dependent additions.
// While |s| stays inside one binade [2^e, 2^(e+1)) of ulp u, s = u S with S a
// whole number and RN(s + x) = u (S + d): d = x/u rounded to the nearest whole
// number, ties by the parity of S.  A run of additions is then a pair of whole
// numbers (the total of the d for an even and for an odd S before the run), and
// such pairs compose associatively.  Runs of kMeanChunk additions are summed in
// any order first, which gives each run's range of s up to the bound E of
// k_mean_scan; a run whose range lies in one binade is composed in parallel
// (k_mean_steps), and k_mean_walk applies the pairs in order, 64 at a time,
// adding one by one only in the runs that may leave their binade, and run by run
// in their batches of 64: a dozen runs an axis where s grows steadily, but a
// twentieth to a half of them where the set is centred and s wanders about zero.
// The chain of additions, one lane per axis, took 1936 us at 300007 particles
// and 27 ms at 2^22.  This takes 110 us at 300007 blob particles (k_mean_walk 89)
// and 460 us at 2^22 (327); k_mean_walk alone takes 1341 us on 300007 and 3.8 ms on
// 10^6 particles of a Plummer sphere about the origin.
constexpr int kMeanChunk = 256;  // one wave per axis, 4 additions a lane
constexpr int kMeanUnsafe = -100000;

struct MeanRun {
  double sum, lo, hi, abs;  // total, least and greatest partial sum (0 included), sum of |x|
};

__device__ __forceinline__ void mean_load(const double* __restrict__ pos, long long n, long long c, double* buf,
                                          int axis, int lane, double (&x)[4]) {
  const long long base = c * kMeanChunk;
  const int m = 3 * (int)(n - base < kMeanChunk ? n - base : kMeanChunk);
  for (int k = threadIdx.x; k < 3 * kMeanChunk; k += 192) buf[k] = k < m ? pos[3 * base + k] : 0.0;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) x[k] = buf[3 * (4 * lane + k) + axis];
}

__global__ __launch_bounds__(192) void k_mean_sums(const double* __restrict__ pos, long long n, long long nrun,
                                                   MeanRun* __restrict__ out) {
  __shared__ double buf[3 * kMeanChunk];
  const int lane = threadIdx.x & 63, axis = threadIdx.x >> 6;
  double x[4];
  mean_load(pos, n, blockIdx.x, buf, axis, lane, x);
  double sum = (x[0] + x[1]) + (x[2] + x[3]), inc = sum;
  double ab = (fabs(x[0]) + fabs(x[1])) + (fabs(x[2]) + fabs(x[3]));
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double v = __shfl_up(inc, o, 64);
    if (lane >= o) inc += v;
  }
  double p = inc - sum, lo = fmin(p, 0.0), hi = fmax(p, 0.0);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    p += x[k];
    lo = fmin(lo, p);
    hi = fmax(hi, p);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, o, 64));
    hi = fmax(hi, __shfl_xor(hi, o, 64));
    ab += __shfl_xor(ab, o, 64);
  }
  const double tot = __shfl(inc, 63, 64);
  // NaN and infinite sums pass through `sum` and make every later run unsafe
  if (lane == 0) out[axis * nrun + blockIdx.x] = MeanRun{tot, lo, hi, ab};
}

// Binade of every run's partial sums, or kMeanUnsafe (one block per axis).
// E bounds the distance of the sequential sum from the sums computed here:
// n additions each rounded by at most 2^-53 of the largest partial sum, and
// this kernel's and k_mean_sums' own additions (a few hundred levels deep for
// the serial parts) by 2^-53 of the sum of |x| each.
__global__ __launch_bounds__(1024) void k_mean_scan(long long n, long long nrun, const MeanRun* __restrict__ run,
                                                    int* __restrict__ expo) {
  __shared__ double sh[3][1024];
  const int tid = threadIdx.x;
  const MeanRun* r = run + blockIdx.x * nrun;
  const long long per = (nrun + 1023) / 1024, b = min(tid * per, nrun), e = min(b + per, nrun);
  double sum = 0.0, ab = 0.0;
  for (long long i = b; i < e; ++i) {
    sum += r[i].sum;
    ab += r[i].abs;
  }
  sh[0][tid] = sum;
  sh[1][tid] = ab;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {  // inclusive scans
    const double v = tid >= o ? sh[0][tid - o] : 0.0, w = tid >= o ? sh[1][tid - o] : 0.0;
    __syncthreads();
    sh[0][tid] += v;
    sh[1][tid] += w;
    __syncthreads();
  }
  const double start = tid > 0 ? sh[0][tid - 1] : 0.0, xabs = sh[1][1023];
  double a = start, big = 0.0;
  for (long long i = b; i < e; ++i) {
    big = fmax(big, fmax(fabs(a + r[i].lo), fabs(a + r[i].hi)));
    a += r[i].sum;
  }
  sh[2][tid] = big;
  __syncthreads();
  for (int s = 512; s > 0; s >>= 1) {
    if (tid < s) sh[2][tid] = fmax(sh[2][tid], sh[2][tid + s]);
    __syncthreads();
  }
  const double E = 0x1p-52 * ((double)n * sh[2][0] + (double)(per + 64) * xabs);
  a = start;
  for (long long i = b; i < e; ++i) {
    double lo = a + r[i].lo - E, hi = a + r[i].hi + E;
    a += r[i].sum;
    if (hi < 0.0) {
      const double t = -lo;
      lo = -hi;
      hi = t;
    }
    int ex = kMeanUnsafe;
    if (lo > 0x1p-900 && hi < 0x1p900) {  // false for NaN
      const int l = ilogb(lo);
      if (hi < ldexp(1.0, l + 1)) ex = l;
    }
    expo[blockIdx.x * nrun + i] = ex;
  }
}

struct MeanStep {
  long long d[2];  // change of S by the parity of S before
};
__device__ __forceinline__ MeanStep mean_then(const MeanStep& a, const MeanStep& b) {
  return MeanStep{{a.d[0] + ((a.d[0] & 1) ? b.d[1] : b.d[0]), a.d[1] + ((a.d[1] & 1) ? b.d[0] : b.d[1])}};
}
__device__ __forceinline__ MeanStep mean_reduce(MeanStep s) {  // lane 0: the lanes' steps in order
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) s = mean_then(s, MeanStep{{__shfl_down(s.d[0], o, 64), __shfl_down(s.d[1], o, 64)}});
  return s;
}

__global__ __launch_bounds__(192) void k_mean_steps(const double* __restrict__ pos, long long n, long long nrun,
                                                    const int* __restrict__ expo, MeanStep* __restrict__ step) {
  __shared__ double buf[3 * kMeanChunk];
  const int lane = threadIdx.x & 63, axis = threadIdx.x >> 6;
  double x[4];
  mean_load(pos, n, blockIdx.x, buf, axis, lane, x);
  const int e = expo[axis * nrun + blockIdx.x];
  if (e == kMeanUnsafe) return;  // uniform over the wave
  MeanStep s{{0, 0}};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    // y in units of the sum's last place; y - rint(y) is exact (y - floor(y) is
    // not just above a negative half), so it shows ties and nothing else
    const double y = ldexp(x[k], 52 - e), f = rint(y), r = y - f;
    const long long i = (long long)f;
    MeanStep t;
    t.d[0] = i;                                              // rint takes a tie to the even side
    t.d[1] = i + (r == 0.5 ? 1 : (r == -0.5 ? -1 : 0));      // an odd S takes the odd side
    s = mean_then(s, t);
  }
  s = mean_reduce(s);
  if (lane == 0) step[axis * nrun + blockIdx.x] = s;
}

__global__ __launch_bounds__(64) void k_mean_walk(const double* __restrict__ pos, long long n, long long nrun,
                                                  const int* __restrict__ expo, const MeanStep* __restrict__ step,
                                                  double* __restrict__ out) {
  __shared__ double buf[kMeanChunk];
  const int lane = threadIdx.x, axis = blockIdx.x;
  expo += axis * nrun;
  step += axis * nrun;
  double s = 0.0;
  // runs past the last one change nothing; unsafe runs have no step
  auto get = [&](long long base, int& e, MeanStep& m) {
    const long long i = base + lane;
    e = i < nrun ? expo[i] : kMeanUnsafe;
    m = i < nrun && e != kMeanUnsafe ? step[i] : MeanStep{{0, 0}};
  };
  auto apply = [&](int e, long long d0, long long d1) {
    const long long S = (long long)ldexp(s, 52 - e);
    s = ldexp((double)(S + ((S & 1) ? d1 : d0)), e - 52);
  };
  int e, en;
  MeanStep m, mn;
  get(0, e, m);
  for (long long base = 0; base < nrun; base += 64) {
    if (base + 64 < nrun) get(base + 64, en, mn);  // in flight during this batch
    const int e0 = __builtin_amdgcn_readfirstlane(e);
    const int cnt = (int)(nrun - base < 64 ? nrun - base : 64);
    if (__all(e0 != kMeanUnsafe && (e == e0 || lane >= cnt))) {
      const MeanStep t = mean_reduce(m);
      apply(e0, __shfl(t.d[0], 0, 64), __shfl(t.d[1], 0, 64));
    } else {
      for (int l = 0; l < cnt; ++l) {
        const int el = __shfl(e, l, 64);
        if (el != kMeanUnsafe) {
          apply(el, __shfl(m.d[0], l, 64), __shfl(m.d[1], l, 64));
          continue;
        }
        const long long first = (base + l) * kMeanChunk;
        const int k = (int)(n - first < kMeanChunk ? n - first : kMeanChunk);
        __syncthreads();
        for (int i = lane; i < k; i += 64) buf[i] = pos[3 * (first + i) + axis];
        __syncthreads();
        int i = 0;
        for (; i + 16 <= k; i += 16) {
          double v[16];
#pragma unroll
          for (int u = 0; u < 16; ++u) v[u] = buf[i + u];
#pragma unroll
          for (int u = 0; u < 16; ++u) s = s + v[u];
        }
        for (; i < k; ++i) s = s + buf[i];
      }
    }
    e = en;
    m = mn;
  }
  if (lane == 0) out[axis] = s / (double)n;
}

__global__ __launch_bounds__(256) void k_maxdev(const double* __restrict__ pos, long long n,
                                                const double* __restrict__ mean,
                                                unsigned long long* __restrict__ mx) {
  __shared__ double red[3][4];
  const double m0 = mean[0], m1 = mean[1], m2 = mean[2];
  double a[3] = {0, 0, 0};
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const double x = fabs(pos[3 * i] - m0), y = fabs(pos[3 * i + 1] - m1), z = fabs(pos[3 * i + 2] - m2);
    a[0] = x > a[0] ? x : a[0];
    a[1] = y > a[1] ? y : a[1];
    a[2] = z > a[2] ? z : a[2];
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const double v = __shfl_xor(a[d], o, 64);
      a[d] = v > a[d] ? v : a[d];
    }
    if ((threadIdx.x & 63) == 0) red[d][threadIdx.x >> 6] = a[d];
  }
  __syncthreads();
  if (threadIdx.x < 3) {  // non-negative doubles order like their bit patterns
    const double* r = red[threadIdx.x];
    double v = r[0];
    for (int w = 1; w < 4; ++w) v = r[w] > v ? r[w] : v;
    atomicMax(&mx[threadIdx.x], (unsigned long long)__double_as_longlong(v));
  }
}

__global__ void k_root(const double* __restrict__ mean, const unsigned long long* __restrict__ mx,
                       double* cx, double* cy, double* cz, double* cr, int* count, int* parent, int* octant,
                       int* ccount, long long n) {
  const double xm = __longlong_as_double((long long)mx[0]);
  const double ym = __longlong_as_double((long long)mx[1]);
  const double zm = __longlong_as_double((long long)mx[2]);
  const double r = (xm > ym ? (xm > zm ? xm : zm) : (ym > zm ? ym : zm)) * 1.001;
  cx[0] = mean[0];
  cy[0] = mean[1];
  cz[0] = mean[2];
  cr[0] = r;
  count[0] = (int)n;
  parent[0] = octant[0] = 0;
  for (int o = 0; o < 8; ++o) ccount[o] = 0;
}

// Moves every particle that is still inside a split cell to its child of the
// level (`cidx`: the previous level's numbering by (cell, octant), unused at
// the root), then finalises the particles whose cell there is a leaf and adds
// the others to the level's (cell, octant) histogram.  On levels of at most
// LDS / 8 cells a block counts in LDS first: added straight into memory, the
// eight counters of the root took all particles' additions (268 us a level on
// average at 300007 blob particles, 3.1 ms at 2^22; now 35 us at 300007).
template <int LDS>
__global__ __launch_bounds__(256) void k_level_octants(const double* __restrict__ pos, int n, int level, int ncell,
                                                       int* __restrict__ pcell, unsigned char* __restrict__ poct,
                                                       unsigned long long* __restrict__ key,
                                                       const int* __restrict__ cidx, int* __restrict__ leaf_of,
                                                       const double* __restrict__ lcx, const double* __restrict__ lcy,
                                                       const double* __restrict__ lcz, const int* __restrict__ lcount,
                                                       int* __restrict__ ccount, int ncrit, int level_base) {
  __shared__ int hist[LDS > 0 ? LDS : 1];
  if constexpr (LDS > 0) {
    for (int j = threadIdx.x; j < 8 * ncell; j += 256) hist[j] = 0;
    __syncthreads();
  }
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += gridDim.x * 256LL) {
    int c = 0;
    if (level > 0) {
      c = pcell[i];
      if (c < 0) continue;
      const int o = poct[i];
      c = cidx[8 * c + o];
      const unsigned long long bit = (unsigned long long)o << (3 * (kMaxSplitLevels - level));
      key[i] = level == 1 ? bit : key[i] | bit;
    }
    if (lcount[c] < ncrit) {
      leaf_of[i] = level_base + c;
      pcell[i] = -1;
      if (level == 0) key[i] = 0;
      continue;
    }
    const int oct = (pos[3 * i] > lcx[c]) + ((pos[3 * i + 1] > lcy[c]) << 1) + ((pos[3 * i + 2] > lcz[c]) << 2);
    poct[i] = (unsigned char)oct;
    pcell[i] = c;
    if constexpr (LDS > 0) atomicAdd(&hist[8 * c + oct], 1);
    else atomicAdd(&ccount[8 * (size_t)c + oct], 1);
  }
  if constexpr (LDS > 0) {
    __syncthreads();
    for (int j = threadIdx.x; j < 8 * ncell; j += 256)
      if (hist[j] > 0) atomicAdd(&ccount[j], hist[j]);
  }
}

struct Occupied {  // an octant with particles becomes a child
  __host__ __device__ int operator()(int count) const { return count > 0 ? 1 : 0; }
};

// Children of the level, numbered by the scan over (parent, octant) slots;
// clears their octant counters.
__global__ void k_make_children(int nparent, const int* __restrict__ ccount, const int* __restrict__ cidx,
                                const double* __restrict__ lcx, const double* __restrict__ lcy,
                                const double* __restrict__ lcz, const double* __restrict__ lr,
                                double* __restrict__ ncx, double* __restrict__ ncy, double* __restrict__ ncz,
                                double* __restrict__ nr, int* __restrict__ ncount, int* __restrict__ nparent_local,
                                int* __restrict__ noctant, int* __restrict__ ncc, int* __restrict__ first_child_local,
                                int* __restrict__ nchild, int* __restrict__ octmask) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nparent) return;
  int first = -1, cnt = 0, mask = 0;
  const double r = lr[c] / 2.0;
  for (int o = 0; o < 8; ++o) {
    const int j = 8 * c + o;
    const int k = ccount[j];
    if (k == 0) continue;
    const int id = cidx[j];
    if (first < 0) first = id;
    ++cnt;
    mask |= 1 << o;
    ncx[id] = lcx[c] + r * ((o & 1) * 2 - 1);
    ncy[id] = lcy[c] + r * ((o & 2) - 1);
    ncz[id] = lcz[c] + r * ((o & 4) / 2 - 1);
    nr[id] = r;
    ncount[id] = k;
    nparent_local[id] = c;
    noctant[id] = o;
    for (int q = 0; q < 8; ++q) ncc[8 * (size_t)id + q] = 0;
  }
  first_child_local[c] = first;
  nchild[c] = cnt;
  octmask[c] = mask;
}

__global__ void k_gather_particles(int n, const int* __restrict__ perm, const double* __restrict__ pos,
                                   const int* __restrict__ leaf_of_orig, double* __restrict__ px,
                                   double* __restrict__ py, double* __restrict__ pz, int* __restrict__ leaf_of) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const int i = perm[j];
  px[j] = pos[3 * (size_t)i];
  py[j] = pos[3 * (size_t)i + 1];
  pz[j] = pos[3 * (size_t)i + 2];
  leaf_of[j] = leaf_of_orig[i];
}

__global__ void k_leaf_starts(int n, const int* __restrict__ leaf_of, int* __restrict__ pstart) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  if (j == 0 || leaf_of[j] != leaf_of[j - 1]) pstart[leaf_of[j]] = j;
}

// An internal cell starts where the leaf at the end of its chain of first
// children does.
__global__ void k_internal_starts(int ncells, const int* __restrict__ nchild, const int* __restrict__ first_child,
                                  int* __restrict__ pstart) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= ncells || nchild[c] == 0) return;
  int l = c;
  while (nchild[l] > 0) l = first_child[l];
  pstart[c] = pstart[l];
}

// One level's cells into the canonical arrays (offset o; parents from po,
// first children from co, both counted inside their own levels).
struct CellArrays {
  double *cx, *cy, *cz, *cr, *crmax;
  int *pcount, *parent, *first_child, *nchild, *octmask, *octant, *level;
};
__global__ void k_place_level(int m, int o, int po, int co, int level, const double* __restrict__ x,
                              const double* __restrict__ y, const double* __restrict__ z,
                              const double* __restrict__ r, const int* __restrict__ count,
                              const int* __restrict__ parent, const int* __restrict__ first_child,
                              const int* __restrict__ nchild, const int* __restrict__ octmask,
                              const int* __restrict__ oct, CellArrays out) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= m) return;
  const int k = o + c;
  out.cx[k] = x[c];
  out.cy[k] = y[c];
  out.cz[k] = z[c];
  out.cr[k] = r[c];
  out.crmax[k] = rmax_of(r[c]);
  out.pcount[k] = count[c];
  out.parent[k] = parent[c] + po;
  out.first_child[k] = first_child[c] < 0 ? first_child[c] : first_child[c] + co;
  out.nchild[k] = nchild[c];
  out.octmask[k] = octmask[c];
  out.octant[k] = oct[c];
  out.level[k] = level;
}

struct IsLeaf {
  __host__ __device__ int operator()(int nchild) const { return nchild == 0 ? 1 : 0; }
};

__global__ void k_leaf_compact(int n, const int* __restrict__ nchild, const int* __restrict__ pos,
                               int* __restrict__ leaves) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c < n && nchild[c] == 0) leaves[pos[c]] = c;
}

// ---------------------------------------------------------------- lists

struct Counts3 {
  int m2l, p2p, nxt;
};
struct Plus3 {
  __host__ __device__ Counts3 operator()(const Counts3& a, const Counts3& b) const {
    return Counts3{a.m2l + b.m2l, a.p2p + b.p2p, a.nxt + b.nxt};
  }
};

// 0: M2L, 1: P2P, 2: split target A, 3: split source B
__device__ __forceinline__ int decide(int A, int B, const double* __restrict__ cx, const double* __restrict__ cy,
                                      const double* __restrict__ cz, const double* __restrict__ rmax,
                                      const int* __restrict__ nchild, const int* __restrict__ pcount,
                                      double theta, int ncrit) {
  const double dx = cx[A] - cx[B];
  const double dy = cy[A] - cy[B];
  const double dz = cz[A] - cz[B];
  const double R = sqrt_rn(dx * dx + dy * dy + dz * dz);
  if (R * theta > (rmax[A] + rmax[B])) return 0;
  const bool la = nchild[A] == 0, lb = nchild[B] == 0;
  if (la && lb) return pcount[B] >= ncrit ? 0 : 1;
  if (lb || (rmax[A] >= rmax[B] && !la)) return 2;
  return 3;
}

__global__ void k_pair_count(int nf, const int2* __restrict__ fr, Counts3* __restrict__ cnt,
                             unsigned char* __restrict__ dec, const double* __restrict__ cx,
                             const double* __restrict__ cy, const double* __restrict__ cz,
                             const double* __restrict__ rmax, const int* __restrict__ nchild,
                             const int* __restrict__ pcount, double theta, int ncrit) {
  const int f = blockIdx.x * blockDim.x + threadIdx.x;
  if (f > nf) return;
  Counts3 c{0, 0, 0};
  if (f < nf) {  // cnt[nf] = 0: the scan's last entry is the total
    const int2 ab = fr[f];
    const int d = decide(ab.x, ab.y, cx, cy, cz, rmax, nchild, pcount, theta, ncrit);
    dec[f] = (unsigned char)d;
    if (d == 0) c.m2l = 1;
    else if (d == 1) c.p2p = 1;
    else if (d == 2) c.nxt = nchild[ab.x];
    else c.nxt = nchild[ab.y];
  }
  cnt[f] = c;
}

// List entries are written as the keys (target << kb) | source that the CSR
// sort orders; the reference stores M2L as (source, target)
// (example/calculate.cpp:95).  maxq: the largest M2L centre offset per axis in
// units of the finer half-width, the field width of the schedule's keys.
__global__ __launch_bounds__(256) void k_pair_emit(int nf, const int2* __restrict__ fr,
                                                   const Counts3* __restrict__ off,
                                                   const unsigned char* __restrict__ dec,
                                                   const int* __restrict__ first_child,
                                                   const int* __restrict__ nchild, const double* __restrict__ cx,
                                                   const double* __restrict__ cy, const double* __restrict__ cz,
                                                   const double* __restrict__ cr, int kb,
                                                   unsigned long long* __restrict__ m2l, long long m2l_base,
                                                   unsigned long long* __restrict__ p2p, long long p2p_base,
                                                   int2* __restrict__ next, int* __restrict__ maxq) {
  const int f = blockIdx.x * blockDim.x + threadIdx.x;
  int q = 0;
  if (f < nf) {
    const int2 ab = fr[f];
    const int d = dec[f];
    const Counts3 o = off[f];
    const unsigned long long key = ((unsigned long long)(unsigned)ab.x << kb) | (unsigned)ab.y;
    if (d == 0) {
      m2l[m2l_base + o.m2l] = key;
      const double rf = fmin(cr[ab.x], cr[ab.y]);
      const double m = fmax(fmax(fabs(cx[ab.x] - cx[ab.y]), fabs(cy[ab.x] - cy[ab.y])), fabs(cz[ab.x] - cz[ab.y]));
      q = (int)fmin(rint(m / rf), 1e9);
    } else if (d == 1) {
      p2p[p2p_base + o.p2p] = key;
    } else if (d == 2) {
      const int fc = first_child[ab.x], k = nchild[ab.x];
      for (int i = 0; i < k; ++i) next[o.nxt + i] = make_int2(fc + i, ab.y);
    } else {
      const int fc = first_child[ab.y], k = nchild[ab.y];
      for (int i = 0; i < k; ++i) next[o.nxt + i] = make_int2(ab.x, fc + i);
    }
  }
  __shared__ int red[4];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) q = max(q, __shfl_xor(q, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = q;
  __syncthreads();
  if (threadIdx.x == 0) {
    q = max(max(red[0], red[1]), max(red[2], red[3]));
    if (q > *maxq) atomicMax(maxq, q);  // a stale read only costs an atomic
  }
}

// CSR from the sorted keys: sources, and the offset of every row (each entry
// sets the rows after its predecessor's up to its own).  With pcount: also the
// particle pairs nA nB of the list, self pairs of a cell with itself excluded.
__global__ __launch_bounds__(256) void k_csr_fill(long long m, int nc, int kb,
                                                  const unsigned long long* __restrict__ key, int* __restrict__ src,
                                                  int* __restrict__ off, const int* __restrict__ pcount,
                                                  unsigned long long* __restrict__ pairs) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  unsigned long long w = 0;
  if (i < m) {
    const unsigned long long k = key[i];
    const int t = (int)(k >> kb), b = (int)(k & ((1ull << kb) - 1));
    src[i] = b;
    const int prev = i > 0 ? (int)(key[i - 1] >> kb) : -1;
    for (int r = prev + 1; r <= t; ++r) off[r] = (int)i;
    if (i == m - 1)
      for (int r = t + 1; r <= nc; ++r) off[r] = (int)m;
    if (pairs) w = (unsigned long long)pcount[t] * (unsigned)pcount[b] - (t == b ? (unsigned)pcount[t] : 0u);
  }
  if (!pairs) return;
  __shared__ unsigned long long red[4];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) w += __shfl_xor(w, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = w;
  __syncthreads();
  if (threadIdx.x == 0) atomicAdd(pairs, red[0] + red[1] + red[2] + red[3]);
}

__global__ void k_fill_off(int n, int* __restrict__ off) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) off[i] = 0;
}

inline int blocks(long long n, int bs) { return (int)((n + bs - 1) / bs); }

template <typename T>
void exclusive_scan_int(Scratch& s, const T* in, T* out, long long n, hipStream_t st) {
  size_t bytes = 0;
  FMM_HIP(rocprim::exclusive_scan(nullptr, bytes, in, out, T(0), (size_t)n, rocprim::plus<T>(), st));
  void* tmp = s.get(bytes);
  FMM_HIP(rocprim::exclusive_scan(tmp, bytes, in, out, T(0), (size_t)n, rocprim::plus<T>(), st));
}

int bits_for(unsigned long long v) {  // bits that hold 0 .. v
  int b = 1;
  while (v >>= 1) ++b;
  return b;
}

void sort_keys(Tree& t, const unsigned long long* in, unsigned long long* out, long long m, int bits,
               hipStream_t st) {
  size_t bytes = 0;
  FMM_HIP(rocprim::radix_sort_keys(nullptr, bytes, in, out, (size_t)m, 0, bits, st));
  void* tmp = t.scratch.get(bytes);
  FMM_HIP(rocprim::radix_sort_keys(tmp, bytes, in, out, (size_t)m, 0, bits, st));
}

// CSR lists from the entry keys (target << kb) | source; `sorted` keeps the
// sorted keys, `total` (optional) adds up the particle pairs.
void build_csr(Tree& t, const unsigned long long* keys, long long m, int kb, DevBuf<unsigned long long>& sorted,
               DevBuf<int>& off, DevBuf<int>& src, unsigned long long* total, hipStream_t st) {
  const int nc = t.ncells;
  off.alloc(nc + 1);
  src.alloc(std::max<long long>(m, 1));
  if (m == 0) {
    k_fill_off<<<blocks(nc + 1, 256), 256, 0, st>>>(nc + 1, off.get());
    return;
  }
  sorted.alloc(m);
  sort_keys(t, keys, sorted.get(), m, 2 * kb, st);
  k_csr_fill<<<blocks(m, 256), 256, 0, st>>>(m, nc, kb, sorted.get(), src.get(), off.get(), t.pcount.get(), total);
}

// Source ranges.  Keys (target << nb) | first source particle of every P2P
// entry, from the sorted entry keys.
__global__ void k_rng_keys(long long m, int kb, int nb, const unsigned long long* __restrict__ entry,
                           const int* __restrict__ pstart, unsigned long long* __restrict__ key) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= m) return;
  const unsigned long long k = entry[i];
  key[i] = ((k >> kb) << nb) | (unsigned)pstart[k & ((1ull << kb) - 1)];
}

// A range starts at an entry that is not the target itself and is the target's
// first, follows the target itself, or does not follow on its predecessor's
// end.  Every source is a leaf, so the cell of an entry is that of its first
// particle.
struct RangeEntry {
  int A, B, start;
};
__device__ __forceinline__ RangeEntry range_entry(unsigned long long k, int nb, const int* __restrict__ leaf_of) {
  const int s = (int)(k & ((1ull << nb) - 1));
  return RangeEntry{(int)(k >> nb), leaf_of[s], s};
}
__global__ void k_rng_flags(long long m, int nb, const unsigned long long* __restrict__ key,
                            const int* __restrict__ leaf_of, const int* __restrict__ pcount, int* __restrict__ flag) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i > m) return;
  int f = 0;  // flag[m] = 0: the scan's last entry is the number of ranges
  if (i < m) {
    const RangeEntry e = range_entry(key[i], nb, leaf_of);
    f = e.B != e.A;
    if (f && i > 0) {
      const RangeEntry p = range_entry(key[i - 1], nb, leaf_of);
      if (p.A == e.A && p.B != p.A && p.start + pcount[p.B] == e.start) f = 0;
    }
  }
  flag[i] = f;
}

__global__ void k_rng_fill(long long m, int nb, int nc, const unsigned long long* __restrict__ key,
                           const int* __restrict__ leaf_of, const int* __restrict__ pcount,
                           const int* __restrict__ flag, const int* __restrict__ pos, int* __restrict__ rstart,
                           int* __restrict__ rlen, int* __restrict__ off) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= m) return;
  const RangeEntry e = range_entry(key[i], nb, leaf_of);
  const int prev = i > 0 ? (int)(key[i - 1] >> nb) : -1;
  for (int r = prev + 1; r <= e.A; ++r) off[r] = pos[i];
  if (i == m - 1)
    for (int r = e.A + 1; r <= nc; ++r) off[r] = pos[m];
  if (e.B == e.A) return;
  const int r = pos[i] + flag[i] - 1;
  if (flag[i]) rstart[r] = e.start;
  atomicAdd(&rlen[r], pcount[e.B]);
}

// Sources of a segment: `seg` (P2PItems::kSegment), or with `even` a
// leaf's sequence of `tot` in as few segments of at most `seg` as hold it, all
// of one length, in whole staged chunks of 128.
__device__ __forceinline__ long long seg_length(long long tot, int seg, int even) {
  if (!even) return seg;
  const long long k = (tot + seg - 1) / seg;
  return ((tot + k - 1) / k + 127) / 128 * 128;
}

// Per leaf: number of P2P segments and of the rows they store (a target a
// segment); both 0 at ncells, so that the scans' last entries are the totals.
__global__ void k_seg_count(int ncells, const int* __restrict__ nchild, const int* __restrict__ pcount,
                            const int* __restrict__ rng_off, const long long* __restrict__ cum,
                            long long* __restrict__ nseg, long long* __restrict__ nrow, int seg, int even) {
  const int A = blockIdx.x * blockDim.x + threadIdx.x;
  if (A > ncells) return;
  long long k = 0;
  if (A < ncells && nchild[A] == 0 && pcount[A] > 0) {
    const long long tot = pcount[A] + cum[rng_off[A + 1]] - cum[rng_off[A]];
    const long long len = seg_length(tot, seg, even);
    k = (tot + len - 1) / len;
  }
  nseg[A] = k;
  nrow[A] = k > 0 ? k * pcount[A] : 0;
}

__global__ void k_widen(long long m, const int* __restrict__ in, long long* __restrict__ out) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i < m) out[i] = in[i];
}

// Items of one leaf: segment s starts at position s * len of the source
// sequence (own particles first, then the ranges in order).
__global__ void k_seg_fill(int ncells, const int* __restrict__ nchild, const int* __restrict__ pcount,
                           const int* __restrict__ rng_off, const long long* __restrict__ cum,
                           const long long* __restrict__ nseg, const long long* __restrict__ seg_off,
                           const long long* __restrict__ row_off, int seg, int even, int* __restrict__ it_leaf,
                           int* __restrict__ it_r, int* __restrict__ it_o, int* __restrict__ it_n,
                           int* __restrict__ it_row) {
  const int A = blockIdx.x * blockDim.x + threadIdx.x;
  if (A >= ncells || nseg[A] == 0) return;
  const int nt = pcount[A], rb = rng_off[A], re = rng_off[A + 1];
  const long long base = cum[rb], tot = nt + cum[re] - base, len = seg_length(tot, seg, even);
  for (long long s = 0; s < nseg[A]; ++s) {
    const long long P = s * len, w = seg_off[A] + s;
    int r, o;
    if (P < nt) {
      r = rb - 1;
      o = (int)P;
    } else {
      // last range r in [rb, re) with cum[r] - base <= P - nt
      const long long q = P - nt + base;
      int lo = rb, hi = re - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (cum[mid] <= q) lo = mid;
        else hi = mid - 1;
      }
      r = lo;
      o = (int)(q - cum[r]);
    }
    it_leaf[w] = A;
    it_r[w] = r;
    it_o[w] = o;
    it_n[w] = (int)((tot - P < len) ? tot - P : len);
    if (it_row) it_row[w] = (int)(row_off[A] + s * nt);
  }
}

}  // namespace

// P2P work items (segments of each leaf's source sequence).  FP32: segments of
// P2PItems::kSegment.  FP64: the same where they fill the GPU many times over;
// smaller sets are cut until there are about kP2PItems items, of at least a
// staged chunk each.  One item a leaf -> this rule, FP64 near field: 2000
// particles (64 leaves) 144 -> 21 us, 10^5 (4096 leaves) 686 -> 364 us, 300007
// blobs 2.53 -> 1.41 ms.  (The FP32 items are not cut: the compensated sums of a
// finer cut differ by 4e-9 of the field.)
constexpr int kP2PItems = 65536;
void build_p2p_items(Tree& t, hipStream_t st) {
  const int nc = t.ncells;
  const long long nr = t.n_rng;
  DevBuf<long long> len, cum, nseg, soff, nrow;
  len.alloc(nr + 1);
  cum.alloc(nr + 1);
  FMM_HIP(hipMemsetAsync(len.get() + nr, 0, sizeof(long long), st));
  if (nr > 0) k_widen<<<blocks(nr, 256), 256, 0, st>>>(nr, t.rng_len.get(), len.get());
  exclusive_scan_int(t.scratch, len.get(), cum.get(), nr + 1, st);
  nseg.alloc(nc + 1);
  soff.alloc(nc + 1);
  nrow.alloc(nc + 1);
  auto cut = [&](P2PItems& I, int seg, int even) {
    k_seg_count<<<blocks(nc + 1, 256), 256, 0, st>>>(nc, t.nchild.get(), t.pcount.get(), t.rng_off.get(), cum.get(),
                                                     nseg.get(), nrow.get(), seg, even);
    exclusive_scan_int(t.scratch, nseg.get(), soff.get(), nc + 1, st);
    long long total = 0, rows = 0;
    FMM_HIP(hipMemcpyAsync(&total, soff.get() + nc, sizeof(long long), hipMemcpyDeviceToHost, st));
    if (even) {
      I.row_off.alloc(nc + 1);
      exclusive_scan_int(t.scratch, nrow.get(), I.row_off.get(), nc + 1, st);
      FMM_HIP(hipMemcpyAsync(&rows, I.row_off.get() + nc, sizeof(long long), hipMemcpyDeviceToHost, st));
    }
    FMM_HIP(hipStreamSynchronize(st));
    FMM_CHECK(total < (1LL << 31), kOutOfMemory, "P2P work items exceed 2^31");
    I.count = total;
    I.split = total > t.nleaves;
    I.rows = I.split && rows <= P2PItems::kMaxRows ? rows : 0;
    const long long na = std::max<long long>(total, 1);
    I.leaf.alloc(na);
    I.r.alloc(na);
    I.o.alloc(na);
    I.n.alloc(na);
    if (I.rows > 0) I.row.alloc(na);
    k_seg_fill<<<blocks(nc, 256), 256, 0, st>>>(nc, t.nchild.get(), t.pcount.get(), t.rng_off.get(), cum.get(),
                                                nseg.get(), soff.get(), I.row_off.get(), seg, even, I.leaf.get(),
                                                I.r.get(), I.o.get(), I.n.get(), I.rows > 0 ? I.row.get() : nullptr);
  };
  cut(t.p2p, P2PItems::kSegment, 0);
  // source sequences in all: the pairs over the mean leaf size
  const double sources = (double)t.p2p_particle_pairs * t.nleaves / (double)t.n;
  const long long seg = 128 * (1 + (long long)(sources / (128.0 * kP2PItems)));
  if (seg < P2PItems::kSegment) cut(t.p2p64, (int)seg, 1);
  FMM_HIP(hipStreamSynchronize(st));  // the temporaries are freed on return
}

// Merged source particle ranges of every P2P target (self excluded), from the
// list's sorted entry keys.
void build_p2p_ranges(Tree& t, const unsigned long long* entry, int kb, hipStream_t st) {
  const int nc = t.ncells;
  const long long m = t.n_p2p;
  t.rng_off.alloc(nc + 1);
  t.n_rng = 0;
  if (m == 0) {
    t.rng_start.alloc(1);
    t.rng_len.alloc(1);
    k_fill_off<<<blocks(nc + 1, 256), 256, 0, st>>>(nc + 1, t.rng_off.get());
    return;
  }
  const int nb = bits_for((unsigned long long)t.n - 1);
  DevBuf<unsigned long long> k0, k1;
  DevBuf<int> fl, ps;
  k0.alloc(m); k1.alloc(m); fl.alloc(m + 1); ps.alloc(m + 1);
  k_rng_keys<<<blocks(m, 256), 256, 0, st>>>(m, kb, nb, entry, t.pstart.get(), k0.get());
  sort_keys(t, k0.get(), k1.get(), m, kb + nb, st);
  k_rng_flags<<<blocks(m + 1, 256), 256, 0, st>>>(m, nb, k1.get(), t.leaf_of.get(), t.pcount.get(), fl.get());
  exclusive_scan_int(t.scratch, fl.get(), ps.get(), m + 1, st);
  int total = 0;
  FMM_HIP(hipMemcpyAsync(&total, ps.get() + m, sizeof(int), hipMemcpyDeviceToHost, st));
  FMM_HIP(hipStreamSynchronize(st));
  t.n_rng = total;
  t.rng_start.alloc(std::max(total, 1));
  t.rng_len.alloc(std::max(total, 1));
  FMM_HIP(hipMemsetAsync(t.rng_len.get(), 0, sizeof(int) * std::max(total, 1), st));
  k_rng_fill<<<blocks(m, 256), 256, 0, st>>>(m, nb, nc, k1.get(), t.leaf_of.get(), t.pcount.get(), fl.get(), ps.get(),
                                             t.rng_start.get(), t.rng_len.get(), t.rng_off.get());
  FMM_HIP(hipStreamSynchronize(st));  // the temporaries are freed on return
}

// Builds the tree of `t` from caller positions (device, [n*3]).
void build_tree_device(Tree& t, const double* d_pos, hipStream_t st) {
  const int n = (int)t.n;
  const int ncrit = (int)t.ncrit;
  DevBuf<double> mean;
  DevBuf<unsigned long long> mx;
  mean.alloc(3);
  mx.alloc(3);
  FMM_HIP(hipMemsetAsync(mx.get(), 0, 3 * sizeof(unsigned long long), st));
  const long long nrun = ((long long)n + kMeanChunk - 1) / kMeanChunk;
  DevBuf<MeanRun> mrun;
  DevBuf<int> mexp;
  DevBuf<MeanStep> mstep;
  mrun.alloc(3 * nrun);
  mexp.alloc(3 * nrun);
  mstep.alloc(3 * nrun);
  k_mean_sums<<<(int)nrun, 192, 0, st>>>(d_pos, n, nrun, mrun.get());
  k_mean_scan<<<3, 1024, 0, st>>>(n, nrun, mrun.get(), mexp.get());
  k_mean_steps<<<(int)nrun, 192, 0, st>>>(d_pos, n, nrun, mexp.get(), mstep.get());
  k_mean_walk<<<3, 64, 0, st>>>(d_pos, n, nrun, mexp.get(), mstep.get(), mean.get());
  k_maxdev<<<std::min(blocks(n, 256), 1024), 256, 0, st>>>(d_pos, n, mean.get(), mx.get());

  // per-level arrays
  struct Level {
    int n = 0;
    DevBuf<double> cx, cy, cz, r;
    DevBuf<int> count, parent, first_child, nchild, octmask, oct;
  };
  std::vector<Level*> lv;
  auto new_level = [&](int m) {
    Level* L = new Level();
    lv.push_back(L);
    L->n = m;
    L->cx.alloc(m); L->cy.alloc(m); L->cz.alloc(m); L->r.alloc(m);
    L->count.alloc(m); L->parent.alloc(m); L->first_child.alloc(m); L->nchild.alloc(m); L->octmask.alloc(m);
    L->oct.alloc(m);
    return L;
  };
  struct Cleanup {
    std::vector<Level*>& v;
    ~Cleanup() { for (auto* p : v) delete p; }
  } cleanup{lv};

  DevBuf<int> pcell, leaf_orig, ccount[2], cidx[2];  // counters and numbering of this level and the last
  DevBuf<unsigned char> poct;
  DevBuf<unsigned long long> key;
  pcell.alloc(n);
  leaf_orig.alloc(n);
  poct.alloc(n);
  key.alloc(n);
  Level* root = new_level(1);
  ccount[0].alloc(8);
  k_root<<<1, 1, 0, st>>>(mean.get(), mx.get(), root->cx.get(), root->cy.get(), root->cz.get(), root->r.get(),
                          root->count.get(), root->parent.get(), root->oct.get(), ccount[0].get(), n);

  std::vector<int> level_off{0};
  int level = 0;
  constexpr int kHist = 4096;  // octant counters of a block (16 KB): levels of up to 512 cells
  while (true) {
    Level* cur = lv.back();
    const int m = cur->n, h = level & 1;
    level_off.push_back(level_off.back() + m);
    auto octants = [&](auto kern, int grid) {
      kern<<<grid, 256, 0, st>>>(d_pos, n, level, m, pcell.get(), poct.get(), key.get(), cidx[h ^ 1].get(),
                                 leaf_orig.get(), cur->cx.get(), cur->cy.get(), cur->cz.get(), cur->count.get(),
                                 ccount[h].get(), ncrit, level_off[level]);
    };
    if (8LL * m <= kHist) octants(k_level_octants<kHist>, std::min(blocks(n, 256), 1024));
    else octants(k_level_octants<0>, std::min(blocks(n, 256), 1 << 16));
    cidx[h].alloc(8 * (size_t)m + 1);
    // numbering of the occupied octants: cidx[j] = how many come before j
    auto occ = rocprim::make_transform_iterator(ccount[h].get(), Occupied());
    size_t bytes = 0;
    FMM_HIP(rocprim::inclusive_scan(nullptr, bytes, occ, cidx[h].get() + 1, 8 * (size_t)m, rocprim::plus<int>(), st));
    void* tmp = t.scratch.get(bytes);
    FMM_HIP(rocprim::inclusive_scan(tmp, bytes, occ, cidx[h].get() + 1, 8 * (size_t)m, rocprim::plus<int>(), st));
    FMM_HIP(hipMemsetAsync(cidx[h].get(), 0, sizeof(int), st));
    int nnext = 0;
    FMM_HIP(hipMemcpyAsync(&nnext, cidx[h].get() + 8 * (size_t)m, sizeof(int), hipMemcpyDeviceToHost, st));
    FMM_HIP(hipStreamSynchronize(st));
    FMM_CHECK(nnext == 0 || level < kMaxSplitLevels, kTreeTooDeep,
              "tree deeper than 21 split levels (coincident particles?)");
    Level* nx = nnext > 0 ? new_level(nnext) : nullptr;
    if (nx) ccount[h ^ 1].alloc(8 * (size_t)nnext);
    // on the last level: no children, their arrays are not touched
    k_make_children<<<blocks(m, 256), 256, 0, st>>>(
        m, ccount[h].get(), cidx[h].get(), cur->cx.get(), cur->cy.get(), cur->cz.get(), cur->r.get(),
        nx ? nx->cx.get() : nullptr, nx ? nx->cy.get() : nullptr, nx ? nx->cz.get() : nullptr,
        nx ? nx->r.get() : nullptr, nx ? nx->count.get() : nullptr, nx ? nx->parent.get() : nullptr,
        nx ? nx->oct.get() : nullptr, ccount[h ^ 1].get(), cur->first_child.get(), cur->nchild.get(),
        cur->octmask.get());
    if (!nx) break;
    ++level;
  }
  t.depth = (int)lv.size();
  t.level_off = level_off;
  t.ncells = level_off.back();
  const int nc = t.ncells;

  // levels into the canonical global arrays
  t.cx.alloc(nc); t.cy.alloc(nc); t.cz.alloc(nc); t.cr.alloc(nc); t.crmax.alloc(nc);
  t.parent.alloc(nc); t.first_child.alloc(nc); t.nchild.alloc(nc); t.octmask.alloc(nc);
  t.level.alloc(nc); t.pstart.alloc(nc); t.pcount.alloc(nc); t.octant.alloc(nc);
  const CellArrays out{t.cx.get(), t.cy.get(), t.cz.get(), t.cr.get(), t.crmax.get(), t.pcount.get(), t.parent.get(),
                       t.first_child.get(), t.nchild.get(), t.octmask.get(), t.octant.get(), t.level.get()};
  for (int l = 0; l < t.depth; ++l) {
    Level* L = lv[l];
    k_place_level<<<blocks(L->n, 256), 256, 0, st>>>(
        L->n, level_off[l], l > 0 ? level_off[l - 1] : 0, level_off[l + 1], l, L->cx.get(), L->cy.get(), L->cz.get(),
        L->r.get(), L->count.get(), L->parent.get(), L->first_child.get(), L->nchild.get(), L->octmask.get(),
        L->oct.get(), out);
  }

  // stable sort of particles by path key
  {
    DevBuf<unsigned long long> k1;
    k1.alloc(n);
    t.perm.alloc(n);
    const unsigned begin_bit = 3u * (unsigned)(kMaxSplitLevels - std::max(level, 1));
    const rocprim::counting_iterator<int> iota(0);
    size_t bytes = 0;
    FMM_HIP(rocprim::radix_sort_pairs(nullptr, bytes, key.get(), k1.get(), iota, t.perm.get(), (size_t)n, begin_bit,
                                      63u, st));
    void* tmp = t.scratch.get(bytes);
    FMM_HIP(rocprim::radix_sort_pairs(tmp, bytes, key.get(), k1.get(), iota, t.perm.get(), (size_t)n, begin_bit, 63u,
                                      st));
    FMM_HIP(hipStreamSynchronize(st));
  }
  t.px.alloc(n); t.py.alloc(n); t.pz.alloc(n); t.leaf_of.alloc(n);
  k_gather_particles<<<blocks(n, 256), 256, 0, st>>>(n, t.perm.get(), d_pos, leaf_orig.get(), t.px.get(),
                                                     t.py.get(), t.pz.get(), t.leaf_of.get());
  k_leaf_starts<<<blocks(n, 256), 256, 0, st>>>(n, t.leaf_of.get(), t.pstart.get());
  k_internal_starts<<<blocks(nc, 256), 256, 0, st>>>(nc, t.nchild.get(), t.first_child.get(), t.pstart.get());
  // leaves in canonical order
  {
    DevBuf<int> lp;
    lp.alloc(nc + 1);
    auto leaf = rocprim::make_transform_iterator(t.nchild.get(), IsLeaf());
    size_t bytes = 0;
    FMM_HIP(rocprim::inclusive_scan(nullptr, bytes, leaf, lp.get() + 1, (size_t)nc, rocprim::plus<int>(), st));
    void* tmp = t.scratch.get(bytes);
    FMM_HIP(rocprim::inclusive_scan(tmp, bytes, leaf, lp.get() + 1, (size_t)nc, rocprim::plus<int>(), st));
    FMM_HIP(hipMemsetAsync(lp.get(), 0, sizeof(int), st));
    FMM_HIP(hipMemcpyAsync(&t.nleaves, lp.get() + nc, sizeof(int), hipMemcpyDeviceToHost, st));
    FMM_HIP(hipStreamSynchronize(st));
    t.leaves.alloc(t.nleaves);
    k_leaf_compact<<<blocks(nc, 256), 256, 0, st>>>(nc, t.nchild.get(), lp.get(), t.leaves.get());
    FMM_HIP(hipStreamSynchronize(st));
  }
}

// Breadth-first dual traversal from (root, root) and CSR lists by target.
void build_lists_device(Tree& t, hipStream_t st) {
  DevBuf<int2> cur, nxt;
  DevBuf<unsigned long long> m2l, p2p, sorted;
  DevBuf<Counts3> cnt, off;
  DevBuf<unsigned char> dec;
  DevBuf<unsigned long long> total;
  DevBuf<int> maxq;
  const int kb = bits_for((unsigned long long)t.ncells - 1);
  long long n_m2l = 0, n_p2p = 0;
  long long cap_m2l = list_entries(t.n), cap_p2p = cap_m2l / 2;
  m2l.alloc(cap_m2l);
  p2p.alloc(cap_p2p);
  cur.alloc(1);
  total.alloc(1);
  maxq.alloc(1);
  FMM_HIP(hipMemsetAsync(cur.get(), 0, sizeof(int2), st));  // the pair (root, root)
  FMM_HIP(hipMemsetAsync(total.get(), 0, sizeof(unsigned long long), st));
  FMM_HIP(hipMemsetAsync(maxq.get(), 0, sizeof(int), st));
  int nf = 1;
  auto grow = [&](DevBuf<unsigned long long>& b, long long& cap, long long used, long long need) {
    if (need <= cap) return;
    const long long c = std::max(need, 2 * cap);
    DevBuf<unsigned long long> nb;
    nb.alloc(c);
    if (used > 0)
      FMM_HIP(hipMemcpyAsync(nb.get(), b.get(), sizeof(unsigned long long) * used, hipMemcpyDeviceToDevice, st));
    FMM_HIP(hipStreamSynchronize(st));
    std::swap(b.p, nb.p);
    std::swap(b.n, nb.n);
    cap = c;
  };
  while (nf > 0) {
    cnt.alloc(nf + 1);
    off.alloc(nf + 1);
    dec.alloc(nf);
    k_pair_count<<<blocks(nf + 1, 256), 256, 0, st>>>(nf, cur.get(), cnt.get(), dec.get(), t.cx.get(), t.cy.get(),
                                                      t.cz.get(), t.crmax.get(), t.nchild.get(), t.pcount.get(),
                                                      t.theta, (int)t.ncrit);
    size_t bytes = 0;
    FMM_HIP(rocprim::exclusive_scan(nullptr, bytes, cnt.get(), off.get(), Counts3{0, 0, 0}, (size_t)nf + 1, Plus3(),
                                    st));
    void* tmp = t.scratch.get(bytes);
    FMM_HIP(rocprim::exclusive_scan(tmp, bytes, cnt.get(), off.get(), Counts3{0, 0, 0}, (size_t)nf + 1, Plus3(), st));
    Counts3 add;
    FMM_HIP(hipMemcpyAsync(&add, off.get() + nf, sizeof(Counts3), hipMemcpyDeviceToHost, st));
    FMM_HIP(hipStreamSynchronize(st));
    FMM_CHECK(add.m2l >= 0 && add.p2p >= 0 && add.nxt >= 0, kOutOfMemory, "traversal frontier exceeds 2^31 pairs");
    grow(m2l, cap_m2l, n_m2l, n_m2l + add.m2l);
    grow(p2p, cap_p2p, n_p2p, n_p2p + add.p2p);
    nxt.alloc(std::max(add.nxt, 1));
    k_pair_emit<<<blocks(nf, 256), 256, 0, st>>>(nf, cur.get(), off.get(), dec.get(), t.first_child.get(),
                                                 t.nchild.get(), t.cx.get(), t.cy.get(), t.cz.get(), t.cr.get(), kb,
                                                 m2l.get(), n_m2l, p2p.get(), n_p2p, nxt.get(), maxq.get());
    n_m2l += add.m2l;
    n_p2p += add.p2p;
    nf = add.nxt;
    std::swap(cur.p, nxt.p);
    std::swap(cur.n, nxt.n);
  }
  FMM_CHECK(n_m2l < (1LL << 31) && n_p2p < (1LL << 31), kOutOfMemory, "more than 2^31 list entries");
  t.n_m2l = n_m2l;
  t.n_p2p = n_p2p;
  FMM_HIP(hipMemcpyAsync(&t.m2l_maxq, maxq.get(), sizeof(int), hipMemcpyDeviceToHost, st));
  build_csr(t, m2l.get(), n_m2l, kb, sorted, t.m2l_off, t.m2l_src, nullptr, st);
  build_csr(t, p2p.get(), n_p2p, kb, sorted, t.p2p_off, t.p2p_src, total.get(), st);
  unsigned long long h = 0;
  FMM_HIP(hipMemcpyAsync(&h, total.get(), sizeof(h), hipMemcpyDeviceToHost, st));
  build_p2p_ranges(t, sorted.get(), kb, st);
  FMM_HIP(hipStreamSynchronize(st));
  t.p2p_particle_pairs = (long long)h;
  build_p2p_items(t, st);
}

}  // namespace fmm
