// Fused energy + forces for fixed-charge LJ + Ewald (real space and PME) on gfx950.
//
// One call evaluates, for an orthorhombic periodic box,
//   E = sum_{i<j, r<=rc, not excluded} [ k q_i q_j erfc(a r)/r + 4 eps_ij s^6 (s^6 - 1) ]
//     + sum_{i<j excluded, r<=rc} k q_i q_j (erfc(a r) - 1)/r
//     + k (E_recip + E_self)                      (smooth PME, any order 3..8)
// with Lorentz-Berthelot mixing, and F = -dE/dr.  It is the composition of the
// reference's MultipolarInteraction(rank 0, with pairs_excl), Vdw(LennardJones)
// and PME(rank 0) (examples/tip3p/model.py:100-123), evaluated without an explicit
// pair list.  Every excluded pair (i != j) of the CSR exclusion list receives the
// erfc - 1 correction, which for rigid water is exactly the reference's
// coulomb_excl_pairs set (examples/tip3p/md.py:152-158).
//
// Data layout: atoms are binned into x-y columns of about one cluster width and
// fine z bins, counting-sorted, and cut per column into clusters of 32
// consecutive atoms (padded), each ordered into four compact groups of 8 slots.  Cluster arrays (TC4 x,
// y, z, q and TC2 sigma/2, 2 sqrt(eps)) are cluster-major, 32 slots per cluster.  Per i-cluster a list of
// the 8-atom j-groups within the cutoff of one of its groups is found per column neighbourhood; the
// pair kernel gives each 64-lane wavefront a share of one cluster's list, four entries at a time, one
// lane per pair of an 8 x 8 block.
// Forces and energies accumulate as int64 fixed point (bitwise independent of
// the order of summation); the reciprocal-space energy is a float64 k-space sum.
// TC = float is the mixed-precision mode, TC = double the all-float64 mode.

#include <string.h>

#include <atomic>
#include <mutex>
#include <type_traits>
#include <vector>

#include "pair_math.h"
#include "pme_core.h"
#include "tff_common.h"
#include "torchff_hip.h"

namespace {

using namespace tffpme;

constexpr int CL = 32;          // atoms per cluster
constexpr int MAXEX = 8;        // exclusion partners per atom kept for the tile masks
constexpr int FB = 256;         // block size of the per-atom kernels
// Fixed-point sums over a whole call go to up to E_SLOTS slots of one 64-byte line each (words: Lennard-Jones,
// Coulomb, listed cluster pairs), added up by the last kernel: same-line atomics serialise at about
// 6 ns each, so a few shared lines cost more than the waves that add to them compute.
constexpr int E_SLOTS = 512;
struct ESlots {
  unsigned long long* p;
  int n;
  __device__ __forceinline__ unsigned long long* line(int k) const { return p + 8 * (long long)(k % n); }
};
constexpr double F_SCALE = 4294967296.0;        // 2^32: forces and energies (kJ/mol, nm)
constexpr double Q_SCALE = 1099511627776.0;     // 2^40: PME charge grid
// padding slots sit at x = PAD_STEP (1 + slot), y = z = PAD_STEP: every padding slot is more
// than PAD_STEP / 2 from every atom and from every other padding slot under any periodic
// shift of at most one box length (boxes shorter than PAD_LIMIT)
constexpr double PAD_STEP = 1.0e6;
constexpr double PAD_LIMIT = 5.0e5;

template <typename T> struct V4 { T x, y, z, w; };
template <typename T> struct V2 { T x, y; };

struct Geo {
  double L[3], invL[3];
  int ncol[2];
  double colw[2];
  int ncl_max;
  long long pair_cap;
  int maxn;  // cluster-pair segment length per i-cluster
  int reach[2];
};

__device__ __forceinline__ long long to_fx(double v, double s) { return __double2ll_rn(v * s); }

// ---------------------------------------------------------------- 1. binning
// Atoms are binned into x-y columns, the columns are scanned, the atoms scattered into their
// column's range, and every column is sorted by (z, atom index) in LDS, so that the order
// (and everything computed from it) does not depend on the order of the atomics.
constexpr int COL_SORT_MAX = 8192;  // atoms per column sorted in LDS (64 KB of keys)

template <typename TI>
__device__ __forceinline__ void wrap_coords(const TI* __restrict__ coords, long long i, const Geo& g, double w[3]) {
  for (int a = 0; a < 3; ++a) {
    double f = (double)coords[3 * i + a] * g.invL[a];
    f -= floor(f);
    w[a] = f * g.L[a];
  }
}

// Column of every atom and its offset within the column: the lanes of a wave that share a
// column reserve one contiguous range with a single atomic (binning water boxes puts hundreds
// of atoms on each column counter, so per-atom atomics would serialise).
template <typename TI>
__global__ __launch_bounds__(FB) void k_bin_atoms(const TI* __restrict__ coords, const TI* __restrict__ q, long long n,
                                                  Geo g, int* __restrict__ col_of, int* __restrict__ off_in_col,
                                                  int* __restrict__ col_count, double* __restrict__ q2part,
                                                  const TI* __restrict__ box_dev, int* __restrict__ status) {
  const long long i = blockIdx.x * (long long)FB + threadIdx.x;
  const int lane = threadIdx.x & (TFF_WAVE - 1);
  const bool valid = i < n;
  if (box_dev && blockIdx.x == 0 && threadIdx.x == 0) {
    // the call was planned (cell grid, capacities, PME geometry) from a host copy of the box: a
    // device box that no longer holds those values marks every result of the call as invalid
    bool same = true;
    for (int k = 0; k < 9; ++k) same = same && box_dev[k] == (k % 4 == 0 ? (TI)g.L[k / 4] : (TI)0);
    if (!same) atomicOr(status, TFF_FUSED_BOX_STALE);
  }
  {
    // sum of q^2 of the block (self energy), one partial per block
    const double qi = valid ? (double)q[i] : 0.0;
    const double t = tff_block_sum(qi * qi);
    if (threadIdx.x == 0) q2part[blockIdx.x] = t;
  }
  int col = -1;
  if (valid) {
    double w[3];
    wrap_coords(coords, i, g, w);
    int cx = (int)(w[0] / g.colw[0]); cx = cx < 0 ? 0 : (cx >= g.ncol[0] ? g.ncol[0] - 1 : cx);
    int cy = (int)(w[1] / g.colw[1]); cy = cy < 0 ? 0 : (cy >= g.ncol[1] ? g.ncol[1] - 1 : cy);
    col = cx * g.ncol[1] + cy;
  }
  int off = 0;
  unsigned long long active = __ballot(valid);
  while (active) {
    const int leader = __ffsll((long long)active) - 1;
    const int c0 = __shfl(col, leader, TFF_WAVE);
    const unsigned long long same = __ballot(valid && col == c0) & active;
    int base = 0;
    if (lane == leader) base = atomicAdd(&col_count[c0], __popcll(same));
    base = __shfl(base, leader, TFF_WAVE);
    if (valid && col == c0) off = base + __popcll(same & ((1ull << lane) - 1ull));
    active &= ~same;
  }
  if (valid) {
    col_of[i] = col;
    off_in_col[i] = off;
  }
}

// exclusive scans over the columns of their atom counts and cluster counts (one workgroup)
__global__ __launch_bounds__(1024) void k_scan_columns(const int* __restrict__ col_count, int ncols,
                                                       int* __restrict__ col_start, int* __restrict__ col_cl_start,
                                                       int* __restrict__ n_clusters, int* __restrict__ status) {
  __shared__ int sa[1024], sc[1024];
  const int t = threadIdx.x;
  const int per = (ncols + 1023) / 1024;
  const int b = t * per, e = b + per < ncols ? b + per : ncols;
  int na = 0, nc = 0;
  bool big = false;
  for (int c = b; c < e; ++c) {
    const int m = col_count[c];
    na += m;
    nc += (m + CL - 1) / CL;
    big = big || m > COL_SORT_MAX;
  }
  if (big) atomicOr(status, TFF_FUSED_COLUMN_OVERFLOW);
  sa[t] = na;
  sc[t] = nc;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {
    const int va = t >= off ? sa[t - off] : 0, vc = t >= off ? sc[t - off] : 0;
    __syncthreads();
    sa[t] += va;
    sc[t] += vc;
    __syncthreads();
  }
  int ra = t > 0 ? sa[t - 1] : 0, rc = t > 0 ? sc[t - 1] : 0;
  for (int c = b; c < e; ++c) {
    const int m = col_count[c];
    col_start[c] = ra;
    col_cl_start[c] = rc;
    ra += m;
    rc += (m + CL - 1) / CL;
  }
  if (t == 1023) {
    col_start[ncols] = sa[1023];
    col_cl_start[ncols] = sc[1023];
    *n_clusters = sc[1023];
  }
}

__global__ __launch_bounds__(FB) void k_scatter_atoms(long long n, const int* __restrict__ col_of,
                                                      const int* __restrict__ off_in_col,
                                                      const int* __restrict__ col_start, int* __restrict__ sorted_orig) {
  long long i = blockIdx.x * (long long)FB + threadIdx.x;
  if (i >= n) return;
  sorted_orig[col_start[col_of[i]] + off_in_col[i]] = (int)i;
}

// One workgroup per column sorts the keys (float bits of the wrapped z << 32 | atom) in LDS.  The
// keys are distinct (the atom index), so the sorted order is unique.  Bucket sort: the keys are
// counted into up to COL_BUCKETS z buckets (the bucket is monotone in the key), the counts
// scanned, the keys placed by bucket, and every key written to its bucket start plus its rank
// among the keys of its bucket; a column whose largest bucket holds more than BUCKET_RANK_MAX
// keys (atoms on shared z planes) is sorted by a bitonic network over the placed keys instead.
// Columns above COL_SORT_MAX atoms are left in scatter order (flagged by the scan).
constexpr int COL_BUCKETS = 2048;
constexpr int BUCKET_RANK_MAX = 32;
constexpr int SORT_THREADS = 256;

template <typename TI>
__device__ __forceinline__ unsigned long long column_key(const TI* __restrict__ coords, int i, const Geo& g) {
  double w[3];
  wrap_coords(coords, i, g, w);
  return ((unsigned long long)__float_as_uint((float)w[2]) << 32) | (unsigned)i;
}
// z >= 0, so the float bits order as the values and the product is monotone in the key
__device__ __forceinline__ int column_bucket(unsigned long long key, float scale, int nb) {
  const int b = (int)(__uint_as_float((unsigned)(key >> 32)) * scale);
  return b < 0 ? 0 : (b < nb - 1 ? b : nb - 1);
}

template <typename TI>
__global__ __launch_bounds__(SORT_THREADS) void k_sort_columns(const TI* __restrict__ coords, Geo g,
                                                               const int* __restrict__ col_start,
                                                               int* __restrict__ sorted_orig, ESlots es) {
  static_assert(COL_BUCKETS <= 8 * SORT_THREADS, "column sort: eight buckets per thread at most");
  __shared__ unsigned long long s_k[COL_SORT_MAX];
  __shared__ int s_c[COL_BUCKETS];
  __shared__ int s_tot[SORT_THREADS / TFF_WAVE], s_max[SORT_THREADS / TFF_WAVE];
  const int col = blockIdx.x;
  for (int k = col * SORT_THREADS + threadIdx.x; k < 8 * es.n; k += gridDim.x * SORT_THREADS) es.p[k] = 0ull;
  const int cs = col_start[col], m = col_start[col + 1] - cs;
  if (m <= 1 || m > COL_SORT_MAX) return;
  const int t = threadIdx.x, lane = t & (TFF_WAVE - 1), wv = t / TFF_WAVE;
  const int nb = m / 2 < 1 ? 1 : (m / 2 < COL_BUCKETS ? m / 2 : COL_BUCKETS);
  const float scale = (float)nb / (float)g.L[2];
  for (int b = t; b < nb; b += SORT_THREADS) s_c[b] = 0;
  __syncthreads();
  for (int k = t; k < m; k += SORT_THREADS)
    atomicAdd(&s_c[column_bucket(column_key(coords, sorted_orig[cs + k], g), scale, nb)], 1);
  __syncthreads();
  // exclusive scan of the bucket sizes (thread t owns buckets [b0, b1)) and the largest bucket
  const int per = (nb + SORT_THREADS - 1) / SORT_THREADS;
  const int b0 = t * per < nb ? t * per : nb, b1 = b0 + per < nb ? b0 + per : nb;
  int sum = 0, mx = 0;
  for (int b = b0; b < b1; ++b) {
    const int c = s_c[b];
    sum += c;
    mx = c > mx ? c : mx;
  }
  int inc = sum;
  for (int o = 1; o < TFF_WAVE; o <<= 1) {
    const int v = __shfl_up(inc, o, TFF_WAVE);
    if (lane >= o) inc += v;
  }
  for (int o = TFF_WAVE / 2; o > 0; o >>= 1) {
    const int v = __shfl_xor(mx, o, TFF_WAVE);
    mx = v > mx ? v : mx;
  }
  if (lane == TFF_WAVE - 1) {
    s_tot[wv] = inc;
    s_max[wv] = mx;
  }
  __syncthreads();
  int run = inc - sum, big = 0;
  for (int v = 0; v < SORT_THREADS / TFF_WAVE; ++v) {
    if (v < wv) run += s_tot[v];
    big = s_max[v] > big ? s_max[v] : big;
  }
  for (int b = b0; b < b1; ++b) {
    const int c = s_c[b];
    s_c[b] = run;
    run += c;
  }
  __syncthreads();
  // place the keys by bucket; afterwards s_c[b] is the end of bucket b
  for (int k = t; k < m; k += SORT_THREADS) {
    const unsigned long long key = column_key(coords, sorted_orig[cs + k], g);
    s_k[atomicAdd(&s_c[column_bucket(key, scale, nb)], 1)] = key;
  }
  __syncthreads();
  if (big <= BUCKET_RANK_MAX) {
    for (int p = t; p < m; p += SORT_THREADS) {
      const unsigned long long key = s_k[p];
      const int b = column_bucket(key, scale, nb);
      const int s = b > 0 ? s_c[b - 1] : 0, e = s_c[b];
      int r = 0;
      for (int q = s; q < e; ++q) r += s_k[q] < key ? 1 : 0;
      sorted_orig[cs + s + r] = (int)(unsigned)(key & 0xffffffffull);
    }
    return;
  }
  // bitonic network over the placed keys, padded to a power of two (pair k -> keys (lo, lo + stride))
  int np = 1;
  while (np < m) np <<= 1;
  for (int k = m + t; k < np; k += SORT_THREADS) s_k[k] = ~0ull;
  __syncthreads();
  for (int size = 2; size <= np; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int k = t; k < (np >> 1); k += SORT_THREADS) {
        const int lo = (k & ~(stride - 1)) * 2 + (k & (stride - 1)), hi = lo + stride;
        const bool asc = (lo & size) == 0;
        const unsigned long long x = s_k[lo], y = s_k[hi];
        if ((x > y) == asc) {
          s_k[lo] = y;
          s_k[hi] = x;
        }
      }
      __syncthreads();
    }
  }
  for (int k = t; k < m; k += SORT_THREADS) sorted_orig[cs + k] = (int)(unsigned)(s_k[k] & 0xffffffffull);
}

// zero several int32 buffers in one launch (lengths in 32-bit words)
struct ClearList {
  int* p[8];
  long long n[8];
  int count;
};
__global__ void k_clear(ClearList c) {
  const long long s = (long long)gridDim.x * blockDim.x;
  for (int b = 0; b < c.count; ++b)
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < c.n[b]; i += s) c.p[b][i] = 0;
}

// ---------------------------------------------------------------- 2. cluster arrays
// Two clusters per wave, one per half (lanes 0..31, 32..63 = slots): a cluster takes 32 consecutive atoms of its
// column's z-sorted range (the last cluster of a column is padded).  The slots are then
// ordered into four spatially compact groups of 8: sort by x and split in halves, sort each
// half by y and split, order each group by z (padding slots, keyed +inf, collect at the end;
// ties broken by slot).  Writes the cluster arrays (TC4 x, y, z, q; TC2 sigma / 2,
// 2 sqrt(eps)), slot_orig / slot_of_orig, the cluster's column, and the bounding boxes (centre,
// half extent) of the cluster and of its four groups (an empty group gets half extent -1),
// widened by a relative epsilon so that float rounding of the tests never drops a pair.
template <typename TI, typename TC>
__global__ __launch_bounds__(FB) void k_build_clusters(const TI* __restrict__ coords, const TI* __restrict__ q,
                                                       const TI* __restrict__ sig, const TI* __restrict__ eps,
                                                       Geo g, const int* __restrict__ ncl_ptr,
                                                       const int* __restrict__ col_cl_start,
                                                       const int* __restrict__ col_start,
                                                       const int* __restrict__ sorted_orig, V4<TC>* __restrict__ xyzq,
                                                       V2<TC>* __restrict__ lj, int* __restrict__ slot_orig,
                                                       int* __restrict__ slot_of_orig, int* __restrict__ cl_col,
                                                       float4* __restrict__ bb_c, float4* __restrict__ bb_h,
                                                       float4* __restrict__ sb_c, float4* __restrict__ sb_h) {
  __shared__ float4 s_p[FB / CL][CL];
  const int c = (blockIdx.x * FB + threadIdx.x) / CL;
  const int s = threadIdx.x & (CL - 1);
  const int w = threadIdx.x / CL;
  if (c >= *ncl_ptr) return;
  // column of cluster c
  int lo = 0, hi = g.ncol[0] * g.ncol[1];
  while (hi - lo > 1) {
    const int mid = (lo + hi) / 2;
    if (col_cl_start[mid] <= c) lo = mid; else hi = mid;
  }
  const int col = lo;
  if (s == 0) cl_col[c] = col;
  const int pos = col_start[col] + (c - col_cl_start[col]) * CL + s;
  const int o = pos < col_start[col + 1] ? sorted_orig[pos] : -1;
  V4<TC> p;
  V2<TC> l;
  if (o >= 0) {
    double wv[3];
    wrap_coords(coords, o, g, wv);
    p = {(TC)wv[0], (TC)wv[1], (TC)wv[2], (TC)q[o]};
    l = {(TC)(0.5 * (double)sig[o]), (TC)(2.0 * sqrt((double)eps[o] > 0 ? (double)eps[o] : 0.0))};
  } else {
    p = {(TC)0, (TC)0, (TC)0, (TC)0};
    l = {(TC)0, (TC)0};
  }
  const float inf = 3.0e38f;
  const float kx = o >= 0 ? (float)p.x : inf, ky = o >= 0 ? (float)p.y : inf, kz = o >= 0 ? (float)p.z : inf;
  // rank by x over all 32 slots
  int rx = 0;
  for (int t = 0; t < CL; ++t) {
    float vx = __shfl(kx, t, CL);
    rx += (vx < kx || (vx == kx && t < s)) ? 1 : 0;
  }
  const int half = rx >= CL / 2;
  int ry = 0;
  for (int t = 0; t < CL; ++t) {
    float vy = __shfl(ky, t, CL);
    int ht = __shfl(half, t, CL);
    ry += (ht == half && (vy < ky || (vy == ky && t < s))) ? 1 : 0;
  }
  const int grp = 2 * half + (ry >= CL / 4);
  int rz = 0;
  for (int t = 0; t < CL; ++t) {
    float vz = __shfl(kz, t, CL);
    int gt = 2 * __shfl(half, t, CL);
    int rt = __shfl(ry, t, CL);
    gt += rt >= CL / 4;
    rz += (gt == grp && (vz < kz || (vz == kz && t < s))) ? 1 : 0;
  }
  const int nl = grp * 8 + rz;
  const int ns = c * CL + nl;
  {
    // padding slots sit far away, each at its own place (see PAD_STEP)
    xyzq[ns] = o >= 0 ? p : V4<TC>{(TC)(PAD_STEP * (1.0 + ns)), (TC)PAD_STEP, (TC)PAD_STEP, (TC)0};
    lj[ns] = l;
    slot_orig[ns] = o;
    if (o >= 0) slot_of_orig[o] = ns;
    s_p[w][nl] = make_float4((float)p.x, (float)p.y, (float)p.z, o >= 0 ? 1.f : 0.f);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // bounding boxes of the ordered slots: thread s of the half wave holds slot s (the xor
  // shuffles below stay inside the half)
  const float4 qv = s_p[w][s];
  const bool v = qv.w != 0.f;
  float mn[3], mx[3], gmn[3], gmx[3];
  const float pv[3] = {qv.x, qv.y, qv.z};
  for (int a = 0; a < 3; ++a) {
    mn[a] = v ? pv[a] : 3.0e38f;
    mx[a] = v ? pv[a] : -3.0e38f;
    for (int off = 4; off > 0; off >>= 1) {
      mn[a] = fminf(mn[a], __shfl_xor(mn[a], off, TFF_WAVE));
      mx[a] = fmaxf(mx[a], __shfl_xor(mx[a], off, TFF_WAVE));
    }
    gmn[a] = mn[a];
    gmx[a] = mx[a];
    for (int off = 16; off > 4; off >>= 1) {
      mn[a] = fminf(mn[a], __shfl_xor(mn[a], off, TFF_WAVE));
      mx[a] = fmaxf(mx[a], __shfl_xor(mx[a], off, TFF_WAVE));
    }
  }
  if (s == 0) {
    bb_c[c] = make_float4(0.5f * (mn[0] + mx[0]), 0.5f * (mn[1] + mx[1]), 0.5f * (mn[2] + mx[2]), 0.f);
    bb_h[c] = make_float4(0.5f * (mx[0] - mn[0]) * 1.0001f + 1e-6f, 0.5f * (mx[1] - mn[1]) * 1.0001f + 1e-6f,
                          0.5f * (mx[2] - mn[2]) * 1.0001f + 1e-6f, 0.f);
  }
  if ((s & 7) == 0) {
    const int gi = c * 4 + s / 8;
    if (gmx[0] < gmn[0]) {
      sb_c[gi] = make_float4(0.f, 0.f, 0.f, 0.f);
      sb_h[gi] = make_float4(-1.f, -1.f, -1.f, 0.f);
    } else {
      sb_c[gi] = make_float4(0.5f * (gmn[0] + gmx[0]), 0.5f * (gmn[1] + gmx[1]), 0.5f * (gmn[2] + gmx[2]), 0.f);
      sb_h[gi] = make_float4(0.5f * (gmx[0] - gmn[0]) * 1.0001f + 1e-6f, 0.5f * (gmx[1] - gmn[1]) * 1.0001f + 1e-6f,
                             0.5f * (gmx[2] - gmn[2]) * 1.0001f + 1e-6f, 0.f);
    }
  }
}

// exclusion partners of every slot as packed (cluster << 5 | slot), -1 = none; padding slots
// have none
__global__ __launch_bounds__(FB) void k_fill_exclusions(const int* __restrict__ ncl_ptr,
                                                        const int* __restrict__ slot_orig,
                                                        const int* __restrict__ slot_of_orig, long long n,
                                                        const int64_t* __restrict__ row_ptr,
                                                        const int64_t* __restrict__ col,
                                                        int* __restrict__ excl_part, int* __restrict__ status) {
  const int sl = blockIdx.x * FB + threadIdx.x;
  if (sl >= *ncl_ptr * CL) return;
  const int i = slot_orig[sl];
  int k = 0;
  if (i >= 0 && col) {
    for (long long e = row_ptr[i]; e < row_ptr[i + 1]; ++e) {
      const long long j = col[e];
      if (j == i || j < 0 || j >= n) continue;
      if (k == MAXEX) {
        atomicOr(status, TFF_FUSED_EXCL_OVERFLOW);
        break;
      }
      excl_part[sl * MAXEX + k++] = slot_of_orig[j];
    }
  }
  for (; k < MAXEX; ++k) excl_part[sl * MAXEX + k] = -1;
}

// ---------------------------------------------------------------- 3. pair list
// Per i-cluster ci a list of entries, one per 8-atom j-group that has at least one group of ci within
// the cutoff: eg = the j-group (cj * 4 + gj, cj >= ci) and ei =
//   bits  0..3   bit gi set when groups gi of ci and gj of cj have bounding boxes within the
//                interaction cutoff (diagonal tiles: gi <= gj only)
//   bits  4..9   periodic shift k_a + 1 (2 bits per axis): x_j + k L is the image of cluster
//                cj closest to cluster ci
//   bit  10      the j-group holds exclusion partners of ci, or belongs to ci itself
//   bit  11      the shift is not the minimum image of every atom pair of the two clusters (small
//                boxes): the pair kernels then take the minimum image per pair
// The 4 * maxn entries of a cluster are filled from both ends: cluster pairs without bits 10 and 11 from
// the front (cnt.x entries, the pair's non-empty j-groups), the others from the back (cnt.y quads, the
// pair's four j-groups each, info 0 where empty).  The pair kernels sum a cluster pair's energies in
// TC before they go on in double; a quad of its own keeps a pair with (large) exclusion terms, or of
// a small box, in one piece, whatever the share of the list that a wave takes.
constexpr unsigned ENT_EXCL = 1u << 10;
constexpr unsigned ENT_MINIMG = 1u << 11;

struct PairList {
  int* g;             // j-groups, 4 * maxn per i-cluster
  unsigned short* i;  // their info
  int2* cnt;          // per i-cluster
  int cap;            // 4 * maxn
};

// One wave per i-cluster.  The lanes sweep the clusters of the neighbouring columns in a fixed order;
// clusters within the list cutoff collect in LDS, and whenever 64 are waiting (and at the end) each
// lane takes one of them, tests its 16 pairs of groups and the wave appends the entries (one ballot
// per j-group).  The order is fixed, so the list is the same on every call.
__global__ __launch_bounds__(FB) void k_pair_list(const int* __restrict__ ncl_ptr, const int* __restrict__ cl_col,
                                                  const int* __restrict__ col_cl_start,
                                                  const float4* __restrict__ bb_c, const float4* __restrict__ bb_h,
                                                  const float4* __restrict__ sb_c, const float4* __restrict__ sb_h,
                                                  Geo g, float rlist2, float cut2, const int* __restrict__ excl_part,
                                                  PairList pl, ESlots es,
                                                  int* __restrict__ status) {
  __shared__ int s_xp[FB / TFF_WAVE][CL * MAXEX];
  __shared__ int s_off[FB / TFF_WAVE][2 * TFF_WAVE], s_cs[FB / TFF_WAVE][2 * TFF_WAVE];
  __shared__ int2 s_tile[FB / TFF_WAVE][2 * TFF_WAVE];
  const int lane = threadIdx.x & (TFF_WAVE - 1);
  const int w = threadIdx.x / TFF_WAVE;
  const int ci = __builtin_amdgcn_readfirstlane(blockIdx.x * (FB / TFF_WAVE) + w);
  const int ncl = *ncl_ptr;
  if (ci >= ncl) return;
  const unsigned long long below = (1ull << lane) - 1ull;
  // j-groups (of clusters other than ci) holding an exclusion partner of an atom of ci, compacted in LDS
  int nxp = 0;
  for (int k = 0; k < MAXEX; ++k) {
    const int v = lane < CL ? excl_part[(ci * CL + lane) * MAXEX + k] : -1;
    const bool keep = v >= 0 && (v >> 5) != ci;
    const unsigned long long m = __ballot(keep);
    if (keep) s_xp[w][nxp + __popcll(m & below)] = v >> 3;
    nxp += __popcll(m);
  }
  tff_wave_sync_lds();
  const int col = cl_col[ci];
  const int cx = col / g.ncol[1], cy = col % g.ncol[1];
  const float4 c0v = bb_c[ci], h0 = bb_h[ci];
  float4 gc[4], gh[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    gc[k] = sb_c[ci * 4 + k];
    gh[k] = sb_h[ci * 4 + k];
  }
  const float Lv[3] = {(float)g.L[0], (float)g.L[1], (float)g.L[2]};
  const float iLv[3] = {(float)g.invL[0], (float)g.invL[1], (float)g.invL[2]};
  int nseg = 0;                    // clusters within the list cutoff
  int nwait = 0;                   // of them in s_tile
  int nfront = 0, nback = 0;       // entries from the front, quads from the back
  const long long ebase = (long long)ci * pl.cap;
  // the first n waiting clusters -> entries
  auto emit = [&](int n) {
    int cj = 0;
    unsigned info = 0, bits = 0;
    if (lane < n) {
      const int2 e = s_tile[w][lane];
      cj = e.x;
      info = (unsigned)e.y;
#pragma unroll
      for (int gj = 0; gj < 4; ++gj) {
        const float4 c1 = sb_c[cj * 4 + gj], h1 = sb_h[cj * 4 + gj];
#pragma unroll
        for (int gi = 0; gi < 4; ++gi) {
          float dx = gc[gi].x - c1.x, dy = gc[gi].y - c1.y, dz = gc[gi].z - c1.z;
          // minimum image of the group centres: a lower bound on the distance of every image
          dx -= Lv[0] * rintf(dx * iLv[0]);
          dy -= Lv[1] * rintf(dy * iLv[1]);
          dz -= Lv[2] * rintf(dz * iLv[2]);
          const float gx = fmaxf(fabsf(dx) - gh[gi].x - h1.x, 0.f);
          const float gy = fmaxf(fabsf(dy) - gh[gi].y - h1.y, 0.f);
          const float gz = fmaxf(fabsf(dz) - gh[gi].z - h1.z, 0.f);
          if (gh[gi].x >= 0.f && h1.x >= 0.f && (ci != cj || gj >= gi) && gx * gx + gy * gy + gz * gz <= cut2)
            bits |= 1u << (gj * 4 + gi);
        }
      }
    }
    unsigned xg = cj == ci ? 15u : 0u;  // j-groups that need the exclusion tests
    for (int t = 0; t < nxp; ++t) {
      const int p = s_xp[w][t];
      xg |= (p >> 2) == cj ? 1u << (p & 3) : 0u;
    }
    unsigned nib_any = 0;
#pragma unroll
    for (int gj = 0; gj < 4; ++gj) nib_any |= (bits >> (4 * gj)) & 15u ? 1u << gj : 0u;
    const bool back = nib_any && (xg || (info & ENT_MINIMG));
    const int nf = back ? 0 : __popc(nib_any);
    int kf = nfront;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const unsigned long long mf = __ballot((nf >> p) & 1);
      kf += __popcll(mf & below) << p;
      nfront += __popcll(mf) << p;
    }
    const unsigned long long mb = __ballot(back);
    const int kb = pl.cap - 4 * (nback + __popcll(mb & below)) - 4;
    nback += __popcll(mb);
#pragma unroll
    for (int gj = 0; gj < 4; ++gj) {
      if (!back && !((nib_any >> gj) & 1u)) continue;  // (back: the empty ones too, with info 0)
      const int k = back ? kb + gj : kf++;
      const unsigned nib = (bits >> (4 * gj)) & 15u;
      pl.g[ebase + k] = cj * 4 + gj;
      pl.i[ebase + k] = (unsigned short)(nib ? info | ((xg >> gj) & 1u ? ENT_EXCL : 0u) | nib : 0u);
    }
  };
  const int nx = 2 * g.reach[0] + 1 >= g.ncol[0] ? g.ncol[0] : 2 * g.reach[0] + 1;
  const int ny = 2 * g.reach[1] + 1 >= g.ncol[1] ? g.ncol[1] : 2 * g.reach[1] + 1;
  const int x0 = nx == g.ncol[0] ? 0 : cx - g.reach[0];
  const int y0 = ny == g.ncol[1] ? 0 : cy - g.reach[1];
  const int ncc = nx * ny;
  // The z window of ci: clusters whose z extent meets [z_lo - rlist, z_hi + rlist] (or its
  // periodic images) can pass the bounding-box test below; every other one fails it.  The
  // clusters of a column are z ordered (their lower and upper z bounds rise along the column), so
  // per column the window is one index range, or two when it wraps round the box; 0.01 nm of slack
  // keeps rounding from dropping a cluster the test would accept.  The accepted clusters and their
  // order (columns in order, clusters ascending) are those of a scan over whole columns.
  const float rl = sqrtf(rlist2) + 0.01f;
  const double zw_lo = (double)(c0v.z - h0.z) - rl, zw_hi = (double)(c0v.z + h0.z) + rl;
  const bool zall = zw_hi - zw_lo >= g.L[2];
  const float za0 = zw_lo < 0 ? 0.f : (float)zw_lo, zb0 = zw_hi > g.L[2] ? (float)g.L[2] : (float)zw_hi;
  const bool zwrap = !zall && (zw_lo < 0 || zw_hi > g.L[2]);
  const float za1 = zw_lo < 0 ? (float)(zw_lo + g.L[2]) : 0.f;  // second interval [za1, zb1]
  const float zb1 = zw_lo < 0 ? (float)g.L[2] : (float)(zw_hi - g.L[2]);
  // Candidates: the neighbouring columns (up to 64 at a time, one per lane), each as up to two
  // cluster ranges inside the window, clipped to cj >= ci, scanned into one flat range that the
  // wave walks 64 clusters at a time (column-major order).
  for (int c0 = 0; c0 < ncc; c0 += TFF_WAVE) {
    const int cc = c0 + lane;
    int r0s = 0, r0n = 0, r1s = 0, r1n = 0;
    if (cc < ncc) {
      int xx = x0 + cc / ny, yy = y0 + cc % ny;
      xx += xx < 0 ? g.ncol[0] : (xx >= g.ncol[0] ? -g.ncol[0] : 0);
      yy += yy < 0 ? g.ncol[1] : (yy >= g.ncol[1] ? -g.ncol[1] : 0);
      const int col_id = xx * g.ncol[1] + yy;
      const int ce = col_cl_start[col_id + 1];
      const int cs = col_cl_start[col_id];
      // first cluster with z max >= a, last cluster with z min <= b (both monotone in the column)
      auto first_ge = [&](float a) {
        int lo = cs, hi = ce;
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (bb_c[mid].z + bb_h[mid].z >= a) hi = mid; else lo = mid + 1;
        }
        return lo;
      };
      auto last_le = [&](float b) {
        int lo = cs - 1, hi = ce - 1;
        while (lo < hi) {
          const int mid = (lo + hi + 1) >> 1;
          if (bb_c[mid].z - bb_h[mid].z <= b) lo = mid; else hi = mid - 1;
        }
        return lo;
      };
      int a0 = cs, e0 = ce, a1 = 0, e1 = 0;  // [start, end) of up to two ranges
      if (!zall && cs < ce) {
        if (!zwrap) {
          a0 = first_ge(za0);
          e0 = last_le(zb0) + 1;
        } else {
          // [0, b] at the column's start, [a, L) at its end; merged when they meet
          const int l0 = last_le(zw_lo < 0 ? zb0 : zb1) + 1;
          const int f1 = first_ge(zw_lo < 0 ? za1 : za0);
          if (f1 > l0) {
            e0 = l0;
            a1 = f1;
            e1 = ce;
          }
        }
      }
      a0 = a0 > ci ? a0 : ci;
      a1 = a1 > ci ? a1 : ci;
      r0s = a0;
      r0n = e0 > a0 ? e0 - a0 : 0;
      r1s = a1;
      r1n = e1 > a1 ? e1 - a1 : 0;
    }
    const int cnt = r0n + r1n;
    int incl = cnt;
#pragma unroll
    for (int off = 1; off < TFF_WAVE; off <<= 1) {
      const int v = __shfl_up(incl, off, TFF_WAVE);
      if (lane >= off) incl += v;
    }
    const int total = __shfl(incl, TFF_WAVE - 1, TFF_WAVE);
    s_off[w][2 * lane] = incl - cnt;
    s_cs[w][2 * lane] = r0s;
    s_off[w][2 * lane + 1] = incl - cnt + r0n;
    s_cs[w][2 * lane + 1] = r1s;
    tff_wave_sync_lds();
    const int nvalid = 2 * (ncc - c0 < TFF_WAVE ? ncc - c0 : TFF_WAVE);
    for (int b = 0; b < total; b += TFF_WAVE) {
      const int k = b + lane;
      unsigned info = 0;
      int cj = -1;
      bool ok = false;
      if (k < total) {
        // last range whose offset is <= k (offsets are non-decreasing; an empty range shares its
        // offset with the next one, which then holds k)
        int lo = 0, hi = nvalid - 1;
        while (lo < hi) {
          const int mid = (lo + hi + 1) >> 1;
          if (s_off[w][mid] <= k) lo = mid; else hi = mid - 1;
        }
        cj = s_cs[w][lo] + (k - s_off[w][lo]);
        const float4 c1 = bb_c[cj], h1 = bb_h[cj];
        const float d[3] = {c0v.x - c1.x, c0v.y - c1.y, c0v.z - c1.z};
        const float hs[3] = {h0.x + h1.x, h0.y + h1.y, h0.z + h1.z};
        float gap2 = 0.f;
        bool minimg = false;
        unsigned shift = 0;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const float kk = rintf(d[a] * iLv[a]);
          const float dm = d[a] - Lv[a] * kk;
          const float gp = fmaxf(fabsf(dm) - hs[a], 0.f);
          gap2 += gp * gp;
          minimg = minimg || !(fabsf(dm) + hs[a] <= 0.49999f * Lv[a]);
          shift |= (unsigned)((int)kk + 1) << (4 + 2 * a);
        }
        ok = gap2 <= rlist2;
        info = shift | (minimg ? ENT_MINIMG : 0u);
      }
      const unsigned long long bm = __ballot(ok);
      const int r = __popcll(bm & below);
      // over the capacity (flagged below) the rest is dropped
      if (ok && nseg + r < g.maxn) s_tile[w][nwait + r] = make_int2(cj, (int)info);
      const int room = g.maxn - nseg, got = __popcll(bm);
      nwait += got < room ? got : (room > 0 ? room : 0);
      nseg += got;
      tff_wave_sync_lds();
      if (nwait >= TFF_WAVE) {
        emit(TFF_WAVE);
        nwait -= TFF_WAVE;
        const int2 tail = s_tile[w][TFF_WAVE + lane];
        tff_wave_sync_lds();
        s_tile[w][lane] = tail;
        tff_wave_sync_lds();
      }
    }
    // the next group of columns rewrites s_off / s_cs
    tff_wave_sync_lds();
  }
  if (nwait > 0) emit(nwait);
  if (lane == 0) {
    if (nseg > g.maxn) atomicOr(status, TFF_FUSED_PAIR_OVERFLOW);
    atomicAdd(es.line(ci) + 2, (unsigned long long)(nseg < g.maxn ? nseg : g.maxn));
    pl.cnt[ci] = make_int2(nfront, nback);
  }
}

// ---------------------------------------------------------------- 4. pair kernels
// Lane maps: lane = 8 ii + jj evaluates i-slot ii of a group of ci against j-slot jj of the j-group.
// Sums over jj (contiguous octets) are DPP adds; sums over ii (stride 8) halve with the gfx950
// half-wave and row swaps: swapping the upper half of one value with the lower half of another and
// adding the two leaves each half with the sum of one of them, so every exchange also scatters.
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ double dpp_f(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
// sum over the 8 lanes sharing lane >> 3 (the result lands in all 8 lanes)
template <typename T>
__device__ __forceinline__ T octet_sum(T v) {
  v += dpp_f<0xB1>(v);   // quad_perm [1,0,3,2]
  v += dpp_f<0x4E>(v);   // quad_perm [2,3,0,1]
  v += dpp_f<0x141>(v);  // row_half_mirror (every lane of a quad holds the quad's sum by now)
  return v;
}
// lanes 0..31: a summed over the lane pair (l, l + 32); lanes 32..63: b summed over (l - 32, l)
__device__ __forceinline__ float half_add(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// even rows of 16 lanes: a summed over the row pair; odd rows: b summed over it
__device__ __forceinline__ float row_add(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ double join_d(unsigned lo, unsigned hi) {
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ double half_add(double a, double b) {
  const unsigned long long x = (unsigned long long)__double_as_longlong(a), y = (unsigned long long)__double_as_longlong(b);
  const auto l = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
  const auto h = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  return join_d(l[0], h[0]) + join_d(l[1], h[1]);
}
__device__ __forceinline__ double row_add(double a, double b) {
  const unsigned long long x = (unsigned long long)__double_as_longlong(a), y = (unsigned long long)__double_as_longlong(b);
  const auto l = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
  const auto h = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  return join_d(l[0], h[0]) + join_d(l[1], h[1]);
}
// one value of each of four entries summed over the 8 lanes sharing lane & 7: the lane gets entry
// 2 (lane >> 5) + ((lane >> 4) & 1)'s sum (both lanes that differ in bit 3 hold it)
template <typename T>
__device__ __forceinline__ T quad_reduce(T f0, T f1, T f2, T f3) {
  const T h = row_add(half_add(f0, f2), half_add(f1, f3));
  return h + dpp_f<0x128>(h);  // row_ror:8
}
template <typename T>
__device__ __forceinline__ T wave_sum_t(T v) {
  v = octet_sum(v);
  v += dpp_f<0x128>(v);
  v = row_add(v, v);
  return half_add(v, v);
}

// v added to an int64 fixed-point accumulator, rounded to the nearest multiple of 2^-32: below 2^19
// the integer is read off the mantissa of v 2^32 + 1.5 2^52 (one fma and one integer subtraction;
// the general double-to-int64 conversion takes about ten float64 instructions); larger values (and
// NaN) take the conversion.  Both round to nearest even.
template <typename T>
__device__ __forceinline__ void acc_add(unsigned long long* p, T v) {
  unsigned long long x;
  if (__builtin_expect(fabs((double)v) < 524288.0, 1))
    x = (unsigned long long)(__double_as_longlong(fma((double)v, F_SCALE, 6755399441055744.0)) - 0x4338000000000000LL);
  else
    x = (unsigned long long)to_fx((double)v, F_SCALE);
  if (v != (T)0) atomicAdd(p, x);
}

// The pair kernels' force accumulators: per group of 8 slots three (backward: GN) lines of 64 bytes, one per
// component.  Memory-side atomics cost one operation per 64-byte line an instruction touches (about
// 24 G lines/s), so an entry costs three line operations; with x, y, z interleaved per slot it cost
// six, and the line rate, not the arithmetic, set the kernel's time.
__device__ __forceinline__ long long acc_slot(int sl, int a) { return (long long)(sl >> 3) * 24 + 8 * a + (sl & 7); }

template <typename TC>
struct TileArgs {
  TC L[3], invL[3];
  TC rc2;
  TC alpha;
  TC coul;
  TC c2alpha;  // (2 / sqrt(pi)) alpha
};

template <typename T> struct V3 { T x, y, z; };

// the periodic shift of an entry along one axis (selected as bits, on the scalar unit)
__device__ __forceinline__ float entry_shift(unsigned info, int axis, float L) {
  const unsigned k = (info >> (4 + 2 * axis)) & 3u;
  const unsigned b = __float_as_uint(L) ^ (k == 0u ? 0x80000000u : 0u);
  return __uint_as_float(k == 1u ? 0u : b);
}
__device__ __forceinline__ double entry_shift(unsigned info, int axis, double L) {
  const unsigned k = (info >> (4 + 2 * axis)) & 3u;
  const unsigned long long b = (unsigned long long)__double_as_longlong(L);
  const unsigned hi = (unsigned)(b >> 32) ^ (k == 0u ? 0x80000000u : 0u);
  return join_d(k == 1u ? 0u : (unsigned)b, k == 1u ? 0u : hi);
}

// exclusion partners of the lane's i atom against j slot sj
__device__ __forceinline__ bool is_partner(const int* __restrict__ excl_part, int sli, int sj) {
  const int4* xp = reinterpret_cast<const int4*>(excl_part + (long long)sli * MAXEX);
  const int4 x0 = xp[0], x1 = xp[1];
  return x0.x == sj || x0.y == sj || x0.z == sj || x0.w == sj || x1.x == sj || x1.y == sj || x1.z == sj || x1.w == sj;
}

// A wave's share of an i-cluster's list: quads [q0, q1) of the nq quads, the first nfq of them from the
// front (unflagged entries), the rest from the back.
struct QuadRange {
  int nfq, q0, q1;
  int2 cnt;
};
__device__ __forceinline__ QuadRange quad_range(const PairList& pl, int ci, int part, int parts) {
  QuadRange r;
  r.cnt = pl.cnt[ci];
  r.nfq = (r.cnt.x + 3) >> 2;
  const int nq = r.nfq + r.cnt.y;
  const int per = (nq + parts - 1) / parts;
  r.q0 = part * per;
  r.q1 = r.q0 + per < nq ? r.q0 + per : nq;
  return r;
}
// four entries: j-groups and infos (past the list's end: info 0 and a valid entry's j-group, so that its
// atoms can be loaded all the same)
struct Quad {
  int g0, g1, g2, g3;
  unsigned i0, i1, i2, i3;
};
__device__ __forceinline__ Quad load_quad(const PairList& pl, int ci, const QuadRange& r, int q) {
  const bool front = q < r.nfq;
  const int k = front ? 4 * q : pl.cap - 4 * (q - r.nfq) - 4;
  const long long b = (long long)ci * pl.cap + k;
  const int4 g = *reinterpret_cast<const int4*>(pl.g + b);
  const uint2 i = *reinterpret_cast<const uint2*>(pl.i + b);
  const int nv = front ? r.cnt.x - k : 4;  // valid entries (at least one)
  return {g.x, nv > 1 ? g.y : g.x, nv > 2 ? g.z : g.x, nv > 3 ? g.w : g.x,
          i.x & 0xffffu, nv > 1 ? i.x >> 16 : 0u, nv > 2 ? i.y & 0xffffu : 0u, nv > 3 ? i.y >> 16 : 0u};
}

// the lane's atom of a j-group
template <typename TC>
struct JAtom {
  V4<TC> p;
  V2<TC> l;
};
template <typename TC>
__device__ __forceinline__ JAtom<TC> load_j(const V4<TC>* __restrict__ xyzq, const V2<TC>* __restrict__ lj, int jg,
                                            unsigned jj) {
  return {(xyzq + (long long)jg * 8)[jj], (lj + (long long)jg * 8)[jj]};
}

template <typename TC>
struct PairSums {
  V3<TC> f0, f1, f2, f3;  // F of the lane's i atoms (groups 0..3)
  TC e_lj, e_c;           // over the consecutive entries of one j-cluster
};

// One entry: the lane's j atom (shifted here) against the groups of ci in the entry's mask; F_j into fj.
// CHECKED: the entry may hold exclusions, lie on the diagonal or need the minimum image per pair
// (tested at run time; uniform over the wave).  The i atoms come from LDS (pi, li: slot ii of group 0):
// kept in registers they cost two waves per SIMD (float64) for two LDS reads per group pair.
template <typename TC, bool CHECKED>
__device__ __forceinline__ V3<TC> entry_steps(unsigned info, int ci, int jg, const V4<TC>* pis, const V2<TC>* lis,
                                              JAtom<TC> j, const int* __restrict__ excl_part, int ii, int jj,
                                              const TileArgs<TC>& ta, PairSums<TC>& s) {
  const bool minimg = CHECKED && (info & ENT_MINIMG) != 0u;
  if (!minimg) {
    j.p.x += entry_shift(info, 0, ta.L[0]);
    j.p.y += entry_shift(info, 1, ta.L[1]);
    j.p.z += entry_shift(info, 2, ta.L[2]);
  }
  V3<TC> fj{(TC)0, (TC)0, (TC)0};
  auto step = [&](int gi, V3<TC>& fi) {
    const V4<TC> pi = pis[gi * 8];
    TC dx = pi.x - j.p.x, dy = pi.y - j.p.y, dz = pi.z - j.p.z;
    if (minimg) {
      dx -= ta.L[0] * rint(dx * ta.invL[0]);
      dy -= ta.L[1] * rint(dy * ta.invL[1]);
      dz -= ta.L[2] * rint(dz * ta.invL[2]);
    }
    // (one order of the products in every variant: rigid molecules repeat its rounding)
    TC r2 = fma(dz, dz, fma(dx, dx, dy * dy));
    bool ok = r2 <= ta.rc2;
    if (minimg) ok = ok && pi.x < (TC)PAD_LIMIT && j.p.x < (TC)PAD_LIMIT;
    if (CHECKED && jg == ci * 4 + gi) ok = ok && jj > ii;
    // about a fifth of the group pairs kept by the bounding-box test hold no pair within the
    // cutoff: the wave skips them (uniform branch)
    if (__builtin_amdgcn_ballot_w64(ok) == 0) return;
    bool excl = false;
    if (CHECKED && (info & ENT_EXCL)) excl = is_partner(excl_part, ci * CL + gi * 8 + ii, jg * 8 + jj);
    // pairs that do not count are moved far away: every term below is then exactly zero
    // (exp underflows, s^6 flushes), except (erfc - 1)/r of an excluded pair beyond the
    // cutoff, which is below 1e-12 q_i q_j (and dropped with its group pair when no pair of it is in
    // range)
    r2 = ok ? r2 : (TC)1e30;
    const TC rinv = rsqrt_t(r2);
    const TC rinv2 = rinv * rinv;
    const TC r = r2 * rinv;
    TC ec, em;
    if (CHECKED)
      erfc_exp_excl(ta.alpha * r, excl, ec, em);
    else
      erfc_exp(ta.alpha * r, ec, em);
    const V2<TC> li = lis[gi * 8];
    const TC qr = pi.w * j.p.w * rinv;
    TC ep4 = li.y * j.l.y;
    if (CHECKED) ep4 = excl ? (TC)0 : ep4;
    const TC sg = li.x + j.l.x;
    const TC s2 = sg * sg * rinv2;
    const TC s6 = s2 * s2 * s2;
    const TC a6 = ep4 * s6;  // 4 eps s^6
    // -dE/dr / r = [k q_i q_j / r (erfc + (2/sqrt pi) a r e^{-a^2 r^2}) + 4 eps s^6 (12 s^6 - 6)] / r^2
    const TC fs = fma(qr, fma(ta.c2alpha * r, em, ec), a6 * fma((TC)12, s6, (TC)-6)) * rinv2;
    s.e_c = fma(qr, ec, s.e_c);
    s.e_lj += fma(a6, s6, -a6);
    // F_i += fs d, F_j -= fs d   (fs = -dE/dr / r)
    fi.x = fma(fs, dx, fi.x);
    fi.y = fma(fs, dy, fi.y);
    fi.z = fma(fs, dz, fi.z);
    fj.x = fma(-fs, dx, fj.x);
    fj.y = fma(-fs, dy, fj.y);
    fj.z = fma(-fs, dz, fj.z);
  };
  if (info & 1u) step(0, s.f0);
  if (info & 2u) step(1, s.f1);
  if (info & 4u) step(2, s.f2);
  if (info & 8u) step(3, s.f3);
  return fj;
}

// One wave per workgroup takes one of `parts` equal shares of an i-cluster's list, four entries at a
// time.  The list holds only the j-groups with a partner (2.9 of the 4 of a listed cluster on average in
// water), so the per-entry work - loads, shift, the sums of F_j, their conversion and the atomics - is
// not spent on the empty ones; what bounds the kernel is vector issue (about 50 instructions per 8 x 8
// block with a pair in range, 38 % of whose lanes are).  Measured alone: float, 96k atoms, 143 -> 121 us
// (5 waves per SIMD), float64, 60k atoms, 396 -> 256 us (two waves per SIMD instead of one; 208 with the pair
// functions of pair_math.h), against one 32 x 32 tile at a time with all 12 F_j components of it reduced in
// every lane; F_i stays in registers for the whole share, F_j of a quad is summed over the 8 lanes sharing
// jj and added to the int64 fixed-point accumulators (entry 2 (lane >> 5) + ((lane >> 4) & 1), slot jj;
// bit 3 picks the components).  Integer sums do not depend on their order and each share is summed
// in a fixed order, so the results are bitwise reproducible.  Charges are pre-multiplied by the
// Coulomb constant on the i side; lj holds (sigma / 2, 2 sqrt(eps)) so that li.y * lJ.y = 4 eps_ij.
template <typename TC>
__device__ __forceinline__ void pairs_body(const int* __restrict__ ncl_ptr, const PairList& pl, int parts,
                                           const V4<TC>* __restrict__ xyzq, const V2<TC>* __restrict__ lj,
                                           const int* __restrict__ excl_part, const TileArgs<TC>& ta,
                                           unsigned long long* __restrict__ facc, ESlots es) {
  __shared__ V4<TC> s_p[CL];
  __shared__ V2<TC> s_l[CL];
  const int lane = threadIdx.x & (TFF_WAVE - 1);
  const int jj = lane & 7, ii = lane >> 3;
  const int ci = blockIdx.x / parts;
  if (ci >= *ncl_ptr) return;
  const QuadRange qr = quad_range(pl, ci, blockIdx.x % parts, parts);
  if (qr.q0 >= qr.q1) return;
  if (lane < CL) {
    V4<TC> p = xyzq[ci * CL + lane];
    p.w *= ta.coul;
    s_p[lane] = p;
    s_l[lane] = lj[ci * CL + lane];
  }
  tff_wave_sync_lds();
  const V4<TC>* pi = s_p + ii;
  const V2<TC>* li = s_l + ii;
  const bool b3 = lane & 8, b4 = lane & 16, b5 = lane & 32;
  PairSums<TC> s{};
  double e_lj = 0.0, e_c = 0.0;
  int cj = -1;
  auto flush_energy = [&](int c) {
    if (c == cj) return;
    cj = c;
    e_lj += (double)s.e_lj;
    e_c += (double)s.e_c;
    s.e_lj = s.e_c = 0;
  };
  for (int q = qr.q0; q < qr.q1; ++q) {
    const Quad d = load_quad(pl, ci, qr, q);
    auto steps = [&](unsigned info, int jg, const JAtom<TC>& j) {
      flush_energy(jg >> 2);
      return info & (ENT_EXCL | ENT_MINIMG)
                 ? entry_steps<TC, true>(info, ci, jg, pi, li, j, excl_part, ii, jj, ta, s)
                 : entry_steps<TC, false>(info, ci, jg, pi, li, j, excl_part, ii, jj, ta, s);
    };
    // the next entry's atoms are loaded while the current one is evaluated
    JAtom<TC> a = load_j(xyzq, lj, d.g0, jj), b = load_j(xyzq, lj, d.g1, jj);
    const V3<TC> f0 = steps(d.i0, d.g0, a);
    a = load_j(xyzq, lj, d.g2, jj);
    const V3<TC> f1 = steps(d.i1, d.g1, b);
    b = load_j(xyzq, lj, d.g3, jj);
    const V3<TC> f2 = steps(d.i2, d.g2, a);
    const V3<TC> f3 = steps(d.i3, d.g3, b);
    const TC hx = quad_reduce(f0.x, f1.x, f2.x, f3.x), hy = quad_reduce(f0.y, f1.y, f2.y, f3.y),
             hz = quad_reduce(f0.z, f1.z, f2.z, f3.z);
    const int g0 = b4 ? d.g1 : d.g0, g1 = b4 ? d.g3 : d.g2;
    unsigned long long* p = facc + (long long)(b5 ? g1 : g0) * 24 + jj;
    acc_add(p + (b3 ? 8 : 0), b3 ? hy : hx);
    if (!b3) acc_add(p + 16, hz);
  }
  flush_energy(-1);
  {
    // F_i: 12 sums over jj; lane (ii, jj) adds values jj and jj + 8 (value 3 g + a: slot g * 8 + ii)
    const TC k0 = octet_sum(s.f0.x), k1 = octet_sum(s.f0.y), k2 = octet_sum(s.f0.z), k3 = octet_sum(s.f1.x);
    const TC k4 = octet_sum(s.f1.y), k5 = octet_sum(s.f1.z), k6 = octet_sum(s.f2.x), k7 = octet_sum(s.f2.y);
    const TC k8 = octet_sum(s.f2.z), k9 = octet_sum(s.f3.x), k10 = octet_sum(s.f3.y), k11 = octet_sum(s.f3.z);
    const bool c0 = jj & 1, c1 = jj & 2, c2 = jj & 4;
    const TC s0 = c0 ? k1 : k0, s1 = c0 ? k3 : k2, s2 = c0 ? k5 : k4, s3 = c0 ? k7 : k6;
    const TC t0 = c1 ? s1 : s0, t1 = c1 ? s3 : s2;
    const TC w0 = c0 ? k9 : k8, w1 = c0 ? k11 : k10;
    unsigned long long* p = facc + (long long)ci * (3 * CL);
    acc_add(p + 8 * jj + ii, c2 ? t1 : t0);
    if (jj < 4) acc_add(p + 8 * (jj + 8) + ii, c1 ? w1 : w0);
  }
  // the wave's energies (integer sums do not depend on their order)
  const double el = wave_sum_t(e_lj), ecl = wave_sum_t(e_c);
  if (lane == 0) {
    unsigned long long* e = es.line(blockIdx.x);
    atomicAdd(e, (unsigned long long)to_fx(el, F_SCALE));
    atomicAdd(e + 1, (unsigned long long)to_fx(ecl, F_SCALE));
  }
}

__global__ __launch_bounds__(TFF_WAVE) __attribute__((amdgpu_waves_per_eu(4))) void k_tiles_f32(
    const int* __restrict__ ncl_ptr, PairList pl, int parts, const V4<float>* __restrict__ xyzq,
    const V2<float>* __restrict__ lj, const int* __restrict__ excl_part, TileArgs<float> ta,
    unsigned long long* __restrict__ facc, ESlots es) {
  // The body needs 89 registers, i.e. 5 waves per SIMD; naming v103 holds it at 4 (104 each) and leaves
  // 96 per SIMD free, so that the workgroups of the reciprocal-space chain find room beside the pair
  // kernel.  Alone the kernel takes 121 us with 5 waves and 129 with 4 (96k atoms); the whole evaluation
  // 258 with 5 and 256 with 4, at 999k atoms 2.00 and 2.06 ms.
  asm volatile("" ::: "v103");
  pairs_body<float>(ncl_ptr, pl, parts, xyzq, lj, excl_part, ta, facc, es);
}
__global__ __launch_bounds__(TFF_WAVE) __attribute__((amdgpu_waves_per_eu(2))) void k_tiles_f64(
    const int* __restrict__ ncl_ptr, PairList pl, int parts, const V4<double>* __restrict__ xyzq,
    const V2<double>* __restrict__ lj, const int* __restrict__ excl_part, TileArgs<double> ta,
    unsigned long long* __restrict__ facc, ESlots es) {
  pairs_body<double>(ncl_ptr, pl, parts, xyzq, lj, excl_part, ta, facc, es);
}

// ---------------------------------------------------------------- 4b. force-matching backward
// For upstream gradients gE (of E) and v (of F = -dE/dr), the vector-Jacobian product of (E, F):
//   dL/dtheta = gE dE/dtheta - d(D_v E)/dtheta,   dL/dr = gE dE/dr - grad(D_v E),
// with D_v E = sum_i v_i . grad_i E.  For a pair (d = r_i - r_j, dv = v_i - v_j, s = d . dv) with
// energy phi(r), f = phi'/r and h = f'/r:  D_v E_pair = f s,  grad_i(f s) = f dv + s h d.
//   Coulomb  phi = k q_i q_j c/r, c = erfc(a r) - [excluded],  g = c + (2/sqrt pi) a r e^{-a^2 r^2}:
//            f = -k q_i q_j g / r^3,  h = k q_i q_j (3 g / r^5 + (4/sqrt pi) a^3 e^{-a^2 r^2} / r^2)
//   LJ       phi = 4 eps (s12 - s6):  f = -4 eps (12 s12 - 6 s6) / r^2,
//            h = 4 eps (168 s12 - 48 s6) / r^4;  d/dsigma_i = 1/2 d/dsigma_ij,
//            d/deps_i = (.)/(2 eps_i) (0 where eps_i = 0).
// Per slot six int64 accumulators: d/dr (3), d/dq, d/dsigma, d/deps.
constexpr int GN = 6;
static_assert(4 * GN == 24, "a cluster column holds 24 backward sums per lane");

// per slot: the upstream force v (x, y, z) and 1 / (2 eps) (w; 0 where eps = 0), from lj's 2 sqrt(eps);
// with status_from set, thread 0 also starts the call's flags from those of the forward call
// whose cluster arrays and pair list are reused
template <typename TI, typename TC>
__global__ __launch_bounds__(FB) void k_fill_vslots(const int* __restrict__ ncl_ptr, const int* __restrict__ slot_orig,
                                                    const TI* __restrict__ v, const V2<TC>* __restrict__ lj,
                                                    V4<TC>* __restrict__ vsl, const int* __restrict__ status_from,
                                                    int* __restrict__ status) {
  const int sl = blockIdx.x * FB + threadIdx.x;
  if (status_from && sl == 0) {
    status[0] = status_from[0];
  }
  if (sl >= *ncl_ptr * CL) return;
  const int i = slot_orig[sl];
  const TC e2 = lj[sl].y;
  const TC ehalf_inv = e2 > (TC)0 ? (TC)2 / (e2 * e2) : (TC)0;
  vsl[sl] = (i >= 0 && v) ? V4<TC>{(TC)v[3 * i], (TC)v[3 * i + 1], (TC)v[3 * i + 2], ehalf_inv}
                          : V4<TC>{(TC)0, (TC)0, (TC)0, ehalf_inv};
}

template <typename T> struct GradSums { T x, y, z, q, s, e; };

// One wave per workgroup over a share of an i-cluster's list, as the forward pair kernel (the tile's
// periodic shift, minimum image per pair on the entries flagged for it); the i-side data of ci's four
// groups stays in LDS, its sums in registers.
// Per pair, in factored form without divisions (Q = q_i q_j, s6 = (sigma_ij / r)^6):
//   f = -k Q g / r^3 - 4 eps s6 (12 s6 - 6) / r^2
//   h =  k Q (3 g / r^3 + (4/sqrt pi) a^3 e^{-a^2 r^2}) / r^2 + 4 eps s6 (168 s6 - 48) / r^4
//   d phi / d sigma_ij = 4 eps (s6 / sigma_ij) (12 s6 - 6),  s6 / sigma_ij = s^4 sigma_ij / r^2,
//   d (f s) / d sigma_ij = -4 eps (s6 / sigma_ij) (144 s6 - 36) s / r^2,
// and 1 / (2 eps) of every slot precomputed (the w component of the per-slot upstream force).
template <typename TC>
__device__ __forceinline__ void grad_body(const int* __restrict__ ncl_ptr, const PairList& pl, int parts,
                                          const V4<TC>* __restrict__ xyzq, const V2<TC>* __restrict__ lj,
                                          const V4<TC>* __restrict__ vsl, const int* __restrict__ excl_part,
                                          const TileArgs<TC>& ta, const double* __restrict__ gE_ptr,
                                          unsigned long long* __restrict__ gacc) {
  __shared__ V4<TC> s_p[CL], s_v[CL];
  __shared__ V2<TC> s_l[CL];
  const int lane = threadIdx.x & (TFF_WAVE - 1);
  const int jj = lane & 7, ii = lane >> 3;
  const int ci = blockIdx.x / parts;
  if (ci >= *ncl_ptr) return;
  const QuadRange qr = quad_range(pl, ci, blockIdx.x % parts, parts);
  if (qr.q0 >= qr.q1) return;
  if (lane < CL) {
    s_p[lane] = xyzq[ci * CL + lane];
    s_v[lane] = vsl[ci * CL + lane];
    s_l[lane] = lj[ci * CL + lane];
  }
  tff_wave_sync_lds();
  const TC gE = gE_ptr ? (TC)gE_ptr[0] : (TC)0;
  const TC c2 = (TC)1.1283791670955126;                     // 2 / sqrt(pi)
  const TC ch = (TC)2 * c2 * ta.alpha * ta.alpha * ta.alpha;  // (4 / sqrt pi) a^3
  const bool b3 = lane & 8, b4 = lane & 16, b5 = lane & 32;
  GradSums<TC> a0{}, a1{}, a2{}, a3{};
  // one entry: the lane's j atom against the groups of ci in the entry's mask (see entry_steps)
  auto entry = [&](auto chk, unsigned info, int jg) {
    constexpr bool CHECKED = decltype(chk)::value;
    const bool minimg = CHECKED && (info & ENT_MINIMG) != 0u;
    JAtom<TC> j = load_j(xyzq, lj, jg, jj);
    const V4<TC> vj = (vsl + (long long)jg * 8)[(unsigned)jj];
    if (!minimg) {
      j.p.x += entry_shift(info, 0, ta.L[0]);
      j.p.y += entry_shift(info, 1, ta.L[1]);
      j.p.z += entry_shift(info, 2, ta.L[2]);
    }
    const TC kqj = ta.coul * j.p.w;
    GradSums<TC> b{};
    auto step = [&](int gi, GradSums<TC>& a) {
      const V4<TC> pi = s_p[gi * 8 + ii];
      TC dx = pi.x - j.p.x, dy = pi.y - j.p.y, dz = pi.z - j.p.z;
      if (minimg) {  // uniform over the wave
        dx -= ta.L[0] * rint(dx * ta.invL[0]);
        dy -= ta.L[1] * rint(dy * ta.invL[1]);
        dz -= ta.L[2] * rint(dz * ta.invL[2]);
      }
      TC r2 = dx * dx + dy * dy + dz * dz;
      // padding slots are out of range of everything, unless wrapped by the per-pair minimum image
      bool ok = r2 <= ta.rc2;
      if (minimg) ok = ok && pi.x < (TC)PAD_LIMIT && j.p.x < (TC)PAD_LIMIT;
      if (CHECKED && jg == ci * 4 + gi) ok = ok && jj > ii;
      if (__builtin_amdgcn_ballot_w64(ok) == 0) return;  // no pair of the two groups in range
      bool excl = false;
      if (CHECKED && (info & ENT_EXCL)) excl = is_partner(excl_part, ci * CL + gi * 8 + ii, jg * 8 + jj);
      const V2<TC> li = s_l[gi * 8 + ii];
      const V4<TC> vi = s_v[gi * 8 + ii];
      const TC kqi = ta.coul * pi.w;
      r2 = ok ? r2 : (TC)1e30;
      const TC rinv = rsqrt_t(r2);
      const TC rinv2 = rinv * rinv;
      const TC u = ta.alpha * (r2 * rinv);
      TC ec, em;
      if (CHECKED)
        erfc_exp_excl(u, excl, ec, em);                      // c = erfc - [excluded]
      else
        erfc_exp(u, ec, em);
      const TC grinv3 = fma(c2 * u, em, ec) * rinv * rinv2;  // g / r^3
      const TC kQ = kqi * j.p.w;
      const TC eps4 = CHECKED && excl ? (TC)0 : li.y * j.l.y;
      const TC sg = li.x + j.l.x;
      const TC tq = sg * rinv2;  // s^2 / sigma_ij
      const TC s2 = sg * tq;
      const TC s4 = s2 * s2;
      const TC s6 = s4 * s2;
      const TC ps = s4 * tq;     // s6 / sigma_ij
      const TC a12 = fma((TC)12, s6, (TC)-6);
      const TC e6 = eps4 * s6;
      const TC f = fma(-kQ, grinv3, -e6 * a12 * rinv2);
      const TC h = fma(kQ * rinv2, fma((TC)3, grinv3, ch * em), e6 * fma((TC)168, s6, (TC)-48) * (rinv2 * rinv2));
      const TC okf = ok ? (TC)1 : (TC)0;
      const TC dvx = vi.x - vj.x, dvy = vi.y - vj.y, dvz = vi.z - vj.z;
      const TC sdv = dx * dvx + dy * dvy + dz * dvz;
      const TC cd = okf * fma(gE, f, -sdv * h), cv = okf * f;
      const TC gx = cd * dx - cv * dvx, gy = cd * dy - cv * dvy, gz = cd * dz - cv * dvz;
      a.x += gx;
      a.y += gy;
      a.z += gz;
      b.x -= gx;
      b.y -= gy;
      b.z -= gz;
      // d/dq_i = k q_j (gE c / r + (s.dv) g / r^3), d/dq_j alike with k q_i
      const TC gq = okf * fma(gE, ec * rinv, sdv * grinv3);
      a.q = fma(kqj, gq, a.q);
      b.q = fma(kqi, gq, b.q);
      const TC rs = sdv * rinv2;
      const TC ts = okf * (TC)0.5 * eps4 * ps * fma(gE, a12, rs * fma((TC)144, s6, (TC)-36));
      a.s += ts;
      b.s += ts;
      const TC te = okf * e6 * fma(gE, s6 - (TC)1, rs * a12);
      a.e = fma(te, vi.w, a.e);
      b.e = fma(te, vj.w, b.e);
    };
    if (info & 1u) step(0, a0);
    if (info & 2u) step(1, a1);
    if (info & 4u) step(2, a2);
    if (info & 8u) step(3, a3);
    return b;
  };
  for (int q = qr.q0; q < qr.q1; ++q) {
    const Quad d = load_quad(pl, ci, qr, q);
    auto steps = [&](unsigned info, int jg) {
      return info & (ENT_EXCL | ENT_MINIMG) ? entry(std::true_type{}, info, jg) : entry(std::false_type{}, info, jg);
    };
    const GradSums<TC> f0 = steps(d.i0, d.g0), f1 = steps(d.i1, d.g1), f2 = steps(d.i2, d.g2), f3 = steps(d.i3, d.g3);
    const TC h0 = quad_reduce(f0.x, f1.x, f2.x, f3.x), h1 = quad_reduce(f0.y, f1.y, f2.y, f3.y),
             h2 = quad_reduce(f0.z, f1.z, f2.z, f3.z), h3 = quad_reduce(f0.q, f1.q, f2.q, f3.q),
             h4 = quad_reduce(f0.s, f1.s, f2.s, f3.s), h5 = quad_reduce(f0.e, f1.e, f2.e, f3.e);
    const int g0 = b4 ? d.g1 : d.g0, g1 = b4 ? d.g3 : d.g2;
    unsigned long long* p = gacc + (long long)(b5 ? g1 : g0) * (8 * GN) + (b3 ? 24 : 0) + jj;
    acc_add(p, b3 ? h3 : h0);
    acc_add(p + 8, b3 ? h4 : h1);
    acc_add(p + 16, b3 ? h5 : h2);
  }
  // the i side: 24 sums over jj; lane (ii, jj) adds values jj, jj + 8, jj + 16 (value 6 g + k: slot g * 8 + ii)
  const TC all[24] = {a0.x, a0.y, a0.z, a0.q, a0.s, a0.e, a1.x, a1.y, a1.z, a1.q, a1.s, a1.e,
                      a2.x, a2.y, a2.z, a2.q, a2.s, a2.e, a3.x, a3.y, a3.z, a3.q, a3.s, a3.e};
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    TC v = 0;
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const TC t = octet_sum(all[8 * r + m]);
      v = jj == m ? t : v;
    }
    const int k = jj + 8 * r;
    acc_add(gacc + (long long)ci * (CL * GN) + 8 * k + ii, v);
  }
}

__global__ __launch_bounds__(TFF_WAVE) __attribute__((amdgpu_waves_per_eu(4))) void k_tiles_grad_f32(
    const int* __restrict__ ncl_ptr, PairList pl, int parts, const V4<float>* __restrict__ xyzq,
    const V2<float>* __restrict__ lj, const V4<float>* __restrict__ vsl, const int* __restrict__ excl_part,
    TileArgs<float> ta, const double* __restrict__ gE_ptr, unsigned long long* __restrict__ gacc) {
  grad_body<float>(ncl_ptr, pl, parts, xyzq, lj, vsl, excl_part, ta, gE_ptr, gacc);
}
__global__ __launch_bounds__(TFF_WAVE) void k_tiles_grad_f64(
    const int* __restrict__ ncl_ptr, PairList pl, int parts, const V4<double>* __restrict__ xyzq,
    const V2<double>* __restrict__ lj, const V4<double>* __restrict__ vsl, const int* __restrict__ excl_part,
    TileArgs<double> ta, const double* __restrict__ gE_ptr, unsigned long long* __restrict__ gacc) {
  grad_body<double>(ncl_ptr, pl, parts, xyzq, lj, vsl, excl_part, ta, gE_ptr, gacc);
}

// ---------------------------------------------------------------- 5. PME on cluster slots
// Owner-computes spreading: one workgroup per BR^3 block ("brick") of grid points.  The
// workgroup lists the clusters whose stencils can reach its brick (column neighbourhood,
// circular interval tests in grid units), accumulates their charges into the brick in LDS
// with int64 fixed-point atomics (order independent), then stores the brick: every grid
// point is written once, so the grid needs neither zeroing nor global atomics.
constexpr int BR = 8;
// A brick's grid points in LDS (the spread kernels): x fastest, rows of BR + 1 and planes of
// (BR + 1) BR + 1 int64 words, so that lanes adding to points at other x, y or z fall on different
// banks (x slowest without padding put every x of a row on one bank: 512 bytes apart).  Measured at
// 96k atoms, the list spread alone: 34.2 us against 41.1.
constexpr int SQ_Y = BR + 1, SQ_Z = SQ_Y * BR + 1;
constexpr int BRICK_MAXC = 1024;
constexpr int SPREAD_CHUNK = 32;  // candidate clusters compacted per round
constexpr int SPREAD_MAXCOL = 64; // candidate columns scanned per round

// Charge-grid fixed point: float mode scales by 2^28 and converts through int32 (a spline-weighted
// charge |q M M M| < 8 e, i.e. |q| < ~36 e for order >= 4, fits); float64 mode scales by 2^40.
constexpr double QF_SCALE = 268435456.0;
__device__ __forceinline__ long long grid_fx(float v) { return (long long)__float2int_rn(v * (float)QF_SCALE); }
__device__ __forceinline__ long long grid_fx(double v) { return to_fx(v, Q_SCALE); }
template <typename TC> constexpr double grid_scale() { return sizeof(TC) == 4 ? QF_SCALE : Q_SCALE; }

// x mod K: two conditional corrections each way cover -2K <= x < 3K (grid indices within a
// few stencil widths of [0, K)); anything further out (tiny grids) takes the division
__device__ __forceinline__ int mod_near(int x, int K) {
  x = x < 0 ? x + K : x;
  x = x < 0 ? x + K : x;
  x = x >= K ? x - K : x;
  x = x >= K ? x - K : x;
  if (x < 0 || x >= K) x = ((x % K) + K) % K;
  return x;
}

// do the circular index intervals [lo, lo + len) and [b0, b0 + b) of Z_K intersect?
__device__ __forceinline__ bool circ_overlap(int lo, int len, int b0, int b, int K) {
  if (len >= K) return true;
  const int d1 = mod_near(b0 - lo, K);
  const int d2 = mod_near(lo - b0, K);
  return d1 < len || d2 < b;
}

// grid-index interval [lo, lo + len) touched by the stencils of atoms with scaled coordinate
// in [slo, shi] (spline order P, anchor of the spline weights in tffpme::anchor_axis)
__device__ __forceinline__ void stencil_interval(float slo, float shi, int P, int& lo, int& len) {
  lo = (int)floorf(slo) - P / 2 - 1;
  int hi = (int)ceilf(shi) + P - P / 2;
  len = hi - lo + 1;
}

// Lists in s_list (at most BRICK_MAXC entries; *s_n gets the full count) the clusters whose
// stencils can reach the brick at B0 of extent Bn.  Called by every thread of the workgroup; *s_n
// must be zero (and visible) on entry.
template <int P>
__device__ __forceinline__ void brick_clusters(const float4* __restrict__ bb_c, const float4* __restrict__ bb_h,
                                               const int* __restrict__ col_cl_start, const Geo& g,
                                               const PmeGeom& pg, const int (&B0)[3], const int (&Bn)[3],
                                               int* s_list, int* s_coff, int* s_ccs, int* s_cln, int* s_n) {
  // candidate columns: those whose x-y extent can reach the brick
  const float kl[3] = {(float)(pg.K[0] * g.invL[0]), (float)(pg.K[1] * g.invL[1]), (float)(pg.K[2] * g.invL[2])};
  int c0[2], nc[2];
  for (int a = 0; a < 2; ++a) {
    double lo = (B0[a] - P / 2 - 2) * g.L[a] / pg.K[a];
    double hi = (B0[a] + Bn[a] + P / 2 + 2) * g.L[a] / pg.K[a];
    int cl = (int)floor(lo / g.colw[a]), ch = (int)floor(hi / g.colw[a]);
    c0[a] = cl;
    nc[a] = ch - cl + 1 < g.ncol[a] ? ch - cl + 1 : g.ncol[a];
  }
  const int ncand_cols = nc[0] * nc[1];
  // the brick's z window (stencil reach plus two grid points), as up to two intervals of [0, L)
  const double zw_lo = (B0[2] - P / 2 - 2) * g.L[2] / pg.K[2];
  const double zw_hi = (B0[2] + Bn[2] + P / 2 + 2) * g.L[2] / pg.K[2];
  const bool zall = zw_hi - zw_lo >= g.L[2];
  const float za0 = zw_lo < 0 ? 0.f : (float)zw_lo, zb0 = zw_hi > g.L[2] ? (float)g.L[2] : (float)zw_hi;
  const bool zwrap = !zall && (zw_lo < 0 || zw_hi > g.L[2]);
  const float za1 = zw_lo < 0 ? (float)(zw_lo + g.L[2]) : 0.f;          // second interval [za1, zb1]
  const float zb1 = zw_lo < 0 ? (float)g.L[2] : (float)(zw_hi - g.L[2]);
  // the candidate columns' cluster sub-ranges inside that window (clusters of a column are z
  // ordered: binary searches, one thread per column), scanned into one flat range (columns in
  // groups of SPREAD_MAXCOL), then every candidate cluster tested in one pass
  for (int g0 = 0; g0 < ncand_cols; g0 += SPREAD_MAXCOL) {
    const int ngc = ncand_cols - g0 < SPREAD_MAXCOL ? ncand_cols - g0 : SPREAD_MAXCOL;
    if (threadIdx.x < ngc) {
      const int cc = g0 + threadIdx.x;
      int xx = (c0[0] + cc / nc[1]) % g.ncol[0];
      if (xx < 0) xx += g.ncol[0];
      int yy = (c0[1] + cc % nc[1]) % g.ncol[1];
      if (yy < 0) yy += g.ncol[1];
      const int col = xx * g.ncol[1] + yy;
      const int cs = col_cl_start[col], ce = col_cl_start[col + 1];
      // first cluster with z max >= a, last cluster with z min <= b (both monotone in the column)
      auto first_ge = [&](float a) {
        int lo = cs, hi = ce;
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (bb_c[mid].z + bb_h[mid].z >= a) hi = mid; else lo = mid + 1;
        }
        return lo;
      };
      auto last_le = [&](float b) {
        int lo = cs - 1, hi = ce - 1;
        while (lo < hi) {
          const int mid = (lo + hi + 1) >> 1;
          if (bb_c[mid].z - bb_h[mid].z <= b) lo = mid; else hi = mid - 1;
        }
        return lo;
      };
      int r0s = cs, r0e = ce, r1s = 0, r1e = 0;  // [start, end) of up to two ranges
      if (!zall && cs < ce) {
        if (!zwrap) {
          r0s = first_ge(za0);
          r0e = last_le(zb0) + 1;
        } else {
          // [0, b] at the column's start, [a, L) at its end; merged when they meet
          const int l0 = last_le(zw_lo < 0 ? zb0 : zb1) + 1;
          const int f1 = first_ge(zw_lo < 0 ? za1 : za0);
          if (f1 <= l0) {
            r0s = cs;
            r0e = ce;
          } else {
            r0s = cs;
            r0e = l0;
            r1s = f1;
            r1e = ce;
          }
        }
      }
      s_ccs[2 * threadIdx.x] = r0s;
      s_cln[2 * threadIdx.x] = r0e > r0s ? r0e - r0s : 0;
      s_ccs[2 * threadIdx.x + 1] = r1s;
      s_cln[2 * threadIdx.x + 1] = r1e > r1s ? r1e - r1s : 0;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      int run = 0;
      for (int t = 0; t < 2 * ngc; ++t) {
        s_coff[t] = run;
        run += s_cln[t];
      }
      s_coff[2 * ngc] = run;
    }
    __syncthreads();
    const int nent = 2 * ngc;
    const int total = s_coff[nent];
    for (int k = threadIdx.x; k < total; k += blockDim.x) {
      int lo = 0, hi = nent - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (s_coff[mid] <= k) lo = mid; else hi = mid - 1;
      }
      const int c = s_ccs[lo] + (k - s_coff[lo]);
      const float4 cc4 = bb_c[c], hh4 = bb_h[c];
      const float cv[3] = {cc4.x, cc4.y, cc4.z}, hv[3] = {hh4.x, hh4.y, hh4.z};
      bool ok = true;
      for (int a = 0; a < 3; ++a) {
        int lo2, len;
        stencil_interval((cv[a] - hv[a]) * kl[a], (cv[a] + hv[a]) * kl[a], P, lo2, len);
        ok = ok && circ_overlap(lo2, len, B0[a], Bn[a], pg.K[a]);
      }
      if (ok) {
        const int q = atomicAdd(s_n, 1);
        if (q < BRICK_MAXC) s_list[q] = c;
      }
    }
    __syncthreads();
  }
}

// DIPOLE: instead of the charges, spread the dipoles q_i v_i . grad_r theta_i(m) (the grid of the
// force-matching backward), from per-slot vectors vsl and the Cartesian-to-grid scale jsc = K / L.
template <typename TC, int P, bool DIPOLE>
__global__ __launch_bounds__(256) void k_spread_bricks(const int* __restrict__ ncl_ptr, const V4<TC>* __restrict__ xyzq,
                                                       const int* __restrict__ slot_orig, const float4* __restrict__ bb_c,
                                                       const float4* __restrict__ bb_h,
                                                       const int* __restrict__ col_cl_start, Geo g, PmeGeom pg,
                                                       unsigned long long* __restrict__ grid, int* __restrict__ status,
                                                       const V4<TC>* __restrict__ vsl, V4<TC> jsc) {
  __shared__ unsigned long long s_q[SQ_Z * BR];
  __shared__ int s_list[BRICK_MAXC];
  __shared__ V4<TC> s_pos[SPREAD_CHUNK * CL];
  __shared__ int s_slot[DIPOLE ? SPREAD_CHUNK * CL : 1];
  __shared__ int s_coff[2 * SPREAD_MAXCOL + 1], s_ccs[2 * SPREAD_MAXCOL], s_cln[2 * SPREAD_MAXCOL];
  __shared__ int s_n, s_na;
  const int K0 = pg.K[0], K1 = pg.K[1], K2 = pg.K[2];
  const int nbx = (K0 + BR - 1) / BR, nby = (K1 + BR - 1) / BR, nbz = (K2 + BR - 1) / BR;
  const int bid = blockIdx.x;
  if (bid >= nbx * nby * nbz) return;
  const int bz = bid % nbz, by = (bid / nbz) % nby, bx = bid / (nbz * nby);
  const int B0[3] = {bx * BR, by * BR, bz * BR};
  const int Bn[3] = {K0 - B0[0] < BR ? K0 - B0[0] : BR, K1 - B0[1] < BR ? K1 - B0[1] : BR,
                     K2 - B0[2] < BR ? K2 - B0[2] : BR};
  for (int k = threadIdx.x; k < SQ_Z * BR; k += blockDim.x) s_q[k] = 0ull;
  if (threadIdx.x == 0) s_n = 0;
  __syncthreads();
  brick_clusters<P>(bb_c, bb_h, col_cl_start, g, pg, B0, Bn, s_list, s_coff, s_ccs, s_cln, &s_n);
  int ncand = s_n;
  if (ncand > BRICK_MAXC) {
    if (threadIdx.x == 0) atomicOr(status, TFF_FUSED_BRICK_OVERFLOW);
    ncand = BRICK_MAXC;
  }
  // Candidate clusters in chunks of SPREAD_CHUNK: the slots whose stencil reaches the brick are
  // compacted into s_pos (a cheap anchor test), then one lane per compacted slot adds its P^3
  // contributions to the brick (LDS int64 atomics: the sums do not depend on the list order).
  for (int r0 = 0; r0 < ncand; r0 += SPREAD_CHUNK) {
    if (threadIdx.x == 0) s_na = 0;
    __syncthreads();
    const int nslot = (ncand - r0 < SPREAD_CHUNK ? ncand - r0 : SPREAD_CHUNK) * CL;
    for (int k = threadIdx.x; k < nslot; k += blockDim.x) {
      const int sl = s_list[r0 + k / CL] * CL + (k % CL);
      if (slot_orig[sl] < 0) continue;
      const V4<TC> p = xyzq[sl];
      const double rr[3] = {(double)p.x, (double)p.y, (double)p.z};
      bool ov = true;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const double sa = (rr[0] * pg.inv[a] + rr[1] * pg.inv[3 + a] + rr[2] * pg.inv[6 + a]) * (double)pg.K[a];
        int base;
        double t;
        anchor_axis(sa, pg.K[a], P, base, t);
        ov = ov && circ_overlap(base, P, B0[a], Bn[a], pg.K[a]);
      }
      if (ov) {
        const int idx = atomicAdd(&s_na, 1);
        s_pos[idx] = p;
        if (DIPOLE) s_slot[idx] = sl;
      }
    }
    __syncthreads();
    const int na = s_na;
    for (int k = threadIdx.x; k < na; k += blockDim.x) {
      const V4<TC> p = s_pos[k];
      TC Mv[3][P], dM[3][P];
      int base[3];
      unsigned int inmask[3];
      const double rr[3] = {(double)p.x, (double)p.y, (double)p.z};
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const double sa = (rr[0] * pg.inv[a] + rr[1] * pg.inv[3 + a] + rr[2] * pg.inv[6 + a]) * (double)pg.K[a];
        double t;
        anchor_axis(sa, pg.K[a], P, base[a], t);
        spline_weights<TC, P>((TC)t, Mv[a], dM[a]);
        unsigned int m = 0;
#pragma unroll
        for (int q = 0; q < P; ++q) {
          int gk = base[a] + q;
          gk = gk >= pg.K[a] ? gk - pg.K[a] : gk;
          if (gk >= B0[a] && gk < B0[a] + Bn[a]) m |= 1u << q;
        }
        inmask[a] = m;
      }
      const TC qi = p.w;
      TC wv[3] = {(TC)0, (TC)0, (TC)0};
      if (DIPOLE) {
        const V4<TC> vv = vsl[s_slot[k]];
        // d theta / d r_a = -K_a / L_a M'_a ... (the weights fall as the scaled coordinate grows)
        wv[0] = -qi * vv.x * jsc.x;
        wv[1] = -qi * vv.y * jsc.y;
        wv[2] = -qi * vv.z * jsc.z;
      }
#pragma unroll
      for (int ka = 0; ka < P; ++ka) {
        if (!((inmask[0] >> ka) & 1u)) continue;
        int gx = base[0] + ka;
        gx = gx >= K0 ? gx - K0 : gx;
        const TC wa = qi * Mv[0][ka];
#pragma unroll
        for (int kb = 0; kb < P; ++kb) {
          if (!((inmask[1] >> kb) & 1u)) continue;
          int gy = base[1] + kb;
          gy = gy >= K1 ? gy - K1 : gy;
          const TC wab = wa * Mv[1][kb];
          // dipole: value(kc) = cz * M_z(kc) + dz * M_z'(kc)
          const TC cz = DIPOLE ? wv[0] * dM[0][ka] * Mv[1][kb] + wv[1] * Mv[0][ka] * dM[1][kb] : (TC)0;
          const TC dz = DIPOLE ? wv[2] * Mv[0][ka] * Mv[1][kb] : (TC)0;
          unsigned long long* row = s_q + (gy - B0[1]) * SQ_Y + (gx - B0[0]);
#pragma unroll
          for (int kc = 0; kc < P; ++kc) {
            if (!((inmask[2] >> kc) & 1u)) continue;
            int gz = base[2] + kc;
            gz = gz >= K2 ? gz - K2 : gz;
            if (DIPOLE)
              atomicAdd(&row[(gz - B0[2]) * SQ_Z], (unsigned long long)to_fx((double)(cz * Mv[2][kc] + dz * dM[2][kc]),
                                                                            Q_SCALE));
            else
              atomicAdd(&row[(gz - B0[2]) * SQ_Z], (unsigned long long)grid_fx(wab * Mv[2][kc]));
          }
        }
      }
    }
    __syncthreads();
  }
  __syncthreads();
  for (int k = threadIdx.x; k < BR * BR * BR; k += blockDim.x) {
    const int lz = k % BR, ly = (k / BR) % BR, lx = k / (BR * BR);
    if (lx < Bn[0] && ly < Bn[1] && lz < Bn[2])
      grid[((long long)(B0[0] + lx) * K1 + (B0[1] + ly)) * K2 + (B0[2] + lz)] = s_q[lz * SQ_Z + ly * SQ_Y + lx];
  }
}

// ---- charge spread of the float path: per-slot spline tables + home-brick lists
// A slot's home brick is the brick holding its stencil base (the grid point of its first spline
// weight on every axis).  k_slot_splines evaluates each slot's spline weights once (the
// arithmetic of k_spread_bricks and k_gather_slots) into wts[sl * WST ...] = M(t_x + k),
// M(t_y + k), M(t_z + k) for k < P, then q, and appends (slot, packed base) to its home brick's
// list (capacity cap per brick; the lanes of a wave that share a home brick reserve one range
// with one atomic).  k_spread_lists then spreads each brick from the lists of the home bricks whose
// stencils can reach it: no search over clusters.  Needs P <= 6 and BR + P <= K_a <= 1023 (every
// stencil meets a brick in one run of grid points; bases fit 10 bits).
template <int P> constexpr int spline_stride() { return (3 * P + 1 + 3) & ~3; }
constexpr int LIST_WST = 20;  // spline_stride<6>(): the table stride of the largest order served

struct BrickGrid {
  int nb[3];  // bricks per axis
  int cap;    // list entries per brick
};

template <int P>
__global__ __launch_bounds__(FB) void k_slot_splines(const int* __restrict__ ncl_ptr, const V4<float>* __restrict__ xyzq,
                                                     const int* __restrict__ slot_orig, PmeGeom pg, BrickGrid bg,
                                                     float* __restrict__ wts, int* __restrict__ bcount,
                                                     int2* __restrict__ blist, int* __restrict__ status) {
  const int sl = blockIdx.x * FB + threadIdx.x;
  const int lane = threadIdx.x & (TFF_WAVE - 1);
  const bool valid = sl < *ncl_ptr * CL && slot_orig[sl] >= 0;
  int hb = -1, packed = 0;
  if (valid) {
    const V4<float> p = xyzq[sl];
    const double rr[3] = {(double)p.x, (double)p.y, (double)p.z};
    int base[3];
    float* w = wts + (size_t)sl * LIST_WST;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const double sa = (rr[0] * pg.inv[a] + rr[1] * pg.inv[3 + a] + rr[2] * pg.inv[6 + a]) * (double)pg.K[a];
      double t;
      float Mv[P], dM[P];
      anchor_axis(sa, pg.K[a], P, base[a], t);
      spline_weights<float, P>((float)t, Mv, dM);
#pragma unroll
      for (int k = 0; k < P; ++k) w[a * P + k] = Mv[k];
    }
    w[3 * P] = p.w;
    hb = ((base[0] / BR) * bg.nb[1] + base[1] / BR) * bg.nb[2] + base[2] / BR;
    packed = base[0] | (base[1] << 10) | (base[2] << 20);
  }
  // wave-aggregated append: group the lanes by home brick (ballots only), then every group's first
  // lane reserves the group's range, all groups at once
  unsigned long long todo = __ballot(valid), grp = 0;
  int leader = 0;
  while (todo) {
    const int l = __ffsll((long long)todo) - 1;
    const int h = __shfl(hb, l, TFF_WAVE);
    const unsigned long long m = __ballot(valid && hb == h);
    todo &= ~m;
    if (valid && hb == h) {
      grp = m;
      leader = l;
    }
  }
  int start = 0;
  if (valid && lane == leader) start = atomicAdd(&bcount[hb], __popcll(grp));
  start = __shfl(start, leader, TFF_WAVE);
  if (valid) {
    const int r = start + __popcll(grp & ((1ull << lane) - 1ull));
    if (r < bg.cap)
      blist[(long long)hb * bg.cap + r] = make_int2(sl, packed);
    else
      atomicOr(status, TFF_FUSED_BRICK_OVERFLOW);
  }
}

// Charge spread from the home-brick lists: one workgroup per BR^3 brick, in rounds of up to 256
// listed slots.  Each thread tests one slot's stencil against the brick (one run of grid points per
// axis) and compacts into LDS the slot's weights over its in-brick runs (q M_x, M_y, M_z, zero past
// the run) and the runs' starts and lengths.  Then lane k takes x point k % P of compacted slot
// k / P and adds its y-z box of points ((q M_x M_y) M_z, the products k_spread_bricks forms) to the
// brick in LDS with int64 fixed-point atomics.  Integer sums do not depend on the order, so the grid
// equals k_spread_bricks' bit for bit; the brick is stored once, so the grid needs neither clearing
// nor global atomics.
// DIPOLE: the dipoles q_i v_i . grad_r theta_i(m) of the force-matching backward instead of the charges
// (per-slot vectors vsl, Cartesian-to-grid scale jsc = K / L), from the lists that the charge spread
// left.  A point gets (X1 Y1 + X2 Y2) Z1 + X2 Y1 Z2 with X1 = w_x M'_x, X2 = M_x, Y1 = M_y, Y2 = w_y M'_y,
// Z1 = M_z, Z2 = w_z M'_z; weights and derivatives are evaluated again per brick that a stencil meets
// (some 4 times; a table of both would be read as often).  Charges: wts holds the weights.
// 96k water atoms, order 5, 96^3: the dipoles alone 44 us, beside the backward's pair kernel 188; k_spread_bricks (a
// search over clusters per brick, one lane per slot, a general double-to-int64 conversion per point) took 251
// beside it, the force-matching step 657 us instead of 644.
constexpr int LIST_ROUND = 256;
template <int P, bool DIPOLE>
__global__ __launch_bounds__(LIST_ROUND) void k_spread_lists(const float* __restrict__ wts,
                                                             const int* __restrict__ bcount,
                                                             const int2* __restrict__ blist, BrickGrid bg,
                                                             PmeGeom pg, unsigned long long* __restrict__ grid,
                                                             const V4<float>* __restrict__ xyzq,
                                                             const V4<float>* __restrict__ vsl, V4<float> jsc) {
  constexpr int NT = LIST_ROUND;
  constexpr int NW = DIPOLE ? 6 * P : 3 * P;  // weights per compacted slot: of its runs, then the runs
  constexpr int REC = (NW + 1 + 3) & ~3;
  constexpr int NC = DIPOLE ? 1 : 2;          // candidates per thread and pass
  __shared__ unsigned long long s_q[SQ_Z * BR];
  __shared__ __align__(16) float s_w[NT][REC];
  __shared__ int s_hoff[28], s_hid[27], s_cnt[27];
  __shared__ int s_na, s_nh;
  const int K0 = pg.K[0], K1 = pg.K[1], K2 = pg.K[2];
  const int bid = blockIdx.x;
  if (bid >= bg.nb[0] * bg.nb[1] * bg.nb[2]) return;
  const int bi[3] = {bid / (bg.nb[2] * bg.nb[1]), (bid / bg.nb[2]) % bg.nb[1], bid % bg.nb[2]};
  const int Ks[3] = {K0, K1, K2};
  int B0[3], Bn[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    B0[a] = bi[a] * BR;
    Bn[a] = Ks[a] - B0[a] < BR ? Ks[a] - B0[a] : BR;
  }
  for (int k = threadIdx.x; k < SQ_Z * BR; k += NT) s_q[k] = 0ull;
  // home bricks whose slots' stencils can reach this brick: per axis the distinct h among b, b - 1,
  // b - 2 (mod the brick count) whose base range plus stencil meets the brick; lane t < 27 of the
  // first wave takes combination t and loads its list length (the other waves skip this scalar
  // work: the CU's scalar unit is shared)
  const int t = threadIdx.x;
  if (t < TFF_WAVE) {
    int hl[3][3], hn[3] = {0, 0, 0};
    for (int a = 0; a < 3; ++a) {
      if (Ks[a] % BR == 0 && bg.nb[a] >= 2) {
        // full bricks: the brick itself and the one below (P <= BR + 1)
        hl[a][0] = bi[a];
        hl[a][1] = bi[a] > 0 ? bi[a] - 1 : bg.nb[a] - 1;
        hn[a] = 2;
        continue;
      }
      for (int d = 0; d < 3; ++d) {
        int h = bi[a] - d;
        while (h < 0) h += bg.nb[a];
        bool dup = false;
        for (int e = 0; e < hn[a]; ++e) dup = dup || hl[a][e] == h;
        const int hB = Ks[a] - h * BR < BR ? Ks[a] - h * BR : BR;
        if (!dup && circ_overlap(h * BR, hB + P - 1, B0[a], Bn[a], Ks[a])) hl[a][hn[a]++] = h;
      }
    }
    const int nh = hn[0] * hn[1] * hn[2];
    if (t < nh) {
      const int x = t / (hn[1] * hn[2]), y = (t / hn[2]) % hn[1], z = t % hn[2];
      const int h = (hl[0][x] * bg.nb[1] + hl[1][y]) * bg.nb[2] + hl[2][z];
      const int c = bcount[h];
      s_hid[t] = h;
      s_cnt[t] = c < bg.cap ? c : bg.cap;
    }
    if (t == 0) s_nh = nh;
  }
  {
    __syncthreads();
    const int nh = s_nh;
    if (t == 0) {
      int run = 0;
      for (int k = 0; k < nh; ++k) {
        s_hoff[k] = run;
        run += s_cnt[k];
      }
      s_hoff[nh] = run;
    }
    __syncthreads();
  }
  const int nh = s_nh, total = s_hoff[nh];
  // candidates in passes of NC NT: each thread loads and tests its two (k and k + NT) and loads the
  // spline tables of those that hit before the first is spread, so the global loads of both rounds
  // overlap
  for (int p0 = 0; p0 < total; p0 += NC * NT) {
    float rec2[NC][REC];
    bool hit2[NC] = {};
    int2 e2[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int k = p0 + c * NT + threadIdx.x;
      e2[c] = make_int2(0, 0);
      if (k < total) {
        int hi = 0;
        for (int j = 1; j < nh; ++j) hi += s_hoff[j] <= k ? 1 : 0;
        e2[c] = blist[(long long)s_hid[hi] * bg.cap + (k - s_hoff[hi])];
      }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int k = p0 + c * NT + threadIdx.x;
      if (k >= total) continue;
      const int2 e = e2[c];
      const int bs[3] = {e.y & 1023, (e.y >> 10) & 1023, (e.y >> 20) & 1023};
      bool hit = true;
      int q0[3], l0[3], nr[3];
      bool small = true;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        // the stencil [bs, bs + P) and the brick [B0, B0 + Bn) as arcs of Z_K: one common run
        int d = B0[a] - bs[a];
        d = d < 0 ? d + Ks[a] : d;  // brick start relative to the stencil start
        if (d < P) {
          q0[a] = d;
          l0[a] = 0;
          nr[a] = P - d < Bn[a] ? P - d : Bn[a];
        } else {
          int f = bs[a] - B0[a];
          f = f < 0 ? f + Ks[a] : f;  // stencil start relative to the brick start
          q0[a] = 0;
          l0[a] = f;
          nr[a] = f < Bn[a] ? (P < Bn[a] - f ? P : Bn[a] - f) : 0;
        }
        hit = hit && nr[a] > 0;
      }
      if (!hit) continue;
      hit2[c] = true;
      if constexpr (DIPOLE) {
        const V4<float> p = xyzq[e.x], vv = vsl[e.x];
        const double rr[3] = {(double)p.x, (double)p.y, (double)p.z};
        // d theta / d r_a = -K_a / L_a M'_a ... (the weights fall as the scaled coordinate grows)
        const float wv[3] = {-p.w * vv.x * jsc.x, -p.w * vv.y * jsc.y, -p.w * vv.z * jsc.z};
        // contributions below 2^10 (weights and derivatives are at most 1) convert by mantissa
        small = fabsf(wv[0]) + fabsf(wv[1]) + fabsf(wv[2]) < 1024.0f;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const double sa = (rr[0] * pg.inv[a] + rr[1] * pg.inv[3 + a] + rr[2] * pg.inv[6 + a]) * (double)pg.K[a];
          int base;
          double t;
          float Mv[P], dM[P];
          anchor_axis(sa, pg.K[a], P, base, t);
          spline_weights<float, P>((float)t, Mv, dM);
#pragma unroll
          for (int i = 0; i < P; ++i) {
            float m = 0.f, d = 0.f;
#pragma unroll
            for (int kk = 0; kk < P; ++kk)
              if (i < nr[a] && q0[a] + i == kk) {
                m = Mv[kk];
                d = wv[a] * dM[kk];
              }
            rec2[c][2 * a * P + i] = m;
            rec2[c][(2 * a + 1) * P + i] = d;
          }
        }
      } else {
        const float* src = wts + (size_t)e.x * LIST_WST;
        float tb[3 * P + 1];
#pragma unroll
        for (int i = 0; i <= 3 * P; ++i) tb[i] = src[i];
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
          for (int i = 0; i < P; ++i) {
            float v = 0.f;
#pragma unroll
            for (int kk = 0; kk < P; ++kk)
              if (i < nr[a] && q0[a] + i == kk) v = tb[a * P + kk];
            // z weights carry the fixed-point scale (a power of two: (a b) 2^28 = a (b 2^28) exactly)
            rec2[c][a * P + i] = a == 0 ? tb[3 * P] * v : (a == 2 ? v * (float)QF_SCALE : v);
          }
      }
      rec2[c][NW] = __int_as_float(l0[0] | (l0[1] << 3) | (l0[2] << 6) | (nr[0] << 9) | (nr[1] << 13) |
                                   (nr[2] << 17) | (small ? 1 << 21 : 0));
#pragma unroll
      for (int i = NW + 1; i < REC; ++i) rec2[c][i] = 0.f;
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (p0 + c * NT >= total) break;
      if (threadIdx.x == 0) s_na = 0;
      __syncthreads();
      // 1. compact
      if (hit2[c]) {
        const int idx = atomicAdd(&s_na, 1);
        float4* dst = reinterpret_cast<float4*>(s_w[idx]);
#pragma unroll
        for (int i = 0; i < REC / 4; ++i)
          dst[i] = make_float4(rec2[c][4 * i], rec2[c][4 * i + 1], rec2[c][4 * i + 2], rec2[c][4 * i + 3]);
      }
      __syncthreads();
      // 2. lane k: x point k % P of compacted slot k / P, its y-z box
      const int nlanes = s_na * P;
      for (int k = threadIdx.x; k < nlanes; k += NT) {
        const int t = k / P, ix = k - t * P;
        const float* w = s_w[t];
        const int meta = __float_as_int(w[NW]);
        const int nx = (meta >> 9) & 15, ny = (meta >> 13) & 15, nz = (meta >> 17) & 15;
        if (ix >= nx) continue;
        const int lx = (meta & 7) + ix, ly0 = (meta >> 3) & 7, lz0 = (meta >> 6) & 7;
        if constexpr (DIPOLE) {
          const float x2 = w[ix], x1 = w[P + ix];
          float z1[P], z2[P];
#pragma unroll
          for (int i = 0; i < P; ++i) {
            z1[i] = w[4 * P + i];
            z2[i] = w[5 * P + i];
          }
          const bool by_mantissa = (meta >> 21) & 1;
#pragma unroll
          for (int iy = 0; iy < P; ++iy) {
            if (iy >= ny) break;
            const float y1 = w[2 * P + iy], y2 = w[3 * P + iy];
            const float cxy = fmaf(x1, y1, x2 * y2), dxy = x2 * y1;
            unsigned long long* row = s_q + lz0 * SQ_Z + (ly0 + iy) * SQ_Y + lx;
#pragma unroll
            for (int iz = 0; iz < P; ++iz) {
              const double v = (double)fmaf(cxy, z1[iz], dxy * z2[iz]);
              unsigned long long b;
              if (__builtin_expect(by_mantissa, 1))
                b = (unsigned long long)(__double_as_longlong(fma(v, Q_SCALE, 6755399441055744.0)) -
                                         0x4338000000000000LL);
              else
                b = (unsigned long long)to_fx(v, Q_SCALE);
              if (iz < nz) atomicAdd(&row[iz * SQ_Z], b);
            }
          }
        } else {
          const float wx = w[ix];
          float wy[P], wz[P];
#pragma unroll
          for (int i = 0; i < P; ++i) {
            wy[i] = w[P + i];
            wz[i] = w[2 * P + i];
          }
#pragma unroll
          for (int iy = 0; iy < P; ++iy) {
            if (iy >= ny) break;
            const float wab = wx * wy[iy];
            long long v[P];
#pragma unroll
            for (int iz = 0; iz < P; ++iz) v[iz] = (long long)__float2int_rn(wab * wz[iz]);
            unsigned long long* row = s_q + lz0 * SQ_Z + (ly0 + iy) * SQ_Y + lx;
#pragma unroll
            for (int iz = 0; iz < P; ++iz)
              if (iz < nz) atomicAdd(&row[iz * SQ_Z], (unsigned long long)v[iz]);
          }
        }
      }
      __syncthreads();
    }
  }
  for (int k = threadIdx.x; k < BR * BR * BR; k += NT) {
    const int lz = k % BR, ly = (k / BR) % BR, lx = k / (BR * BR);
    if (lx < Bn[0] && ly < Bn[1] && lz < Bn[2])
      grid[((long long)(B0[0] + lx) * K1 + (B0[1] + ly)) * K2 + (B0[2] + lz)] = s_q[lz * SQ_Z + ly * SQ_Y + lx];
  }
}

template <typename TC, int P>
__global__ __launch_bounds__(FB) void k_gather_slots(const int* __restrict__ ncl_ptr, const TC* __restrict__ phi_grid,
                                                     const V4<TC>* __restrict__ xyzq, const int* __restrict__ slot_orig,
                                                     PmeGeom g, double coul, unsigned long long* __restrict__ facc) {
  int sl = blockIdx.x * FB + threadIdx.x;
  if (sl >= *ncl_ptr * CL || slot_orig[sl] < 0) return;
  V4<TC> p = xyzq[sl];
  TC Mv[3][P], dM[3][P];
  int base[3];
  const double r[3] = {(double)p.x, (double)p.y, (double)p.z};
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    double s = (r[0] * g.inv[a] + r[1] * g.inv[3 + a] + r[2] * g.inv[6 + a]) * (double)g.K[a];
    double t;
    anchor_axis(s, g.K[a], P, base[a], t);
    spline_weights<TC, P>((TC)t, Mv[a], dM[a]);
  }
  const int K1 = g.K[1], K2 = g.K[2];
  TC du0 = 0, du1 = 0, du2 = 0;
  int gx = base[0];
#pragma unroll 1
  for (int a = 0; a < P; ++a) {
    int gy = base[1];
    TC t0 = 0, t1 = 0, t2 = 0;
#pragma unroll
    for (int b = 0; b < P; ++b) {
      const TC* row = phi_grid + ((long long)gx * K1 + gy) * K2;
      int gz = base[2];
      TC s0 = 0, s1 = 0;
#pragma unroll
      for (int c = 0; c < P; ++c) {
        TC v = row[gz];
        s0 += v * Mv[2][c];
        s1 += v * dM[2][c];
        gz = gz + 1 == K2 ? 0 : gz + 1;
      }
      t0 += Mv[1][b] * s0;
      t1 += dM[1][b] * s0;
      t2 += Mv[1][b] * s1;
      gy = gy + 1 == K1 ? 0 : gy + 1;
    }
    du0 += dM[0][a] * t0;
    du1 += Mv[0][a] * t1;
    du2 += Mv[0][a] * t2;
    gx = gx + 1 == g.K[0] ? 0 : gx + 1;
  }
  // dE/dr = k q grad phi; weights depend on -s, ds_a/dr_j = K_a inv[j][a]
  const double kq = coul * (double)p.w;
  const double d0 = -(double)du0 * g.K[0], d1 = -(double)du1 * g.K[1], d2 = -(double)du2 * g.K[2];
  const double gxr = d0 * g.inv[0] + d1 * g.inv[1] + d2 * g.inv[2];
  const double gyr = d0 * g.inv[3] + d1 * g.inv[4] + d2 * g.inv[5];
  const double gzr = d0 * g.inv[6] + d1 * g.inv[7] + d2 * g.inv[8];
  // force = -dE/dr into the slot's reciprocal-space accumulator (one thread per slot; the pair
  // kernel, which may run concurrently, adds into the other accumulator)
  facc[3 * sl + 0] = (unsigned long long)to_fx(-kq * gxr, F_SCALE);
  facc[3 * sl + 1] = (unsigned long long)to_fx(-kq * gyr, F_SCALE);
  facc[3 * sl + 2] = (unsigned long long)to_fx(-kq * gzr, F_SCALE);
}

// Backward gather, one thread per slot: from the potential grid Phi (of the charges) and Psi (of
// the dipoles q v . grad theta), the reciprocal-space parts
//   dL/dq_i = k [gE phi(r_i) - v_i . grad phi(r_i) - psi(r_i)],
//   dL/dr_i = k q_i [gE grad phi(r_i) - H_phi(r_i) v_i - grad psi(r_i)]
// (orthorhombic box: d s_a / d r_a = K_a / L_a), as int64 fixed point into gpme (4 per slot).
template <typename TC, int P>
__global__ __launch_bounds__(FB) void k_gather_grad(const int* __restrict__ ncl_ptr, const TC* __restrict__ phi_grid,
                                                    const TC* __restrict__ psi_grid, const V4<TC>* __restrict__ xyzq,
                                                    const V4<TC>* __restrict__ vsl, const int* __restrict__ slot_orig,
                                                    PmeGeom g, double coul, const double* __restrict__ gE_ptr,
                                                    unsigned long long* __restrict__ gpme) {
  const int sl = blockIdx.x * FB + threadIdx.x;
  if (sl >= *ncl_ptr * CL || slot_orig[sl] < 0) return;
  const V4<TC> p = xyzq[sl];
  const V4<TC> v = vsl[sl];
  TC M[3][P], D1[3][P], D2[3][P];
  int base[3];
  const double r[3] = {(double)p.x, (double)p.y, (double)p.z};
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double sa = (r[0] * g.inv[a] + r[1] * g.inv[3 + a] + r[2] * g.inv[6 + a]) * (double)g.K[a];
    double t;
    anchor_axis(sa, g.K[a], P, base[a], t);
    spline_weights2<TC, P>((TC)t, M[a], D1[a], D2[a]);
  }
  const int K1 = g.K[1], K2 = g.K[2];
  // separable sums over z, then y, then x (derivatives in t; d/ds = -d/dt)
  double phi = 0, px = 0, py = 0, pz = 0, hxx = 0, hyy = 0, hzz = 0, hxy = 0, hxz = 0, hyz = 0;
  double psi = 0, sx = 0, sy = 0, sz = 0;
  int gx = base[0];
#pragma unroll 1
  for (int a = 0; a < P; ++a) {
    double ty0 = 0, ty1 = 0, ty2 = 0, tz1 = 0, tz2 = 0, tyz = 0, uy0 = 0, uy1 = 0, uz1 = 0;
    int gy = base[1];
#pragma unroll
    for (int b = 0; b < P; ++b) {
      const long long row = ((long long)gx * K1 + gy) * K2;
      double z0 = 0, z1 = 0, z2 = 0, w0 = 0, w1 = 0;
      int gz = base[2];
#pragma unroll
      for (int c = 0; c < P; ++c) {
        const double f = (double)phi_grid[row + gz], q = (double)psi_grid[row + gz];
        z0 += (double)M[2][c] * f;
        z1 += (double)D1[2][c] * f;
        z2 += (double)D2[2][c] * f;
        w0 += (double)M[2][c] * q;
        w1 += (double)D1[2][c] * q;
        gz = gz + 1 == K2 ? 0 : gz + 1;
      }
      const double my = M[1][b], dy = D1[1][b], ddy = D2[1][b];
      ty0 += my * z0;
      ty1 += dy * z0;
      ty2 += ddy * z0;
      tz1 += my * z1;
      tz2 += my * z2;
      tyz += dy * z1;
      uy0 += my * w0;
      uy1 += dy * w0;
      uz1 += my * w1;
      gy = gy + 1 == K1 ? 0 : gy + 1;
    }
    const double mx = M[0][a], dx = D1[0][a], ddx = D2[0][a];
    phi += mx * ty0;
    px += dx * ty0;
    py += mx * ty1;
    pz += mx * tz1;
    hxx += ddx * ty0;
    hyy += mx * ty2;
    hzz += mx * tz2;
    hxy += dx * ty1;
    hxz += dx * tz1;
    hyz += mx * tyz;
    psi += mx * uy0;
    sx += dx * uy0;
    sy += mx * uy1;
    sz += mx * uz1;
    gx = gx + 1 == g.K[0] ? 0 : gx + 1;
  }
  const double j0 = g.K[0] * g.inv[0], j1 = g.K[1] * g.inv[4], j2 = g.K[2] * g.inv[8];
  // Cartesian gradient (first derivatives change sign from t to s) and Hessian
  const double gp[3] = {-px * j0, -py * j1, -pz * j2};
  const double gs[3] = {-sx * j0, -sy * j1, -sz * j2};
  const double H[3][3] = {{hxx * j0 * j0, hxy * j0 * j1, hxz * j0 * j2},
                          {hxy * j0 * j1, hyy * j1 * j1, hyz * j1 * j2},
                          {hxz * j0 * j2, hyz * j1 * j2, hzz * j2 * j2}};
  const double gE = gE_ptr ? gE_ptr[0] : 0.0;
  const double vv[3] = {(double)v.x, (double)v.y, (double)v.z};
  const double q = (double)p.w;
  const double dq = coul * (gE * phi - (vv[0] * gp[0] + vv[1] * gp[1] + vv[2] * gp[2]) - psi);
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double hv = H[a][0] * vv[0] + H[a][1] * vv[1] + H[a][2] * vv[2];
    gpme[4 * (long long)sl + a] = (unsigned long long)to_fx(coul * q * (gE * gp[a] - hv - gs[a]), F_SCALE);
  }
  gpme[4 * (long long)sl + 3] = (unsigned long long)to_fx(dq, F_SCALE);
}

// word k of the slots, summed by the first wave of a workgroup (the result is valid there)
__device__ __forceinline__ long long slot_sum(const ESlots& es, int k) {
  long long v = 0;
  if (threadIdx.x < TFF_WAVE) {
    for (int j = threadIdx.x; j < es.n; j += TFF_WAVE) v += (long long)es.p[8 * j + k];
    for (int o = TFF_WAVE / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, TFF_WAVE);
  }
  return v;
}

// gradients back in the caller's atom order (pair + reciprocal accumulators; self energy
// -k alpha / sqrt(pi) sum q^2 contributes gE * (-2 k alpha / sqrt(pi)) q_i to dL/dq_i)
template <typename TI>
__global__ __launch_bounds__(FB) void k_finalize_grad(const int* __restrict__ ncl_ptr, const int* __restrict__ slot_orig,
                                                      const unsigned long long* __restrict__ gacc,
                                                      const unsigned long long* __restrict__ gpme,
                                                      const TI* __restrict__ q, double coul, double alpha,
                                                      const double* __restrict__ gE_ptr, TI* __restrict__ dr,
                                                      TI* __restrict__ dq, TI* __restrict__ dsig, TI* __restrict__ deps,
                                                      ESlots es,
                                                      int* __restrict__ status, int* __restrict__ status_host) {
  const int sl = blockIdx.x * FB + threadIdx.x;
  const int s1 = blockIdx.x == 0 ? (int)slot_sum(es, 2) : 0;
  if (sl == 0) {
    // every kernel that sets a flag ran before this one on the stream; word 0 last, after a
    // system-scope fence: a host that sees it sees word 1
    status[1] = s1;
    if (status_host) {
      status_host[1] = s1;
      __threadfence_system();
      status_host[0] = status[0];
    }
  }
  if (sl >= *ncl_ptr * CL) return;
  const int i = slot_orig[sl];
  if (i < 0) return;
  const long long b6 = (long long)(sl >> 3) * (8 * GN) + (sl & 7), b4 = 4 * (long long)sl;
  if (dr)
    for (int a = 0; a < 3; ++a) dr[3 * i + a] = (TI)((double)(long long)(gacc[b6 + 8 * a] + gpme[b4 + a]) / F_SCALE);
  if (dq) {
    const double gE = gE_ptr ? gE_ptr[0] : 0.0;
    dq[i] = (TI)((double)(long long)(gacc[b6 + 24] + gpme[b4 + 3]) / F_SCALE -
                 gE * 2.0 * coul * alpha * 0.5641895835477563 * (double)q[i]);
  }
  if (dsig) dsig[i] = (TI)((double)(long long)gacc[b6 + 32] / F_SCALE);
  if (deps) deps[i] = (TI)((double)(long long)gacc[b6 + 40] / F_SCALE);
}

// ---------------------------------------------------------------- 6. finalize
// Forces (pair + reciprocal accumulators) back in the caller's atom order; block 0 also sums
// the energy terms:
// out = [Lennard-Jones, real-space Coulomb, reciprocal, self, total].
template <typename TI>
__global__ __launch_bounds__(FB) void k_finalize(const int* __restrict__ ncl_ptr, const int* __restrict__ slot_orig,
                                                 const unsigned long long* __restrict__ facc,
                                                 const unsigned long long* __restrict__ facc_pme, TI* __restrict__ forces,
                                                 ESlots es,
                                                 const double* __restrict__ kparts, int nk,
                                                 const double* __restrict__ qparts, int nq, double coul,
                                                 double alpha, double* __restrict__ out, const int* __restrict__ status,
                                                 int* __restrict__ status_out, int* __restrict__ status_host) {
  const int sl = blockIdx.x * FB + threadIdx.x;
  const int s1 = blockIdx.x == 0 ? (int)slot_sum(es, 2) : 0;
  if (sl == 0) {
    // every kernel that sets a flag ran before this one on the stream (after the join)
    const int s0 = status[0];
    status_out[0] = s0;
    status_out[1] = s1;
    if (status_host) {
      // word 0 last, after a system-scope fence: a host that sees it sees word 1
      status_host[1] = s1;
      __threadfence_system();
      status_host[0] = s0;
    }
  }
  if (sl < *ncl_ptr * CL) {
    const int i = slot_orig[sl];
    if (i >= 0)
      for (int a = 0; a < 3; ++a)
        forces[3 * i + a] = (TI)((double)(long long)(facc[acc_slot(sl, a)] + facc_pme[3 * sl + a]) / F_SCALE);
  }
  if (blockIdx.x != 0) return;
  const double ek = tff_sum_partials(kparts, nk);
  const double q2 = tff_sum_partials(qparts, nq);
  const long long sl_lj = slot_sum(es, 0), sl_c = slot_sum(es, 1);
  if (threadIdx.x != 0) return;
  out[0] = (double)sl_lj / F_SCALE;
  out[1] = (double)sl_c / F_SCALE;
  out[2] = coul * ek;
  out[3] = -coul * alpha * 0.5641895835477563 * q2;
  out[4] = out[0] + out[1] + out[2] + out[3];
}



// ---------------------------------------------------------------- host side

bool make_geo(const TffBox& box, long long n, double list_cutoff, Geo& g) {
  const double* b = box.b;
  if (!box.periodic || b[1] != 0 || b[2] != 0 || b[3] != 0 || b[5] != 0 || b[6] != 0 || b[7] != 0) return false;
  for (int a = 0; a < 3; ++a) {
    g.L[a] = b[4 * a];
    if (!(g.L[a] > 0)) return false;
    g.invL[a] = 1.0 / g.L[a];
  }
  const double vol = g.L[0] * g.L[1] * g.L[2];
  const double rho = (double)(n > 0 ? n : 1) / vol;
  const double a = cbrt((double)CL / rho);  // edge of a cube holding one cluster
  for (int k = 0; k < 2; ++k) {
    int nc = (int)floor(g.L[k] / a);
    if (nc < 1) nc = 1;
    if (nc > 1024) nc = 1024;
    g.ncol[k] = nc;
    g.colw[k] = g.L[k] / nc;
    // clusters |d| columns apart are at least (|d| - 1) column widths apart
    g.reach[k] = (int)floor(list_cutoff / g.colw[k]) + 1;
  }
  g.ncl_max = (int)((n + CL - 1) / CL) + g.ncol[0] * g.ncol[1];
  // cluster pairs per i-cluster (half list): clusters whose cube of edge a lies within the
  // dilated cube of edge a + 2 rlist, with a 2.5x margin for cluster shapes, in multiples of 64
  double dil = (a + 2.0 * list_cutoff) / a;
  int maxn = (int)ceil(dil * dil * dil * 1.25 / 64.0) * 64;
  if (maxn < 128) maxn = 128;
  if (maxn > g.ncl_max) maxn = ((g.ncl_max + 63) / 64) * 64;
  g.maxn = maxn;
  g.pair_cap = (long long)g.ncl_max * maxn;
  return true;
}

// Waves per i-cluster of the pair kernels: about 9000 waves in all (two rounds of the device's 4096 resident
// ones), so that a small system still spreads over the device; one wave per cluster where the clusters
// alone are enough.  Every further wave pays its start, the i atoms and the F_i sums again.  Measured
// (pair kernel, float): 96k atoms 131 us at 3 waves per cluster, 138 at 6, 150 at 11; 999k atoms
// 1.45 ms at 1, 1.54 at 4.
int pair_parts(const Geo& g) {
  const int p = (9000 + g.ncl_max - 1) / g.ncl_max;
  return p > 32 ? 32 : p;
}

// z extent of the reciprocal-space array: even K2 uses the real-input half spectrum
int spectrum_nz(const int K[3]) { return K[2] % 2 == 0 ? K[2] / 2 + 1 : K[2]; }

struct FusedWs {
  int *col_of, *off_in_col, *col_count, *col_start, *sorted_orig, *col_cl_start, *ncl, *cl_col, *slot_orig,
      *excl_part, *slot_of_orig;
  int* st;  // the forward call's status words while it runs (copied out by k_finalize)
  PairList pl;
  void *xyzq, *lj;
  float4 *bb_c, *bb_h, *sb_c, *sb_h;
  unsigned long long *facc, *facc_pme, *grid;
  void* work;
  double *kparts, *qparts;
  ESlots es;
  // float compute only: per-slot spline tables and home-brick lists of the charge spread
  float* wts;
  int* bcount;
  int2* blist;
  BrickGrid bg;
  // backward only
  void* vsl;
  unsigned long long *gacc, *gpme, *grid_d;
  size_t bytes;
  int nk, parts, nq;
};

FusedWs carve(void* base, long long n, const Geo& g, const int K[3], size_t tc, bool grad = false) {
  FusedWs w{};
  size_t off = 0;
  char* p = (char*)base;
  auto take = [&](size_t b) {
    char* r = p ? p + off : nullptr;
    off += tff_align(b > 0 ? b : 1);
    return r;
  };
  size_t nn = (size_t)(n > 0 ? n : 1);
  size_t slots = (size_t)g.ncl_max * CL;
  size_t ng = (size_t)K[0] * K[1] * K[2];
  int ncols = g.ncol[0] * g.ncol[1];
  w.col_of = (int*)take(4 * nn);
  w.off_in_col = (int*)take(4 * nn);
  // dead after the scatter; the column sort clears the slots
  w.es.p = (unsigned long long*)w.off_in_col;
  w.es.n = (int)(tff_align(4 * nn) / 64 < (size_t)E_SLOTS ? tff_align(4 * nn) / 64 : (size_t)E_SLOTS);
  w.col_count = (int*)take(4 * (size_t)(ncols + 1));
  w.col_start = (int*)take(4 * (size_t)(ncols + 1));
  w.sorted_orig = (int*)take(4 * nn);
  w.col_cl_start = (int*)take(4 * (size_t)(ncols + 1));
  w.ncl = (int*)take(32);
  w.st = w.ncl ? w.ncl + 4 : nullptr;
  w.cl_col = (int*)take(4 * (size_t)g.ncl_max);
  w.slot_orig = (int*)take(4 * slots);
  w.excl_part = (int*)take(4 * slots * MAXEX);
  w.xyzq = take(4 * tc * slots);
  w.lj = take(2 * tc * slots);
  w.bb_c = (float4*)take(16 * (size_t)g.ncl_max);
  w.bb_h = (float4*)take(16 * (size_t)g.ncl_max);
  w.sb_c = (float4*)take(16 * 4 * (size_t)g.ncl_max);
  w.sb_h = (float4*)take(16 * 4 * (size_t)g.ncl_max);
  w.slot_of_orig = (int*)take(4 * nn);
  w.pl.cap = 4 * g.maxn;  // 4 j-groups per listed cluster pair
  w.pl.g = (int*)take(4 * 4 * (size_t)g.pair_cap);
  w.pl.i = (unsigned short*)take(2 * 4 * (size_t)g.pair_cap);
  w.pl.cnt = (int2*)take(8 * (size_t)g.ncl_max);
  w.facc = (unsigned long long*)take(8 * 3 * slots);
  w.facc_pme = (unsigned long long*)take(8 * 3 * slots);
  w.parts = pair_parts(g);
  w.grid = (unsigned long long*)take(8 * ng);
  w.work = take(2 * tc * ng);
  PassCfg px = pass_cfg(1, K[0], K[1] * spectrum_nz(K), 2 * tc);
  w.nk = px.tiles;
  w.kparts = (double*)take(8 * (size_t)w.nk);
  w.nq = (int)((nn + FB - 1) / FB);
  w.qparts = (double*)take(8 * (size_t)w.nq);
  if (tc == 4) {
    for (int a = 0; a < 3; ++a) w.bg.nb[a] = (K[a] + BR - 1) / BR;
    const long long nbr = (long long)w.bg.nb[0] * w.bg.nb[1] * w.bg.nb[2];
    // four times the mean occupancy (plus a margin) per brick; more sets TFF_FUSED_BRICK_OVERFLOW
    w.bg.cap = (int)(4 * ((long long)nn + nbr - 1) / nbr + 64);
    w.wts = (float*)take(4 * (size_t)LIST_WST * slots);
    w.bcount = (int*)take(4 * (size_t)nbr);
    w.blist = (int2*)take(8 * (size_t)nbr * w.bg.cap);
  }
  if (grad) {
    w.vsl = take(4 * tc * slots);
    w.gacc = (unsigned long long*)take(8 * GN * slots);
    w.gpme = (unsigned long long*)take(8 * 4 * slots);
    w.grid_d = (unsigned long long*)take(8 * ng);
  }
  w.bytes = off;
  return w;
}

// the list spread serves the float path for orders up to 6 on grids with BR + P <= K_a <= 1023
bool spread_from_lists(int P, const int K[3]) {
  if (P > 6) return false;
  for (int a = 0; a < 3; ++a)
    if (K[a] < BR + P || K[a] > 1023) return false;
  return true;
}

template <typename TC>
int launch_pme_slots(int order, const FusedWs& w, const Geo& g, const PmeGeom& pg, int nslots, const TC* phi,
                     double coul, bool spread, int* status, hipStream_t st) {
  unsigned nb = (unsigned)((nslots + FB - 1) / FB);
  const unsigned nbricks = (unsigned)(((pg.K[0] + BR - 1) / BR) * ((pg.K[1] + BR - 1) / BR) * ((pg.K[2] + BR - 1) / BR));
#define TFF_SP(P)                                                                                               \
  if (spread && sizeof(TC) == 4 && spread_from_lists(P, pg.K)) {                                                \
    hipLaunchKernelGGL((k_slot_splines<P < 7 ? P : 6>), dim3(nb), dim3(FB), 0, st, w.ncl,                      \
                       (const V4<float>*)w.xyzq, w.slot_orig, pg, w.bg, w.wts, w.bcount, w.blist, status);      \
    hipLaunchKernelGGL((k_spread_lists<P < 7 ? P : 6, false>), dim3(nbricks), dim3(LIST_ROUND), 0, st,       \
                       (const float*)w.wts,                                                                      \
                       (const int*)w.bcount, (const int2*)w.blist, w.bg, pg, w.grid,                          \
                       (const V4<float>*)nullptr, (const V4<float>*)nullptr, V4<float>{});                    \
  } else if (spread)                                                                                            \
    hipLaunchKernelGGL((k_spread_bricks<TC, P, false>), dim3(nbricks), dim3(256), 0, st, w.ncl,               \
                       (const V4<TC>*)w.xyzq, w.slot_orig, w.bb_c, w.bb_h, w.col_cl_start, g, pg, w.grid, status, \
                       (const V4<TC>*)nullptr, V4<TC>{});                                                        \
  else                                                                                                          \
    hipLaunchKernelGGL((k_gather_slots<TC, P>), dim3(nb), dim3(FB), 0, st, w.ncl, phi, (const V4<TC>*)w.xyzq,   \
                       w.slot_orig, pg, coul, w.facc_pme)
  switch (order) {
    case 3: TFF_SP(3); break;
    case 4: TFF_SP(4); break;
    case 5: TFF_SP(5); break;
    case 6: TFF_SP(6); break;
    case 7: TFF_SP(7); break;
    case 8: TFF_SP(8); break;
    default: tff_set_error("fused: unsupported spline order %d (3..8)", order); return TFF_ERR_UNSUPPORTED;
  }
#undef TFF_SP
  return TFF_OK;
}

// Per-device auxiliary stream (default priority) and fork / join events.  The fork makes the
// auxiliary stream wait for the work enqueued so far on the caller's stream; the join makes
// the caller's stream wait for the auxiliary work, so the call stays ordered on the caller's
// stream (and can be captured into a graph).  The mutex covers each record / wait pair.
struct AuxStream {
  hipStream_t s = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
};
std::mutex g_aux_mu;
AuxStream g_aux[64];

// 0: the reciprocal-space chain runs on the caller's stream, in order (a timing aid); 2: the charge
// spread runs on the caller's stream before the fork, the FFT and the gather on the auxiliary
// stream; 3: the whole chain runs on the auxiliary stream; 1: 3 below SPREAD_FIRST_ATOMS, 2 from
// there on (beside the pair kernel a spread gets few registers and leaves the FFT and the gather to run
// after it).  Measured per evaluation (mixed, launched one by one, as 3 and as 2): 96k atoms 0.242 and
// 0.266 ms, 192k 0.453 and 0.433, 300k 0.583 and 0.601, 480k 0.975 and 0.878, 999k 2.06 and 2.07; replayed as a
// graph 96k 0.260 and 0.279, 192k 0.416 and 0.442.
constexpr long long SPREAD_FIRST_ATOMS = 300000;
std::atomic<int> g_overlap{1};

// *sp: the auxiliary stream, waiting for the work enqueued so far on st (st itself when the
// overlap is off); false when the stream or its events could not be set up
// creates the auxiliary stream and its events of device dev once (caller holds g_aux_mu)
bool aux_stream_setup_locked(int dev) {
  AuxStream& a = g_aux[dev];
  if (!a.s) {
    if (hipStreamCreateWithFlags(&a.s, hipStreamNonBlocking) != hipSuccess) return false;
    if (hipEventCreateWithFlags(&a.fork, hipEventDisableTiming) != hipSuccess) return false;
    if (hipEventCreateWithFlags(&a.join, hipEventDisableTiming) != hipSuccess) return false;
  }
  return true;
}

bool aux_stream_fork(hipStream_t st, hipStream_t* sp) {
  *sp = st;
  if (!g_overlap.load()) return true;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return false;
  std::lock_guard<std::mutex> lk(g_aux_mu);
  AuxStream& a = g_aux[dev];
  if (!aux_stream_setup_locked(dev)) return false;
  if (hipEventRecord(a.fork, st) != hipSuccess) return false;
  if (hipStreamWaitEvent(a.s, a.fork, 0) != hipSuccess) return false;
  *sp = a.s;
  return true;
}

void aux_stream_join(hipStream_t st, hipStream_t sp) {
  if (sp == st) return;
  int dev = 0;
  hipGetDevice(&dev);
  std::lock_guard<std::mutex> lk(g_aux_mu);
  AuxStream& a = g_aux[dev];
  hipEventRecord(a.join, a.s);
  hipStreamWaitEvent(st, a.join, 0);
}

// Reciprocal-space convolution of a fixed-point grid: forward transforms, influence function with
// the k-space energy partials, inverse transforms; the real potential grid phi_out may alias
// grid_in (it is written by the last pass only).
template <typename TC>
void run_recip_fft(const FusedWs& w, const int K[3], const TffBox& box, double alpha, const FftPlan* pl,
                   const TC* mx, const TC* my, const TC* mz, const unsigned long long* grid_in,
                   double grid_inv_scale, TC* phi_out, double* kparts, const char* prof_name, hipStream_t st) {
  ConvArgs cv{};
  for (int a = 0; a < 3; ++a) cv.K[a] = K[a];
  for (int k = 0; k < 9; ++k) cv.inv[k] = box.inv[k];
  cv.vol = box.det;
  cv.alpha = alpha;
  cv.grid_fixed = 1;
  cv.grid_inv_scale = grid_inv_scale;
  const size_t ce = 2 * sizeof(TC);
  // real-input transforms along z when K2 is even (half spectrum, K2 / 2 + 1 planes), else complex
  const bool rz = K[2] % 2 == 0;
  const int nzc = spectrum_nz(K);
  cv.nz = nzc;
  cv.half = rz ? 1 : 0;
  PassCfg cz = pass_cfg(K[0] * K[1], K[2], 1, ce);
  PassCfg cy = pass_cfg(K[0], K[1], nzc, ce);
  PassCfg cxp = pass_cfg(1, K[0], K[1] * nzc, ce);
  FftPlan pzh;
  make_plan(rz ? K[2] / 2 : 1, pzh);
  const ZPlanCfg zc = zcfg(K[0] * K[1], K[2], ce);
  {
    void* tok = tff_prof_begin(prof_name, st);
    if (rz)
      hipLaunchKernelGGL(k_fft_z_r2c<TC>, dim3(zc.blocks), dim3(FFT_THREADS), zc.lds, st, grid_in, (cx<TC>*)w.work,
                         K[0] * K[1], K[2], zc.AB, zc.ab_shift, pzh, 1, cv.grid_inv_scale);
    else
      hipLaunchKernelGGL((k_fft_pass<TC, PASS_Z_FWD>), dim3(cz.tiles), dim3(FFT_THREADS), cz.lds, st, grid_in, w.work,
                         cz.pa, pl[2], cv, mx, my, mz, 1, kparts);
    hipLaunchKernelGGL((k_fft_pass<TC, PASS_Y_FWD>), dim3(cy.tiles), dim3(FFT_THREADS), cy.lds, st, w.work, w.work,
                       cy.pa, pl[1], cv, mx, my, mz, 1, kparts);
    hipLaunchKernelGGL((k_fft_pass<TC, PASS_X_CONV>), dim3(cxp.tiles), dim3(FFT_THREADS), cxp.lds, st, w.work,
                       w.work, cxp.pa, pl[0], cv, mx, my, mz, 1, kparts);
    hipLaunchKernelGGL((k_fft_pass<TC, PASS_Y_INV>), dim3(cy.tiles), dim3(FFT_THREADS), cy.lds, st, w.work, w.work,
                       cy.pa, pl[1], cv, mx, my, mz, 1, kparts);
    if (rz)
      hipLaunchKernelGGL(k_fft_z_c2r<TC>, dim3(zc.blocks), dim3(FFT_THREADS), zc.lds, st, (const cx<TC>*)w.work, phi_out,
                         K[0] * K[1], K[2], zc.AB, zc.ab_shift, pzh);
    else
      hipLaunchKernelGGL((k_fft_pass<TC, PASS_Z_INV>), dim3(cz.tiles), dim3(FFT_THREADS), cz.lds, st, w.work, phi_out,
                         cz.pa, pl[2], cv, mx, my, mz, 1, kparts);
    tff_prof_end(tok, st);
  }
}

// Everything of one forward call up to the join of the reciprocal-space chain: reads the inputs,
// writes only the workspace (status words in w.st), so the same launch sequence can be captured
// once into a graph and replayed for every call with the same inputs and workspace.
template <typename TI, typename TC>
int run_fused_core(const TI* coords, const TI* q, const TI* sig, const TI* eps, long long n, const TffBox& box,
                   const Geo& g, const int64_t* row_ptr, const int64_t* col, double cutoff, double list_cutoff,
                   double alpha, double coul, const int K[3], int order, const TC* mx, const TC* my, const TC* mz,
                   const TI* box_dev, const FusedWs& w, hipStream_t st) {
  if (order < 3 || order > 8) {  // checked before any launch: the stream fork below must be joined
    tff_set_error("fused: unsupported spline order %d (3..8)", order);
    return TFF_ERR_UNSUPPORTED;
  }
  int* status = w.st;
  const unsigned nbA = (unsigned)((n + FB - 1) / FB);
  const int nslots = g.ncl_max * CL;
  const unsigned nbS = (unsigned)((nslots + FB - 1) / FB);
  const int ncols = g.ncol[0] * g.ncol[1];
  {
    ClearList cl{};
    auto add = [&](void* p, long long words) {
      cl.p[cl.count] = (int*)p;
      cl.n[cl.count] = words;
      ++cl.count;
    };
    add(w.col_count, ncols + 1);
    add(status, 2);
    add(w.facc, 6LL * nslots);
    add(w.slot_orig, nslots);
    if (w.bcount) add(w.bcount, (long long)w.bg.nb[0] * w.bg.nb[1] * w.bg.nb[2]);
    hipLaunchKernelGGL(k_clear, dim3(1024), dim3(256), 0, st, cl);
  }
  // 1. sort
  hipLaunchKernelGGL(k_bin_atoms<TI>, dim3(nbA), dim3(FB), 0, st, coords, q, n, g, w.col_of, w.off_in_col,
                     w.col_count, w.qparts, box_dev, status);
  hipLaunchKernelGGL(k_scan_columns, dim3(1), dim3(1024), 0, st, w.col_count, ncols, w.col_start, w.col_cl_start,
                     w.ncl, status);
  hipLaunchKernelGGL(k_scatter_atoms, dim3(nbA), dim3(FB), 0, st, n, w.col_of, w.off_in_col, w.col_start,
                     w.sorted_orig);
  hipLaunchKernelGGL(k_sort_columns<TI>, dim3(ncols), dim3(SORT_THREADS), 0, st, coords, g, w.col_start, w.sorted_orig, w.es);
  // 2. cluster arrays
  const unsigned nbW = (unsigned)(((long long)g.ncl_max * TFF_WAVE + FB - 1) / FB);
  const unsigned nbB = (unsigned)(((long long)g.ncl_max * CL + FB - 1) / FB);  // two clusters per wave
  hipLaunchKernelGGL((k_build_clusters<TI, TC>), dim3(nbB), dim3(FB), 0, st, coords, q, sig, eps, g, w.ncl,
                     w.col_cl_start, w.col_start, w.sorted_orig, (V4<TC>*)w.xyzq, (V2<TC>*)w.lj, w.slot_orig,
                     w.slot_of_orig, w.cl_col, w.bb_c, w.bb_h, w.sb_c, w.sb_h);
  // 3. PME on the auxiliary stream (needs only the cluster arrays), concurrent with 4-5; the
  // exclusion table (needed from the pair search on) beside the first reciprocal-space kernels
  PmeGeom pg = make_geom(box, K, order, alpha);
  FftPlan pl[3];
  for (int a = 0; a < 3; ++a) make_plan(K[a], pl[a]);
  const int mode = g_overlap.load();
  const bool spread_first = mode == 2 || (mode == 1 && n >= SPREAD_FIRST_ATOMS);
  auto fill_exclusions = [&](hipStream_t s) {
    hipLaunchKernelGGL(k_fill_exclusions, dim3(nbS), dim3(FB), 0, s, w.ncl, w.slot_orig, w.slot_of_orig, n, row_ptr,
                       col, w.excl_part, status);
  };
  auto spread = [&](hipStream_t s) {
    void* tok = tff_prof_begin("fused_spread", s);
    const int rc = launch_pme_slots<TC>(order, w, g, pg, nslots, nullptr, coul, true, status, s);
    tff_prof_end(tok, s);
    return rc;
  };
  hipStream_t sp = st;
  if (!aux_stream_fork(st, &sp)) {
    tff_set_error("fused: could not create the auxiliary stream");
    return TFF_ERR_LAUNCH;
  }
  if (spread_first) {
    // the spread alone on the caller's stream, the exclusion table beside it; the FFT and the
    // gather fork after the spread
    fill_exclusions(sp);
    const int rc = spread(st);
    if (rc) return rc;
    aux_stream_join(st, sp);
    if (!aux_stream_fork(st, &sp)) {
      tff_set_error("fused: could not create the auxiliary stream");
      return TFF_ERR_LAUNCH;
    }
  } else {
    const int rc = spread(sp);
    if (rc) return rc;
  }
  TC* phi = (TC*)w.grid;  // the real potential grid reuses the charge grid's memory after the z pass
  run_recip_fft<TC>(w, K, box, alpha, pl, mx, my, mz, w.grid, 1.0 / grid_scale<TC>(), phi, w.kparts, "fused_fft", sp);
  {
    void* tok = tff_prof_begin("fused_gather", sp);
    int rc = launch_pme_slots<TC>(order, w, g, pg, nslots, phi, coul, false, status, sp);
    tff_prof_end(tok, sp);
    if (rc) return rc;
  }
  if (!spread_first) fill_exclusions(st);
  // 4. cluster pairs
  {
    void* tok = tff_prof_begin("fused_cluster_pairs", st);
    float rl2 = (float)(list_cutoff * list_cutoff);
    // group pairs are pruned at the interaction cutoff itself: pairs between rc and the list
    // cutoff contribute nothing to this evaluation
    hipLaunchKernelGGL(k_pair_list, dim3(nbW), dim3(FB), 0, st, w.ncl, w.cl_col, w.col_cl_start, w.bb_c, w.bb_h,
                       w.sb_c, w.sb_h, g, rl2, (float)(cutoff * cutoff), w.excl_part, w.pl,
                       w.es, status);
    tff_prof_end(tok, st);
  }
  // 5. tiles
  {
    TileArgs<TC> ta;
    for (int a = 0; a < 3; ++a) {
      ta.L[a] = (TC)g.L[a];
      ta.invL[a] = (TC)g.invL[a];
    }
    ta.rc2 = (TC)(cutoff * cutoff);
    ta.alpha = (TC)alpha;
    ta.coul = (TC)coul;
    ta.c2alpha = (TC)(1.1283791670955126 * alpha);
    void* tok = tff_prof_begin("fused_tiles", st);
    const dim3 nw((unsigned)((long long)g.ncl_max * w.parts));
    if constexpr (sizeof(TC) == 4)
      hipLaunchKernelGGL(k_tiles_f32, nw, dim3(TFF_WAVE), 0, st, w.ncl, w.pl, w.parts, (const V4<float>*)w.xyzq,
                         (const V2<float>*)w.lj, w.excl_part, ta, w.facc, w.es);
    else
      hipLaunchKernelGGL(k_tiles_f64, nw, dim3(TFF_WAVE), 0, st, w.ncl, w.pl, w.parts, (const V4<double>*)w.xyzq,
                         (const V2<double>*)w.lj, w.excl_part, ta, w.facc, w.es);
    tff_prof_end(tok, st);
  }
  aux_stream_join(st, sp);
  TFF_CHECK_LAUNCH("fused energy+forces");
  return TFF_OK;
}

// 6. outputs, after the reciprocal-space work: forces in atom order, energy terms, status words
template <typename TI>
int launch_fused_finalize(const FusedWs& w, const Geo& g, double coul, double alpha, double* energies, TI* forces,
                          int* status_out, int* status_host, hipStream_t st) {
  const unsigned nbS = (unsigned)(((long long)g.ncl_max * CL + FB - 1) / FB);
  hipLaunchKernelGGL(k_finalize<TI>, dim3(nbS), dim3(FB), 0, st, w.ncl, w.slot_orig, w.facc, w.facc_pme, forces, w.es,
                     w.kparts, w.nk, w.qparts, w.nq, coul, alpha, energies, w.st, status_out, status_host);
  TFF_CHECK_LAUNCH("fused energy+forces");
  return TFF_OK;
}

// Force-matching backward: rebuilds the cluster pair list (not stored from the forward call),
// then the pair backward, the charge and dipole reciprocal convolutions and the gather.
template <typename TI, typename TC>
int run_fused_grad(const TI* coords, const TI* q, const TI* sig, const TI* eps, long long n, const TffBox& box,
                   const Geo& g, const int64_t* row_ptr, const int64_t* col, double cutoff, double list_cutoff,
                   double alpha, double coul, const int K[3], int order, const TC* mx, const TC* my, const TC* mz,
                   const double* gE, const TI* gF, TI* dr, TI* dq, TI* dsig, TI* deps, int* status, const TI* box_dev,
                   int* status_host, const FusedWs& w, bool reuse, hipStream_t st) {
  if (order < 3 || order > 8) {
    tff_set_error("fused: unsupported spline order %d (3..8)", order);
    return TFF_ERR_UNSUPPORTED;
  }
  const unsigned nbA = (unsigned)((n + FB - 1) / FB);
  const int nslots = g.ncl_max * CL;
  const unsigned nbS = (unsigned)((nslots + FB - 1) / FB);
  const int ncols = g.ncol[0] * g.ncol[1];
  {
    ClearList cl{};
    auto add = [&](void* p, long long words) {
      cl.p[cl.count] = (int*)p;
      cl.n[cl.count] = words;
      ++cl.count;
    };
    if (!reuse) {
      add(w.col_count, ncols + 1);
      add(status, 2);
      add(w.slot_orig, nslots);
      // the brick counters of the charge spread (float: the forward's list spread runs again)
      if (w.bcount) add(w.bcount, (long long)w.bg.nb[0] * w.bg.nb[1] * w.bg.nb[2]);
    }
    add(w.gacc, 2LL * GN * nslots);
    hipLaunchKernelGGL(k_clear, dim3(1024), dim3(256), 0, st, cl);
  }
  const unsigned nbW = (unsigned)(((long long)g.ncl_max * TFF_WAVE + FB - 1) / FB);
  // reuse: the cluster arrays, the exclusion table and the pair list are those the forward call
  // left in the workspace (for the same inputs); otherwise they are rebuilt here
  if (!reuse) {
    hipLaunchKernelGGL(k_bin_atoms<TI>, dim3(nbA), dim3(FB), 0, st, coords, q, n, g, w.col_of, w.off_in_col,
                       w.col_count, w.qparts, box_dev, status);
    hipLaunchKernelGGL(k_scan_columns, dim3(1), dim3(1024), 0, st, w.col_count, ncols, w.col_start,
                       w.col_cl_start, w.ncl, status);
    hipLaunchKernelGGL(k_scatter_atoms, dim3(nbA), dim3(FB), 0, st, n, w.col_of, w.off_in_col, w.col_start,
                       w.sorted_orig);
    hipLaunchKernelGGL(k_sort_columns<TI>, dim3(ncols), dim3(SORT_THREADS), 0, st, coords, g, w.col_start,
                       w.sorted_orig, w.es);
    const unsigned nbB = (unsigned)(((long long)g.ncl_max * CL + FB - 1) / FB);  // two clusters per wave
    hipLaunchKernelGGL((k_build_clusters<TI, TC>), dim3(nbB), dim3(FB), 0, st, coords, q, sig, eps, g, w.ncl,
                       w.col_cl_start, w.col_start, w.sorted_orig, (V4<TC>*)w.xyzq, (V2<TC>*)w.lj, w.slot_orig,
                       w.slot_of_orig, w.cl_col, w.bb_c, w.bb_h, w.sb_c, w.sb_h);
  }
  hipLaunchKernelGGL((k_fill_vslots<TI, TC>), dim3(nbS), dim3(FB), 0, st, w.ncl, w.slot_orig, gF, (const V2<TC>*)w.lj,
                     (V4<TC>*)w.vsl, reuse ? (const int*)w.st : nullptr, status);
  // the reciprocal-space part (charge and dipole grids, both transforms, the gather) needs only
  // the cluster arrays and the per-slot upstream forces: it runs on the auxiliary stream beside the
  // pair search and the pair kernel, joined before the final kernel
  hipStream_t sp = st;
  if (!aux_stream_fork(st, &sp)) {
    tff_set_error("fused backward: could not create the auxiliary stream");
    return TFF_ERR_LAUNCH;
  }
  // the pair search and the pair kernel are enqueued first, so that the pair kernel starts as soon
  // as the caller's stream reaches it rather than after the host has enqueued the reciprocal chain
  if (!reuse) {
    hipLaunchKernelGGL(k_fill_exclusions, dim3(nbS), dim3(FB), 0, st, w.ncl, w.slot_orig, w.slot_of_orig, n,
                       row_ptr, col, w.excl_part, status);
    hipLaunchKernelGGL(k_pair_list, dim3(nbW), dim3(FB), 0, st, w.ncl, w.cl_col, w.col_cl_start, w.bb_c, w.bb_h,
                       w.sb_c, w.sb_h, g, (float)(list_cutoff * list_cutoff), (float)(cutoff * cutoff), w.excl_part,
                       w.pl, w.es, status);
  }
  {
    TileArgs<TC> ta;
    for (int a = 0; a < 3; ++a) {
      ta.L[a] = (TC)g.L[a];
      ta.invL[a] = (TC)g.invL[a];
    }
    ta.rc2 = (TC)(cutoff * cutoff);
    ta.alpha = (TC)alpha;
    ta.coul = (TC)coul;
    ta.c2alpha = (TC)(1.1283791670955126 * alpha);
    void* tok = tff_prof_begin("fused_grad_tiles", st);
    const dim3 nw((unsigned)((long long)g.ncl_max * w.parts));
    if constexpr (sizeof(TC) == 4)
      hipLaunchKernelGGL(k_tiles_grad_f32, nw, dim3(TFF_WAVE), 0, st, w.ncl, w.pl, w.parts, (const V4<float>*)w.xyzq,
                         (const V2<float>*)w.lj, (const V4<float>*)w.vsl, w.excl_part, ta, gE, w.gacc);
    else
      hipLaunchKernelGGL(k_tiles_grad_f64, nw, dim3(TFF_WAVE), 0, st, w.ncl, w.pl, w.parts, (const V4<double>*)w.xyzq,
                         (const V2<double>*)w.lj, (const V4<double>*)w.vsl, w.excl_part, ta, gE, w.gacc);
    tff_prof_end(tok, st);
  }
  PmeGeom pg = make_geom(box, K, order, alpha);
  FftPlan pl[3];
  for (int a = 0; a < 3; ++a) make_plan(K[a], pl[a]);
  const unsigned nbricks = (unsigned)(((K[0] + BR - 1) / BR) * ((K[1] + BR - 1) / BR) * ((K[2] + BR - 1) / BR));
  V4<TC> jsc{(TC)(K[0] * box.inv[0]), (TC)(K[1] * box.inv[4]), (TC)(K[2] * box.inv[8]), (TC)0};
  TC* phi = (TC*)w.grid;
  TC* psi = (TC*)w.grid_d;
  const unsigned nb = (unsigned)((nslots + FB - 1) / FB);
  auto spread_dipoles = [&] {
    auto go = [&](auto order_c) {
      constexpr int P = decltype(order_c)::value;
      if constexpr (sizeof(TC) == 4 && P < 7) {
        if (spread_from_lists(P, K)) {
          hipLaunchKernelGGL((k_spread_lists<P, true>), dim3(nbricks), dim3(LIST_ROUND), 0, sp, (const float*)w.wts,
                             (const int*)w.bcount, (const int2*)w.blist, w.bg, pg, w.grid_d,
                             (const V4<float>*)w.xyzq, (const V4<float>*)w.vsl, jsc);
          return;
        }
      }
      hipLaunchKernelGGL((k_spread_bricks<TC, P, true>), dim3(nbricks), dim3(256), 0, sp, w.ncl,
                         (const V4<TC>*)w.xyzq, w.slot_orig, w.bb_c, w.bb_h, w.col_cl_start, g, pg, w.grid_d, status,
                         (const V4<TC>*)w.vsl, jsc);
    };
    switch (order) {
      case 3: go(std::integral_constant<int, 3>{}); break;
      case 4: go(std::integral_constant<int, 4>{}); break;
      case 5: go(std::integral_constant<int, 5>{}); break;
      case 6: go(std::integral_constant<int, 6>{}); break;
      case 7: go(std::integral_constant<int, 7>{}); break;
      default: go(std::integral_constant<int, 8>{}); break;
    }
  };
  // the potential grid phi of the charges: the forward call's, left in place (reuse), or made
  // again by the forward's own spread and transforms, so that both give the same bits
  if (!reuse) {
    const int rc = launch_pme_slots<TC>(order, w, g, pg, nslots, (const TC*)nullptr, coul, true, status, sp);
    if (rc) {
      aux_stream_join(st, sp);
      return rc;
    }
    run_recip_fft<TC>(w, K, box, alpha, pl, mx, my, mz, w.grid, 1.0 / grid_scale<TC>(), phi, w.kparts,
                      "fused_grad_fft", sp);
  }
  spread_dipoles();
  run_recip_fft<TC>(w, K, box, alpha, pl, mx, my, mz, w.grid_d, 1.0 / Q_SCALE, psi, w.kparts, "fused_grad_fft", sp);
#define TFF_GRAD_GATHER(P)                                                                                       \
  hipLaunchKernelGGL((k_gather_grad<TC, P>), dim3(nb), dim3(FB), 0, sp, w.ncl, phi, psi, (const V4<TC>*)w.xyzq, \
                     (const V4<TC>*)w.vsl, w.slot_orig, pg, coul, gE, w.gpme)
  switch (order) {
    case 3: TFF_GRAD_GATHER(3); break;
    case 4: TFF_GRAD_GATHER(4); break;
    case 5: TFF_GRAD_GATHER(5); break;
    case 6: TFF_GRAD_GATHER(6); break;
    case 7: TFF_GRAD_GATHER(7); break;
    default: TFF_GRAD_GATHER(8); break;
  }
#undef TFF_GRAD_GATHER
  aux_stream_join(st, sp);
  hipLaunchKernelGGL(k_finalize_grad<TI>, dim3(nbS), dim3(FB), 0, st, w.ncl, w.slot_orig, w.gacc, w.gpme, q, coul,
                     alpha, gE, dr, dq, dsig, deps, w.es, status, status_host);
  TFF_CHECK_LAUNCH("fused energy+forces backward");
  return TFF_OK;
}

}  // namespace

extern "C" void tff_fused_set_overlap(int mode) { g_overlap.store(mode >= 0 && mode <= 3 ? mode : 1); }

extern "C" size_t tff_fused_workspace_bytes(int compute_dtype, long long natoms, const double* box_host,
                                            double list_cutoff, int K0, int K1, int K2) {
  TffBox box = tff_make_box(box_host);
  Geo g;
  if (!make_geo(box, natoms, list_cutoff, g)) return 0;
  int K[3] = {K0, K1, K2};
  return carve(nullptr, natoms, g, K, compute_dtype == TFF_F64 ? 8 : 4).bytes;
}

namespace {
// checks shared by the forward and backward entry points
int fused_check(const TffBox& box, long long natoms, double cutoff, double list_cutoff, double ewald_alpha,
                const int K[3], int order, const int64_t* excl_row_ptr, const int64_t* excl_col, Geo& g) {
  if (!make_geo(box, natoms, list_cutoff, g)) {
    tff_set_error("fused: needs an orthorhombic periodic box (diagonal box matrix)");
    return TFF_ERR_UNSUPPORTED;
  }
  if (natoms <= 0 || !(cutoff > 0) || list_cutoff < cutoff || ewald_alpha < 0) {
    tff_set_error("fused: invalid arguments");
    return TFF_ERR_ARG;
  }
  if ((excl_row_ptr == nullptr) != (excl_col == nullptr)) {
    tff_set_error("fused: exclusion row_ptr and col must be given together");
    return TFF_ERR_ARG;
  }
  for (int a = 0; a < 3; ++a) {
    FftPlan p;
    if (K[a] < order || K[a] > 4096 || !make_plan(K[a], p)) {
      tff_set_error("fused: PME grid size %d must be 2^a 3^b 5^c and >= the spline order", K[a]);
      return TFF_ERR_UNSUPPORTED;
    }
  }
  for (int a = 0; a < 3; ++a)
    if (2.0 * list_cutoff > g.L[a]) {
      tff_set_error("fused: the box (%.4g nm) must exceed twice the list cutoff (%.4g nm) for the minimum image",
                    g.L[a], list_cutoff);
      return TFF_ERR_UNSUPPORTED;
    }
  return TFF_OK;
}
}  // namespace

extern "C" size_t tff_fused_backward_workspace_bytes(int compute_dtype, long long natoms, const double* box_host,
                                                     double list_cutoff, int K0, int K1, int K2) {
  TffBox box = tff_make_box(box_host);
  Geo g;
  if (!make_geo(box, natoms, list_cutoff, g)) return 0;
  int K[3] = {K0, K1, K2};
  return carve(nullptr, natoms, g, K, compute_dtype == TFF_F64 ? 8 : 4, true).bytes;
}

namespace {
int fused_backward(int io_dtype, int compute_dtype, const void* coords, const void* charges, const void* sigma,
                   const void* epsilon, long long natoms, const double* box_host, const int64_t* excl_row_ptr,
                   const int64_t* excl_col, double cutoff, double list_cutoff, double ewald_alpha,
                   double coul_constant, int K0, int K1, int K2, int order, const void* xmoduli,
                   const void* ymoduli, const void* zmoduli, const double* grad_energy, const void* grad_forces,
                   void* grad_coords, void* grad_charges, void* grad_sigma, void* grad_epsilon, int32_t* status_out,
                   const void* box_device, int32_t* status_host, void* workspace, size_t workspace_bytes,
                   bool reuse, hipStream_t stream) {
  TffBox box = tff_make_box(box_host);
  Geo g;
  int K[3] = {K0, K1, K2};
  int rc = fused_check(box, natoms, cutoff, list_cutoff, ewald_alpha, K, order, excl_row_ptr, excl_col, g);
  if (rc) return rc;
  if (!coords || !charges || !sigma || !epsilon || !status_out || !xmoduli || !ymoduli || !zmoduli) {
    tff_set_error("fused backward: invalid arguments");
    return TFF_ERR_ARG;
  }
  size_t tc = compute_dtype == TFF_F64 ? 8 : 4;
  size_t need = carve(nullptr, natoms, g, K, tc, true).bytes;
  if (!workspace || workspace_bytes < need) {
    tff_set_error("fused backward: workspace too small (%zu < %zu)", workspace_bytes, need);
    return TFF_ERR_WORKSPACE;
  }
  FusedWs w = carve(workspace, natoms, g, K, tc, true);
#define TFF_RUN(TI, TC)                                                                                            \
  return run_fused_grad<TI, TC>((const TI*)coords, (const TI*)charges, (const TI*)sigma, (const TI*)epsilon,       \
                                natoms, box, g, excl_row_ptr, excl_col, cutoff, list_cutoff, ewald_alpha,          \
                                coul_constant, K, order, (const TC*)xmoduli, (const TC*)ymoduli,                  \
                                (const TC*)zmoduli, grad_energy, (const TI*)grad_forces, (TI*)grad_coords,         \
                                (TI*)grad_charges, (TI*)grad_sigma, (TI*)grad_epsilon, (int*)status_out,        \
                                (const TI*)box_device, (int*)status_host, w, reuse, stream)
  if (io_dtype == TFF_F64 && compute_dtype == TFF_F32) TFF_RUN(double, float);
  if (io_dtype == TFF_F32 && compute_dtype == TFF_F32) TFF_RUN(float, float);
  if (io_dtype == TFF_F64 && compute_dtype == TFF_F64) TFF_RUN(double, double);
  if (io_dtype == TFF_F32 && compute_dtype == TFF_F64) TFF_RUN(float, double);
#undef TFF_RUN
  tff_set_error("fused backward: unsupported dtype combination");
  return TFF_ERR_ARG;
}
}  // namespace

extern "C" int tff_fused_energy_forces_backward(
    int io_dtype, int compute_dtype, const void* coords, const void* charges, const void* sigma, const void* epsilon,
    long long natoms, const double* box_host, const int64_t* excl_row_ptr, const int64_t* excl_col, double cutoff,
    double list_cutoff, double ewald_alpha, double coul_constant, int K0, int K1, int K2, int order,
    const void* xmoduli, const void* ymoduli, const void* zmoduli, const double* grad_energy,
    const void* grad_forces, void* grad_coords, void* grad_charges, void* grad_sigma, void* grad_epsilon,
    int32_t* status_out, const void* box_device, int32_t* status_host, void* workspace, size_t workspace_bytes,
    hipStream_t stream) {
  return fused_backward(io_dtype, compute_dtype, coords, charges, sigma, epsilon, natoms, box_host, excl_row_ptr,
                        excl_col, cutoff, list_cutoff, ewald_alpha, coul_constant, K0, K1, K2, order, xmoduli,
                        ymoduli, zmoduli, grad_energy, grad_forces, grad_coords, grad_charges, grad_sigma,
                        grad_epsilon, status_out, box_device, status_host, workspace, workspace_bytes, false, stream);
}

extern "C" int tff_fused_energy_forces_backward_reuse(
    int io_dtype, int compute_dtype, const void* coords, const void* charges, const void* sigma, const void* epsilon,
    long long natoms, const double* box_host, const int64_t* excl_row_ptr, const int64_t* excl_col, double cutoff,
    double list_cutoff, double ewald_alpha, double coul_constant, int K0, int K1, int K2, int order,
    const void* xmoduli, const void* ymoduli, const void* zmoduli, const double* grad_energy,
    const void* grad_forces, void* grad_coords, void* grad_charges, void* grad_sigma, void* grad_epsilon,
    int32_t* status_out, const void* box_device, int32_t* status_host, void* workspace, size_t workspace_bytes,
    hipStream_t stream) {
  return fused_backward(io_dtype, compute_dtype, coords, charges, sigma, epsilon, natoms, box_host, excl_row_ptr,
                        excl_col, cutoff, list_cutoff, ewald_alpha, coul_constant, K0, K1, K2, order, xmoduli,
                        ymoduli, zmoduli, grad_energy, grad_forces, grad_coords, grad_charges, grad_sigma,
                        grad_epsilon, status_out, box_device, status_host, workspace, workspace_bytes, true, stream);
}

namespace {
// ---------------------------------------------------------------- graph replay of the forward core
// The forward core (19 kernels on two streams) is captured once per key into a HIP graph and
// replayed; k_finalize, which writes the caller's outputs, is launched after the replay, so every
// call still returns its own output buffers.  A key holds everything the captured launches read:
// the device, the input and workspace addresses, the box, every scalar parameter and the stream
// schedule.  Replays read the inputs at their addresses when they run, so coordinates updated in
// place are picked up.  Launched one by one, the pair search waits behind the reciprocal-space
// kernels of the other stream; the same kernels replayed give bitwise equal results.
constexpr int GRAPH_CACHE = 8;  // captured forward cores kept per device (least recently used evicted)

struct FusedKey {
  int dev, io, cd, order, K[3], mode;
  long long natoms;
  const void* p[11];  // coords, charges, sigma, epsilon, excl row_ptr, excl col, x/y/z moduli, box_device, workspace
  double d[13];       // box, cutoff, list cutoff, alpha, Coulomb constant
};

struct GraphEntry {
  FusedKey key;
  hipGraphExec_t ex;
  unsigned long long used;
};

std::atomic<int> g_graphs_mode{1};
std::mutex g_graph_mu;
std::vector<GraphEntry> g_graphs[64];
unsigned long long g_graph_clock = 0;
hipStream_t g_capture_stream[64];
FusedKey g_seen[64];  // per device: the key of the last call that found no graph
bool g_seen_valid[64];

// a graph is captured and launched for a call on st: by the mode (0: never; 1: float32 arithmetic
// below SPREAD_FIRST_ATOMS atoms; 2: always), no event timing requested, st not itself being
// captured (an enclosing capture records the kernels one by one instead).  Measured per evaluation in a
// back-to-back loop (cutoff 0.9 nm, from 192k atoms on 1.0), graph and one by one, us: mixed 900 atoms 145 and
// 163, 3k 147 and 165, 12k 153 and 160, 60k 194 and 182, 96k 241 and 228, 192k 416 and 453, 300k 580 and 583,
// 999k 2050 and 2055; fp64 900 atoms 136 and 152, 3k 144 and 155, 12k 174 and 171, 60k 317 and 322, 96k 429 and
// 449.  (The line was drawn with slower pair kernels: most fp64 boxes would gain by a graph now, mixed ones of 60k
// to 96k atoms by going without.)
bool graphs_usable(hipStream_t st, bool f32, long long n) {
  const int mode = g_graphs_mode.load();
  if (mode == 0 || (mode == 1 && !(f32 && n < SPREAD_FIRST_ATOMS)) || tff_prof_active()) return false;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &cs) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return cs == hipStreamCaptureStatusNone;
}

// Captures key's forward core into a new cache entry (caller holds g_graph_mu) when the previous
// uncached key seen on this device was the same key: a key seen once (inputs at new addresses on
// every call, one-off calls) is not captured.  *ex stays null when the call should run without a
// graph; a failure of launch_core itself is returned.
template <typename F>
int graph_capture(const FusedKey& key, F&& launch_core, hipGraphExec_t* ex) {
  *ex = nullptr;
  if (!g_seen_valid[key.dev] || memcmp(&g_seen[key.dev], &key, sizeof key) != 0) {
    g_seen[key.dev] = key;
    g_seen_valid[key.dev] = true;
    return TFF_OK;
  }
  std::vector<GraphEntry>& cache = g_graphs[key.dev];
  hipStream_t& cs = g_capture_stream[key.dev];
  if (!cs && hipStreamCreateWithFlags(&cs, hipStreamNonBlocking) != hipSuccess) {
    cs = nullptr;
    (void)hipGetLastError();
    return TFF_OK;
  }
  {
    // the auxiliary stream is created outside the capture
    std::lock_guard<std::mutex> lk2(g_aux_mu);
    if (!aux_stream_setup_locked(key.dev)) return TFF_OK;
  }
  if (hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal) != hipSuccess) {
    (void)hipGetLastError();
    return TFF_OK;
  }
  const int rc = launch_core(cs);
  hipGraph_t graph = nullptr;
  const hipError_t e = hipStreamEndCapture(cs, &graph);
  if (rc != TFF_OK || e != hipSuccess || !graph) {
    if (graph) hipGraphDestroy(graph);
    (void)hipGetLastError();
    return rc;
  }
  hipGraphExec_t g = nullptr;
  const hipError_t ei = hipGraphInstantiate(&g, graph, nullptr, nullptr, 0);
  hipGraphDestroy(graph);
  if (ei != hipSuccess || !g) {
    (void)hipGetLastError();
    return TFF_OK;
  }
  if ((int)cache.size() >= GRAPH_CACHE) {
    size_t v = 0;
    for (size_t k = 1; k < cache.size(); ++k)
      if (cache[k].used < cache[v].used) v = k;
    // a launch of the evicted graph may still be queued: let it finish first
    (void)hipDeviceSynchronize();
    hipGraphExecDestroy(cache[v].ex);
    cache.erase(cache.begin() + (long)v);
  }
  cache.push_back({key, g, ++g_graph_clock});
  g_seen_valid[key.dev] = false;
  *ex = g;
  return TFF_OK;
}

// Launches the executable graph of key on st, from the cache or newly captured (graph_capture).
// The launch happens under the cache's lock, so no other thread evicts the graph meanwhile.
// *launched stays false when this call should run without a graph.
template <typename F>
int graph_launch(const FusedKey& key, F&& launch_core, hipStream_t st, bool* launched) {
  *launched = false;
  std::lock_guard<std::mutex> lk(g_graph_mu);
  hipGraphExec_t ex = nullptr;
  for (GraphEntry& e : g_graphs[key.dev])
    if (memcmp(&e.key, &key, sizeof key) == 0) {
      e.used = ++g_graph_clock;
      ex = e.ex;
      break;
    }
  if (!ex) {
    const int rc = graph_capture(key, launch_core, &ex);
    if (rc || !ex) return rc;
  }
  if (hipGraphLaunch(ex, st) != hipSuccess) {
    tff_set_error("fused: graph launch failed: %s", hipGetErrorString(hipGetLastError()));
    return TFF_ERR_LAUNCH;
  }
  *launched = true;
  return TFF_OK;
}

template <typename TI, typename TC>
int fused_forward_t(int io_dtype, int compute_dtype, const TI* coords, const TI* q, const TI* sig, const TI* eps,
                    long long n, const double* box_host, const TffBox& box, const Geo& g, const int64_t* row_ptr,
                    const int64_t* col, double cutoff, double list_cutoff, double alpha, double coul,
                    const int K[3], int order, const TC* mx, const TC* my, const TC* mz, double* energies,
                    TI* forces, int* status_out, const TI* box_dev, int* status_host, void* workspace,
                    const FusedWs& w, bool graphs, hipStream_t st) {
  auto core = [&](hipStream_t s) {
    return run_fused_core<TI, TC>(coords, q, sig, eps, n, box, g, row_ptr, col, cutoff, list_cutoff, alpha, coul, K,
                                  order, mx, my, mz, box_dev, w, s);
  };
  if (graphs && graphs_usable(st, sizeof(TC) == 4, n)) {
    FusedKey key;
    memset(&key, 0, sizeof key);  // padding included, the key is compared bytewise
    if (hipGetDevice(&key.dev) != hipSuccess || key.dev < 0 || key.dev >= 64) {
      tff_set_error("fused: no current device");
      return TFF_ERR_LAUNCH;
    }
    key.io = io_dtype;
    key.cd = compute_dtype;
    key.order = order;
    for (int a = 0; a < 3; ++a) key.K[a] = K[a];
    key.mode = g_overlap.load();
    key.natoms = n;
    const void* ptrs[11] = {coords, q, sig, eps, row_ptr, col, mx, my, mz, box_dev, workspace};
    for (int k = 0; k < 11; ++k) key.p[k] = ptrs[k];
    for (int k = 0; k < 9; ++k) key.d[k] = box_host[k];
    key.d[9] = cutoff;
    key.d[10] = list_cutoff;
    key.d[11] = alpha;
    key.d[12] = coul;
    bool launched = false;
    const int rc = graph_launch(key, core, st, &launched);
    if (rc) return rc;
    if (launched) return launch_fused_finalize<TI>(w, g, coul, alpha, energies, forces, status_out, status_host, st);
  }
  const int rc = core(st);
  if (rc) return rc;
  return launch_fused_finalize<TI>(w, g, coul, alpha, energies, forces, status_out, status_host, st);
}

int fused_forward(int io_dtype, int compute_dtype, const void* coords, const void* charges, const void* sigma,
                  const void* epsilon, long long natoms, const double* box_host, const int64_t* excl_row_ptr,
                  const int64_t* excl_col, double cutoff, double list_cutoff, double ewald_alpha,
                  double coul_constant, int K0, int K1, int K2, int order, const void* xmoduli, const void* ymoduli,
                  const void* zmoduli, double* energies_out, void* forces_out, int32_t* status_out,
                  const void* box_device, int32_t* status_host, void* workspace, size_t workspace_bytes, bool graphs,
                  hipStream_t stream) {
  TffBox box = tff_make_box(box_host);
  Geo g;
  if (!make_geo(box, natoms, list_cutoff, g)) {
    tff_set_error("fused: needs an orthorhombic periodic box (diagonal box matrix)");
    return TFF_ERR_UNSUPPORTED;
  }
  if (natoms <= 0 || !coords || !charges || !sigma || !epsilon || !energies_out || !forces_out || !status_out ||
      !xmoduli || !ymoduli || !zmoduli || !(cutoff > 0) || list_cutoff < cutoff || ewald_alpha < 0) {
    tff_set_error("fused: invalid arguments");
    return TFF_ERR_ARG;
  }
  if ((excl_row_ptr == nullptr) != (excl_col == nullptr)) {
    tff_set_error("fused: exclusion row_ptr and col must be given together");
    return TFF_ERR_ARG;
  }
  int K[3] = {K0, K1, K2};
  for (int a = 0; a < 3; ++a) {
    FftPlan p;
    if (K[a] < order || K[a] > 4096 || !make_plan(K[a], p)) {
      tff_set_error("fused: PME grid size %d must be 2^a 3^b 5^c and >= the spline order", K[a]);
      return TFF_ERR_UNSUPPORTED;
    }
  }
  for (int a = 0; a < 3; ++a)
    if (2.0 * list_cutoff > g.L[a]) {
      tff_set_error("fused: the box (%.4g nm) must exceed twice the list cutoff (%.4g nm) for the minimum image",
                    g.L[a], list_cutoff);
      return TFF_ERR_UNSUPPORTED;
    }
  size_t tc = compute_dtype == TFF_F64 ? 8 : 4;
  size_t need = carve(nullptr, natoms, g, K, tc).bytes;
  if (!workspace || workspace_bytes < need) {
    tff_set_error("fused: workspace too small (%zu < %zu)", workspace_bytes, need);
    return TFF_ERR_WORKSPACE;
  }
  FusedWs w = carve(workspace, natoms, g, K, tc);
#define TFF_RUN(TI, TC)                                                                                          \
  return fused_forward_t<TI, TC>(io_dtype, compute_dtype, (const TI*)coords, (const TI*)charges, (const TI*)sigma, \
                                 (const TI*)epsilon, natoms, box_host, box, g, excl_row_ptr, excl_col, cutoff,     \
                                 list_cutoff, ewald_alpha, coul_constant, K, order, (const TC*)xmoduli,            \
                                 (const TC*)ymoduli, (const TC*)zmoduli, energies_out, (TI*)forces_out,            \
                                 (int*)status_out, (const TI*)box_device, (int*)status_host, workspace, w, graphs, \
                                 stream)
  if (io_dtype == TFF_F64 && compute_dtype == TFF_F32) TFF_RUN(double, float);
  if (io_dtype == TFF_F32 && compute_dtype == TFF_F32) TFF_RUN(float, float);
  if (io_dtype == TFF_F64 && compute_dtype == TFF_F64) TFF_RUN(double, double);
  if (io_dtype == TFF_F32 && compute_dtype == TFF_F64) TFF_RUN(float, double);
#undef TFF_RUN
  tff_set_error("fused: unsupported dtype combination");
  return TFF_ERR_ARG;
}
}  // namespace

extern "C" void tff_fused_set_graphs(int mode) { g_graphs_mode.store(mode >= 0 && mode <= 2 ? mode : 1); }

extern "C" int tff_fused_energy_forces(int io_dtype, int compute_dtype, const void* coords, const void* charges,
                                       const void* sigma, const void* epsilon, long long natoms,
                                       const double* box_host, const int64_t* excl_row_ptr,
                                       const int64_t* excl_col, double cutoff, double list_cutoff,
                                       double ewald_alpha, double coul_constant, int K0, int K1, int K2, int order,
                                       const void* xmoduli, const void* ymoduli, const void* zmoduli,
                                       double* energies_out, void* forces_out, int32_t* status_out,
                                       const void* box_device, int32_t* status_host, void* workspace,
                                       size_t workspace_bytes, hipStream_t stream) {
  return fused_forward(io_dtype, compute_dtype, coords, charges, sigma, epsilon, natoms, box_host, excl_row_ptr,
                       excl_col, cutoff, list_cutoff, ewald_alpha, coul_constant, K0, K1, K2, order, xmoduli,
                       ymoduli, zmoduli, energies_out, forces_out, status_out, box_device, status_host, workspace,
                       workspace_bytes, true, stream);
}

// ---------------------------------------------------------------- allocation-free variant
// The workspace of tff_fused_energy_forces_noalloc is this array: each device holds one copy for
// the life of the process.  Host code never passes the array's name to a kernel (on the host it
// is only a stand-in for the symbol): the entry point looks up the device address of its copy
// with hipGetSymbolAddress once per device, at its first call there, and uses that address.
// Every call on one device shares the copy (and keeps the previous call's contents; every kernel
// of the call clears or overwrites what it reads first), so calls that overlap on one device race.
static __device__ __align__(256) unsigned char scratch[TFF_FUSED_SCRATCH_BYTES];

namespace {
std::mutex g_scratch_mu;
void* g_scratch_ptr[64];

// device address of this device's scratch copy and the auxiliary stream, set up once per device
int scratch_setup(void** out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    tff_set_error("fused noalloc: no current device");
    return TFF_ERR_LAUNCH;
  }
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
      void* p = nullptr;
      const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      if (e != hipSuccess || !p) {
        tff_set_error("fused noalloc: hipGetSymbolAddress of the scratch array failed (%s)", hipGetErrorString(e));
        return TFF_ERR_LAUNCH;
      }
      g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
  }
  std::lock_guard<std::mutex> lk(g_aux_mu);
  if (!aux_stream_setup_locked(dev)) {
    tff_set_error("fused noalloc: could not create the auxiliary stream");
    return TFF_ERR_LAUNCH;
  }
  return TFF_OK;
}
}  // namespace

extern "C" int tff_fused_energy_forces_noalloc(int io_dtype, int compute_dtype, const void* coords,
                                               const void* charges, const void* sigma, const void* epsilon,
                                               long long natoms, const double* box_host,
                                               const int64_t* excl_row_ptr, const int64_t* excl_col, double cutoff,
                                               double list_cutoff, double ewald_alpha, double coul_constant, int K0,
                                               int K1, int K2, int order, const void* xmoduli, const void* ymoduli,
                                               const void* zmoduli, double* energies_out, void* forces_out,
                                               int32_t* status_out, const void* box_device, int32_t* status_host,
                                               hipStream_t stream) {
  const size_t need = tff_fused_workspace_bytes(compute_dtype, natoms, box_host, list_cutoff, K0, K1, K2);
  if (need > TFF_FUSED_SCRATCH_BYTES) {
    tff_set_error("fused noalloc: this system needs %zu bytes of scratch, above the %zu of the static array "
                  "(use tff_fused_energy_forces with a workspace)", need, (size_t)TFF_FUSED_SCRATCH_BYTES);
    return TFF_ERR_WORKSPACE;
  }
  void* ws = nullptr;
  const int rc = scratch_setup(&ws);
  if (rc) return rc;
  return fused_forward(io_dtype, compute_dtype, coords, charges, sigma, epsilon, natoms, box_host, excl_row_ptr,
                       excl_col, cutoff, list_cutoff, ewald_alpha, coul_constant, K0, K1, K2, order, xmoduli,
                       ymoduli, zmoduli, energies_out, forces_out, status_out, box_device, status_host, ws,
                       (size_t)TFF_FUSED_SCRATCH_BYTES, false, stream);
}
