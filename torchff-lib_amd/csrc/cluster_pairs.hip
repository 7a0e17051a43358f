// Cluster-pair neighbour list in the reference's five-tensor format, its decoding into atom
// pairs, and the nonbonded energy / forces evaluated directly on it (no (P, 2) pair list).
//
// Format (torchff/nblist.py:260-344; csrc/nblist/nblist_cluster_pairs_cuda.cu:18-525, which the
// reference's setup.py does not build, and the commented schemas of
// csrc/nonbonded/nonbonded_interface.cpp:5-8):
//   sorted_atom_indices (N, int32)     slot -> atom; cluster c owns slots 32c .. 32c + 31
//   cluster_exclusions (2, E, int32)   cluster pairs (x, y), x <= y, whose 32 x 32 block holds an
//                                      excluded atom pair, plus every diagonal (x, x)
//   bitmask_exclusions (E, 32, uint32) word [e][l], bit k: skip (slot 32x + l, slot 32y + k)
//                                      (excluded, an empty slot, or k <= l on the diagonal)
//   interacting_clusters (M, int32)    row -> cluster x
//   interacting_atoms (M, 32, int32)   atoms of clusters y > x (not in x's exclusion set) whose
//                                      minimum-image distance to x's bounding sphere is within the
//                                      cutoff, 32 per row in cluster-then-slot order, -1 padded
// Every atom pair within the cutoff and not excluded is visited exactly once: clusters listed in
// x's exclusion set through their bitmask block, all others through x's rows.
//
// Build (deterministic: counting passes, scans, then writes at fixed offsets):
//   k_cp_keys / k_cp_scan / k_cp_scatter / k_cp_rank  cell sort (cells cs x cs x cs/10 as in the
//        reference, z fastest; refined when they would hold more than 8 atoms on average), the
//        atoms of a cell ordered by index;
//   k_cp_bounds      half a wave per cluster: minimum-image offsets from the first atom, bounding
//                    box centre and enclosing radius;
//   k_cp_excl        half a wave per cluster: distinct partner clusters y >= x of its exclusions;
//   k_cp_rows<WRITE> a workgroup per cluster: sphere tests against the clusters above it, then
//                    atom tests; the count pass sizes the rows, the write pass fills them.
// The sphere tests are exact for the fractional-rounding minimum image while the radii plus the
// cutoff stay below half the smallest box height; beyond that the candidates are kept untested
// (the traversal applies the exact cutoff test to every pair).
//
// Traversal (decode and nonbonded): half a wave per entry (exclusion blocks first, then rows);
// lane l holds atom i of slot 32x + l and atom j of column l, and walks the 32 columns by
// shuffles.  Pairs come out in entry, lane, column order at offsets from a count pass and a scan.

#include <cmath>
#include <type_traits>

#include "pair_math.h"
#include "tff_common.h"
#include "torchff_hip.h"

namespace {

constexpr int CPW = 32;        // atoms per cluster / row width of the format
constexpr int CPB = 256;       // threads per workgroup (4 waves, 8 half-waves)
constexpr int CP_EXMAX = 16;   // exclusion partners per atom
constexpr int CP_XCL = 32;     // distinct exclusion partner clusters per cluster
constexpr int CP_MAXBLK = 4096;

enum { CP_FLAG_EXCL_ATOM = 1, CP_FLAG_EXCL_CLUSTER = 2 };

__device__ __forceinline__ int half_lane() { return threadIdx.x & 31; }
__device__ __forceinline__ int half_index() { return (blockIdx.x * CPB + threadIdx.x) >> 5; }
__device__ __forceinline__ int half_count() { return (gridDim.x * CPB) >> 5; }
// bits of this half-wave in a wave-wide ballot
__device__ __forceinline__ unsigned half_ballot(bool v) {
  const unsigned long long b = __builtin_amdgcn_ballot_w64(v);
  return (unsigned)(b >> (threadIdx.x & 32));
}
__device__ __forceinline__ int half_min(int v) {
  for (int o = 16; o > 0; o >>= 1) {
    const int w = __shfl_xor(v, o, 32);
    v = w < v ? w : v;
  }
  return v;
}
__device__ __forceinline__ double half_max(double v) {
  for (int o = 16; o > 0; o >>= 1) {
    const double w = __shfl_xor(v, o, 32);
    v = w > v ? w : v;
  }
  return v;
}
__device__ __forceinline__ double half_minf(double v) {
  for (int o = 16; o > 0; o >>= 1) {
    const double w = __shfl_xor(v, o, 32);
    v = w < v ? w : v;
  }
  return v;
}

struct CpGeom {
  TffBox box;
  double rc2;
  double rc;
  double half_h;  // half the smallest box height
  int nc[3];
  int natoms;
  int nclusters;
};

template <typename T>
__device__ __forceinline__ void load_xyz(const T* c, int a, double& x, double& y, double& z) {
  x = (double)c[3 * a];
  y = (double)c[3 * a + 1];
  z = (double)c[3 * a + 2];
}

// ---------------------------------------------------------------- cell sort
template <typename T>
__global__ void k_cp_keys(const T* __restrict__ coords, CpGeom g, int* __restrict__ cell_of,
                          int* __restrict__ count, int* __restrict__ flags) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) flags[0] = 0;
  if (i >= g.natoms) return;
  double x, y, z;
  load_xyz(coords, i, x, y, z);
  const double f[3] = {x * g.box.inv[0] + y * g.box.inv[3] + z * g.box.inv[6],
                       x * g.box.inv[1] + y * g.box.inv[4] + z * g.box.inv[7],
                       x * g.box.inv[2] + y * g.box.inv[5] + z * g.box.inv[8]};
  int c[3];
  for (int k = 0; k < 3; ++k) {
    const double fk = f[k] - floor(f[k]);
    const int ck = (int)(fk * g.nc[k]);
    c[k] = ck < 0 ? 0 : (ck >= g.nc[k] ? g.nc[k] - 1 : ck);
  }
  const int cell = (c[0] * g.nc[1] + c[1]) * g.nc[2] + c[2];
  cell_of[i] = cell;
  atomicAdd(&count[cell], 1);
}

// exclusive scan of cnt[0..m) into off[0..m] (off[m] = total), one workgroup of 1024 threads
template <typename C, typename O>
__global__ __launch_bounds__(1024) void k_cp_scan(const C* __restrict__ cnt, long long m, O* __restrict__ off) {
  tff_block_scan_1024<C, O>(cnt, m, off, true);
}

// the same over many workgroups: the sums of CP_SCAN entries each, then every workgroup adds up the
// sums before its own (42k cells: two launches of 3 us; one workgroup walking them took 25)
constexpr int CP_SCAN = 4096;
template <typename C, typename O>
__global__ __launch_bounds__(1024) void k_cp_scan_sums(const C* __restrict__ cnt, long long m, O* __restrict__ sums) {
  const long long base = (long long)blockIdx.x * CP_SCAN;
  O v = 0;
  for (int k = threadIdx.x; k < CP_SCAN; k += 1024) v += base + k < m ? (O)cnt[base + k] : (O)0;
  __shared__ O s_w[1024 / TFF_WAVE];
  for (int o = TFF_WAVE / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, TFF_WAVE);
  if (threadIdx.x % TFF_WAVE == 0) s_w[threadIdx.x / TFF_WAVE] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    O t = 0;
    for (int w = 0; w < 1024 / TFF_WAVE; ++w) t += s_w[w];
    sums[blockIdx.x] = t;
  }
}
template <typename C, typename O>
__global__ __launch_bounds__(1024) void k_cp_scan_tiles(const C* __restrict__ cnt, long long m,
                                                        const O* __restrict__ sums, O* __restrict__ off) {
  __shared__ O s_w[1024 / TFF_WAVE], s_t[1024 / TFF_WAVE];
  const int t = threadIdx.x, lane = t % TFF_WAVE, wv = t / TFF_WAVE;
  O before = 0;
  for (int b = t; b < (int)blockIdx.x; b += 1024) before += sums[b];
  for (int o = TFF_WAVE / 2; o > 0; o >>= 1) before += __shfl_xor(before, o, TFF_WAVE);
  const long long i0 = (long long)blockIdx.x * CP_SCAN + 4 * t;
  O v[4], local = 0;
  for (int k = 0; k < 4; ++k) {
    v[k] = i0 + k < m ? (O)cnt[i0 + k] : (O)0;
    local += v[k];
  }
  O incl = local;
  for (int o = 1; o < TFF_WAVE; o <<= 1) {
    const O x = __shfl_up(incl, o, TFF_WAVE);
    if (lane >= o) incl += x;
  }
  if (lane == 0) s_t[wv] = before;
  if (lane == TFF_WAVE - 1) s_w[wv] = incl;
  __syncthreads();
  O run = incl - local;
  for (int w = 0; w < 1024 / TFF_WAVE; ++w) run += s_t[w] + (w < wv ? s_w[w] : (O)0);
  for (int k = 0; k < 4; ++k) {
    if (i0 + k < m) off[i0 + k] = run;
    run += v[k];
    if (i0 + k == m - 1) off[m] = run;
  }
}

// (the counts are used up)
__global__ void k_cp_scatter(int n, const int* __restrict__ cell_of, const int* __restrict__ start,
                             int* __restrict__ count, int* __restrict__ seg) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int c = cell_of[i];
  seg[start[c] + atomicSub(&count[c], 1) - 1] = i;
}

// place each atom at its rank by index within its cell
__global__ void k_cp_rank(int n, const int* __restrict__ cell_of, const int* __restrict__ start,
                          const int* __restrict__ seg, int* __restrict__ sorted, int* __restrict__ inv) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int c = cell_of[i];
  const int b = start[c], e = start[c + 1];
  int r = 0;
  for (int k = b; k < e; ++k) r += seg[k] < i;
  sorted[b + r] = i;
  inv[i] = b + r;
}

// ---------------------------------------------------------------- cluster bounds
template <typename T>
__global__ __launch_bounds__(CPB) void k_cp_bounds(const T* __restrict__ coords, CpGeom g,
                                                   const int* __restrict__ sorted, double4* __restrict__ sphere) {
  const int l = half_lane();
  for (int c = half_index(); c < g.nclusters; c += half_count()) {
    const int slot = c * CPW + l;
    const bool ok = slot < g.natoms;
    double x = 0, y = 0, z = 0;
    if (ok) load_xyz(coords, sorted[slot], x, y, z);
    const double ax = __shfl(x, 0, 32), ay = __shfl(y, 0, 32), az = __shfl(z, 0, 32);
    double dx = x - ax, dy = y - ay, dz = z - az;
    tff_min_image_d(g.box, dx, dy, dz);
    const double lo[3] = {half_minf(ok ? dx : 1e300), half_minf(ok ? dy : 1e300), half_minf(ok ? dz : 1e300)};
    const double hi[3] = {half_max(ok ? dx : -1e300), half_max(ok ? dy : -1e300), half_max(ok ? dz : -1e300)};
    const double mx = 0.5 * (lo[0] + hi[0]), my = 0.5 * (lo[1] + hi[1]), mz = 0.5 * (lo[2] + hi[2]);
    const double ex = dx - mx, ey = dy - my, ez = dz - mz;
    const double r = half_max(ok ? sqrt(ex * ex + ey * ey + ez * ez) : 0.0);
    if (l == 0) sphere[c] = make_double4(ax + mx, ay + my, az + mz, r * (1.0 + 1e-12) + 1e-12);
  }
}

// ---------------------------------------------------------------- exclusion blocks
// the smallest partner cluster above `last` among atom i's exclusions (INT_MAX if none)
__device__ __forceinline__ int next_partner(int i, int x, int last, const long long* __restrict__ rp,
                                            const long long* __restrict__ col, const int* __restrict__ inv,
                                            int natoms, int* flags) {
  int best = 0x7fffffff;
  if (i < 0 || !rp) return best;  // no exclusion list: only the diagonal block
  const long long b = rp[i], e = rp[i + 1];
  if (e - b > CP_EXMAX && flags) {  // (negative entries are padding)
    bool more = false;
    for (long long k = b + CP_EXMAX; k < e; ++k) more |= col[k] >= 0;
    if (more) atomicOr(flags, CP_FLAG_EXCL_ATOM);
  }
  for (long long k = b; k < e && k < b + CP_EXMAX; ++k) {
    const long long j = col[k];
    if (j < 0 || j >= natoms) continue;
    const int cy = inv[j] / CPW;
    if (cy >= x && cy > last && cy < best) best = cy;
  }
  return best;
}

__global__ __launch_bounds__(CPB) void k_cp_excl(CpGeom g, const int* __restrict__ sorted,
                                                 const int* __restrict__ inv, const long long* __restrict__ rp,
                                                 const long long* __restrict__ col, int* __restrict__ xlist,
                                                 int* __restrict__ xcount, int* __restrict__ flags) {
  const int l = half_lane();
  for (int x = half_index(); x < g.nclusters; x += half_count()) {
    const int slot = x * CPW + l;
    const int i = slot < g.natoms ? sorted[slot] : -1;
    int n = 0;
    if (l == 0) xlist[x * CP_XCL] = x;  // the diagonal block is always present
    n = 1;
    int last = x;
    while (true) {
      const int nx = half_min(next_partner(i, x, last, rp, col, inv, g.natoms, flags));
      if (nx == 0x7fffffff) break;
      if (n >= CP_XCL) {
        if (l == 0) atomicOr(flags, CP_FLAG_EXCL_CLUSTER);
        break;
      }
      if (l == 0) xlist[x * CP_XCL + n] = nx;
      ++n;
      last = nx;
    }
    if (l == 0) xcount[x] = n;
  }
}

// One half-wave per cluster x: the blocks of its partner clusters.  Lane l sets its word's bits from its own
// atom's exclusions (their slots by `inv`) rather than searching them for each of the 32 columns
// (96k water atoms: 5 us instead of 29).
__global__ __launch_bounds__(CPB) void k_cp_excl_emit(CpGeom g, const int* __restrict__ sorted,
                                                      const int* __restrict__ inv,
                                                      const long long* __restrict__ rp,
                                                      const long long* __restrict__ col,
                                                      const int* __restrict__ xlist, const int* __restrict__ xcount,
                                                      const int* __restrict__ xoff, int ecap,
                                                      int* __restrict__ coo, unsigned* __restrict__ mask) {
  const int l = half_lane();
  for (int x = half_index(); x < g.nclusters; x += half_count()) {
    const int slot = x * CPW + l;
    const int i = slot < g.natoms ? sorted[slot] : -1;
    const int n = xcount[x], o0 = xoff[x];
    const long long b = rp && i >= 0 ? rp[i] : 0, e = rp && i >= 0 ? rp[i + 1] : 0;
    for (int k = 0; k < n; ++k) {
      const int o = o0 + k;
      if (o >= ecap) break;
      const int y = xlist[x * CP_XCL + k];
      const int left = g.natoms - y * CPW;  // atoms from this cluster on
      unsigned m = i < 0 ? 0xffffffffu : left < CPW ? 0xffffffffu << left : 0u;
      if (x == y) m |= 0xffffffffu >> (31 - l);  // columns c <= l
      for (long long k2 = b; k2 < e; ++k2) {
        const long long j = col[k2];
        if (j < 0 || j >= g.natoms) continue;
        const int sj = inv[j];
        if (sj / CPW == y) m |= 1u << (sj % CPW);
      }
      mask[(size_t)o * CPW + l] = m;
      if (l == 0) {
        coo[o] = x;
        coo[ecap + o] = y;
      }
    }
  }
}

// ---------------------------------------------------------------- interacting rows
// One workgroup per cluster x, CP_TILE clusters y > x at a time: the sphere tests fill a bit mask, its bits
// become an ordered candidate list, the 8 half-waves take the candidates in turn for the atom tests
// (a 32-bit hit mask each), and a scan of their counts gives every candidate its place in the rows.
// Bound by the latency of the candidates' two dependent loads (slot -> atom -> position): 96k water
// atoms, count and write pass 29 and 33 us; with one half-wave walking all of a cluster's candidates
// the 1500 waves took 89 and 94.
constexpr int CP_TILE = 2048;

template <typename T, bool WRITE>
__global__ __launch_bounds__(CPB) void k_cp_rows(const T* __restrict__ coords, CpGeom g,
                                                 const int* __restrict__ sorted,
                                                 const double4* __restrict__ sphere,
                                                 const int* __restrict__ xlist, const int* __restrict__ xcount,
                                                 int* __restrict__ natoms_of, const long long* __restrict__ row_off,
                                                 long long mcap, int* __restrict__ ic, int* __restrict__ ia) {
  __shared__ unsigned s_word[CP_TILE / 32], s_hit[CP_TILE];
  __shared__ unsigned short s_cand[CP_TILE];
  __shared__ int s_pos[CP_TILE], s_sum[CPB / TFF_WAVE], s_ncand, s_ex[CP_XCL];
  const int t = threadIdx.x, l = half_lane(), hw = t >> 5, lane = t & (TFF_WAVE - 1);
  for (int x = blockIdx.x; x < g.nclusters; x += gridDim.x) {
    const double4 sx = sphere[x];
    const int nx = xcount[x];
    __syncthreads();
    if (t < nx) s_ex[t] = xlist[x * CP_XCL + t];
    __syncthreads();
    const bool all_atoms = sx.w + g.rc > g.half_h;
    const double rr2 = (sx.w + g.rc) * (sx.w + g.rc);
    long long total = 0;  // atoms of the tiles so far
    const long long base = WRITE ? row_off[x] : 0;
    for (int y0 = x + 1; y0 < g.nclusters; y0 += CP_TILE) {
      const int ny = g.nclusters - y0 < CP_TILE ? g.nclusters - y0 : CP_TILE, nw = (ny + 31) / 32;
      for (int w = hw; w < nw; w += CPB / 32) {
        const int y = y0 + 32 * w + l;
        bool inc = false;
        if (y < g.nclusters) {
          bool ex = false;
          for (int k = 1; k < nx; ++k) ex |= s_ex[k] == y;
          if (!ex) {
            const double4 sy = sphere[y];
            const double bound = sx.w + sy.w + g.rc;
            if (bound > g.half_h) {
              inc = true;
            } else {
              double dx = sx.x - sy.x, dy = sx.y - sy.y, dz = sx.z - sy.z;
              tff_min_image_d(g.box, dx, dy, dz);
              inc = dx * dx + dy * dy + dz * dz <= bound * bound;
            }
          }
        }
        const unsigned m = half_ballot(inc);
        if (l == 0) s_word[w] = m;
      }
      __syncthreads();
      if (t < TFF_WAVE) {  // the candidates in order (CP_TILE / 32 = one wave of words)
        unsigned m = t < nw ? s_word[t] : 0u;
        const int n = __builtin_popcount(m);
        int incl = n;
        for (int o = 1; o < TFF_WAVE; o <<= 1) {
          const int v = __shfl_up(incl, o, TFF_WAVE);
          if (t >= o) incl += v;
        }
        int k = incl - n;
        for (; m; m &= m - 1) s_cand[k++] = (unsigned short)(32 * t + __builtin_ctz(m));
        if (t == TFF_WAVE - 1) s_ncand = incl;
      }
      __syncthreads();
      const int nc = s_ncand;
      for (int k = hw; k < nc; k += CPB / 32) {
        const int slot = (y0 + s_cand[k]) * CPW + l;
        bool hit = false;
        if (slot < g.natoms) {
          if (all_atoms) {
            hit = true;
          } else {
            double px, py, pz;
            load_xyz(coords, sorted[slot], px, py, pz);
            double dx = px - sx.x, dy = py - sx.y, dz = pz - sx.z;
            tff_min_image_d(g.box, dx, dy, dz);
            hit = dx * dx + dy * dy + dz * dz <= rr2;
          }
        }
        const unsigned hb = half_ballot(hit);
        if (l == 0) s_hit[k] = hb;
      }
      __syncthreads();
      // places of the candidates: each thread sums CP_TILE / CPB neighbours
      constexpr int PER = CP_TILE / CPB;
      int sum = 0;
      for (int k = PER * t; k < PER * (t + 1) && k < nc; ++k) sum += __builtin_popcount(s_hit[k]);
      int incl = sum;
      for (int o = 1; o < TFF_WAVE; o <<= 1) {
        const int v = __shfl_up(incl, o, TFF_WAVE);
        if (lane >= o) incl += v;
      }
      if (lane == TFF_WAVE - 1) s_sum[t / TFF_WAVE] = incl;
      __syncthreads();
      int tile = 0, before = incl - sum;
      for (int w = 0; w < CPB / TFF_WAVE; ++w) {
        if (w < t / TFF_WAVE) before += s_sum[w];
        tile += s_sum[w];
      }
      if (WRITE) {
        for (int k = PER * t; k < PER * (t + 1) && k < nc; ++k) {
          s_pos[k] = before;
          before += __builtin_popcount(s_hit[k]);
        }
        __syncthreads();
        for (int k = hw; k < nc; k += CPB / 32) {
          const unsigned hb = s_hit[k];
          if ((hb >> l) & 1u) {
            const long long ord = total + s_pos[k] + __builtin_popcount(hb & ((1u << l) - 1u));
            const long long row = base + ord / CPW;
            if (row < mcap) ia[row * CPW + ord % CPW] = sorted[(y0 + s_cand[k]) * CPW + l];
          }
        }
      }
      total += tile;
      __syncthreads();  // the lists are free for the next tile
    }
    const long long rows = (total + CPW - 1) / CPW;
    if (!WRITE) {
      if (t == 0) natoms_of[x] = (int)rows;
    } else {
      for (long long r = t; r < rows; r += CPB)
        if (base + r < mcap) ic[base + r] = x;
      // pad the last row
      const long long last = total % CPW;
      if (last && t >= last && t < CPW && base + rows - 1 < mcap) ia[(base + rows - 1) * CPW + t] = -1;
    }
  }
}
static_assert(CP_TILE / 32 == TFF_WAVE && CP_TILE <= 65536, "one wave lists the candidates, in 16 bits");

__global__ void k_cp_fill(int* p, long long from, long long to, int v) {
  for (long long k = from + blockIdx.x * (long long)blockDim.x + threadIdx.x; k < to;
       k += (long long)gridDim.x * blockDim.x)
    p[k] = v;
}

// row offsets of the clusters, and the totals
__global__ __launch_bounds__(1024) void k_cp_rows_scan(const int* __restrict__ rows, int nclusters,
                                                       const int* __restrict__ xoff, const int* __restrict__ flags,
                                                       long long* __restrict__ row_off,
                                                       long long* __restrict__ out) {
  const long long total = tff_block_scan_1024<int, long long>(rows, nclusters, row_off, true);
  if (threadIdx.x == 0) {
    out[0] = xoff[nclusters];
    out[1] = total;
    out[2] = flags[0];
  }
}

// the sorted atoms, and -1 behind the last entry of each array
__global__ void k_cp_pad(const int* __restrict__ sorted, int natoms, const int* __restrict__ xoff,
                         const long long* __restrict__ row_off, int nclusters, int* __restrict__ sorted_out,
                         long long ecap, int* __restrict__ coo, unsigned* __restrict__ mask, long long mcap,
                         int* __restrict__ ic, int* __restrict__ ia) {
  const long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x, nt = (long long)gridDim.x * blockDim.x;
  const long long E = xoff[nclusters], M = row_off[nclusters];
  for (long long k = t; k < natoms; k += nt) sorted_out[k] = sorted[k];
  for (long long k = E + t; k < ecap; k += nt) coo[k] = coo[ecap + k] = -1;
  for (long long k = E * CPW + t; k < ecap * CPW; k += nt) mask[k] = 0xffffffffu;
  for (long long k = M + t; k < mcap; k += nt) ic[k] = -1;
  for (long long k = M * CPW + t; k < mcap * CPW; k += nt) ia[k] = -1;
}

// ---------------------------------------------------------------- exclusion lists
// Symmetric CSR of a COO pair list for the build, by counting (two atomics per pair): pairs with a negative
// index are left out, an index past the atoms sets the status; a row's repeated partners are
// dropped, its tail filled with -1 (17 distinct ones are kept: more than the build accepts).  Rows come
// in any order, which neither the partner clusters nor the masks depend on.  Replaces a sort and a
// unique of 2 E keys and twenty elementwise launches (96k pairs: 26 us instead of 180).
__device__ __forceinline__ bool coo_pair(const long long* __restrict__ p, long long E, int rows2, long long k,
                                         long long n, long long& i, long long& j, long long* __restrict__ status) {
  i = rows2 ? p[k] : p[2 * k];
  j = rows2 ? p[E + k] : p[2 * k + 1];
  if (i < 0 || j < 0) return false;
  if (i >= n || j >= n) {
    if (status) status[0] = 1;
    return false;
  }
  return true;
}
__global__ void k_cp_csr_count(const long long* __restrict__ p, long long E, int rows2, long long n,
                               int* __restrict__ cnt, long long* __restrict__ status) {
  for (long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x; k < E; k += (long long)gridDim.x * blockDim.x) {
    long long i, j;
    if (!coo_pair(p, E, rows2, k, n, i, j, status)) continue;
    atomicAdd(&cnt[i], 1);
    atomicAdd(&cnt[j], 1);
  }
}
__global__ void k_cp_csr_fill(const long long* __restrict__ p, long long E, int rows2, long long n,
                              int* __restrict__ cnt, const long long* __restrict__ rp, long long* __restrict__ col) {
  for (long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x; k < E; k += (long long)gridDim.x * blockDim.x) {
    long long i, j;
    if (!coo_pair(p, E, rows2, k, n, i, j, nullptr)) continue;
    col[rp[i] + atomicSub(&cnt[i], 1) - 1] = j;
    col[rp[j] + atomicSub(&cnt[j], 1) - 1] = i;
  }
}
__global__ void k_cp_csr_unique(long long n, const long long* __restrict__ rp, long long* __restrict__ col) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const long long b = rp[i], e = rp[i + 1];
  long long w = b;
  for (long long k = b; k < e; ++k) {
    const long long j = col[k];
    bool seen = w - b > CP_EXMAX;
    for (long long m = b; m < w && !seen; ++m) seen = col[m] == j;
    if (!seen) col[w++] = j;
  }
  for (; w < e; ++w) col[w] = -1;
}

// ---------------------------------------------------------------- traversal
struct Entries {
  const int* sorted;
  const int* coo;      // (2, E)
  long long E;
  const unsigned* mask;
  const int* ic;       // (M)
  const int* ia;       // (M, 32)
  long long M;
};

// the atom of a slot, -1 for a slot past the end or an index out of range
__device__ __forceinline__ int slot_atom(const int* __restrict__ sorted, long long slot, int natoms) {
  if (slot >= natoms) return -1;
  const int a = sorted[slot];
  return a >= 0 && a < natoms ? a : -1;
}

// lane's atom i, column atom j and skip mask for entry e; false if the entry is padding
__device__ __forceinline__ bool entry_atoms(const Entries& en, long long e, int natoms, int nclusters, int l, int& i,
                                            int& j, unsigned& skip) {
  if (e < en.E) {
    const int x = en.coo[e], y = en.coo[en.E + e];
    if (x < 0 || y < 0 || x > y || y >= nclusters) return false;
    i = slot_atom(en.sorted, (long long)x * CPW + l, natoms);
    j = slot_atom(en.sorted, (long long)y * CPW + l, natoms);
    skip = en.mask[e * CPW + l];
    return true;
  }
  const long long r = e - en.E;
  const int x = en.ic[r];
  if (x < 0 || x >= nclusters) return false;
  i = slot_atom(en.sorted, (long long)x * CPW + l, natoms);
  j = en.ia[r * CPW + l];
  if (j >= natoms) j = -1;
  skip = 0;
  return true;
}

enum { TR_COUNT = 0, TR_WRITE = 1 };

template <typename T, int MODE>
__global__ __launch_bounds__(CPB) void k_cp_decode(const T* __restrict__ coords, CpGeom g, Entries en,
                                                   int* __restrict__ cnt, const long long* __restrict__ off,
                                                   long long cap, int* __restrict__ pairs) {
  const int l = half_lane();
  const long long total = en.E + en.M;
  for (long long e = half_index(); e < total; e += half_count()) {
    int i = -1, j = -1;
    unsigned skip = 0xffffffffu;
    const bool live = entry_atoms(en, e, g.natoms, g.nclusters, l, i, j, skip);
    double xi = 0, yi = 0, zi = 0, xj = 0, yj = 0, zj = 0;
    if (live && i >= 0) load_xyz(coords, i, xi, yi, zi);
    if (live && j >= 0) load_xyz(coords, j, xj, yj, zj);
    int n = 0;
    unsigned hits = 0;
    for (int c = 0; c < CPW; ++c) {
      const int jc = __shfl(j, c, 32);
      const double dx0 = xi - __shfl(xj, c, 32), dy0 = yi - __shfl(yj, c, 32), dz0 = zi - __shfl(zj, c, 32);
      double dx = dx0, dy = dy0, dz = dz0;
      tff_min_image_d(g.box, dx, dy, dz);
      const bool ok = live && i >= 0 && jc >= 0 && !((skip >> c) & 1u) && dx * dx + dy * dy + dz * dz <= g.rc2;
      hits |= (unsigned)ok << c;
      n += ok;
    }
    if (MODE == TR_COUNT) {
      int s = n;
      for (int o = 16; o > 0; o >>= 1) s += __shfl_xor(s, o, 32);
      if (l == 0) cnt[e] = s;
    } else {
      // lanes below this one write first
      int pre = n;
      for (int o = 1; o < 32; o <<= 1) {
        const int v = __shfl_up(pre, o, 32);
        if (l >= o) pre += v;
      }
      long long p = off[e] + pre - n;
      for (int c = 0; c < CPW; ++c) {
        const int jc = __shfl(j, c, 32);
        if ((hits >> c) & 1u) {
          if (p < cap) {
            pairs[2 * p] = i;
            pairs[2 * p + 1] = jc;
          }
          ++p;
        }
      }
    }
  }
}

__global__ void k_cp_npairs(const long long* __restrict__ off, long long total, long long cap, int* __restrict__ np,
                            int* __restrict__ pairs) {
  const long long n = off[total];
  if (blockIdx.x == 0 && threadIdx.x == 0) np[0] = (int)n;
  // -1 padding after the last pair
  for (long long k = n + blockIdx.x * (long long)blockDim.x + threadIdx.x; k < cap;
       k += (long long)gridDim.x * blockDim.x) {
    pairs[2 * k] = -1;
    pairs[2 * k + 1] = -1;
  }
}

// ---------------------------------------------------------------- nonbonded terms
// 16-lane row rotation: lane l takes the value of lane l - K of its row
template <int K>
__device__ __forceinline__ int ror(int v) { return __builtin_amdgcn_mov_dpp(v, 0x120 + K, 0xf, 0xf, true); }
template <int K>
__device__ __forceinline__ float ror(float v) { return __int_as_float(ror<K>(__float_as_int(v))); }
template <int K>
__device__ __forceinline__ double ror(double v) {
  return __hiloint2double(ror<K>(__double2hiint(v)), ror<K>(__double2loint(v)));
}
__device__ __forceinline__ void half_sync() {  // the wave's own LDS writes before its reads
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// 1 / sqrt(x), sqrt(x) and a / b to within an ulp (float: the hardware's, corrected by one step whose
// residual is exact; zero, infinite and denormal x as the hardware gives them)
__device__ __forceinline__ float cp_rsqrt(float x) {
  const float y = __builtin_amdgcn_rsqf(x), h = x * y;
  const float e = fmaf(-h, y, 1.0f) - fmaf(x, y, -h) * y;
  return fabsf(e) < 1.0f ? fmaf(0.5f * y, e, y) : y;
}
__device__ __forceinline__ double cp_rsqrt(double x) { return rsqrt_t(x); }
__device__ __forceinline__ float cp_sqrt(float x) {
  const float s = __builtin_amdgcn_sqrtf(x), h = 0.5f * __builtin_amdgcn_rsqf(x);
  float f = fmaf(fmaf(-s, s, x), h, s);
  const bool mid = x > 1e-30f && x < 1e30f;
  if (__builtin_amdgcn_ballot_w64(!mid && x != 0.0f)) {  // rare
    asm volatile("");                                    // (kept a branch)
    f = mid ? f : sqrtf(x);
  }
  return x == 0.0f ? x : f;
}
__device__ __forceinline__ double cp_sqrt(double x) { return sqrt(x); }
__device__ __forceinline__ float cp_div(float a, float b) {
  const float y = __builtin_amdgcn_rcpf(b), d = a * y;
  return fabsf(d) < INFINITY ? fmaf(fmaf(-b, d, a), y, d) : d;
}
__device__ __forceinline__ double cp_div(double a, double b) { return a / b; }

// Accumulators: CH doubles per atom (x, y, z, q and, with the Lennard-Jones gradients, sigma, eps, -, -),
// one 32 or 64 byte piece of a line each.
template <bool LJG>
struct CpCh {
  static constexpr int ST = LJG ? 8 : 4;  // doubles per atom
  static constexpr int N = LJG ? 6 : 4;   // of them in use
};

// The atoms `a` (one per lane of the half-wave, -1 for none) with N channels each, added to the
// accumulators: through LDS, so that the lanes of one instruction hold the channels of few atoms.  An
// atomic costs a memory-side operation per line it touches: one per atom here, one per atom and
// channel when each lane adds its own atom's.
template <bool LJG>
__device__ __forceinline__ void cp_flush(int a, const double (&v)[CpCh<LJG>::N], double* __restrict__ s,
                                         double* __restrict__ acc) {
  constexpr int ST = CpCh<LJG>::ST, N = CpCh<LJG>::N, PAD = ST + 1;
  const int l = half_lane();
  half_sync();
#pragma unroll
  for (int k = 0; k < N; ++k) s[l * PAD + k] = v[k];
  half_sync();
  const int k = l % ST;
#pragma unroll
  for (int r = 0; r < ST; ++r) {
    const int m = r * (CPW / ST) + l / ST;
    const int am = __shfl(a, m, 32);
    if (k < N && am >= 0) {
      const double x = s[m * PAD + k];
      if (x != 0.0) atomicAdd(&acc[(size_t)am * ST + k], x);
    }
  }
}

// nonbonded energy and gradients on the cluster pairs: k q_i q_j (1/r - [1/rc]) + 4 eps s^6 (s^6 - 1),
// sigma and eps by Lorentz-Berthelot, the same pair term as compute_nonbonded_energy_from_atom_pairs.
// GRAD: 0 energy only, 1 with coordinates and charges, 2 with sigma and epsilon too.
//
// A half-wave takes a run of consecutive entries (they mostly share their cluster x, whose atoms' sums
// stay in registers, float64, until x changes).  Its two rows of 16 lanes take 16 of the column atoms
// each, which then go round the row by DPP together with their sums, 16 steps, twice: no shuffle and no
// reduction per column.  A column's sums are T for CP_CHAIN steps and float64 from there on: for 32 terms of
// like size their squared rounding error is 140 (in units of a rounding of one term), where a butterfly over
// the rows has 160 and one sum over all steps 527.  (List and terms of the call below: 463 us with one sum,
// 470 with chains of 8, 474 of 4, which spill.)
// The pair predicate is that of the decoded list, in float64: T = float decides by its own r^2
// unless that is within its error bound `tol_k` (|x_i| + |x_j| + box) of rc^2.
// Bound by the arithmetic of the candidate pairs (of 32 x 32 per entry about one in five is within the
// cutoff; some 150 instructions a step).  96k water atoms, float, all gradients: 283 us (energy alone
// 150); one column per step by shuffles, a butterfly per gradient and an atomic per atom and channel
// took 683.  Testing all pairs first and working off each lane's hits, with the column sums in LDS, took
// 828: the fullest lane of 64 has nearly all 32 columns.
// ORTHO: the box is orthorhombic.
constexpr int CP_CHAIN = 8;
template <typename T, int GRAD, bool ORTHO>
__global__ __launch_bounds__(CPB) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 3))) void k_cp_nonbonded(
    const T* __restrict__ coords, CpGeom g, Entries en, int run, const T* __restrict__ q, const T* __restrict__ sig,
    const T* __restrict__ eps, double coul, int do_shift, T tol_k, T tol_l, double* __restrict__ e_part,
    double* __restrict__ acc) {
  constexpr bool LJG = GRAD == 2;
  constexpr int N = GRAD ? CpCh<LJG>::N : 1;
  __shared__ double s_fl[GRAD ? (CPB / 32) * CPW * (CpCh<LJG>::ST + 1) : 1];
  double* s = s_fl + (GRAD ? (threadIdx.x >> 5) * CPW * (CpCh<LJG>::ST + 1) : 0);
  const int l = half_lane(), l16 = l & 15;
  const long long total = en.E + en.M;
  const T shift = do_shift ? (T)(1.0 / g.rc) : (T)0, kc = (T)coul, rc2 = (T)g.rc2;
  const T b0 = (T)g.box.b[0], b1 = (T)g.box.b[4], b2 = (T)g.box.b[8];
  const T v0 = (T)g.box.inv[0], v1 = (T)g.box.inv[4], v2 = (T)g.box.inv[8];
  double e_acc = 0.0;
  const long long runs = (total + run - 1) / run;
  for (long long r0 = half_index() & ~1; r0 < runs; r0 += half_count()) {  // both halves of a wave together
    const long long e0 = (r0 + (half_index() & 1)) * run;
    double fi[N];
    for (int k = 0; k < N; ++k) fi[k] = 0.0;
    int i = -1, x_of = -1;
    T xi = 0, yi = 0, zi = 0, qi = 0, si = 0, ei = 0;
    for (int n = 0; n < run; ++n) {
      const long long e = e0 + n;
      int in = -1, j = -1, x = -1;
      unsigned skip = 0xffffffffu;
      if (e < total && entry_atoms(en, e, g.natoms, g.nclusters, l, in, j, skip))
        x = e < en.E ? en.coo[e] : en.ic[e - en.E];
      if (x < 0) {  // past the end or padding
        in = i;
        x = x_of;
        j = -1;
      }
      if (x != x_of) {
        if constexpr (GRAD != 0) {
          if (x_of >= 0) {
            fi[3] *= coul;
            cp_flush<LJG>(i, fi, s, acc);
          }
          for (int k = 0; k < N; ++k) fi[k] = 0.0;
        }
        x_of = x;
        i = in;
        if (i >= 0) {
          xi = coords[3 * i]; yi = coords[3 * i + 1]; zi = coords[3 * i + 2];
          qi = q[i]; si = (T)0.5 * sig[i]; ei = eps[i];
        }
      }
      T xj = 0, yj = 0, zj = 0, qj = 0, sj = 0, ej = 0;
      if (j >= 0) {
        xj = coords[3 * j]; yj = coords[3 * j + 1]; zj = coords[3 * j + 2];
        qj = q[j]; sj = (T)0.5 * sig[j]; ej = eps[j];
      }
      skip |= half_ballot(j < 0);
      if (i < 0) skip = 0xffffffffu;
      // r^2 (T) below r2_in is within the cutoff, above r2_out it is not
      T r2_in = rc2, r2_out = rc2;
      if constexpr (sizeof(T) == 4) {
        T m = fabs(xj) + fabs(yj) + fabs(zj);
        for (int o = 16; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 32));  // (a NaN fails its own tests)
        const T tol = tol_k * (fabs(xi) + fabs(yi) + fabs(zi) + m + tol_l);
        r2_in = rc2 - tol;
        r2_out = rc2 + tol;
      }
      double gd[N];  // the column's sums, float64 over chains of CP_CHAIN steps
      for (int k = 0; k < N; ++k) gd[k] = 0.0;
      for (int h = 0; h < 2; ++h) {
        // bit 31 - k of `todo`: the pair of step k (column (l16 - k) & 15 of the row's block)
        const unsigned m16 = ((l >> 4) ^ h ? skip >> 16 : skip) & 0xffffu;
        int todo = (int)(~((m16 | m16 << 16) >> l16) << 15);
        for (int c0 = 0; c0 < 16; c0 += CP_CHAIN) {
          T gj[N];
          for (int k = 0; k < N; ++k) gj[k] = 0;
          for (int c = 0; c < CP_CHAIN; ++c) {
            T dx = xi - xj, dy = yi - yj, dz = zi - zj;
            if constexpr (ORTHO) {  // tff_min_image, its branches taken
              dx *= v0; dy *= v1; dz *= v2;
              dx = (dx - rint(dx)) * b0; dy = (dy - rint(dy)) * b1; dz = (dz - rint(dz)) * b2;
            } else {
              tff_min_image<T>(g.box, dx, dy, dz);
            }
            T r2 = dx * dx + dy * dy + dz * dz;
            bool ok = todo < 0;
            if constexpr (sizeof(T) == 8) {
              double ax = (double)xi - (double)xj, ay = (double)yi - (double)yj, az = (double)zi - (double)zj;
              tff_min_image_d(g.box, ax, ay, az);
              ok = ok && ax * ax + ay * ay + az * az <= g.rc2;
            } else {
              if (ok && !(r2 < r2_in || r2 > r2_out)) {
                double ax = (double)xi - (double)xj, ay = (double)yi - (double)yj, az = (double)zi - (double)zj;
                tff_min_image_d(g.box, ax, ay, az);
                ok = ax * ax + ay * ay + az * az <= g.rc2;
              } else {
                ok = ok && r2 < r2_in;
              }
            }
            if (ok) {
              const T rinv = cp_rsqrt(r2), rinv2 = rinv * rinv;
              const T qq = qi * qj * kc, ph = rinv - shift;
              T en_ = qq * ph;
              T dr = -qq * rinv * rinv2;
              const T sij = si + sj, eij = cp_sqrt(ei * ej);
              const T sr2 = sij * sij * rinv2, s6 = sr2 * sr2 * sr2;
              en_ += (T)4 * eij * s6 * (s6 - (T)1);
              const T w = (T)24 * eij * s6 * ((T)2 * s6 - (T)1);
              dr -= w * rinv2;
              e_acc += (double)en_;
              if constexpr (GRAD != 0) {
                fi[0] += (double)(dr * dx);
                fi[1] += (double)(dr * dy);
                fi[2] += (double)(dr * dz);
                fi[3] += (double)(qj * ph);  // times k at the end
                gj[0] -= dr * dx;
                gj[1] -= dr * dy;
                gj[2] -= dr * dz;
                gj[3] += qi * ph;
              }
              if constexpr (LJG) {
                const T ds = cp_div(w, sij) * (T)0.5;
                const T de = eij > (T)0 ? cp_div((T)4 * s6 * (s6 - (T)1) * (T)0.5, eij) : (T)0;
                fi[4] += (double)ds;
                fi[5] += (double)(de * ej);
                gj[4] += ds;
                gj[5] += de * ei;
              }
            }
            if constexpr (GRAD != 0)
              for (int k = 0; k < N; ++k) gj[k] = ror<1>(gj[k]);
            sj = ror<1>(sj);
            ej = ror<1>(ej);
            xj = ror<1>(xj);
            yj = ror<1>(yj);
            zj = ror<1>(zj);
            qj = ror<1>(qj);
            todo <<= 1;
          }
          if constexpr (GRAD != 0)
            for (int k = 0; k < N; ++k) gd[k] = ror<CP_CHAIN>(gd[k]) + (double)gj[k];
        }
        // the other row's columns and their sums (twice: every lane ends with its own column)
        xj = __shfl_xor(xj, 16, 32);
        yj = __shfl_xor(yj, 16, 32);
        zj = __shfl_xor(zj, 16, 32);
        qj = __shfl_xor(qj, 16, 32);
        sj = __shfl_xor(sj, 16, 32);
        ej = __shfl_xor(ej, 16, 32);
        if constexpr (GRAD != 0)
          for (int k = 0; k < N; ++k) gd[k] = __shfl_xor(gd[k], 16, 32);
      }
      if constexpr (GRAD != 0) {
        gd[3] *= coul;
        cp_flush<LJG>(j, gd, s, acc);
      }
    }
    if constexpr (GRAD != 0)
      if (x_of >= 0) {
        fi[3] *= coul;
        cp_flush<LJG>(i, fi, s, acc);
      }
  }
  const double sum = tff_block_sum(e_acc);
  if (threadIdx.x == 0) e_part[blockIdx.x] = sum;
}

// energy (block 0) and the requested gradients from the accumulators (st doubles per atom)
template <typename T>
struct CpOut {
  T *energy, *g_xyz, *g_q, *g_sig, *g_eps, *forces;
};
template <typename T>
__global__ __launch_bounds__(256) void k_cp_finish(const double* __restrict__ part, int nparts,
                                                   const double* __restrict__ acc, int st, long long n, double scale,
                                                   CpOut<T> o) {
  for (long long k = blockIdx.x * 256LL + threadIdx.x; k < n; k += (long long)gridDim.x * 256) {
    const double* a = acc + k * st;
    if (o.g_xyz)
      for (int c = 0; c < 3; ++c) o.g_xyz[3 * k + c] = (T)(a[c] * scale);
    if (o.forces)
      for (int c = 0; c < 3; ++c) o.forces[3 * k + c] += (T)(a[c] * -scale);
    if (o.g_q) o.g_q[k] = (T)(a[3] * scale);
    if (o.g_sig) o.g_sig[k] = (T)(a[4] * scale);
    if (o.g_eps) o.g_eps[k] = (T)(a[5] * scale);
  }
  if (o.energy && blockIdx.x == 0) {
    const double s = tff_sum_partials(part, nparts);
    if (threadIdx.x == 0) o.energy[0] = (T)(s * scale);
  }
}

__global__ void k_cp_zero_d(double* p, long long n) {
  for (long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x; k < n; k += (long long)gridDim.x * blockDim.x)
    p[k] = 0.0;
}

// ---------------------------------------------------------------- host side
int make_geom(const double* box_host, long long natoms, double cutoff, double cell_size, CpGeom& g) {
  if (!box_host || natoms < 1 || natoms > 0x3fffffffLL || !(cutoff > 0) || !(cell_size > 0)) {
    tff_set_error("cluster pairs: invalid arguments (box, 1 <= natoms < 2^30, cutoff > 0, cell_size > 0)");
    return TFF_ERR_ARG;
  }
  g.box = tff_make_box(box_host);
  if (!(g.box.det > 0)) {
    tff_set_error("cluster pairs: the box must have a positive volume");
    return TFF_ERR_ARG;
  }
  double h[3];
  for (int a = 0; a < 3; ++a) {
    const double c0 = g.box.inv[a], c1 = g.box.inv[3 + a], c2 = g.box.inv[6 + a];
    h[a] = 1.0 / sqrt(c0 * c0 + c1 * c1 + c2 * c2);
  }
  g.half_h = 0.5 * (h[0] < h[1] ? (h[0] < h[2] ? h[0] : h[2]) : (h[1] < h[2] ? h[1] : h[2]));
  if (cutoff > g.half_h) {
    tff_set_error("cluster pairs: cutoff %g exceeds half the smallest box height %g", cutoff, g.half_h);
    return TFF_ERR_ARG;
  }
  const double w[3] = {cell_size, cell_size, cell_size / 10.0};
  long long nc[3];
  for (int a = 0; a < 3; ++a) {
    nc[a] = (long long)floor(h[a] / w[a]);
    if (nc[a] < 1) nc[a] = 1;
    if (nc[a] > 4096) nc[a] = 4096;
  }
  // refine along z while the cells would hold more than 8 atoms on average
  while (natoms > 8LL * nc[0] * nc[1] * nc[2] && nc[2] < 1 << 20) nc[2] *= 2;
  if (nc[0] * nc[1] * nc[2] > (1LL << 28)) {
    tff_set_error("cluster pairs: cell grid too large (cell_size %g)", cell_size);
    return TFF_ERR_ARG;
  }
  for (int a = 0; a < 3; ++a) g.nc[a] = (int)nc[a];
  g.rc = cutoff;
  g.rc2 = cutoff * cutoff;
  g.natoms = (int)natoms;
  g.nclusters = (int)((natoms + CPW - 1) / CPW);
  return TFF_OK;
}

struct BuildWs {
  int* cell_of;
  int* count;    // ncell
  int* start;    // ncell + 1
  int* sums;     // a scan's partial sums
  int* seg;
  int* sorted;
  int* inv;
  double4* sphere;
  int* xlist;    // C * CP_XCL
  int* xcount;   // C
  int* xoff;     // C + 1
  int* rows;     // C
  long long* row_off;  // C + 1
  int* flags;
  size_t bytes;
};

BuildWs carve_build(void* base, const CpGeom& g) {
  BuildWs w{};
  size_t off = 0;
  char* p = (char*)base;
  auto take = [&](size_t b) {
    char* r = p ? p + off : nullptr;
    off += tff_align(b > 0 ? b : 1);
    return r;
  };
  const size_t n = (size_t)g.natoms, c = (size_t)g.nclusters;
  const size_t ncell = (size_t)g.nc[0] * g.nc[1] * g.nc[2];
  w.cell_of = (int*)take(4 * n);
  w.count = (int*)take(4 * ncell);
  w.start = (int*)take(4 * (ncell + 1));
  w.sums = (int*)take(4 * (ncell / CP_SCAN + 1));
  w.seg = (int*)take(4 * n);
  w.sorted = (int*)take(4 * n);
  w.inv = (int*)take(4 * n);
  w.sphere = (double4*)take(sizeof(double4) * c);
  w.xlist = (int*)take(4 * c * CP_XCL);
  w.xcount = (int*)take(4 * c);
  w.xoff = (int*)take(4 * (c + 1));
  w.rows = (int*)take(4 * c);
  w.row_off = (long long*)take(8 * (c + 1));
  w.flags = (int*)take(4 * 4);
  w.bytes = off;
  return w;
}

unsigned grid_for(long long items_per_half, long long n) {
  long long b = (n * items_per_half + (CPB / 32) - 1) / (CPB / 32);
  if (b < 1) b = 1;
  if (b > CP_MAXBLK) b = CP_MAXBLK;
  return (unsigned)b;
}

// exclusive scan (off[m] = total); sums: at least m / CP_SCAN + 1 entries, or null
template <typename C, typename O>
void scan_counts(const C* cnt, long long m, O* off, O* sums, hipStream_t st) {
  if (m <= 2 * CP_SCAN || !sums) {
    hipLaunchKernelGGL((k_cp_scan<C, O>), dim3(1), dim3(1024), 0, st, cnt, m, off);
    return;
  }
  const dim3 grid((unsigned)((m + CP_SCAN - 1) / CP_SCAN));
  hipLaunchKernelGGL((k_cp_scan_sums<C, O>), grid, dim3(1024), 0, st, cnt, m, sums);
  hipLaunchKernelGGL((k_cp_scan_tiles<C, O>), grid, dim3(1024), 0, st, cnt, m, (const O*)sums, off);
}

template <typename T>
int run_build(const T* coords, const CpGeom& g, const long long* rp, const long long* col, const BuildWs& w,
              long long* counts_out, hipStream_t st) {
  const int n = g.natoms;
  const long long ncell = (long long)g.nc[0] * g.nc[1] * g.nc[2];
  const unsigned nb = (unsigned)((n + 255) / 256);
  auto fill = [&](int* p, long long cnt) {
    long long b = (cnt + 255) / 256;
    if (b > 4096) b = 4096;
    if (b < 1) b = 1;
    hipLaunchKernelGGL(k_cp_fill, dim3((unsigned)b), dim3(256), 0, st, p, 0LL, cnt, 0);
  };
  fill(w.count, ncell);
  hipLaunchKernelGGL(k_cp_keys<T>, dim3(nb), dim3(256), 0, st, coords, g, w.cell_of, w.count,
                     w.flags);
  scan_counts(w.count, ncell, w.start, w.sums, st);
  hipLaunchKernelGGL(k_cp_scatter, dim3(nb), dim3(256), 0, st, n, w.cell_of, w.start, w.count, w.seg);
  hipLaunchKernelGGL(k_cp_rank, dim3(nb), dim3(256), 0, st, n, w.cell_of, w.start, w.seg, w.sorted, w.inv);
  const unsigned gc = grid_for(1, g.nclusters);
  const unsigned gx = (unsigned)(g.nclusters < 65536 ? g.nclusters : 65536);  // a workgroup per cluster
  hipLaunchKernelGGL(k_cp_bounds<T>, dim3(gc), dim3(CPB), 0, st, coords, g, w.sorted, w.sphere);
  hipLaunchKernelGGL(k_cp_excl, dim3(gc), dim3(CPB), 0, st, g, w.sorted, w.inv, rp, col, w.xlist, w.xcount,
                     w.flags);
  hipLaunchKernelGGL((k_cp_scan<int, int>), dim3(1), dim3(1024), 0, st, w.xcount, (long long)g.nclusters, w.xoff);
  hipLaunchKernelGGL((k_cp_rows<T, false>), dim3(gx), dim3(CPB), 0, st, coords, g, w.sorted, w.sphere, w.xlist,
                     w.xcount, w.rows, (const long long*)nullptr, 0LL, (int*)nullptr, (int*)nullptr);
  hipLaunchKernelGGL(k_cp_rows_scan, dim3(1), dim3(1024), 0, st, w.rows, g.nclusters, w.xoff, w.flags, w.row_off,
                     counts_out);
  TFF_CHECK_LAUNCH("cluster pairs build");
  return TFF_OK;
}

template <typename T>
int run_emit(const T* coords, const CpGeom& g, const long long* rp, const long long* col, const BuildWs& w,
             int* sorted_out, int* coo_out, unsigned* mask_out, long long ecap, int* ic_out, int* ia_out,
             long long mcap, hipStream_t st) {
  const unsigned gc = grid_for(1, g.nclusters);
  const unsigned gx = (unsigned)(g.nclusters < 65536 ? g.nclusters : 65536);  // a workgroup per cluster
  hipLaunchKernelGGL(k_cp_pad, dim3(512), dim3(256), 0, st, w.sorted, g.natoms, w.xoff, w.row_off, g.nclusters,
                     sorted_out, ecap, coo_out, mask_out, mcap, ic_out, ia_out);
  hipLaunchKernelGGL(k_cp_excl_emit, dim3(gc), dim3(CPB), 0, st, g, w.sorted, w.inv, rp, col, w.xlist,
                     w.xcount, w.xoff, (int)ecap, coo_out, mask_out);
  hipLaunchKernelGGL((k_cp_rows<T, true>), dim3(gx), dim3(CPB), 0, st, coords, g, w.sorted, w.sphere, w.xlist,
                     w.xcount, (int*)nullptr, (const long long*)w.row_off, mcap, ic_out, ia_out);
  TFF_CHECK_LAUNCH("cluster pairs emit");
  return TFF_OK;
}

struct TravWs {
  int* cnt;
  long long* off;
  double* e_part;
  double* acc;  // 8 doubles per atom
  size_t bytes;
};

TravWs carve_trav(void* base, long long natoms, long long entries) {
  TravWs w{};
  size_t off = 0;
  char* p = (char*)base;
  auto take = [&](size_t b) {
    char* r = p ? p + off : nullptr;
    off += tff_align(b > 0 ? b : 1);
    return r;
  };
  w.cnt = (int*)take(4 * (size_t)entries);
  w.off = (long long*)take(8 * ((size_t)entries + 1));
  w.e_part = (double*)take(8 * (size_t)CP_MAXBLK);
  w.acc = (double*)take(64 * (size_t)natoms);
  w.bytes = off;
  return w;
}

int check_entries(const Entries& en, const char* name) {
  if (!en.sorted || en.E < 0 || en.M < 0 || (en.E > 0 && (!en.coo || !en.mask)) || (en.M > 0 && (!en.ic || !en.ia)) ||
      en.E + en.M > 0x7fffffffLL) {
    tff_set_error("%s: invalid cluster-pair arguments", name);
    return TFF_ERR_ARG;
  }
  return TFF_OK;
}

}  // namespace

extern "C" size_t tff_exclusions_csr_workspace_bytes(long long natoms) {
  if (natoms < 1 || natoms > 0x3fffffffLL) return 0;
  return tff_align(4 * (size_t)natoms) + 8 * ((size_t)natoms / CP_SCAN + 1);
}

extern "C" int tff_exclusions_csr(const int64_t* pairs, long long num_pairs, int two_rows, long long natoms,
                                  int64_t* row_ptr, int64_t* col, long long* status, void* workspace,
                                  size_t workspace_bytes, hipStream_t stream) {
  if (num_pairs < 0 || num_pairs > 0x3fffffffLL || (num_pairs > 0 && (!pairs || !col)) || natoms < 1 ||
      natoms > 0x3fffffffLL || !row_ptr || !status) {
    tff_set_error("tff_exclusions_csr: invalid arguments");
    return TFF_ERR_ARG;
  }
  if (!workspace || workspace_bytes < tff_exclusions_csr_workspace_bytes(natoms)) {
    tff_set_error("tff_exclusions_csr: workspace too small (%zu < %zu)", workspace_bytes,
                  tff_exclusions_csr_workspace_bytes(natoms));
    return TFF_ERR_WORKSPACE;
  }
  int* cnt = (int*)workspace;
  long long* sums = (long long*)((char*)workspace + tff_align(4 * (size_t)natoms));
  const long long* p = reinterpret_cast<const long long*>(pairs);
  long long* rp = reinterpret_cast<long long*>(row_ptr);
  long long* cl = reinterpret_cast<long long*>(col);
  auto blocks = [](long long n) { return dim3((unsigned)(n < 256 ? 1 : n > 256 * 4096LL ? 4096 : (n + 255) / 256)); };
  hipLaunchKernelGGL(k_cp_fill, blocks(natoms), dim3(256), 0, stream, cnt, 0LL, natoms, 0);
  hipLaunchKernelGGL(k_cp_csr_count, blocks(num_pairs), dim3(256), 0, stream, p, num_pairs, two_rows, natoms, cnt,
                     status);
  scan_counts(cnt, natoms, rp, sums, stream);
  hipLaunchKernelGGL(k_cp_csr_fill, blocks(num_pairs), dim3(256), 0, stream, p, num_pairs, two_rows, natoms, cnt,
                     (const long long*)rp, cl);
  hipLaunchKernelGGL(k_cp_csr_unique, dim3((unsigned)((natoms + 255) / 256)), dim3(256), 0, stream, natoms,
                     (const long long*)rp, cl);
  TFF_CHECK_LAUNCH("exclusion lists");
  return TFF_OK;
}

extern "C" size_t tff_cluster_pairs_workspace_bytes(long long natoms, const double* box_host, double cutoff,
                                                    double cell_size) {
  CpGeom g{};
  if (make_geom(box_host, natoms, cutoff, cell_size, g)) return 0;
  return carve_build(nullptr, g).bytes;
}

extern "C" int tff_cluster_pairs_build(int dtype, const void* coords, long long natoms, const double* box_host,
                                       double cutoff, double cell_size, const int64_t* excl_row_ptr,
                                       const int64_t* excl_col, long long* counts_out, void* workspace,
                                       size_t workspace_bytes, hipStream_t stream) {
  CpGeom g{};
  int rc = make_geom(box_host, natoms, cutoff, cell_size, g);
  if (rc) return rc;
  if (!coords || !counts_out || (!excl_row_ptr) != (!excl_col) || (dtype != TFF_F32 && dtype != TFF_F64)) {
    tff_set_error("tff_cluster_pairs_build: invalid arguments");
    return TFF_ERR_ARG;
  }
  const BuildWs w = carve_build(workspace, g);
  if (!workspace || workspace_bytes < w.bytes) {
    tff_set_error("tff_cluster_pairs_build: workspace too small (%zu < %zu)", workspace_bytes, w.bytes);
    return TFF_ERR_WORKSPACE;
  }
  const long long* rp = reinterpret_cast<const long long*>(excl_row_ptr);
  const long long* col = reinterpret_cast<const long long*>(excl_col);
  if (dtype == TFF_F64) return run_build<double>((const double*)coords, g, rp, col, w, counts_out, stream);
  return run_build<float>((const float*)coords, g, rp, col, w, counts_out, stream);
}

extern "C" int tff_cluster_pairs_emit(int dtype, const void* coords, long long natoms, const double* box_host,
                                      double cutoff, double cell_size, const int64_t* excl_row_ptr,
                                      const int64_t* excl_col, int32_t* sorted_atom_indices,
                                      int32_t* cluster_exclusions, uint32_t* bitmask_exclusions,
                                      long long excl_capacity, int32_t* interacting_clusters,
                                      int32_t* interacting_atoms, long long row_capacity, void* workspace,
                                      size_t workspace_bytes, hipStream_t stream) {
  CpGeom g{};
  int rc = make_geom(box_host, natoms, cutoff, cell_size, g);
  if (rc) return rc;
  if (!coords || !sorted_atom_indices || excl_capacity < 0 || row_capacity < 0 ||
      (excl_capacity > 0 && (!cluster_exclusions || !bitmask_exclusions)) ||
      (row_capacity > 0 && (!interacting_clusters || !interacting_atoms)) || excl_capacity > 0x7fffffffLL ||
      (!excl_row_ptr) != (!excl_col) || (dtype != TFF_F32 && dtype != TFF_F64)) {
    tff_set_error("tff_cluster_pairs_emit: invalid arguments");
    return TFF_ERR_ARG;
  }
  const BuildWs w = carve_build(workspace, g);
  if (!workspace || workspace_bytes < w.bytes) {
    tff_set_error("tff_cluster_pairs_emit: workspace too small (%zu < %zu)", workspace_bytes, w.bytes);
    return TFF_ERR_WORKSPACE;
  }
  const long long* rp = reinterpret_cast<const long long*>(excl_row_ptr);
  const long long* col = reinterpret_cast<const long long*>(excl_col);
  if (dtype == TFF_F64)
    return run_emit<double>((const double*)coords, g, rp, col, w, sorted_atom_indices, cluster_exclusions,
                            bitmask_exclusions, excl_capacity, interacting_clusters, interacting_atoms, row_capacity,
                            stream);
  return run_emit<float>((const float*)coords, g, rp, col, w, sorted_atom_indices, cluster_exclusions,
                         bitmask_exclusions, excl_capacity, interacting_clusters, interacting_atoms, row_capacity,
                         stream);
}

extern "C" size_t tff_cluster_pairs_traverse_workspace_bytes(long long natoms, long long num_exclusion_blocks,
                                                             long long num_rows) {
  if (natoms < 0 || num_exclusion_blocks < 0 || num_rows < 0) return 0;
  return carve_trav(nullptr, natoms, num_exclusion_blocks + num_rows).bytes;
}

extern "C" int tff_cluster_pairs_decode(int dtype, const void* coords, long long natoms, const double* box_host,
                                        double cutoff, const int32_t* sorted_atom_indices,
                                        const int32_t* cluster_exclusions, const uint32_t* bitmask_exclusions,
                                        long long num_exclusion_blocks, const int32_t* interacting_clusters,
                                        const int32_t* interacting_atoms, long long num_rows, int32_t* pairs_out,
                                        long long pair_capacity, int32_t* npairs_out, void* workspace,
                                        size_t workspace_bytes, hipStream_t stream) {
  CpGeom g{};
  int rc = make_geom(box_host, natoms, cutoff, cutoff, g);
  if (rc) return rc;
  const Entries en{(const int*)sorted_atom_indices, (const int*)cluster_exclusions, num_exclusion_blocks,
                   (const unsigned*)bitmask_exclusions, (const int*)interacting_clusters,
                   (const int*)interacting_atoms, num_rows};
  if ((rc = check_entries(en, "tff_cluster_pairs_decode"))) return rc;
  if (!coords || !npairs_out || pair_capacity < 0 || (pair_capacity > 0 && !pairs_out) ||
      (dtype != TFF_F32 && dtype != TFF_F64)) {
    tff_set_error("tff_cluster_pairs_decode: invalid arguments");
    return TFF_ERR_ARG;
  }
  const long long total = num_exclusion_blocks + num_rows;
  const TravWs w = carve_trav(workspace, natoms, total);
  if (!workspace || workspace_bytes < w.bytes) {
    tff_set_error("tff_cluster_pairs_decode: workspace too small (%zu < %zu)", workspace_bytes, w.bytes);
    return TFF_ERR_WORKSPACE;
  }
  const unsigned gt = grid_for(1, total);
  if (dtype == TFF_F64) {
    hipLaunchKernelGGL((k_cp_decode<double, TR_COUNT>), dim3(gt), dim3(CPB), 0, stream, (const double*)coords, g, en,
                       w.cnt, (const long long*)nullptr, 0LL, (int*)nullptr);
  } else {
    hipLaunchKernelGGL((k_cp_decode<float, TR_COUNT>), dim3(gt), dim3(CPB), 0, stream, (const float*)coords, g, en,
                       w.cnt, (const long long*)nullptr, 0LL, (int*)nullptr);
  }
  long long* sums = total / CP_SCAN < CP_MAXBLK ? (long long*)w.e_part : nullptr;
  scan_counts(w.cnt, total, w.off, sums, stream);
  if (pair_capacity > 0) {
    if (dtype == TFF_F64)
      hipLaunchKernelGGL((k_cp_decode<double, TR_WRITE>), dim3(gt), dim3(CPB), 0, stream, (const double*)coords, g,
                         en, w.cnt, (const long long*)w.off, pair_capacity, (int*)pairs_out);
    else
      hipLaunchKernelGGL((k_cp_decode<float, TR_WRITE>), dim3(gt), dim3(CPB), 0, stream, (const float*)coords, g, en,
                         w.cnt, (const long long*)w.off, pair_capacity, (int*)pairs_out);
  }
  long long pb = (pair_capacity + 255) / 256;
  if (pb > 4096) pb = 4096;
  if (pb < 1) pb = 1;
  hipLaunchKernelGGL(k_cp_npairs, dim3((unsigned)pb), dim3(256), 0, stream, (const long long*)w.off, total,
                     pair_capacity, (int*)npairs_out, (int*)pairs_out);
  TFF_CHECK_LAUNCH("cluster pairs decode");
  return TFF_OK;
}

extern "C" int tff_cluster_pairs_nonbonded(int dtype, const void* coords, long long natoms, const double* box_host,
                                           const void* charges, const void* sigma, const void* epsilon,
                                           double coul_constant, double cutoff, int do_shift,
                                           const int32_t* sorted_atom_indices, const int32_t* cluster_exclusions,
                                           const uint32_t* bitmask_exclusions, long long num_exclusion_blocks,
                                           const int32_t* interacting_clusters, const int32_t* interacting_atoms,
                                           long long num_rows, double scale, void* energy_out, void* grad_coords,
                                           void* grad_charges, void* grad_sigma, void* grad_epsilon,
                                           void* forces_accum, void* workspace, size_t workspace_bytes,
                                           hipStream_t stream) {
  CpGeom g{};
  int rc = make_geom(box_host, natoms, cutoff, cutoff, g);
  if (rc) return rc;
  const Entries en{(const int*)sorted_atom_indices, (const int*)cluster_exclusions, num_exclusion_blocks,
                   (const unsigned*)bitmask_exclusions, (const int*)interacting_clusters,
                   (const int*)interacting_atoms, num_rows};
  if ((rc = check_entries(en, "tff_cluster_pairs_nonbonded"))) return rc;
  if (!coords || !charges || !sigma || !epsilon || (dtype != TFF_F32 && dtype != TFF_F64)) {
    tff_set_error("tff_cluster_pairs_nonbonded: invalid arguments");
    return TFF_ERR_ARG;
  }
  const long long total = num_exclusion_blocks + num_rows;
  const TravWs w = carve_trav(workspace, natoms, total);
  if (!workspace || workspace_bytes < w.bytes) {
    tff_set_error("tff_cluster_pairs_nonbonded: workspace too small (%zu < %zu)", workspace_bytes, w.bytes);
    return TFF_ERR_WORKSPACE;
  }
  const int grad = grad_sigma || grad_epsilon ? 2 : (grad_coords || forces_accum || grad_charges ? 1 : 0);
  const int stride = grad == 2 ? 8 : 4;
  auto blocks = [](long long n) {
    const long long b = (n + 255) / 256;
    return dim3((unsigned)(b < 1 ? 1 : b > 4096 ? 4096 : b));
  };
  if (grad) hipLaunchKernelGGL(k_cp_zero_d, blocks(stride * natoms), dim3(256), 0, stream, w.acc, stride * natoms);
  // runs of up to 16 entries, shorter ones while there are fewer than 8192 half-waves of them
  int run = (int)(total / 8192);
  run = run < 1 ? 1 : run > 16 ? 16 : run;
  const unsigned gt = grid_for(1, (total + run - 1) / run);
  // float r^2 against the exact one: each component is off by at most 8 2^-24 (|d| + box) times the
  // condition of the change to fractional coordinates; where the cutoff is half the box, two images
  // are equally far and only the exact test is taken
  double box_l = 0, cond = 1;
  for (int a = 0; a < 3; ++a) {
    double s = 0;
    for (int b = 0; b < 3; ++b) {
      s += fabs(g.box.b[3 * a + b]);
      double c = 0;
      for (int k = 0; k < 3; ++k) c += fabs(g.box.inv[3 * a + k]) * (fabs(g.box.b[3 * k]) + fabs(g.box.b[3 * k + 1]) + fabs(g.box.b[3 * k + 2]));
      if (c > cond) cond = c;
    }
    if (s > box_l) box_l = s;
  }
  const double tol_k = g.rc > 0.998 * g.half_h ? INFINITY : 64.0 / 16777216.0 * g.rc * cond;
  auto go = [&](auto tag) {
    using TT = decltype(tag);
    const TT *c = (const TT*)coords, *q = (const TT*)charges, *sg = (const TT*)sigma, *ep = (const TT*)epsilon;
    auto launch = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(gt), dim3(CPB), 0, stream, c, g, en, run, q, sg, ep, coul_constant, do_shift,
                         (TT)tol_k, (TT)box_l, w.e_part, w.acc);
    };
    auto pick = [&](auto box) {
      constexpr bool B = decltype(box)::value;
      if (grad == 2)
        launch(k_cp_nonbonded<TT, 2, B>);
      else if (grad == 1)
        launch(k_cp_nonbonded<TT, 1, B>);
      else
        launch(k_cp_nonbonded<TT, 0, B>);
    };
    if (g.box.ortho)
      pick(std::true_type{});
    else
      pick(std::false_type{});
    const CpOut<TT> o{(TT*)energy_out, (TT*)grad_coords, (TT*)grad_charges, (TT*)grad_sigma, (TT*)grad_epsilon,
                      (TT*)forces_accum};
    hipLaunchKernelGGL(k_cp_finish<TT>, blocks(grad ? natoms : 1), dim3(256), 0, stream, (const double*)w.e_part,
                       (int)gt, (const double*)w.acc, stride, grad ? natoms : 0LL, scale, o);
  };
  if (dtype == TFF_F64)
    go(double{});
  else
    go(float{});
  TFF_CHECK_LAUNCH("nonbonded from cluster pairs");
  return TFF_OK;
}
