// Direct (FFT-free) Ewald reciprocal sum: the reference's ewald_long_range / ewald_long_range_all
// (csrc/ewald/ewald.cu:9-171, 304-610; torchff/ewald.py:60-110).  Point charges here; with point
// dipoles and quadrupoles further down.
//
//   integer vectors m of the half space (m_x > 0, or m_x = 0 and m_y > 0, or m_x = m_y = 0 and
//   m_z > 0) with |m_a| <= kmax; k = B^-1 m (the columns of B^-1 are the reciprocal lattice
//   vectors of the row-major lattice B; k . r = m . s, s = r B^-1 the fractional coordinates);
//   G(k) = exp(-pi^2 k^2 / alpha^2) / k^2;  S(k) = sum_j q_j exp(2 pi i m . s_j);
//   E   = 1/(pi V) sum_k G |S|^2 - alpha/sqrt(pi) sum_j q_j^2,
//   phi_i = 2/(pi V) sum_k G (Re S cos theta_i + Im S sin theta_i) - 2 alpha/sqrt(pi) q_i,
//   F_i = -dE/dr_i = 4 q_i / V sum_k G k (Re S sin theta_i - Im S cos theta_i),  theta_i = 2 pi m . s_i.
//
// Layout: per atom and axis the phases exp(2 pi i h s_a), h = -kmax..kmax (one sincos each, in the
// input precision); one workgroup of 16 waves per (m_x, m_y) line, the lanes of a wave taking the
// m_z values of a few atoms and the waves a share of the atoms (fixed-order reduction), G S stored per
// vector; one workgroup per atom for the potential and force, the lanes taking the m_z values and its
// waves the lines (or the lanes striding over all k; reading G S through L1 / L2), and wave sums at the end.  Every sum runs in a fixed order, in float64.

#include <type_traits>

#include "tff_common.h"
#include "torchff_hip.h"

namespace {

constexpr int EW_WAVES = 16;  // waves per line workgroup
constexpr int EW_MAXK = 31;  // 2 kmax + 1 lanes

template <typename T> struct CX { T x, y; };

__device__ __forceinline__ void sincos_pi2(double v, double& s, double& c) { sincospi(2.0 * v, &s, &c); }
__device__ __forceinline__ void sincos_pi2(float v, float& s, float& c) { sincospif(2.0f * v, &s, &c); }

// fractional coordinates and the per-axis phase tables tab[(a * N + j) * W + (h + kmax)]
template <typename T>
__global__ void k_ewald_phases(const T* __restrict__ coords, long long n, TffBox box, int kmax,
                               CX<T>* __restrict__ tab) {
  const int W = 2 * kmax + 1;
  const long long total = n * 3 * W;
  for (long long idx = blockIdx.x * (long long)blockDim.x + threadIdx.x; idx < total;
       idx += (long long)gridDim.x * blockDim.x) {
    const int h = (int)(idx % W) - kmax;
    const long long ja = idx / W;
    const int a = (int)(ja / n);
    const long long j = ja - (long long)a * n;
    const double r[3] = {(double)coords[3 * j], (double)coords[3 * j + 1], (double)coords[3 * j + 2]};
    double s = r[0] * box.inv[a] + r[1] * box.inv[3 + a] + r[2] * box.inv[6 + a];
    s -= floor(s);  // the phase of an integer multiple does not change; keeps h s small
    // h s reduced to [-1/2, 1/2) before the transcendental (exact: h is an integer)
    double v = (double)h * s;
    v -= rint(v);
    T sn, cs;
    sincos_pi2((T)v, sn, cs);
    tab[idx] = {cs, sn};
  }
}

__device__ __forceinline__ void line_of(int line, int kmax, int& mx, int& my) {
  if (line <= kmax) {
    mx = 0;
    my = line;
  } else {
    const int t = line - (kmax + 1);
    mx = 1 + t / (2 * kmax + 1);
    my = t % (2 * kmax + 1) - kmax;
  }
}

// ------------------------------------------------------------------ multipoles (ranks 1, 2)
// Point dipoles p and Cartesian quadrupoles theta (3 x 3 row-major) enter through
// L(k) = q - (4 pi^2/3) k.theta.k + i 2 pi k.p and S(k) = sum_j L_j exp(2 pi i k.r_j)
// (torchff/ewald.py:75-97).  With A_i = G S* exp(2 pi i k.r_i) summed over the half space,
//   potential  = dE/dq      = 2/(pi V) sum Re A - 2 a q/sqrt(pi)
//   field      = -dE/dp     = 4/V sum k Im A + 4 a^3/(3 sqrt(pi)) p
//   field grad = -3 dE/dth  = 8 pi/V sum Re A k k^T + 16 a^5/(15 sqrt(pi)) theta
//   force      = -dE/dr     = 4/V sum k Im(L_i A_i),
// the force contracting a second multipole set X in place of L when one is given (the
// backward of ewald_long_range_all contracts one structure factor with two sets).
struct EwMp {
  const void* q;   // N, NULL = zero
  const void* p;   // N x 3, NULL = zero
  const void* th;  // N x 9, NULL = zero
};

template <typename T>
__device__ __forceinline__ double ew_load(const void* a, long long k) {
  return (double)((const T*)a)[k];
}

// real and imaginary parts of L(k) for atom j (RANK: 0 charges, 1 and dipoles, 2 and quadrupoles)
template <typename T, int RANK>
__device__ __forceinline__ void ew_L(const EwMp& m, long long j, double kx, double ky, double kz, double& lr,
                                     double& li) {
  lr = m.q ? ew_load<T>(m.q, j) : 0.0;
  li = 0.0;
  if (RANK >= 1 && m.p)
    li = 2.0 * M_PI * (kx * ew_load<T>(m.p, 3 * j) + ky * ew_load<T>(m.p, 3 * j + 1) + kz * ew_load<T>(m.p, 3 * j + 2));
  if (RANK >= 2 && m.th) {
    const double k[3] = {kx, ky, kz};
    double acc = 0.0;
#pragma unroll
    for (int x = 0; x < 3; ++x)
#pragma unroll
      for (int y = 0; y < 3; ++y) acc += k[x] * ew_load<T>(m.th, 9 * j + 3 * x + y) * k[y];
    lr -= 4.0 * M_PI * M_PI / 3.0 * acc;
  }
}

__device__ __forceinline__ void ew_k(const TffBox& box, int mx, int my, int mz, double& kx, double& ky, double& kz) {
  kx = box.inv[0] * mx + box.inv[1] * my + box.inv[2] * mz;
  ky = box.inv[3] * mx + box.inv[4] * my + box.inv[5] * mz;
  kz = box.inv[6] * mx + box.inv[7] * my + box.inv[8] * mz;
}

// S(k) of one (m_x, m_y) line per workgroup and the line's energy partial.  W = 2 kmax + 1 lanes hold one
// atom's m_z = -kmax .. kmax, a wave takes as many atoms at once as fit (64 / W).  Bound by the latency of the
// phase loads: 2700 atoms, dipoles, kmax 10, float64: 51 us; one atom per wave step, 43 lanes
// idle, took 127.
template <typename T, int RANK>
__global__ __launch_bounds__(EW_WAVES * TFF_WAVE) void k_ewald_structure(EwMp src, long long n, int kmax, TffBox box,
                                                                         double alpha,
                                                                         const CX<T>* __restrict__ tab,
                                                                         double* __restrict__ S,
                                                                         double* __restrict__ eline) {
  __shared__ double red[EW_WAVES][2][TFF_WAVE];
  const int line = blockIdx.x;
  const int lane = threadIdx.x & (TFF_WAVE - 1), wv = threadIdx.x / TFF_WAVE;
  const int W = 2 * kmax + 1, G = TFF_WAVE / W;
  int mx, my;
  line_of(line, kmax, mx, my);
  const int grp = lane / W, hz = lane - grp * W, mz = hz - kmax;
  double kx, ky, kz;
  ew_k(box, mx, my, mz, kx, ky, kz);
  double sr = 0, si = 0;
  // quadrupoles: four atoms at once spilled (12000 atoms, kmax 16: 3.34 ms, 2.87 one by one)
  constexpr int UNROLL = RANK < 2 ? 4 : 1;
  if (grp < G) {
#pragma unroll UNROLL
    for (long long j = wv * G + grp; j < n; j += EW_WAVES * G) {
      const CX<T> tx = tab[(0 * n + j) * W + mx + kmax];
      const CX<T> ty = tab[(1 * n + j) * W + my + kmax];
      const CX<T> tz = tab[(2 * n + j) * W + hz];
      const double ax = (double)tx.x * ty.x - (double)tx.y * ty.y, ay = (double)tx.x * ty.y + (double)tx.y * ty.x;
      const double c = ax * tz.x - ay * tz.y, s = ax * tz.y + ay * tz.x;
      double lr, li;
      ew_L<T, RANK>(src, j, kx, ky, kz, lr, li);
      sr += lr * c - li * s;
      si += lr * s + li * c;
    }
  }
  red[wv][0][lane] = sr;
  red[wv][1][lane] = si;
  __syncthreads();
  if (wv != 0) return;
  const bool lane_ok = lane < W;
  sr = si = 0;
  if (lane_ok) {
    for (int w = 0; w < EW_WAVES; ++w)
      for (int g = 0; g < G; ++g) {
        sr += red[w][0][g * W + lane];
        si += red[w][1][g * W + lane];
      }
  }
  // half space: m_x = m_y = 0 keeps m_z > 0 only
  const bool valid = lane_ok && !(mx == 0 && my == 0 && mz <= 0);
  double e = 0, g = 0;
  if (valid) {
    const double k2 = kx * kx + ky * ky + kz * kz;
    g = exp(-M_PI * M_PI * k2 / (alpha * alpha)) / k2;
    e = g * (sr * sr + si * si);
  }
  // G S: the per-atom pass then needs no transcendental per k
  if (lane_ok) {
    S[2 * ((size_t)line * W + lane)] = g * sr;
    S[2 * ((size_t)line * W + lane) + 1] = g * si;
  }
  e = tff_wave_sum(e);
  if (lane == 0) eline[line] = e;
}

// one atom's multipoles in registers
struct EwAtom {
  double q, p[3], th[9];
};

template <typename T>
__device__ __forceinline__ EwAtom ew_atom(const EwMp& m, long long j) {
  EwAtom a{};
  if (m.q) a.q = ew_load<T>(m.q, j);
  if (m.p)
    for (int k = 0; k < 3; ++k) a.p[k] = ew_load<T>(m.p, 3 * j + k);
  if (m.th)
    for (int k = 0; k < 9; ++k) a.th[k] = ew_load<T>(m.th, 9 * j + k);
  return a;
}

// Potential, field, field gradient (incl. the self terms) and force of one atom per workgroup of up to
// EW_AWAVES waves; the energy by block 0.  W lanes hold the m_z of a line, so that a lane's z phase and its part of k
// stay in registers and a step loads the two line phases and G S only.  Bound by FP64 arithmetic (some
// 35 operations per atom and k) and, for few atoms, by the waves in flight: hence several per atom below
// 8192 atoms.  2700 atoms, dipoles, kmax 10, float64: 38 us; a wave per atom striding over all k, with two
// integer divisions and a z phase load each, took 51.
// FLAT: where one line leaves too many lanes idle (33 to EW_FLAT - 1 values of m_z), the lanes stride over all k
// instead, line and m_z advanced without a division.  12000 atoms, ranks 0, 1, 2, the whole call in ms: kmax 16
// (33 values) 1.48, 2.09, 4.07, by lines 1.66, 2.39, 4.52; kmax 25 (51) 3.67, 4.98, 9.48, by lines 3.57, 5.10, 9.76; kmax
// 28 (57) 4.69, 6.34, 12.0, by lines 4.30, 6.12, 11.8.
constexpr int EW_AWAVES = 8;
constexpr int EW_FLAT = 53;

template <typename T, int RANK, bool FLAT>
__global__ __launch_bounds__(EW_AWAVES * TFF_WAVE) void k_ewald_atoms(EwMp src, EwMp con, long long n, int kmax,
                                                                      TffBox box, double alpha, int nlines,
                                                                      const CX<T>* __restrict__ tab,
                                                                      const double* __restrict__ S,
                                                                      const double* __restrict__ eline,
                                                                      double* __restrict__ energy,
                                                                      T* __restrict__ pot, T* __restrict__ field,
                                                                      T* __restrict__ fgrad, T* __restrict__ forces) {
  __shared__ double red[EW_AWAVES][13];
  const long long i = blockIdx.x;
  const int lane = threadIdx.x & (TFF_WAVE - 1), wv = threadIdx.x / TFF_WAVE, nw = blockDim.x / TFF_WAVE;
  const int W = 2 * kmax + 1, G = TFF_WAVE / W;
  const double V = box.det;
  const double rpi = 1.0 / sqrt(M_PI), a2 = alpha * alpha;
  if (blockIdx.x == 0 && energy) {
    double e = 0, self = 0;
    for (int l = threadIdx.x; l < nlines; l += blockDim.x) e += eline[l];
    for (long long j = threadIdx.x; j < n; j += blockDim.x) {
      const EwAtom a = ew_atom<T>(src, j);
      self += a.q * a.q;
      for (int k = 0; k < 3; ++k) self += 2.0 * a2 / 3.0 * a.p[k] * a.p[k];
      for (int k = 0; k < 9; ++k) self += 8.0 * a2 * a2 / 45.0 * a.th[k] * a.th[k];
    }
    e = tff_block_sum(e);
    self = tff_block_sum(self);
    if (threadIdx.x == 0) *energy = e / (M_PI * V) - alpha * rpi * self;
  }
  if (i >= n || (!pot && !field && !fgrad && !forces)) return;
  const EwAtom X = ew_atom<T>(con, i);  // the contracted set, loaded once
  const bool xp = RANK >= 1 && con.p != nullptr, xt = RANK >= 2 && con.th != nullptr;
  const CX<T>* tx = tab + (0 * n + i) * W;
  const CX<T>* ty = tab + (1 * n + i) * W;
  double sar = 0, fa[3] = {0, 0, 0}, eg[6] = {0, 0, 0, 0, 0, 0}, fk[3] = {0, 0, 0};
  const float inv_w = 1.0f / (float)W;
  const double2* GS = reinterpret_cast<const double2*>(S);  // G S (0 outside the half space)
  // vector (line, m_z): z phase az_, m_z's part of k zx, zy, zz
  auto step = [&](int line, const CX<T>& az_, double zx, double zy, double zz, const double2& Sk) {
    // line_of with the division by W in float (exact for fewer than 2^20 lines)
    const int t = line - (kmax + 1), row = (int)(((float)t + 0.5f) * inv_w);
    const int mx = t < 0 ? 0 : 1 + row, my = t < 0 ? line : t - row * W - kmax;
    const CX<T> ax_ = tx[mx + kmax], ay_ = ty[my + kmax];
    const double ax = (double)ax_.x * ay_.x - (double)ax_.y * ay_.y,
                 ay = (double)ax_.x * ay_.y + (double)ax_.y * ay_.x;
    const double c = ax * az_.x - ay * az_.y, s = ax * az_.y + ay * az_.x;
    const double kx = box.inv[0] * mx + box.inv[1] * my + zx;
    const double ky = box.inv[3] * mx + box.inv[4] * my + zy;
    const double kz = box.inv[6] * mx + box.inv[7] * my + zz;
    const double Ar = Sk.x * c + Sk.y * s, Ai = Sk.x * s - Sk.y * c;
    sar += Ar;
    fa[0] += kx * Ai;
    fa[1] += ky * Ai;
    fa[2] += kz * Ai;
    if (fgrad) {
      eg[0] += Ar * kx * kx;
      eg[1] += Ar * ky * ky;
      eg[2] += Ar * kz * kz;
      eg[3] += Ar * kx * ky;
      eg[4] += Ar * kx * kz;
      eg[5] += Ar * ky * kz;
    }
    if (RANK >= 1 && forces) {  // (of charges alone: q times the field's sums)
      double lr = X.q, li = 0.0;
      if (xp) li = 2.0 * M_PI * (kx * X.p[0] + ky * X.p[1] + kz * X.p[2]);
      if (xt) {
        const double kv[3] = {kx, ky, kz};
        double acc = 0.0;
#pragma unroll
        for (int x = 0; x < 3; ++x)
#pragma unroll
          for (int y = 0; y < 3; ++y) acc += kv[x] * X.th[3 * x + y] * kv[y];
        lr -= 4.0 * M_PI * M_PI / 3.0 * acc;
      }
      const double im = lr * Ai + li * Ar;
      fk[0] += kx * im;
      fk[1] += ky * im;
      fk[2] += kz * im;
    }
  };
  if constexpr (FLAT) {
    const CX<T>* tz = tab + (2 * n + i) * W;
    const int stride = nw * TFF_WAVE, dl = stride / W, dh = stride - dl * W;
    int k = wv * TFF_WAVE + lane, line = k / W, h = k - line * W;
#pragma unroll 2
    for (; k < nlines * W; k += stride) {
      const int mz = h - kmax;
      step(line, tz[h], box.inv[2] * mz, box.inv[5] * mz, box.inv[8] * mz, GS[k]);
      line += dl;
      h += dh;
      if (h >= W) {
        h -= W;
        ++line;
      }
    }
  } else {
    const int grp = lane / W, h = lane - grp * W, mz = h - kmax;
    if (grp < G) {
      const CX<T> az = tab[(2 * n + i) * W + h];
      const double zx = box.inv[2] * mz, zy = box.inv[5] * mz, zz = box.inv[8] * mz;
#pragma unroll 2
      for (int line = wv * G + grp; line < nlines; line += nw * G)
        step(line, az, zx, zy, zz, GS[(size_t)line * W + h]);
    }
  }
  auto put = [&](int k, double v) {
    v = tff_wave_sum(v);
    if (lane == 0) red[wv][k] = v;
  };
  put(0, sar);
  for (int k = 0; k < 3; ++k) put(1 + k, fa[k]);
  if (RANK >= 1 && forces)
    for (int k = 0; k < 3; ++k) put(4 + k, fk[k]);
  if (fgrad)
    for (int k = 0; k < 6; ++k) put(7 + k, eg[k]);
  __syncthreads();
  if (threadIdx.x != 0) return;
  auto get = [&](int k) {
    double v = 0;
    for (int w = 0; w < nw; ++w) v += red[w][k];
    return v;
  };
  const EwAtom A = ew_atom<T>(src, i);
  if (pot) pot[i] = (T)(2.0 / (M_PI * V) * get(0) - 2.0 * alpha * rpi * A.q);
  if (field) {
    const double cf = 4.0 * alpha * a2 * rpi / 3.0;
    for (int x = 0; x < 3; ++x) field[3 * i + x] = (T)(4.0 / V * get(1 + x) + cf * A.p[x]);
  }
  if (fgrad) {
    const double cg = 16.0 * alpha * a2 * a2 * rpi / 15.0;
    const int map[9] = {0, 3, 4, 3, 1, 5, 4, 5, 2};
    for (int k = 0; k < 9; ++k) fgrad[9 * i + k] = (T)(8.0 * M_PI / V * get(7 + map[k]) + cg * A.th[k]);
  }
  if (forces)
    for (int x = 0; x < 3; ++x)
      forces[3 * i + x] = (T)(4.0 / V * (RANK >= 1 ? get(4 + x) : X.q * get(1 + x)));
}

struct EwaldWs {
  void* tab;
  double* S;
  double* eline;
  size_t bytes;
};

EwaldWs ewald_carve(void* base, long long n, int kmax, size_t tsize) {
  EwaldWs w{};
  size_t off = 0;
  char* p = (char*)base;
  auto take = [&](size_t b) {
    char* r = p ? p + off : nullptr;
    off += tff_align(b > 0 ? b : 1);
    return r;
  };
  const size_t W = 2 * (size_t)kmax + 1;
  const size_t nlines = (size_t)(kmax + 1) + (size_t)kmax * W;
  w.tab = take(2 * tsize * 3 * (size_t)n * W);
  w.S = (double*)take(16 * nlines * W);
  w.eline = (double*)take(8 * nlines);
  w.bytes = off;
  return w;
}

template <typename T>
int run_ewald(const T* coords, const EwMp& src, const EwMp& con, long long n, const TffBox& box, int kmax,
              double alpha, double* energy, T* pot, T* field, T* fgrad, T* forces, const EwaldWs& w, hipStream_t st) {
  const int W = 2 * kmax + 1;
  const int nlines = (kmax + 1) + kmax * W;
  const long long total = n * 3 * W;
  const unsigned g1 = (unsigned)((total + 255) / 256 < 8192 ? (total + 255) / 256 : 8192);
  hipLaunchKernelGGL(k_ewald_phases<T>, dim3(g1 > 0 ? g1 : 1), dim3(256), 0, st, coords, n, box, kmax,
                     (CX<T>*)w.tab);
  const unsigned g3 = (unsigned)(n > 0 ? n : 1);  // one workgroup per atom
  const long long waves = 8192 / (n > 0 ? n : 1);
  const unsigned nw = (unsigned)(waves < 1 ? 1 : waves > EW_AWAVES ? EW_AWAVES : waves);
  auto go = [&](auto rank) {
    constexpr int R = decltype(rank)::value;
    hipLaunchKernelGGL((k_ewald_structure<T, R>), dim3(nlines), dim3(EW_WAVES * TFF_WAVE), 0, st, src, n, kmax, box,
                       alpha, (const CX<T>*)w.tab, w.S, w.eline);
    auto atoms = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(g3), dim3(nw * TFF_WAVE), 0, st, src, con, n, kmax, box, alpha, nlines,
                         (const CX<T>*)w.tab, (const double*)w.S, (const double*)w.eline, energy, pot, field, fgrad,
                         forces);
    };
    atoms(2 * W > TFF_WAVE && W < EW_FLAT ? k_ewald_atoms<T, R, true> : k_ewald_atoms<T, R, false>);
  };
  if (src.th || con.th)
    go(std::integral_constant<int, 2>{});
  else if (src.p || con.p)
    go(std::integral_constant<int, 1>{});
  else
    go(std::integral_constant<int, 0>{});
  TFF_CHECK_LAUNCH("ewald");
  return TFF_OK;
}

}  // namespace

extern "C" size_t tff_ewald_workspace_bytes(int dtype, long long natoms, int kmax) {
  if (natoms < 1 || kmax < 1 || kmax > EW_MAXK) return 0;
  return ewald_carve(nullptr, natoms, kmax, dtype == TFF_F64 ? 8 : 4).bytes;
}

extern "C" int tff_ewald(int dtype, const void* coords, const void* charges, long long natoms, const double* box_host,
                         int kmax, double alpha, double* energy_out, void* potential_out, void* forces_out,
                         void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (!coords || !charges || natoms < 1 || !box_host || kmax < 1 || kmax > EW_MAXK || !(alpha > 0) ||
      (dtype != TFF_F32 && dtype != TFF_F64)) {
    tff_set_error("ewald: invalid arguments (natoms >= 1, box, 1 <= kmax <= %d, alpha > 0, dtype 0/1)", EW_MAXK);
    return TFF_ERR_ARG;
  }
  const TffBox box = tff_make_box(box_host);
  if (!(box.det > 0)) {
    tff_set_error("ewald: the box must have a positive volume");
    return TFF_ERR_ARG;
  }
  const EwaldWs w = ewald_carve(workspace, natoms, kmax, dtype == TFF_F64 ? 8 : 4);
  if (!workspace || workspace_bytes < w.bytes) {
    tff_set_error("ewald: workspace too small (%zu < %zu)", workspace_bytes, w.bytes);
    return TFF_ERR_WORKSPACE;
  }
  const EwMp src{charges, nullptr, nullptr};
  if (dtype == TFF_F64)
    return run_ewald<double>((const double*)coords, src, src, natoms, box, kmax, alpha, energy_out,
                             (double*)potential_out, nullptr, nullptr, (double*)forces_out, w, stream);
  return run_ewald<float>((const float*)coords, src, src, natoms, box, kmax, alpha, energy_out,
                          (float*)potential_out, nullptr, nullptr, (float*)forces_out, w, stream);
}

extern "C" int tff_ewald_multipole(int dtype, const void* coords, long long natoms, const double* box_host, int kmax,
                                   double alpha, const void* charges, const void* dipoles, const void* quadrupoles,
                                   const void* c_charges, const void* c_dipoles, const void* c_quadrupoles,
                                   double* energy_out, void* potential_out, void* field_out, void* field_grad_out,
                                   void* forces_out, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (!coords || natoms < 1 || !box_host || kmax < 1 || kmax > EW_MAXK || !(alpha > 0) ||
      (dtype != TFF_F32 && dtype != TFF_F64)) {
    tff_set_error("ewald: invalid arguments (natoms >= 1, box, 1 <= kmax <= %d, alpha > 0, dtype 0/1)", EW_MAXK);
    return TFF_ERR_ARG;
  }
  const TffBox box = tff_make_box(box_host);
  if (!(box.det > 0)) {
    tff_set_error("ewald: the box must have a positive volume");
    return TFF_ERR_ARG;
  }
  const EwaldWs w = ewald_carve(workspace, natoms, kmax, dtype == TFF_F64 ? 8 : 4);
  if (!workspace || workspace_bytes < w.bytes) {
    tff_set_error("ewald: workspace too small (%zu < %zu)", workspace_bytes, w.bytes);
    return TFF_ERR_WORKSPACE;
  }
  const EwMp src{charges, dipoles, quadrupoles};
  const bool own = !c_charges && !c_dipoles && !c_quadrupoles;
  const EwMp con = own ? src : EwMp{c_charges, c_dipoles, c_quadrupoles};
  if (dtype == TFF_F64)
    return run_ewald<double>((const double*)coords, src, con, natoms, box, kmax, alpha, energy_out,
                                (double*)potential_out, (double*)field_out, (double*)field_grad_out,
                                (double*)forces_out, w, stream);
  return run_ewald<float>((const float*)coords, src, con, natoms, box, kmax, alpha, energy_out,
                             (float*)potential_out, (float*)field_out, (float*)field_grad_out, (float*)forces_out, w,
                             stream);
}
