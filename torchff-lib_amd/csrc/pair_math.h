// Pair arithmetic shared by the fused and the serving kernels.
#pragma once

#include <hip/hip_runtime.h>

// erfc(u) and exp(-u^2) for u >= 0.
// float: exp(-u^2) = 2^(-u^2 log2 e) through the hardware base-2 exponential (relative error
// below 7e-7 for u <= 3 from the rounding of the argument); erfc(u) exp(u^2) = sum_k c_k t^k,
// t = 1 / (1 + 0.39 u) (hardware reciprocal), a degree-8 polynomial fitted to the scaled
// complementary error function on [0, 3.6] by iteratively reweighted least squares (relative
// error 1.3e-9 in exact arithmetic, about 1.5e-6 evaluated in float32, against
// scipy.special.erfc).  The fit is kept this accurate because rigid molecules put every
// intramolecular pair at the same u, where a polynomial error would add up coherently over the
// exclusion corrections.
__device__ __forceinline__ float erfc_scaled(float u) {
  const float t = __builtin_amdgcn_rcpf(fmaf(0.39f, u, 1.0f));
  float p = 9.27117256e-02f;
  p = fmaf(p, t, -5.29840954e-01f);
  p = fmaf(p, t, 1.06552963e+00f);
  p = fmaf(p, t, -8.61721388e-01f);
  p = fmaf(p, t, 7.81784359e-01f);
  p = fmaf(p, t, -4.21555312e-02f);
  p = fmaf(p, t, 2.82117988e-01f);
  p = fmaf(p, t, 2.10995424e-01f);
  return fmaf(p, t, 5.78745155e-04f);
}
__device__ __forceinline__ void erfc_exp(float u, float& ec, float& em) {
  em = __builtin_amdgcn_exp2f(u * u * -1.44269502f);
  ec = erfc_scaled(u) * em;
}
// double: both from one argument, without a branch.  -u^2 = n ln 2 + r with u^2 unrounded (the library call
// on the rounded square is off by up to u^2 ulp), exp(r) a degree-11 polynomial; (u + K) erfc(u) exp(u^2) a
// degree-23 polynomial in t = (A u - K) / (u + K) = A - K (A + 1) / (u + K), which maps [0, 27.9] onto
// [-1, 1]: both are Chebyshev interpolants computed in 60 digits, 3e-18 and 3e-17 off in exact
// arithmetic.  The factor u + K leaves the polynomial to run from 2.4 to 0.6; erfc(u) exp(u^2) alone
// runs from 1 to 0.02, where its even and odd parts cancel (3.7e-15 off for u in [10, 20]).  It is the
// factor 1 + 2 u of Shepherd and Laframboise, Math. Comp. 36, 1981, in a form whose reciprocal t needs
// anyway; K = 151 / 64 and A were chosen among short numbers so that the constant term is a double to
// 3e-20.  The reciprocal, the constant and linear terms and exp(r) carry their roundings along.  u is
// cut at 27.5, where both results are 0 already (a padding pair at 1e15 stays exactly 0).
// Relative errors against 28 digits (this arithmetic on the host), rms and largest: erfc 5.8e-17 and 2.1e-16
// for u in [0, 3.6] (C library 8.4e-17, 4.7e-16), at most 7.8e-17 and 3.0e-16 on [3.6, 26] (library
// 8.8e-17, 3.2e-16); exp(-u^2) 5.0e-17 and 1.6e-16 throughout (library call 2.8e-16, 1.0e-15 on [0, 3.6]).
// Bound by the FP64 rate: one evaluation of 60k water atoms takes 392 us with the library's functions, 374 us
// with these (372 us with the polynomial for erfc(u) exp(u^2) alone).
// Each coefficient is the scalar addend of a v_fma: left to itself the compiler moves it into a
// vector register first, one move per fma (3.7 us instead of 2.75 before the last corrections).
__device__ __forceinline__ double fma_coef(double a, double b, double c) {
  double d;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(c));
  return d;
}
static __device__ constexpr double EXP_C[12] = {
    0x1.0000000000000p+0, 0x1.0000000000000p+0, 0x1.0000000000011p-1, 0x1.5555555555562p-3,
    0x1.555555554f0ccp-5, 0x1.111111110db75p-7, 0x1.6c16c187fc3e6p-10, 0x1.a01a01b802660p-13,
    0x1.a01991aba6f13p-16, 0x1.71dde76a2f6d2p-19, 0x1.28b40639f7187p-22, 0x1.af785e0a5dff9p-26};
static __device__ constexpr double ERFCX_K = 2.359375, ERFCX_A = 1.16888427734375;
static __device__ constexpr double ERFCX_C[24] = {
    0x1.1c08996a7f535p+0, -0x1.8db9f04495585p-1, 0x1.7eece391e3014p-2, -0x1.acfb97a3f0883p-4,
    0x1.8d76d6840b2f1p-9, 0x1.114fd1049d386p-7, -0x1.3d0b470d9a8cap-10, -0x1.ca64e770e7228p-11,
    0x1.1aaaa78517553p-13, 0x1.04979d2286077p-13, -0x1.5866a7aae1bb6p-18, -0x1.44959b93d7645p-16,
    -0x1.832bd42588626p-19, 0x1.535dc11cf178ep-19, 0x1.3398120a23249p-20, -0x1.031b85d7f71edp-23,
    -0x1.0f910b0826991p-22, -0x1.0a2409b18687fp-24, 0x1.13cf99d0fa925p-25, 0x1.92ccb01864b9bp-26,
    -0x1.8023504096768p-31, -0x1.214244ff06bf4p-28, -0x1.5bdc4714cdf1ap-32, 0x1.7c0b3c7a2ada2p-32};
__device__ __forceinline__ void erfc_exp(double u, double& ec, double& em) {
  u = __hiloint2double(u > 27.5 ? 0x403b8000 : __double2hiint(u), __double2loint(u));  // high word only; a NaN stays one
  // n = rint(-u^2 log2 e): the integer is the low word of its sum with 1.5 2^52; ln 2 in two parts, the first of
  // 42 bits, so that n times it is exact
  const double nm = fma(u * u, -1.4426950408889634, 6755399441055744.0), n = nm - 6755399441055744.0;
  const int ni = __double2loint(nm);
  const double r = fma(n, -0x1.ef35793c7673p-45, fma(-u, u, n * -0x1.62e42fefa38p-1));
  double g = EXP_C[11];
#pragma unroll
  for (int k = 10; k >= 1; --k) g = fma_coef(g, r, EXP_C[k]);
  const double p = fma(g, r, 1.0), h = g * r;  // exp(r), exp(r) - 1
  em = ldexp(p, ni);
  // w + wl = 1 / (u + K): w the float reciprocal, off by e (at most 2e-7), wl = w (e + e^2); w's 24 bits
  // make its product with K and the subtraction from 1 exact
  const double w = (double)__builtin_amdgcn_rcpf((float)(u + ERFCX_K));
  const double e = fma(-w, u, fma(-w, ERFCX_K, 1.0)), wl = fma(e, e, e) * w;
  const double t = fma(-ERFCX_K * (ERFCX_A + 1.0), wl, fma(-ERFCX_K * (ERFCX_A + 1.0), w, ERFCX_A));
  const double t2 = t * t;
  double a = ERFCX_C[22], b = ERFCX_C[23];  // even and odd powers: two chains
#pragma unroll
  for (int k = 20; k >= 2; k -= 2) {
    a = fma_coef(a, t2, ERFCX_C[k]);
    b = fma_coef(b, t2, ERFCX_C[k + 1]);
  }
  // f + fl = (u + K) erfc(u) exp(u^2), constant and linear terms last
  const double c1t = ERFCX_C[1] * t, s = fma(fma(b, t, a), t2, c1t), f = ERFCX_C[0] + s;
  const double fl = ((ERFCX_C[0] - f) + s) + fma(ERFCX_C[1], t, -c1t);
  const double q = f * w, ql = fma(fl, w, fma(f, wl, fma(f, w, -q)));
  ec = ldexp(q + fma(q, h, ql * p), ni);
}
// the same with 1 subtracted from erfc where excl is set (float: in one rounding)
__device__ __forceinline__ void erfc_exp_excl(float u, bool excl, float& ec, float& em) {
  em = __builtin_amdgcn_exp2f(u * u * -1.44269502f);
  ec = fmaf(erfc_scaled(u), em, excl ? -1.f : 0.f);
}
__device__ __forceinline__ void erfc_exp_excl(double u, bool excl, double& ec, double& em) {
  erfc_exp(u, ec, em);
  ec = excl ? ec - 1.0 : ec;
}
// hardware reciprocal square root (1 ulp; Lennard-Jones raises the error to 12 ulp of s^12)
__device__ __forceinline__ float rsqrt_t(float x) { return __builtin_amdgcn_rsqf(x); }
// double: v_rsq_f64 (1e-7 off) and one third-order step (5e-17 rms, 1.4e-16 at most; 1 / sqrt: 7e-17,
// 1.6e-16); 0, infinity and NaN keep the hardware's value, which is the right one
__device__ __forceinline__ double rsqrt_t(double x) {
  const double y = __builtin_amdgcn_rsq(x), e = fma(-x * y, y, 1.0);
  const double z = fma(y * e, fma(e, 0.375, 0.5), y);
  return fabs(e) < 1.0 ? z : y;
}
// For pair functions that hold float to the library's accuracy: the library in float, the above in double.
__device__ __forceinline__ void erfc_exp_full(float u, float& ec, float& em) {
  ec = erfc(u);
  em = exp(-u * u);
}
__device__ __forceinline__ void erfc_exp_full(double u, double& ec, double& em) { erfc_exp(u, ec, em); }
__device__ __forceinline__ float rsqrt_full(float x) { return 1.0f / sqrt(x); }
__device__ __forceinline__ double rsqrt_full(double x) { return rsqrt_t(x); }
