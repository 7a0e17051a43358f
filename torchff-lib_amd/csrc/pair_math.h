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
// double: both from one argument, without a branch.  -u^2 = n ln 2 + r with the rounding of u^2 taken
// into r (the library call on the rounded square is off by up to u^2 ulp), exp(r) a degree-11
// polynomial; erfc(u) exp(u^2) a degree-21 polynomial in t = (1.28125 u - 3.75) / (u + 3.75), which
// maps [0, 26.67] onto [-1, 1]: both are Chebyshev interpolants computed in 60 digits, 3e-18 and 4e-18
// off in exact arithmetic.  u is cut at 27.5, where both results are 0 already (a padding pair at 1e15
// stays exactly 0).  Measured against 25-digit values for u in [0, 3.6], rms and largest: erfc 9.7e-17
// and 3.2e-16 (library 9.8e-17, 3.4e-16), exp(-u^2) 5.0e-17 and 1.4e-16 (library 2.8e-16, 1.0e-15);
// over r in [0.9, 9] A at alpha 0.3 A^-1 the pair energies are off by 5.8e-16 rms and their forces by
// 5.2e-16 (library 6.2e-16, 5.7e-16).  Bound by the FP64 rate: erfc, exp and 1 / sqrt of a million
// pairs took 5.4 us with the library's, 3.2 us with these (k_tiles_f64 of 60k water atoms 256 -> 190 us).
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
static __device__ constexpr double ERFCX_C[22] = {
    0x1.76eb8a31072c7p-3, -0x1.2ef15ea35aa48p-2, 0x1.d37d59145d1aep-3, -0x1.34696a5469df1p-3,
    0x1.58bb04227d1b5p-4, -0x1.403d71bd5537ap-5, 0x1.dc2a28605774fp-7, -0x1.04408f6e53ca3p-8,
    0x1.396ede3f17fbcp-11, 0x1.009e30e82b512p-14, -0x1.d97c3d57c13bbp-15, 0x1.1413239c0c019p-17,
    0x1.80d1790065794p-19, -0x1.30947befef2fcp-20, -0x1.d8805c68c88f3p-24, 0x1.f05ff1829a28ep-24,
    0x1.56ec6dfa80deep-29, -0x1.8e2cfdf20744fp-27, 0x1.35ce6dd1300acp-35, 0x1.358385ec92ffdp-30,
    -0x1.40d78682a7ecfp-39, -0x1.52433b61b276dp-34};
__device__ __forceinline__ void erfc_exp(double u, double& ec, double& em) {
  u = u > 27.5 ? 27.5 : u;  // (a NaN stays one)
  const double u2 = u * u, lo = fma(u, u, -u2);
  const double n = rint(u2 * -1.4426950408889634);
  const double r = fma(n, -0x1.abc9e3b39803fp-56, fma(n, -0x1.62e42fefa39efp-1, -u2)) - lo;
  double p = EXP_C[11];
#pragma unroll
  for (int k = 10; k >= 0; --k) p = fma_coef(p, r, EXP_C[k]);
  em = ldexp(p, (int)n);
  const double d = u + 3.75;
  double w = __builtin_amdgcn_rcp(d);  // off by at most 5e-8
  const double e = fma(-d, w, 1.0);
  w = fma(w * e, e + 1.0, w);
  // t = (1.28125 u - 3.75) / (u + 3.75), corrected by the roundings of numerator, denominator and quotient
  const double num = fma(u, 1.28125, -3.75), dlo = u - (d - 3.75), nlo = fma(u, 1.28125, -(num + 3.75));
  double t = num * w;
  t = fma(fma(-t, d, num) + fma(-t, dlo, nlo), w, t);
  const double t2 = t * t;
  double a = ERFCX_C[20], b = ERFCX_C[21];  // even and odd powers: two chains
#pragma unroll
  for (int k = 18; k >= 0; k -= 2) {
    a = fma_coef(a, t2, ERFCX_C[k]);
    b = fma_coef(b, t2, ERFCX_C[k + 1]);
  }
  const double f = fma(b, t, a);
  ec = fma(f, em, fma(b, t, a - f) * em);
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
