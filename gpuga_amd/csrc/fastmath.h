// Device math used by every kernel.
//
//  * ldu(): load through the constant address space.  With a wave-uniform
//    index the compiler issues a scalar load (s_load) and keeps the value in
//    SGPRs, so branches on it are scalar; used only for buffers that no
//    kernel writes while it runs (the training-set tables).
//  * exp2 / log2 / reciprocal: the CDNA transcendental instructions
//    (v_exp_f32, v_log_f32, v_rcp_f32, about 1 ulp on normal inputs), and
//    tanh from them (the NN2B tabulation's hidden layers).
//  * cos(pi t), sin(pi t) for t in [0, 1] (the cutoff taper): reduced to
//    y = pi (t - 1/2) in [-pi/2, pi/2] and evaluated from the Taylor series of
//    sin y (to y^11) and cos y (to y^12), whose truncation errors on that
//    interval are below 6e-8 and 7e-9.
#pragma once

#include <hip/hip_runtime.h>

namespace gpuga {

template <class T>
__device__ __forceinline__ T ldu(const T* p, long i)
{
#if defined(__HIP_DEVICE_COMPILE__)
  typedef const __attribute__((address_space(4))) T CT;
  return ((CT*)p)[i];
#else
  return p[i];
#endif
}

// ldu() when the index is wave-uniform (U), an ordinary per-lane load otherwise.
template <bool U, class T>
__device__ __forceinline__ T ldx(const T* p, long i)
{
  if constexpr (U) return ldu(p, i);
  else return p[i];
}

constexpr float LOG2E = 1.4426950408889634f;
constexpr float PI_F = 3.14159265358979f;

__device__ __forceinline__ float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float flog2(float x) { return __builtin_amdgcn_logf(x); }
__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }

// tanh x = 1 - 2 / (e^(2x) + 1) from exp2 and the reciprocal: absolute
// error about 2e-7 (the subtraction from 1 sets it near x = 0); -1 and +1
// for large |x| (e^(2x) flushes to 0 or overflows to +inf)
__device__ __forceinline__ float ftanh(float x)
{
  return 1.0f - 2.0f * frcp(fexp2(x * (2.0f * LOG2E)) + 1.0f);
}

// tanh x = sgn(x) (1 - e) / (1 + e) and s = (1 - tanh^2 x) / 4 = e / (1 + e)^2
// with e = exp(-2 |x|): about 1e-7 absolute, the derivative without a
// difference of nearly equal numbers.  (A quarter of it: callers multiply once,
// at the end.)
__device__ __forceinline__ void tanh_sech2(float x, float& t, float& s)
{
  const float e = fexp2(-2.0f * LOG2E * __builtin_fabsf(x));
  const float r = frcp(1.0f + e);
  t = __builtin_copysignf((1.0f - e) * r, x);
  s = e * r * r;
}

// tanh x = sgn(x) (1 - 2 r) and s = (1 - tanh^2 x) / 4 = r (1 - r) with
// r = 1 / (exp(2 |x|) + 1): the error of ftanh, the derivative as above.
__device__ __forceinline__ void ftanh_sech2(float x, float& t, float& s)
{
  const float r = frcp(fexp2(2.0f * LOG2E * __builtin_fabsf(x)) + 1.0f);
  t = __builtin_copysignf(fmaf(-2.0f, r, 1.0f), x);
  s = fmaf(-r, r, r);
}

// The same with tanh to about 1e-7 of its value: below 1/2 as x + x^3 p(x^2)
// (p: least-maximum fit of degree 3, 1.5e-8 of tanh x).
__device__ __forceinline__ void tanh_sech2_relative(float x, float& t, float& s)
{
  ftanh_sech2(x, t, s);
  const float y = x * x;
  float p = fmaf(0.01724139f, y, -0.05304545f);
  p = fmaf(p, y, 0.13325878f);
  p = fmaf(p, y, -0.33333144f);
  t = __builtin_fabsf(x) < 0.5f ? fmaf(x * y, p, x) : t;
}

// sin(pi t) and cos(pi t) for 0 <= t <= 1
__device__ __forceinline__ void sincospi01(float t, float& s, float& c)
{
  const float y = PI_F * (t - 0.5f);
  const float y2 = y * y;
  float ps = -1.0f / 39916800.0f;
  ps = ps * y2 + 1.0f / 362880.0f;
  ps = ps * y2 - 1.0f / 5040.0f;
  ps = ps * y2 + 1.0f / 120.0f;
  ps = ps * y2 - 1.0f / 6.0f;
  const float siny = y + y * y2 * ps;
  float pc = 1.0f / 479001600.0f;
  pc = pc * y2 - 1.0f / 3628800.0f;
  pc = pc * y2 + 1.0f / 40320.0f;
  pc = pc * y2 - 1.0f / 720.0f;
  pc = pc * y2 + 1.0f / 24.0f;
  pc = pc * y2 - 0.5f;
  const float cosy = 1.0f + y2 * pc;
  s = cosy;  // sin(pi t) = cos(y)
  c = -siny; // cos(pi t) = -sin(y)
}

} // namespace gpuga
