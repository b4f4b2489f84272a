// Device helpers of the stage kernels (march.hip, tile.hip): lane shifts,
// row addressing, and the stencils' arithmetic in FP64 and FP32.
#pragma once

#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>
#include <type_traits>

#include "march.hpp"
#include "sbfs_internal.hpp"
#include "stencils.hpp"

namespace sbfs {

// value of the neighbouring lane (l-1 / l+1) through DPP wave shifts; the
// lane shifted in from outside the wavefront reads 0 (bound_ctrl), so the
// destination needs no clearing move first (every shift runs with all lanes
// active, where this equals keeping an old value of 0)
__device__ __forceinline__ double from_left(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  int lo = (int)(unsigned)(b & 0xffffffffull), hi = (int)(unsigned)(b >> 32);
  lo = __builtin_amdgcn_update_dpp(0, lo, 0x138, 0xf, 0xf, true);  // wave_shr:1
  hi = __builtin_amdgcn_update_dpp(0, hi, 0x138, 0xf, 0xf, true);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

__device__ __forceinline__ double from_right(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  int lo = (int)(unsigned)(b & 0xffffffffull), hi = (int)(unsigned)(b >> 32);
  lo = __builtin_amdgcn_update_dpp(0, lo, 0x130, 0xf, 0xf, true);  // wave_shl:1
  hi = __builtin_amdgcn_update_dpp(0, hi, 0x130, 0xf, 0xf, true);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// Two ways to address a wave-uniform row, so that every access is a scalar
// base plus the lane's byte offset:
//  * RowRef: the field's base and a 32-bit byte offset of lane 0's element,
//    plus the lane offset; rows of one layout share one offset for all
//    their fields, where a 64-bit row address per field and row costs
//    several scalar operations: a row step of the mixed marching body has 372
//    scalar instructions with it instead of 777, and a wavefront issues one
//    instruction at a time (k_march_mixed 55.5 -> 50 us at 1024 x 1500, together
//    with the tables in FP32; k_tile 27.9 -> 27.4 at 512 x 512).  Lanes whose
//    column lies before the array wrap the 32-bit offset; they are the masked
//    halo lanes and access nothing.
//  * the row's 64-bit address, pinned to SGPRs (readfirstlane of a uniform
//    value), plus the lane offset: the mixed marching body's for fields of
//    4 GiB or more.
// Both go through a global-address-space pointer, so the accesses stay
// global_load / global_store (a generic pointer made from an integer would
// compile to flat accesses, which also count against the LDS wait counter).
template <typename T>
using GlobalBytes =
    __attribute__((address_space(1))) typename std::conditional<std::is_const<T>::value, const char, char>::type;

template <typename T>
__device__ __forceinline__ T& lane_at(T* row, unsigned loff) {
  const unsigned long long u = (unsigned long long)row;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)u);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32));
  GlobalBytes<T>* base = (GlobalBytes<T>*)(((unsigned long long)hi << 32) | lo);
  return *(T*)(base + loff);
}

template <typename T>
struct RowRef {
  T* base;
  unsigned off;
  __device__ __forceinline__ RowRef operator+(int d) const { return {base, off + (unsigned)(d * (int)sizeof(T))}; }
};
template <typename T>
__device__ __forceinline__ T& lane_at(RowRef<T> r, unsigned loff) {
  GlobalBytes<T>* base = (GlobalBytes<T>*)r.base;
  return *(T*)(base + (r.off + loff));
}

// the lane's element of a row as a global pointer (for streaming stores)
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T* lane_gp(RowRef<T> r, unsigned loff) {
  GlobalBytes<T>* base = (GlobalBytes<T>*)r.base;
  return (__attribute__((address_space(1))) T*)(base + (r.off + loff));
}

// A wave-uniform value pinned to SGPRs.  FP64 arithmetic has no scalar
// form, so a constant such as dt * gamma is formed on the vector unit and
// would otherwise hold a VGPR pair for the whole kernel.
__device__ __forceinline__ double uni(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readfirstlane((int)b);
  const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ __forceinline__ float uni(float x) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}

__device__ __forceinline__ int wrap_r(int j, int ny) {
  while (j < 1) j += ny;
  while (j > ny) j -= ny;
  return j;
}

enum { T_RHF, T_RHC, T_RJF, T_RJC, T_QF, T_QC, T_EQF, T_ECY, T_CYC, T_CYF, T_DFX, T_DCX, T_HXXF, T_HXXC, T_N };

// Arithmetic of the interface and momentum stencils.  FP64 is the reference's
// arithmetic, expression for expression (stencils.hpp); FP32 is the mixed-
// precision step's, with the hardware's reciprocal, square root, exponential
// and logarithm (v_rcp_f32, v_sqrt_f32, v_exp_f32, v_log_f32, about an ulp
// each).  __fdividef, __fsqrt_rn and __logf do not map to these without
// fast-math flags: they compile to the IEEE sequences (11, 6 and 13 VALU
// instructions).
// The FP64 parts (the density-weighted updates, the Poisson right-hand
// side, the folded projection) divide by the column width and hy as the
// reference does in the FP64 body; the mixed body, whose error budget is
// FP32's, multiplies by the stored reciprocals (rhf, 1/hy) instead (per_h,
// per_hy in march_body).
template <typename R>
struct Arith;

template <>
struct Arith<double> {
  static __device__ __forceinline__ double left(double v) { return from_left(v); }
  static __device__ __forceinline__ double right(double v) { return from_right(v); }
  static __device__ __forceinline__ double div(double a, double b) { return a / b; }
  static __device__ __forceinline__ double sqr(double x) { return sqrt(x); }
  static __device__ __forceinline__ double eps() { return DBL_EPSILON; }
  // 0.5 (1 + tanh(beta sf)) (update/main.c:18-35)
  static __device__ __forceinline__ double indicator(double sf) { return 0.5 * (1. + tanh(kVofBeta * sf)); }
  // -0.5 / beta ln(1 / vof - 1) (curvature_tensor.c:92)
  static __device__ __forceinline__ double intercept(double v) { return -0.5 / kVofBeta * log(1. / v - 1.); }
};

template <>
struct Arith<float> {
  static __device__ __forceinline__ float left(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
  }
  static __device__ __forceinline__ float right(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));
  }
  static __device__ __forceinline__ float div(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
  static __device__ __forceinline__ float sqr(float x) { return __builtin_amdgcn_sqrtf(x); }
  static __device__ __forceinline__ float eps() { return (float)DBL_EPSILON; }
  // tanh from one exponential: 1 - 2 / (e^{2|x|} + 1), sign restored
  static __device__ __forceinline__ float indicator(float sf) {
    const float x = (float)kVofBeta * sf;
    const float t = 1.f - 2.f * __builtin_amdgcn_rcpf(__expf(2.f * fabsf(x)) + 1.f);
    return 0.5f * (1.f + copysignf(t, x));
  }
  // 0.5 / beta (ln vof - ln(1 - vof)) from base-2 logarithms; 1 - vof in
  // FP64 keeps the band edge
  static __device__ __forceinline__ float intercept(double v) {
    constexpr float c = (float)(0.5 / kVofBeta * 0.69314718055994530942);
    return c * (__builtin_amdgcn_logf((float)v) - __builtin_amdgcn_logf((float)(1. - v)));
  }
};

template <typename R>
struct V3R {
  R x, y, z;
};

// THINC face value from the upwind cell, averaged over the 2-point Gauss
// rule (update/fluxx.c:53-68, fluxy.c:53-68); the band test reads the FP64 vof
template <typename R, bool XFACE>
__device__ __forceinline__ R thinc_flux(R vel, double v, V3R<R> n) {
  using A = Arith<R>;
  const R h = vel < R(0) ? R(-0.5) : R(+0.5);
  if (!in_band(v)) return vel * R(v);
  const R gp = R(kGaussP), gw = R(kGaussW);
  R fl = R(0);
  if (XFACE) {
    fl += gw * A::indicator(n.x * h + n.y * -gp + n.z);
    fl += gw * A::indicator(n.x * h + n.y * +gp + n.z);
  } else {
    fl += gw * A::indicator(n.x * -gp + n.y * h + n.z);
    fl += gw * A::indicator(n.x * +gp + n.y * h + n.z);
  }
  return vel * fl;
}

template <typename R>
__device__ __forceinline__ R mixr(double ratio, double lo, double hi, R v) {
  R r = R(1) + (R(ratio) - R(1)) * v;
  r = fmax(R(lo), r);
  r = fmin(R(hi), r);
  return r;
}

}  // namespace sbfs
