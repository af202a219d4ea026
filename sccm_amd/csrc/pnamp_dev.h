// pnamp_dev.h -- complex FP64 helpers and wavefront reductions shared by the
// HIP sources of the PNAMP library (gfx950, 64-lane wavefronts).
#pragma once
#include <hip/hip_runtime.h>

namespace pnamp_dev {

__device__ __forceinline__ double2 cz() { return make_double2(0.0, 0.0); }
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 cneg(double2 a) { return make_double2(-a.x, -a.y); }
__device__ __forceinline__ double2 cconj(double2 a) { return make_double2(a.x, -a.y); }
__device__ __forceinline__ double2 cscale(double s, double2 a) { return make_double2(s * a.x, s * a.y); }
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ void cfma(double2 &acc, double2 a, double2 b) {
  acc.x = fma(a.x, b.x, acc.x);
  acc.x = fma(-a.y, b.y, acc.x);
  acc.y = fma(a.x, b.y, acc.y);
  acc.y = fma(a.y, b.x, acc.y);
}
__device__ __forceinline__ void cfms(double2 &acc, double2 a, double2 b) {  // acc -= a * b
  acc.x = fma(-a.x, b.x, acc.x);
  acc.x = fma(a.y, b.y, acc.x);
  acc.y = fma(-a.x, b.y, acc.y);
  acc.y = fma(-a.y, b.x, acc.y);
}
__device__ __forceinline__ void rfma(double2 &acc, double a, double2 b) {  // acc += a * b, a real
  acc.x = fma(a, b.x, acc.x);
  acc.y = fma(a, b.y, acc.y);
}
// 1 / d for a positive normal d: the hardware reciprocal estimate (v_rcp_f64)
// refined by two Newton-Raphson steps r <- r + r (1 - d r), each of which
// about doubles the number of correct bits (a few instructions instead of the
// scaled division sequence; within an ulp or two of the rounded quotient)
__device__ __forceinline__ double rcp_nr(double d) {
  double r = __builtin_amdgcn_rcp(d);
  double e = fma(-d, r, 1.0);
  r = fma(r, e, r);
  e = fma(-d, r, 1.0);
  return fma(r, e, r);
}
__device__ __forceinline__ double2 crecip_nr(double2 a) {
  const double r = rcp_nr(a.x * a.x + a.y * a.y);
  return make_double2(a.x * r, -a.y * r);
}
// Read-only view in the constant address space: wave-uniform reads through it
// become scalar loads (a generic pointer that stores in the kernel might
// alias is read with per-lane vector loads)
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(4))) T *ro_const(const T *q) {
  return (const __attribute__((address_space(4))) T *)q;
}
__device__ __forceinline__ double cabs1(double2 a) { return fabs(a.x) + fabs(a.y); }
__device__ __forceinline__ double2 cexpi(double t) {
  double s, c;
  sincos(t, &s, &c);
  return make_double2(c, s);
}
// A DPP move and the unsigned maximum with it; lanes without a DPP source read
// 0, the identity of an unsigned maximum.
template <int CTRL, int RM>
__device__ __forceinline__ unsigned dpp_umax(unsigned v) {
  return max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, RM, 0xF, false));
}

// Pivot key from the high word of a non-negative double (sign 0, 11 exponent
// and 20 mantissa bits: unsigned order is numeric order) with the low KB bits
// replaced by (2^KB - 1 - idx): the largest magnitude to 2^-(20-KB) relative,
// ties to the smallest index.  A NaN or infinite magnitude wins.
template <int KB>
__device__ __forceinline__ unsigned pivot_key_hi(double mag, int idx) {
  return ((unsigned)((unsigned long long)__double_as_longlong(mag) >> 32) & ~((1u << KB) - 1u)) |
         ((1u << KB) - 1u - (unsigned)idx);
}

// Maximum over each aligned group of eight lanes, on all eight (quad
// exchanges, then the half-row mirror).
__device__ __forceinline__ unsigned oct_umax(unsigned v) {
  v = dpp_umax<0xB1, 0xF>(v);   // quad_perm [1,0,3,2]
  v = dpp_umax<0x4E, 0xF>(v);   // quad_perm [2,3,0,1]
  v = dpp_umax<0x141, 0xF>(v);  // row_half_mirror
  return v;
}

}  // namespace pnamp_dev
