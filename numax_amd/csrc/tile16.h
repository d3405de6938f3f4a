// 16 x 16 tiles on MFMA and on 16-lane rows, and correctly rounded quotients:
// what the triangular, Cholesky, LU and QR kernels share.
#pragma once

#include "nmx_internal.h"

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
template <typename T>
struct Acc {
  typedef f4 type;
};
template <>
struct Acc<double> {
  typedef d4 type;
};
__device__ __forceinline__ d4 mma(double a, double b, d4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f4 mma(float a, float b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
// row of output item e of lane l; also the contraction index of step e
template <typename T>
__device__ __forceinline__ int acc_row(int lane, int e) {
  return sizeof(T) == 8 ? (lane >> 4) + 4 * e : 4 * (lane >> 4) + e;
}

template <int L>
__device__ __forceinline__ float row_bcast(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + L, 0xF, 0xF, true));
}
template <int L>
__device__ __forceinline__ double row_bcast(double v) {
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, 0x150 + L, 0xF, 0xF, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), 0x150 + L, 0xF, 0xF, true);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

template <typename T>
__device__ __forceinline__ bool finite(T v) {
  return fabs(v) <= (sizeof(T) == 8 ? (T)1.7976931348623157e308 : (T)3.4028234663852886e38f);
}

// s += x(lane I of the 16-lane row) * y, the broadcast as the DPP operand of the
// multiply-add.  s_nop 1: the two wait states between a vector write and a DPP
// read of the same register.
template <int I>
__device__ __forceinline__ void fmac_bcast(float& s, float x, float y) {
  asm volatile("s_nop 1\nv_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(s) : "v"(x), "v"(y), "n"(I));
}
template <int I>
__device__ __forceinline__ void fmac_bcast(double& s, double x, double y) {
  asm volatile("s_nop 1\nv_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(s) : "v"(x), "v"(y), "n"(I));
}

// d0 .. d3 += x(lanes I .. I + 3 of the 16-lane row) * y, as above
#define NMX_FMAC_LANES4(TYPE, D0, D1, D2, D3, X, Y, I)                                     \
  asm volatile("s_nop 1\n"                                                                 \
               "v_fmac_" TYPE "_dpp %0, %4, %5 row_newbcast:%6 row_mask:0xf bank_mask:0xf\n" \
               "v_fmac_" TYPE "_dpp %1, %4, %5 row_newbcast:%7 row_mask:0xf bank_mask:0xf\n" \
               "v_fmac_" TYPE "_dpp %2, %4, %5 row_newbcast:%8 row_mask:0xf bank_mask:0xf\n" \
               "v_fmac_" TYPE "_dpp %3, %4, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n" \
               : "+v"(D0), "+v"(D1), "+v"(D2), "+v"(D3)                                    \
               : "v"(X), "v"(Y), "n"(I), "n"((I) + 1), "n"((I) + 2), "n"((I) + 3))
template <int I>
__device__ __forceinline__ void fmac_lanes4(float& d0, float& d1, float& d2, float& d3, float x, float y) {
  NMX_FMAC_LANES4("f32", d0, d1, d2, d3, x, y, I);
}
template <int I>
__device__ __forceinline__ void fmac_lanes4(double& d0, double& d1, double& d2, double& d3, double x, double y) {
  NMX_FMAC_LANES4("f64", d0, d1, d2, d3, x, y, I);
}

// x / d, correctly rounded, from r = 1 / d correctly rounded: two corrections
// of the product by its residual (Markstein; the first leaves it within an ulp,
// the second rounds).  For operands whose quotient and residuals stay normal:
// d and x in the ranges below.  A quarter of a division's instructions.
template <typename T>
__device__ __forceinline__ T plain_quotient(T x, T d, T r) {
  T q = x * r;
  q = __builtin_elementwise_fma(__builtin_elementwise_fma(-q, d, x), r, q);
  return __builtin_elementwise_fma(__builtin_elementwise_fma(-q, d, x), r, q);
}
// and zeros (with their sign), infinities and NaNs
__device__ __forceinline__ double quotient(double x, double d, double r) {
  return __builtin_amdgcn_div_fixup(plain_quotient(x, d, r), d, x);
}
__device__ __forceinline__ float quotient(float x, float d, float r) {
  return __builtin_amdgcn_div_fixupf(plain_quotient(x, d, r), d, x);
}
// 1 / d, correctly rounded unless d's significand is all ones (Markstein):
// Newton's step from a value within an ulp.  d in the range below.
__device__ __forceinline__ double reciprocal(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
  return __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
}
__device__ __forceinline__ bool plain_divisor(double d) { return fabs(d) >= 1e-90 && fabs(d) <= 1e90; }
__device__ __forceinline__ bool plain_divisor(float d) { return fabsf(d) >= 1e-9f && fabsf(d) <= 1e9f; }
__device__ __forceinline__ bool plain_dividend(double x) { return (fabs(x) >= 1e-180 && fabs(x) <= 1e180) || x == 0; }
// a dividend's magnitude as an exponent; 0 for zeros, infinities and NaNs
__device__ __forceinline__ int magnitude(double x) { return __builtin_amdgcn_frexp_exp(x); }
__device__ __forceinline__ int magnitude(float x) { return __builtin_amdgcn_frexp_expf(x); }
template <typename T>
constexpr int plain_magnitude() { return sizeof(T) == 8 ? 600 : 90; }  // dividends of 2^-this .. 2^this

// acc += x(lane K of the 16-lane row) * y for four registers, the broadcast as
// the multiply-add's DPP operand (the compiler makes a move of it, which would
// double the instructions and keep R broadcast values live).  s_nop 1: the two
// wait states between a vector write and a DPP read of the same register.
#define NMX_FMAC_DPP4(TYPE, D0, D1, D2, D3, X0, X1, X2, X3, S0, S1, S2, S3, CONS)                                  \
  asm volatile("s_nop 1\n"                                                                                         \
               "v_fmac_" TYPE "_dpp %0, %4, %8 row_newbcast:%12 row_mask:0xf bank_mask:0xf\n"                      \
               "v_fmac_" TYPE "_dpp %1, %5, %9 row_newbcast:%12 row_mask:0xf bank_mask:0xf\n"                      \
               "v_fmac_" TYPE "_dpp %2, %6, %10 row_newbcast:%12 row_mask:0xf bank_mask:0xf\n"                     \
               "v_fmac_" TYPE "_dpp %3, %7, %11 row_newbcast:%12 row_mask:0xf bank_mask:0xf\n"                     \
               : "+v"(D0), "+v"(D1), "+v"(D2), "+v"(D3)                                                            \
               : "v"(X0), "v"(X1), "v"(X2), "v"(X3), "v"(S0), "v"(S1), "v"(S2), "v"(S3), "n"(CONS))
template <int K>
__device__ __forceinline__ void fmac_bcast4(float& d0, float& d1, float& d2, float& d3, float x0, float x1, float x2,
                                            float x3, float s0, float s1, float s2, float s3) {
  NMX_FMAC_DPP4("f32", d0, d1, d2, d3, x0, x1, x2, x3, s0, s1, s2, s3, K);
}
template <int K>
__device__ __forceinline__ void fmac_bcast4(double& d0, double& d1, double& d2, double& d3, double x0, double x1,
                                            double x2, double x3, double s0, double s1, double s2, double s3) {
  NMX_FMAC_DPP4("f64", d0, d1, d2, d3, x0, x1, x2, x3, s0, s1, s2, s3, K);
}
// x -= x(lane K) * s in place, four registers
#define NMX_FMAC_DPP4_SELF(TYPE, X0, X1, X2, X3, S, CONS)                                     \
  asm volatile("s_nop 1\n"                                                                    \
               "v_fmac_" TYPE "_dpp %0, %0, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n"  \
               "v_fmac_" TYPE "_dpp %1, %1, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n"  \
               "v_fmac_" TYPE "_dpp %2, %2, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n"  \
               "v_fmac_" TYPE "_dpp %3, %3, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n"  \
               : "+v"(X0), "+v"(X1), "+v"(X2), "+v"(X3)                                       \
               : "v"(S), "n"(CONS))
template <int K>
__device__ __forceinline__ void fmac_self4(float& x0, float& x1, float& x2, float& x3, float s) {
  NMX_FMAC_DPP4_SELF("f32", x0, x1, x2, x3, s, K);
}
template <int K>
__device__ __forceinline__ void fmac_self4(double& x0, double& x1, double& x2, double& x3, double s) {
  NMX_FMAC_DPP4_SELF("f64", x0, x1, x2, x3, s, K);
}

}  // namespace
