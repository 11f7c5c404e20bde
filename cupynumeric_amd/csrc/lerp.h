// Weighted sum of two neighbouring elements, the interpolation step of a quantile: shared by the
// kernels that read a sorted array (quantile.hip) and those that select from an unsorted one (select.hip).
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cpn {

// The reference's expression in the arithmetic of `T`'s array type; the result as float64.
template <typename T>
struct Lerp {  // integers and bool bytes: promoted to float64
  static __device__ __forceinline__ double eval(T l, T r, double gamma)
  {
#pragma clang fp contract(off)  // two rounded products and a rounded sum, never a fused multiply-add
    const double a = (1.0 - gamma) * static_cast<double>(l);
    const double b = gamma * static_cast<double>(r);
    return a + b;
  }
};
template <>
struct Lerp<double> {
  static __device__ __forceinline__ double eval(double l, double r, double gamma)
  {
#pragma clang fp contract(off)
    const double a = (1.0 - gamma) * l;
    const double b = gamma * r;
    return a + b;
  }
};
template <>
struct Lerp<float> {
  static __device__ __forceinline__ double eval(float l, float r, double gamma)
  {
#pragma clang fp contract(off)
    const float m1 = static_cast<float>(1.0 - gamma), g = static_cast<float>(gamma);  // the scalars take the array's type
    const float a = m1 * l;
    const float b = g * r;
    return static_cast<double>(a + b);
  }
};
// float16 arithmetic as NumPy does it: operands widened to float32, one operation, rounded back
// (a product of two float16 numbers is exact in float32).  The scalars are rounded from float64 once.
__device__ __forceinline__ float half_round(float v) { return __half2float(__float2half(v)); }
__device__ __forceinline__ float half_of_double(double v)
{
  float f = __double2float_rz(v);
  if (v == v && static_cast<double>(f) != v) {  // inexact: round to odd first, then the proper rounding is exact
    uint32_t bits;
    __builtin_memcpy(&bits, &f, 4);
    bits |= 1u;
    __builtin_memcpy(&f, &bits, 4);
  }
  return half_round(f);
}
template <>
struct Lerp<__half> {
  static __device__ __forceinline__ double eval(__half l, __half r, double gamma)
  {
#pragma clang fp contract(off)
    const float m1 = half_of_double(1.0 - gamma), g = half_of_double(gamma);
    const float a  = half_round(m1 * __half2float(l));
    const float b  = half_round(g * __half2float(r));
    return static_cast<double>(half_round(a + b));
  }
};

}  // namespace cpn
