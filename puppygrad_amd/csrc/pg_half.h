// f32 values as two f16 numbers, and activation matrices that are kept that way.
#pragma once
#include <hip/hip_runtime.h>

#include "pg_cut.h"

namespace pgk {
namespace {

typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));

// Two values times a power of two as two f16 numbers each, two to a register (a in the low half): hi = f16(x), lo =
// f16(x - hi), rounded to nearest, the difference exact.  hi + lo is x to 2^-23 of its binade's lower end or better where
// |x| >= 2^-2 (three of four values exactly), and to 2^-25 below that.
__device__ __forceinline__ void halves2(float a, float b, float mul, unsigned& hi, unsigned& lo) {
  a *= mul, b *= mul;
  const h2v h = __builtin_convertvector(f2{a, b}, h2v);
  const h2v l = __builtin_convertvector(f2{a - (float)h.x, b - (float)h.y}, h2v);
  hi = __builtin_bit_cast(unsigned, h), lo = __builtin_bit_cast(unsigned, l);
}
// The same of values that are right past f32: what f32 would have rounded away is in lo.
__device__ __forceinline__ void halves2(double a, double b, unsigned& hi, unsigned& lo) {
  const h2v h = __builtin_convertvector(f2{(float)a, (float)b}, h2v);
  const h2v l = __builtin_convertvector(f2{(float)(a - (double)(float)h.x), (float)(b - (double)(float)h.y)}, h2v);
  hi = __builtin_bit_cast(unsigned, h), lo = __builtin_bit_cast(unsigned, l);
}
// An activation matrix in half form: as in cut form (pg_cut.h) with two parts for three and a power of two in front of every column:
// part p of element (m, k) is the (k % 8)-th f16 of the 16 bytes at ((k / 8 * 2 + p) * cut_rows(M) + m) * 16.
// Columns k .. k + 3 (k a multiple of 4) of row m of a matrix with room for mp rows.
__device__ __forceinline__ void store_half4(void* to, int mp, size_t m, size_t k, f4 v, float mul) {
  unsigned h0, l0, h1, l1;
  halves2(v.x, v.y, mul, h0, l0);
  halves2(v.z, v.w, mul, h1, l1);
  char* at = static_cast<char*>(to) + (k >> 3) * 2 * mp * 16 + m * 16 + (k & 4) * 2;
  *reinterpret_cast<u2v*>(at) = u2v{h0, h1};
  *reinterpret_cast<u2v*>(at + (size_t)mp * 16) = u2v{l0, l1};
}
// The same of values with what f32 rounded away, times a power of two a column.
__device__ __forceinline__ void store_half4(void* to, int mp, size_t m, size_t k, f4 v, f4 rest, f4 mul) {
  unsigned h[2], l[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const float a = v[2 * e] * mul[2 * e], b = v[2 * e + 1] * mul[2 * e + 1];
    const h2v hi = __builtin_convertvector(f2{a, b}, h2v);
    const h2v lo = __builtin_convertvector(f2{fmaf(rest[2 * e], mul[2 * e], a - (float)hi.x), fmaf(rest[2 * e + 1], mul[2 * e + 1], b - (float)hi.y)}, h2v);
    h[e] = __builtin_bit_cast(unsigned, hi), l[e] = __builtin_bit_cast(unsigned, lo);
  }
  char* at = static_cast<char*>(to) + (k >> 3) * 2 * mp * 16 + m * 16 + (k & 4) * 2;
  *reinterpret_cast<u2v*>(at) = u2v{h[0], h[1]};
  *reinterpret_cast<u2v*>(at + (size_t)mp * 16) = u2v{l[0], l[1]};
}
// One value of it.
__device__ __forceinline__ void store_half1(void* to, int mp, size_t m, size_t k, float v, float mul) {
  unsigned h, l;
  halves2(v, 0.0f, mul, h, l);
  char* at = static_cast<char*>(to) + (k >> 3) * 2 * mp * 16 + m * 16 + (k & 7) * 2;
  *reinterpret_cast<unsigned short*>(at) = (unsigned short)h;
  *reinterpret_cast<unsigned short*>(at + (size_t)mp * 16) = (unsigned short)l;
}

}  // namespace
}  // namespace pgk
