// f32 values as three bf16 numbers, and activation matrices that are kept that way.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

namespace pgk {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned u2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ unsigned pk_bf16(float a, float b) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector(f2{a, b}, bf16x2));
}
// Two values as three bf16 each whose sum is the value, two to a register (a in the low half): rounded to
// nearest, every difference exact.  A value that is infinite as bf16 gives NaN in the second and third part.
__device__ __forceinline__ void cut2(float a, float b, unsigned& hi, unsigned& mid, unsigned& lo) {
  hi = pk_bf16(a, b);
  const float a1 = a - __uint_as_float(hi << 16), b1 = b - __uint_as_float(hi & 0xffff0000u);
  mid = pk_bf16(a1, b1);
  const float a2 = a1 - __uint_as_float(mid << 16), b2 = b1 - __uint_as_float(mid & 0xffff0000u);
  lo = pk_bf16(a2, b2);
}
// An activation matrix in cut form: its values as the three bf16 numbers of cut2, eight columns of a row to 16 bytes, the
// rows of such an octet next to each other, the parts of an octet one after the other: part p of element (m, k) is the
// (k % 8)-th bf16 of the 16 bytes at ((k / 8 * 3 + p) * cut_rows(M) + m) * 16.  That is the operand of a matrix
// instruction as it is, so that the blocks which read the matrix need not each cut it again (the cut is all that a
// block's vector units do: 37 rows x 1280 cut by 256 blocks take 7 us of a 13 us launch).
// A value that is infinite as bf16 is its first part alone where it is not finite, else cut downward, so that the
// parts of every finite value are finite and their sum is the value.
__device__ __forceinline__ void cut_safe2(float a, float b, unsigned (&part)[3]) {
  cut2(a, b, part[0], part[1], part[2]);
  if ((part[0] & 0x7f80u) != 0x7f80u && (part[0] & 0x7f800000u) != 0x7f800000u) return;
  unsigned p[2][3];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const float x = e ? b : a;
    const bool finite = fabsf(x) < INFINITY;
    p[e][0] = x != x ? 0x7fc00000u : __float_as_uint(x) & 0xffff0000u;
    const float x1 = finite ? x - __uint_as_float(p[e][0]) : 0.0f;
    p[e][1] = __float_as_uint(x1) & 0xffff0000u;
    p[e][2] = __float_as_uint(x1 - __uint_as_float(p[e][1])) & 0xffff0000u;
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) part[i] = (p[0][i] >> 16) | p[1][i];
}
// Columns k .. k + 3 (k a multiple of 4) of row m of a matrix with room for mp rows.
__device__ __forceinline__ void store_cut4(void* to, int mp, size_t m, size_t k, f4 v) {
  unsigned ab[3], cd[3];
  cut_safe2(v.x, v.y, ab);
  cut_safe2(v.z, v.w, cd);
  char* at = static_cast<char*>(to) + (k >> 3) * 3 * mp * 16 + m * 16 + (k & 4) * 2;
#pragma unroll
  for (int p = 0; p < 3; ++p) *reinterpret_cast<u2v*>(at + (size_t)p * mp * 16) = u2v{ab[p], cd[p]};
}
// One value of it.
__device__ __forceinline__ void store_cut1(void* to, int mp, size_t m, size_t k, float v) {
  unsigned part[3];
  cut_safe2(v, 0.0f, part);
  char* at = static_cast<char*>(to) + (k >> 3) * 3 * mp * 16 + m * 16 + (k & 7) * 2;
#pragma unroll
  for (int p = 0; p < 3; ++p) *reinterpret_cast<unsigned short*>(at + (size_t)p * mp * 16) = (unsigned short)part[p];
}
__device__ __forceinline__ float cut_form_value(const void* from, int mp, size_t m, size_t k) {
  const char* at = static_cast<const char*>(from) + (k >> 3) * 3 * mp * 16 + m * 16 + (k & 7) * 2;
  float v[3];
#pragma unroll
  for (int p = 0; p < 3; ++p) v[p] = __uint_as_float((unsigned)*reinterpret_cast<const unsigned short*>(at + (size_t)p * mp * 16) << 16);
  return v[0] + (v[1] + v[2]);
}

}  // namespace
}  // namespace pgk
