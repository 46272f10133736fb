// Sums and maxima over the lanes of a wavefront without a trip through LDS: __shfl_xor is one (about 100 clocks before
// the next step can start, 0.25 us for the six of a wavefront, which a launch of 4 to 8 us waits for once to three
// times); moves within a row of 16 lanes ride on the addition itself, and rows are brought together by a swap.  All lanes
// have to be active, and all get the result.
// The order of the additions is that of __shfl_xor by 32, 16, 8, 4, 2 and 1, to the last bit: a stream that is drawn
// over a whole row walks 50257 ids by value, neighbours 10^-5 apart, and where a logit's last bit swaps two of them it
// takes another id, and other ids from there on.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

namespace pgk {
namespace {

// The value of a lane of the same row of 16: 0xB1 lane ^ 1, 0x4E lane ^ 2, 0x1B lane ^ 3, 0x141 lane ^ 7, 0x140 lane ^ 15,
// 0x128 lane ^ 8, and 0x124 lane - 4, which serves as lane ^ 4 where lanes 8 apart hold the same.
template <int CTRL>
__device__ __forceinline__ float row_lane(float x) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xf, 0xf, true));
}
struct AddLanes {
  __device__ __forceinline__ float operator()(float a, float b) const { return a + b; }
};
struct MaxLanes {
  __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); }
};
// over each 8 neighbouring lanes: lane ^ 4, ^ 2, ^ 1
template <typename Op>
__device__ __forceinline__ float lanes8(float v, Op op) {
  v = op(v, row_lane<0x1B>(row_lane<0x141>(v)));
  v = op(v, row_lane<0x4E>(v));
  return op(v, row_lane<0xB1>(v));
}
// over each 16: lane ^ 8, ^ 4, ^ 2, ^ 1
template <typename Op>
__device__ __forceinline__ float lanes16(float v, Op op) {
  v = op(v, row_lane<0x128>(v));
  v = op(v, row_lane<0x124>(v));
  v = op(v, row_lane<0x4E>(v));
  return op(v, row_lane<0xB1>(v));
}
// over each 16 the other way round: lane ^ 1, ^ 2, ^ 4, ^ 8 (mirrors: the lanes in between hold the same)
template <typename Op>
__device__ __forceinline__ float lanes16_up(float v, Op op) {
  v = op(v, row_lane<0xB1>(v));
  v = op(v, row_lane<0x4E>(v));
  v = op(v, row_lane<0x141>(v));
  return op(v, row_lane<0x140>(v));
}
// with the lane 16 (32) away
template <typename Op>
__device__ __forceinline__ float with_lane16(float v, Op op) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
template <typename Op>
__device__ __forceinline__ float with_lane32(float v, Op op) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float wave_sum(float v) {
  return lanes16(with_lane16(with_lane32(v, AddLanes{}), AddLanes{}), AddLanes{});
}
// of a * b: the first addition takes this lane's product unrounded (what a product met by __shfl_xor is compiled to)
__device__ __forceinline__ float wave_sum_of_products(float a, float b) {
  const unsigned p = __float_as_uint(a * b);
  const auto r = __builtin_amdgcn_permlane32_swap(p, p, false, false);
  const float other = __uint_as_float((threadIdx.x & 32) ? r[0] : r[1]);
  return lanes16(with_lane16(fmaf(a, b, other), AddLanes{}), AddLanes{});
}
__device__ __forceinline__ float wave_max(float v) {
  return lanes16(with_lane16(with_lane32(v, MaxLanes{}), MaxLanes{}), MaxLanes{});
}
// The better of all lanes' (value, index) pairs; take(v, i, ov, oi): whether (ov, oi) is better than (v, i).
template <typename Take>
__device__ __forceinline__ void wave_best(float& v, unsigned& i, Take take) {
  auto with = [&](float ov, unsigned oi) {
    if (take(v, i, ov, oi)) v = ov, i = oi;
  };
  auto in_row = [](unsigned x, auto ctrl) {
    return (unsigned)__builtin_amdgcn_mov_dpp((int)x, decltype(ctrl)::value, 0xf, 0xf, true);
  };
  auto step = [&](auto ctrl) {
    const float ov = __uint_as_float(in_row(__float_as_uint(v), ctrl));
    with(ov, in_row(i, ctrl));
  };
  step(std::integral_constant<int, 0xB1>{});
  step(std::integral_constant<int, 0x4E>{});
  step(std::integral_constant<int, 0x141>{});
  step(std::integral_constant<int, 0x140>{});
  {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(i, i, false, false);
    v = __uint_as_float(a[0]), i = b[0];
    with(__uint_as_float(a[1]), b[1]);
  }
  {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(i, i, false, false);
    v = __uint_as_float(a[0]), i = b[0];
    with(__uint_as_float(a[1]), b[1]);
  }
}

// The value the lane 32 away holds (v_permlane32_swap: one VALU instruction, no LDS trip).
__device__ __forceinline__ float other_half(float x) {
  typedef unsigned u2x __attribute__((ext_vector_type(2)));
  const u2x r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  // r.x holds lanes 0..31 of x in both halves, r.y lanes 32..63
  return (threadIdx.x & 32) ? __uint_as_float(r.x) : __uint_as_float(r.y);
}

}  // namespace
}  // namespace pgk
