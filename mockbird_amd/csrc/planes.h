// Floats as sums of bf16 planes, the operands of the matrix unit's bf16
// products that stand for fp32 ones.
//  - three planes (split3): x = h + m + l exactly.  h = bf16(x) and m =
//    bf16(x - h), rounded to nearest even: the remainders are exact and of
//    either sign, |m| <= 2^-8 |x| and |l| <= 2^-17 |x|, and l has 7 bits at
//    most.  (bf16 ends at 2^-133: of values below 2^-110, whose bits go on
//    below it, that much is lost.)  A magnitude that rounds past the largest
//    bf16 (above (2 - 2^-8) 2^127) has no h: its planes, as an infinity's, give
//    NaN, and kernels that split their operands themselves take such sums
//    again in fp32; planes that are stored (SAT) stop h at the largest bf16,
//    which leaves the sum exact.
//  - two planes (split2): h = bf16(x), l = bf16(x - h), rounded to nearest
//    even: x to within about 2^-17.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace mb {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

// bf16(a), bf16(b) packed as (b << 16 | a), and what they leave of a and b.
// SAT: stopped at the largest bf16.
template <bool SAT = false>
__device__ __forceinline__ uint32_t high_pair(float& a, float& b) {
  constexpr float top = 0x1.fep127f;
  f32x2_t v = {a, b};
  if (SAT) v = f32x2_t{__builtin_amdgcn_fmed3f(a, -top, top), __builtin_amdgcn_fmed3f(b, -top, top)};
  const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
  a -= __uint_as_float(h << 16);
  b -= __uint_as_float(h & 0xffff0000u);
  return h;
}
// Two floats' three planes.
template <bool SAT = false>
__device__ __forceinline__ void split3_pair(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = high_pair<SAT>(a, b);
  m = high_pair(a, b);
  l = __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
// Two floats' two planes, likewise.
__device__ __forceinline__ void split2_pair(float a, float b, uint32_t& h, uint32_t& l) {
  h = high_pair(a, b);
  l = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){a, b}, bf16x2_t));
}

// Eight values' planes, packed as MFMA operands.
struct Planes {
  bf16x8_t p[3];
};
template <bool SAT = false>
__device__ __forceinline__ Planes split3(const float (&v)[8]) {
  uint32_t w[3][4];
#pragma unroll
  for (int i = 0; i < 4; i++) split3_pair<SAT>(v[2 * i], v[2 * i + 1], w[0][i], w[1][i], w[2][i]);
  Planes r;
#pragma unroll
  for (int k = 0; k < 3; k++)
    r.p[k] = __builtin_bit_cast(bf16x8_t, make_uint4(w[k][0], w[k][1], w[k][2], w[k][3]));
  return r;
}
// Four values' P planes, 8 bytes each, to be stored.
template <int P>
__device__ __forceinline__ void split4(const float4& v, uint2 (&o)[P]) {
  if constexpr (P == 3) {
    split3_pair<true>(v.x, v.y, o[0].x, o[1].x, o[2].x);
    split3_pair<true>(v.z, v.w, o[0].y, o[1].y, o[2].y);
  } else {
    split2_pair(v.x, v.y, o[0].x, o[1].x);
    split2_pair(v.z, v.w, o[0].y, o[1].y);
  }
}

// Index of the 16-byte chunk (row, k = 8 chunk .. + 7, plane p) of a planes
// operand of 32 nkb columns (gemm_planes.hip).
__device__ __forceinline__ int64_t plane_chunk(int64_t row, int chunk, int nkb, int planes, int p) {
  return (((row >> 4) * nkb + (chunk >> 2)) * planes + p) * 64 + (chunk & 3) * 16 + (row & 15);
}

// f(i, j) for the plane pairs of a product of an operand of I planes by one
// of J that are kept, the smallest first.  Plane i weighs at most 2^-8 and
// 2^-17 of the value; with three planes on either side the pairs beyond i + j
// = 2 add up to at most 2^-24 (1 + 2^-9) of the product (reached within 1 %
// by 1 + 0x7fc0 2^-23; 0.09 2^-24 rms over random operands, 0 in the mean),
// with two the pair (1, 1) is below 2^-16.
template <int I, int J, class F>
__device__ __forceinline__ void plane_products(F f) {
  using std::integral_constant;
  constexpr int top = (I > J ? I : J) - 1;
  auto at = [&](auto i, auto j) {
    constexpr int a = decltype(i)::value, b = decltype(j)::value;
    if constexpr (a < I && b < J && a + b <= top) f(i, j);
  };
  integral_constant<int, 0> c0;
  integral_constant<int, 1> c1;
  integral_constant<int, 2> c2;
  at(c2, c0); at(c0, c2); at(c1, c1); at(c1, c0); at(c0, c1); at(c0, c0);
}

}  // namespace mb
