// Floats as sums of bf16 planes, the operands of the matrix unit's bf16
// products that stand for fp32 ones.
//  - three planes (split3): x = h + m + l exactly.  Cutting the low 16 bits
//    leaves 8 significant bits, the remainder (exact) has at most 16, and
//    cutting that one leaves at most 8.  Overflow cannot happen, as rounding
//    to bf16 could; below 2^-110 the low plane may be denormal.
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

// Two floats' three planes, each packed as (b << 16 | a).
__device__ __forceinline__ void split3_pair(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  const uint32_t ua = __float_as_uint(a), ub = __float_as_uint(b);
  h = __builtin_amdgcn_perm(ub, ua, 0x07060302u);
  const float ra = a - __uint_as_float(ua & 0xffff0000u), rb = b - __uint_as_float(ub & 0xffff0000u);
  const uint32_t ma = __float_as_uint(ra), mb = __float_as_uint(rb);
  m = __builtin_amdgcn_perm(mb, ma, 0x07060302u);
  const float la = ra - __uint_as_float(ma & 0xffff0000u), lb = rb - __uint_as_float(mb & 0xffff0000u);
  l = __builtin_amdgcn_perm(__float_as_uint(lb), __float_as_uint(la), 0x07060302u);
}
// Two floats' two planes, likewise.
__device__ __forceinline__ void split2_pair(float a, float b, uint32_t& h, uint32_t& l) {
  h = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){a, b}, bf16x2_t));
  const f32x2_t rest = {a - __uint_as_float(h << 16), b - __uint_as_float(h & 0xffff0000u)};
  l = __builtin_bit_cast(uint32_t, __builtin_convertvector(rest, bf16x2_t));
}

// Eight values' planes, packed as MFMA operands.
struct Planes {
  bf16x8_t p[3];
};
__device__ __forceinline__ Planes split3(const float (&v)[8]) {
  uint32_t w[3][4];
#pragma unroll
  for (int i = 0; i < 4; i++) split3_pair(v[2 * i], v[2 * i + 1], w[0][i], w[1][i], w[2][i]);
  Planes r;
#pragma unroll
  for (int k = 0; k < 3; k++)
    r.p[k] = __builtin_bit_cast(bf16x8_t, make_uint4(w[k][0], w[k][1], w[k][2], w[k][3]));
  return r;
}
// Four values' P planes, 8 bytes each.
template <int P>
__device__ __forceinline__ void split4(const float4& v, uint2 (&o)[P]) {
  if constexpr (P == 3) {
    split3_pair(v.x, v.y, o[0].x, o[1].x, o[2].x);
    split3_pair(v.z, v.w, o[0].y, o[1].y, o[2].y);
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
// of J that are kept, the smallest first.  Plane i weighs about 2^-8i; with
// three planes on either side pairs beyond i + j = 2 are below 2^-24 of the
// product, with two the pair (1, 1) below 2^-16.
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
