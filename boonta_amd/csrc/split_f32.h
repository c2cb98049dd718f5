// fp32 products on the bf16 matrix cores: an fp32 value times 2^24 is the sum
// of three bf16 values (each piece the bf16 nearest to what the pieces before
// it leave), exactly: the second leaves at most 2^-17 of the value's power of
// two, seven bits of its 24, and the scale keeps every piece of every value,
// fp32 subnormals among them, at or above 2^-125, a normal bf16 number.  A
// product of two values is eight of their nine piece products, smallest first;
// the one left out is at most 2^-34 of the product.  (Six leave out up to 2^-24,
// half an fp32 ulp.)  bf16 piece products are exact in the MFMA, so what is
// rounded is the fp32 accumulator: eight roundings per 16 reduction elements,
// as many as v_mfma_f32_32x32x2_f32 has.  The sums come out times 2^48: the
// caller scales them back, and forms those that are not finite (a value from
// 2^104 on, a sum from 2^80 on, infinities and NaN) again in fp32.
#pragma once
#include "common.h"

namespace ppo {

typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));

// The three bf16 pieces of 8 values (one lane's share of a 16-deep MFMA operand).
struct Split8 {
  bf16x8 p[3];
};

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  const floatx2 v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// The bf16 values nearest to x and y, which keep what those leave (exactly).
__device__ __forceinline__ bf16x8 split_piece(floatx4& x, floatx4& y) {
  uintx4 w;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    floatx4& v = i < 2 ? x : y;
    const int e = 2 * (i & 1);
    const uint32_t u = pack_bf16(v[e], v[e + 1]);
    w[i] = u;
    v[e] -= __uint_as_float(u << 16);
    v[e + 1] -= __uint_as_float(u & 0xffff0000u);
  }
  return __builtin_bit_cast(bf16x8, w);
}

constexpr float SPLIT_SCALE = 0x1p24f;     // of each operand
constexpr float SPLIT_UNSCALE = 0x1p-48f;  // of a sum of products

__device__ __forceinline__ Split8 split8(floatx4 x, floatx4 y) {
  Split8 s;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    x[i] *= SPLIT_SCALE;
    y[i] *= SPLIT_SCALE;
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) s.p[q] = split_piece(x, y);
  return s;
}

// Product t (0 .. SPLIT_PRODUCTS - 1, smallest first) of a 32 x 32 x 16 block.
constexpr int SPLIT_PRODUCTS = 8;

__device__ __forceinline__ constexpr int split_product_a(int t) {
  return t == 0 || t == 2 ? 2 : t == 1 || t == 4 || t == 5 ? 1 : 0;
}
__device__ __forceinline__ constexpr int split_product_b(int t) {
  return t == 1 || t == 3 ? 2 : t == 0 || t == 4 || t == 6 ? 1 : 0;
}

__device__ __forceinline__ floatx16 split_mfma(int t, const Split8& a, const Split8& b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.p[split_product_a(t)], b.p[split_product_b(t)], c, 0, 0, 0);
}

}  // namespace ppo
