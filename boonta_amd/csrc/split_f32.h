// fp32 products on the bf16 matrix cores: an fp32 value is the sum of three
// bf16 values (each piece the bf16 nearest to what the pieces before it leave,
// so the 24 significand bits are covered exactly), and a product of two
// values is six of their nine piece products, smallest first; the three left
// out are below 2^-26 of the product.  bf16 piece products are exact in the
// MFMA, so what is rounded is the fp32 accumulator alone: six roundings per 16
// reduction elements where v_mfma_f32_32x32x2_f32 has eight.
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

__device__ __forceinline__ Split8 split8(floatx4 x, floatx4 y) {
  Split8 s;
#pragma unroll
  for (int q = 0; q < 3; ++q) s.p[q] = split_piece(x, y);
  return s;
}

// Product t (0 .. SPLIT_PRODUCTS - 1, smallest first) of a 32 x 32 x 16 block.
constexpr int SPLIT_PRODUCTS = 6;

__device__ __forceinline__ constexpr int split_product_a(int t) { return t == 0 ? 2 : t == 2 || t == 3 ? 1 : 0; }
__device__ __forceinline__ constexpr int split_product_b(int t) { return t == 1 ? 2 : t == 2 || t == 4 ? 1 : 0; }

__device__ __forceinline__ floatx16 split_mfma(int t, const Split8& a, const Split8& b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.p[split_product_a(t)], b.p[split_product_b(t)], c, 0, 0, 0);
}

}  // namespace ppo
