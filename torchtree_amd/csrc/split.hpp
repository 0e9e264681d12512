// Split-precision products of the dense-state kernels (HX_F32_BF16X3).
#pragma once

#include <hip/hip_runtime.h>

#include <stdint.h>

namespace hx {

using f32x4 = float __attribute__((ext_vector_type(4)));

// ---- split-precision products on the BF16 matrix cores
//
// A float x is carried as hi = bf16(x) and lo = bf16(x - hi) (both rounded to nearest even;
// x - hi is exact in FP32), which keeps 16 significant bits: |x - hi - lo| <= 2^-17 |x|.
// A product of two such operands is formed as lo_a hi_b + hi_a lo_b + hi_a hi_b on
// v_mfma_f32_16x16x32_bf16 (8 operand values per lane, K = 32) or v_mfma_f32_16x16x16_bf16
// (4 per lane, K = 16), accumulating in FP32; the dropped lo_a lo_b term is below 2^-16 of
// the product. Operand and accumulator lanes follow the FP32 instruction's: A[i][k] in lane
// i + 16 (k / n), element k % n, B[k][j] in lane j + 16 (k / n), and the FP32 16x16
// accumulator (checked on the device by hx_selftest_mfma_layout). Every caller builds A and
// B with the same map from (lane group, element) to the contraction index, so the sum runs
// over the same index pairs as the FP32 products.
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
template <int N>
struct BfPack;
template <>
struct BfPack<8> {
  bf16x8_t hi, lo;
};
template <>
struct BfPack<4> {
  bf16x4_t hi, lo;
};

// hi and lo halves of x, as one 32-bit word (hi in the low 16 bits): the form kept in LDS and
// in the padded copies of P, so that an operand is assembled without converting again
__device__ __forceinline__ uint32_t bf_pair(float x) {
  const __bf16 hi = (__bf16)x;
  const __bf16 lo = (__bf16)(x - (float)hi);
  return (uint32_t)__builtin_bit_cast(uint16_t, hi) |
         ((uint32_t)__builtin_bit_cast(uint16_t, lo) << 16);
}
__device__ __forceinline__ __bf16 pair_hi(uint32_t p) {
  return __builtin_bit_cast(__bf16, (uint16_t)(p & 0xffffu));
}
__device__ __forceinline__ __bf16 pair_lo(uint32_t p) {
  return __builtin_bit_cast(__bf16, (uint16_t)(p >> 16));
}

template <int N>
__device__ __forceinline__ void pack_set(BfPack<N>& b, int e, float x) {
  const __bf16 hi = (__bf16)x;
  b.hi[e] = hi;
  b.lo[e] = (__bf16)(x - (float)hi);
}
template <int N>
__device__ __forceinline__ void pack_set_pair(BfPack<N>& b, int e, uint32_t p) {
  b.hi[e] = pair_hi(p);
  b.lo[e] = pair_lo(p);
}

__device__ __forceinline__ f32x4 mma3(const BfPack<8>& a, const BfPack<8>& b,
                                              f32x4 c) {
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.lo, b.hi, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.hi, b.lo, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.hi, b.hi, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mma3(const BfPack<4>& a, const BfPack<4>& b,
                                              f32x4 c) {
  c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a.lo, b.hi, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a.hi, b.lo, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a.hi, b.hi, c, 0, 0, 0);
}

// The state contractions (forward, transpose) take KV values per lane; in the split form
// they go as packs of KB = 8 (one K = 32 instruction covers four lane groups of 8 states)
// or KB = 4 for KV = 4, NB packs per lane, values past KV zero.
template <int KV>
struct SplitShape {
  static constexpr int KB = KV <= 4 ? 4 : 8;
  static constexpr int NB = (KV + KB - 1) / KB;
};

}  // namespace hx
