// Device helpers shared by the fused attention kernels.
#pragma once
#include "ktir_common.h"

namespace ktir {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr float LOG2E = 1.44269504088896341f;

template <bool BF16>
__device__ __forceinline__ f32x16_t mfma_at(const uint4& a, const uint4& b, f32x16_t c) {
  if constexpr (BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), c,
                                                  0, 0, 0);
}

// (a, b) rounded to nearest-even in the operand type, packed low/high
template <bool BF16>
__device__ __forceinline__ uint32_t cvt2(float a, float b) {
  const f32x2_t v = {a, b};
  if constexpr (BF16) return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
  else return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
}

// the two operand-type values of a packed word, back in f32
template <bool BF16>
__device__ __forceinline__ f32x2_t uncvt2(uint32_t w) {
  if constexpr (BF16) return f32x2_t{__uint_as_float(w << 16), __uint_as_float(w & 0xffff0000u)};
  else return __builtin_convertvector(__builtin_bit_cast(f16x2_t, w), f32x2_t);
}

// P is carried into the P @ V product as hi + lo, both in the operand type
// (hi = P rounded, lo = the rounded remainder), so the product keeps about
// 16 significant bits of P instead of the operand type's 8 (bf16) / 11 (f16).
template <bool BF16>
__device__ __forceinline__ void split4(const float* p, uint32_t& h0, uint32_t& h1, uint32_t& l0, uint32_t& l1) {
  h0 = cvt2<BF16>(p[0], p[1]);
  h1 = cvt2<BF16>(p[2], p[3]);
  const f32x2_t a = uncvt2<BF16>(h0), b = uncvt2<BF16>(h1);
  l0 = cvt2<BF16>(__fsub_rn(p[0], a.x), __fsub_rn(p[1], a.y));
  l1 = cvt2<BF16>(__fsub_rn(p[2], b.x), __fsub_rn(p[3], b.y));
}

// the packed values of w with 0 in the place of infinities and NaN
template <bool BF16>
__device__ __forceinline__ uint32_t finite2(uint32_t w) {
  constexpr uint32_t E = BF16 ? 0x7f80u : 0x7c00u;
  const uint32_t lo = (w & E) == E ? 0u : w & 0xffffu, hi = ((w >> 16) & E) == E ? 0u : w & 0xffff0000u;
  return lo | hi;
}

// the smallest f16 in the place of a leading term 0 whose value is positive
__device__ __forceinline__ void lift4(const float* p, uint32_t (&t)[2]) {
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    if (p[2 * k] > 0.f && !(t[k] & 0xffffu)) t[k] |= 1u;
    if (p[2 * k + 1] > 0.f && !(t[k] >> 16)) t[k] |= 0x10000u;
  }
}

// v_permlane32_swap: lanes 32-63 of a trade places with lanes 0-31 of b, so
// afterwards lanes 0-31 hold a of both half-waves (own in a, the other
// half's in b) and lanes 32-63 hold b of both (the other half's in a)
__device__ __forceinline__ void swap32(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// value of the other half-wave's lane l ^ 32
__device__ __forceinline__ float other_half(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float((threadIdx.x & 32) ? r[0] : r[1]);
}

// max / sum of x over the lane pair (l, l ^ 32): after v_permlane32_swap the
// two results hold the pair's two values in either order, so one maximum or
// add of them gives both lanes the same result (IEEE add commutes)
__device__ __forceinline__ float pair_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __builtin_elementwise_maximum(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pair_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __fadd_rn(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// arith.maximumf: NaN-propagating maximum (v_maximum3_f32 on gfx950)
__device__ __forceinline__ float fmax_nan(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ float fmax3_nan(float a, float b, float c) { return fmax_nan(fmax_nan(a, b), c); }

// x = -inf in the lanes of mask, in place (v_cndmask_b32 on x's own
// register: the caller's S values keep the registers the MFMAs wrote)
// -inf where `kill` holds: a plain select, so the compiler inserts the wait
// states between an MFMA result and this VALU read itself
__device__ __forceinline__ float mask_ninf(float x, bool kill) { return kill ? -__builtin_inff() : x; }

// e^x as 2^(x log2 e) on the hardware exp2 (v_exp_f32)
__device__ __forceinline__ float exp_f(float x) { return __builtin_amdgcn_exp2f(__fmul_rn(x, LOG2E)); }

// ds_read_b64_tr_b16: in each 16-lane group, member t receives element t % 4
// of the 4-element chunks addressed by members 4s + t / 4, s = 0..3
__device__ __forceinline__ uint2 ds_tr16(const uint16_t* p) {
  const s16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)p);
  return __builtin_bit_cast(uint2, v);
}

}  // namespace ktir
