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

// P in the P V products of ktir_attn_tile.hip and ktir_pattn_split.hip.  The
// loop holds P in f32; here it enters as terms of a 16-bit type whose products
// are exact and are summed in f32.
//   bf16: the terms have f32's exponents; three of them hold P's 24 bits.
//   f16: P lies in (0, e^P_LAG], relative to a base that the row max passes by
//   at most P_LAG.  Times P_SCALE = 2^13 (e^2 2^13 < 65504; O carries the
//   factor to the end) two f16 terms hold 23 bits of a P from P_SMALL on.  Below
//   that the second term is subnormal, so a step with a smaller P, other than
//   0, also adds what the two terms leave of each P, as three bf16 terms, times
//   V as two (exact: f16 has 11 bits, bf16 8).  Without it a key of weight
//   e^-16 counts nothing where the heaviest one has V = 0.
template <bool BF16>
constexpr float P_LAG = BF16 ? 8.f : 2.f;
template <bool BF16>
constexpr float P_SCALE = BF16 ? 1.f : 8192.f;
constexpr float P_SMALL = 0x1p-15f;

// four values times P_SCALE as PARTS terms of the type, largest first: t[p]
// holds (x0, x1) and (x2, x3) packed; what is left of them in x
template <bool BF16, int PARTS, bool REST>
__device__ __forceinline__ void p_split(float* x, uint32_t (&t)[PARTS][2]) {
  constexpr float S = P_SCALE<BF16>;
#pragma unroll
  for (int p = 0; p < PARTS; ++p) {
    t[p][0] = BF16 || p ? cvt2<BF16>(x[0], x[1]) : cvt2<BF16>(__fmul_rn(x[0], S), __fmul_rn(x[1], S));
    t[p][1] = BF16 || p ? cvt2<BF16>(x[2], x[3]) : cvt2<BF16>(__fmul_rn(x[2], S), __fmul_rn(x[3], S));
    if (REST || p + 1 < PARTS) {
      const f32x2_t a = uncvt2<BF16>(t[p][0]), b = uncvt2<BF16>(t[p][1]);
      const float h[4] = {a.x, a.y, b.x, b.y};
#pragma unroll
      for (int k = 0; k < 4; ++k) x[k] = BF16 || p ? __fsub_rn(x[k], h[k]) : __builtin_fmaf(x[k], S, -h[k]);   // exact
    }
  }
}

// eight values as three bf16 terms each, packed for an MFMA
__device__ __forceinline__ void p_split_bf(float* x, uint4 (&t)[3]) {
  uint32_t lo[3][2], hi[3][2];
  p_split<true, 3, false>(x, lo);
  p_split<true, 3, false>(x + 4, hi);
#pragma unroll
  for (int q = 0; q < 3; ++q) t[q] = make_uint4(lo[q][0], lo[q][1], hi[q][0], hi[q][1]);
}

// o + V^T P^T of 16 keys (a: V^T fragment).  INF_V: only the first term of P,
// which has P's sign, meets the infinities and NaN of V; the others would make
// NaN of an infinity.
template <bool BF16, int PARTS, bool INF_V>
__device__ __forceinline__ f32x16_t pv_mfma(uint4 a, const uint32_t (&t0)[PARTS][2], const uint32_t (&t1)[PARTS][2], f32x16_t o) {
  uint4 af = a;
  if constexpr (INF_V) af = make_uint4(finite2<BF16>(a.x), finite2<BF16>(a.y), finite2<BF16>(a.z), finite2<BF16>(a.w));
#pragma unroll
  for (int q = PARTS - 1; q >= 0; --q) o = mfma_at<BF16>(q ? af : a, make_uint4(t0[q][0], t0[q][1], t1[q][0], t1[q][1]), o);
  return o;
}

// the same for f16 V as two bf16 terms and P (or the rest of it) as three
template <bool INF_V>
__device__ __forceinline__ f32x16_t pv_mfma_bf(uint4 a, const uint4 (&t)[3], f32x16_t o) {
  const uint32_t w[4] = {a.x, a.y, a.z, a.w};
  uint32_t vh[4], vf[4], vl[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const f32x2_t v = uncvt2<false>(w[k]);
    vh[k] = cvt2<true>(v.x, v.y);
    const f32x2_t h = uncvt2<true>(vh[k]);
    vl[k] = cvt2<true>(__fsub_rn(v.x, h.x), __fsub_rn(v.y, h.y));
    vf[k] = vh[k];
    if constexpr (INF_V) {
      vf[k] = finite2<true>(vh[k]);
      vl[k] = finite2<true>(vl[k]);                // infinity - infinity
    }
  }
  const uint4 h = make_uint4(vh[0], vh[1], vh[2], vh[3]), f = make_uint4(vf[0], vf[1], vf[2], vf[3]),
              lo = make_uint4(vl[0], vl[1], vl[2], vl[3]);
#pragma unroll
  for (int q = 2; q >= 0; --q) {
    o = mfma_at<true>(lo, t[q], o);
    o = mfma_at<true>(q ? f : h, t[q], o);
  }
  return o;
}

// the smallest of N values, none of them negative, that is not 0 (any value
// above 1 where all are)
template <int N>
__device__ __forceinline__ float least_positive(const float* x) {
  uint32_t m = 0xffffffffu;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const uint32_t u = __float_as_uint(x[i]) - 1u;
    m = u < m ? u : m;
  }
  return __uint_as_float(m < 0x40000000u ? m : 0x40000000u);
}

// Slot permutation of the 16-byte chunks of a K or V row in LDS: 8 chunks for
// 128-byte rows (64 columns), 16 for 256-byte rows (128 columns).  Both are
// XORs of row bits chosen so that 8 rows' same chunk (ds_read_b128 of K) and 4
// rows' 32-byte pieces (ds_read_b64_tr_b16 of V) lie in distinct banks.
template <int D>
__device__ __forceinline__ int kv_swz(int r) {
  if constexpr (D == 64)
    return ((r & 1) << 1) ^ ((r & 2) << 1) ^ ((r >> 2) & 1) ^ (((r >> 3) & 1) << 1);
  else
    return ((r & 1) ? 4 : 0) ^ ((r & 2) ? 10 : 0) ^ ((r & 4) ? 1 : 0) ^ ((r & 8) ? 8 : 0);
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

// the NaN-propagating minimum of three
__device__ __forceinline__ float fmin3_nan(float a, float b, float c) {
  return __builtin_elementwise_minimum(__builtin_elementwise_minimum(a, b), c);
}

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
