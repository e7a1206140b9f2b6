// Device helpers shared by the MFMA matmul kernels.
#pragma once
#include "ktir_common.h"

namespace ktir {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bfx8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

template <bool BF16>
__device__ __forceinline__ f32x16 mfma32(const uint4& a, const uint4& b, f32x16 c) {
  if constexpr (BF16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bfx8, a), __builtin_bit_cast(bfx8, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
  }
}

// one result element of dtype DT (f32, f16 or bf16, round to nearest even)
template <int DT>
__device__ __forceinline__ void mm_put(uint64_t ptr, int64_t off, float v) {
  if constexpr (DT == KTIR_F32)
    ((KTIR_G(float)*)ptr)[off] = v;
  else if constexpr (DT == KTIR_F16)
    ((KTIR_G(_Float16)*)ptr)[off] = (_Float16)v;
  else
    ((KTIR_G(uint16_t)*)ptr)[off] = (uint16_t)(__float_as_uint(round_bf16(v)) >> 16);
}

typedef short mm_s16x4 __attribute__((ext_vector_type(4)));

// slot permutation of the 16 chunks of a 256-byte LDS row r (an XOR of row
// bits; conflict-free for ds_read_b64_tr_b16 column reads and ds_read_b128
// row reads)
__device__ __forceinline__ int swz16(int r) {
  return ((r & 1) ? 4 : 0) ^ ((r & 2) ? 10 : 0) ^ ((r & 4) ? 1 : 0) ^ ((r & 8) ? 8 : 0);
}

__device__ __forceinline__ int swz_a(int r) { return (r & 7) ^ ((r >> 3) & 1); }

__device__ __forceinline__ uint2 mm_tr16(const uint16_t* p) {
  const mm_s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) mm_s16x4*)p);
  return __builtin_bit_cast(uint2, v);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t mm_rsrc(const uint16_t* base, int64_t hi_elems) {
  int64_t bytes = hi_elems * 2;
  if (bytes < 0) bytes = 0;
  if (bytes > 0xffffffffll) bytes = 0xffffffffll;
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)(uint32_t)bytes, 0x00020000);
}

}  // namespace ktir
