// What the row kernels share: the position of a row, the row instructions
// between two folds, and the plan of the fixed-form kernels (softmax and
// norm-scale rows).
#pragma once
#include "ktir_program_impl.h"

namespace ktir {

typedef float gf2 __attribute__((ext_vector_type(2)));
typedef uint32_t gu4 __attribute__((ext_vector_type(4)));

// x / s for a row scalar s with r = 1/s correctly rounded: q = x r, then one
// Markstein correction q + (x - s q) r (fused); within one ulp of x / s and
// nearly always its correct rounding.  Operands near the ends of the
// exponent range take __fdiv_rn.
__device__ __forceinline__ float div_by(float x, float s, float r) {
  const float q = x * r;
  const float res = __builtin_fmaf(-s, q, x);
  return __builtin_fmaf(res, r, q);
}

// A leaf of a row program (outer dims only; rows have unit inner stride).
struct RwLeaf {
  uint64_t ptr, lane_base;
  int64_t base, lane_stride, lo, hi;
  int64_t strides[KTIR_MAX_DIMS - 1];   // outer dims
  int32_t dtype, esize;
};

// Position of row r: its lane (core) and its index in each outer dim.  Rows,
// lanes and dims are below 2^31 (checked at launch): 32-bit division.
struct RwPos {
  int32_t lane;
  int32_t idx[KTIR_MAX_DIMS - 1];
};

template <typename PL>
__device__ __forceinline__ RwPos rw_pos(const PL& SP, int64_t r, int32_t rows_per_lane) {
  RwPos p;
  const uint32_t ru = (uint32_t)r, rpl = (uint32_t)rows_per_lane;
  const uint32_t lane = ru / rpl;
  uint32_t t = ru - lane * rpl;
  p.lane = (int32_t)lane;
  const int nd = __builtin_amdgcn_readfirstlane(SP.nd);
#pragma unroll
  for (int d = KTIR_MAX_DIMS - 2; d >= 0; --d) {
    p.idx[d] = 0;
    if (d < nd - 1) {
      const uint32_t ext = (uint32_t)__builtin_amdgcn_readfirstlane((int)SP.shape[d]);
      const uint32_t q = t / ext;
      p.idx[d] = (int32_t)(t - q * ext);
      t = q;
    }
  }
  return p;
}

// element offset of column 0 of the row at p in leaf L
__device__ __forceinline__ int64_t rw_row_base(const RwLeaf& L, const RwPos& p) {
  int64_t e = L.lane_base ? uni(((const KTIR_G(int64_t)*)L.lane_base)[p.lane]) : L.base + (int64_t)p.lane * L.lane_stride;
#pragma unroll
  for (int d = 0; d < KTIR_MAX_DIMS - 1; ++d) e += (int64_t)p.idx[d] * L.strides[d];
  return e;
}

template <typename PL, typename RR>
__device__ __forceinline__ void rw_row_exec(const PL& SP, const ktir_instr_t in, RR& rr, int64_t lane) {
  const int op = in.op;
  const float a = rr.get(in.a), b = rr.get(in.b);
  float v;
  if (op >= KTIR_OP_NEGF && op < KTIR_OP_ADDF) {
    v = unop_simple(op, in.dt, a);
  } else if (op >= KTIR_OP_ADDI) {
    v = __int_as_float(binop_i_simple(op, __float_as_int(a), __float_as_int(b)));
  } else if (op >= KTIR_OP_ADDF) {
    v = binop_f_simple(op, in.dt, a, b);
  } else {
    switch (op) {
      case KTIR_OP_CONST: v = __int_as_float(in.imm); break;
      case KTIR_OP_LANE: {
        const double d = ((const KTIR_G(double)*)uni((int64_t)SP.lane_scalars))[lane * uni(SP.n_lane_scalars) + in.aux];
        v = is_float_dt(in.dt) ? round_to((float)d, in.dt) : __int_as_float((int)(long long)d);
        break;
      }
      case KTIR_OP_CAST: v = cast_val(a, in.aux, in.dt); break;
      case KTIR_OP_BITCAST: v = a; break;
      case KTIR_OP_SELECT: v = __float_as_int(a) ? b : rr.get(in.c); break;
      case KTIR_OP_FMA: v = round_to(__fadd_rn(__fmul_rn(a, b), rr.get(in.c)), in.dt); break;
      case KTIR_OP_CMPF: v = __int_as_float(cmp_f(in.aux, a, b)); break;
      case KTIR_OP_CMPI: v = __int_as_float(cmp_i(in.aux, __float_as_int(a), __float_as_int(b))); break;
      default: v = 0.f;
    }
  }
  rr.set(in.dst, __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))));
}

constexpr int RF_MAX_ROW = 8;
enum { RF_SOFTMAX = 1, RF_NORM = 2, RF_SOFTMAX16 = 3, RF_NORM16 = 4 };

struct RfPlan {
  int32_t nd, has_w, w_first, n_row0, n_row1, numf;   // numf: softmax16's max ignores NaN
  int64_t shape[KTIR_MAX_DIMS];
  uint64_t lane_scalars;
  int64_t n_lane_scalars;
  RwLeaf x, w, y;
  int8_t fold0, fold1;        // registers the folds write
  int8_t m, s;                // softmax: the subtracted register and the divisor; norm-scale: s the multiplier
  int32_t pad1;
  ktir_instr_t row0[RF_MAX_ROW], row1[RF_MAX_ROW];   // after the first and the second fold
};

template <int DT>
__device__ __forceinline__ void rf_unpack(const gu4 c, float (&v)[8]) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t u = c[k];
    if (DT == KTIR_BF16) {
      v[2 * k] = __uint_as_float(u << 16);
      v[2 * k + 1] = __uint_as_float(u & 0xffff0000u);
    } else {
      v[2 * k] = (float)__builtin_bit_cast(_Float16, (uint16_t)(u & 0xffffu));
      v[2 * k + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(u >> 16));
    }
  }
}

// eight values rounded to nearest-even in DT, packed
template <int DT>
__device__ __forceinline__ gu4 rf_pack(const float (&v)[8]) {
  gu4 c;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (DT == KTIR_BF16)
      c[k] = (__float_as_uint(round_bf16(v[2 * k])) >> 16) | (__float_as_uint(round_bf16(v[2 * k + 1])) & 0xffff0000u);
    else
      c[k] = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v[2 * k]) |
             ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v[2 * k + 1]) << 16);
  }
  return c;
}

// as rf_pack, f16 pairs converted by one instruction (v_cvt_pk_f16_f32, round
// to nearest even); the row kernels whose register count it does not raise
template <int DT>
__device__ __forceinline__ gu4 rf_pack2(const float (&v)[8]) {
  if (DT == KTIR_BF16) return rf_pack<DT>(v);
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  gu4 c;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const f2 x = {v[2 * k], v[2 * k + 1]};
    c[k] = __builtin_bit_cast(uint32_t, __builtin_convertvector(x, h2));
  }
  return c;
}

// Row registers in lanes 0..7 of one vector register: a read is one lane
// access and a write one lane select, with no selection over the register
// number.
struct RowLanes {
  int v, lane;
  __device__ __forceinline__ float get(int i) const { return __int_as_float(__builtin_amdgcn_readlane(v, i)); }
  __device__ __forceinline__ void set(int i, float x) {
    const int u = __builtin_amdgcn_readfirstlane(__float_as_int(x));
    v = lane == i ? u : v;
  }
};

}  // namespace ktir
