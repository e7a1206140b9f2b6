// Sums and differences of two products, elementwise: out = a*b +- c*d, and
// the pair out1 = a*b +- c*d, out2 = a*d +- c*b in one pass over the four
// inputs (a rotation: both halves of a rotary position embedding).
//
// Bound: bytes.  A pair moves 6 elements (the angles of a rotary embedding
// come back from L2, so 4 reach memory) for 6 operations; per element the
// conversions of 16-bit types to the f32 the operations run in, and back, are
// most of the instructions.  The straight line is what matters: as a chain of
// interpreted register ops (prog_map_n) 40 heads x 4096 x 128 f16 took 46.8 us
// for each half, two launches, 93 us; the pair in one launch takes 20.3 us
// (84 MB read and written, 4.1 TB/s; the least at a large copy's rate is 15).
#include "ktir_program_impl.h"

namespace ktir {

typedef uint32_t ru4 __attribute__((ext_vector_type(4)));

// the inputs' and outputs' leaves and the sign bit each product gets before
// the sum (second output: products a*d and c*b)
struct RotPlan {
  int32_t leaf[4], out[2], n_out;
  uint32_t neg[4];
};

template <int DT>
struct RotRaw {
  ru4 w[DT == KTIR_F32 ? 2 : 1];
};

template <int DT>
__device__ __forceinline__ RotRaw<DT> rot_load(const ktir_leaf_t& L, int64_t e) {
  RotRaw<DT> r;
  const KTIR_G(ru4)* p = (const KTIR_G(ru4)*)((const KTIR_G(uint8_t)*)L.ptr + e * (DT == KTIR_F32 ? 4 : 2));
  r.w[0] = p[0];
  if (DT == KTIR_F32) r.w[DT == KTIR_F32 ? 1 : 0] = p[1];
  return r;
}

// a chunk some of whose elements lie outside the allocation: those read as 0
template <int DT>
__device__ __forceinline__ RotRaw<DT> rot_load_edge(const ktir_leaf_t& L, int64_t e0) {
  uint32_t v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int64_t e = e0 + i;
    const bool in = e >= L.lo && e < L.hi;
    if (DT == KTIR_F32) v[i] = in ? ((const KTIR_G(uint32_t)*)L.ptr)[e] : 0u;
    else v[i] = in ? ((const KTIR_G(uint16_t)*)L.ptr)[e] : 0u;
  }
  RotRaw<DT> r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (DT == KTIR_F32) {
      r.w[0][i] = v[i];
      r.w[DT == KTIR_F32 ? 1 : 0][i] = v[4 + i];
    } else {
      r.w[0][i] = v[2 * i] | (v[2 * i + 1] << 16);
    }
  }
  return r;
}

template <int DT>
__device__ __forceinline__ float rot_elem(const RotRaw<DT>& r, int i) {
  if (DT == KTIR_F32) return __uint_as_float(i < 4 ? r.w[0][i & 3] : r.w[DT == KTIR_F32 ? 1 : 0][i & 3]);
  const uint32_t u = r.w[0][i >> 1];
  if (DT == KTIR_BF16) return __uint_as_float(i & 1 ? u & 0xffff0000u : u << 16);
  return (float)__builtin_bit_cast(_Float16, (uint16_t)(i & 1 ? u >> 16 : u & 0xffffu));
}

template <int DT>
__device__ __forceinline__ float rot_sum(float a, float b, float c, float d, uint32_t n0, uint32_t n1) {
  const float x = round_to(mul_keep(a, b), DT), y = round_to(mul_keep(c, d), DT);
  return __fadd_rn(__uint_as_float(__float_as_uint(x) ^ n0), __uint_as_float(__float_as_uint(y) ^ n1));
}

template <int DT>
__device__ __forceinline__ void rot_store(const ktir_leaf_t& L, int64_t e0, const float (&v)[8]) {
  if (e0 >= L.lo && e0 + 8 <= L.hi) {
    if (DT == KTIR_F32) {
      KTIR_G(ru4)* p = (KTIR_G(ru4)*)((KTIR_G(float)*)L.ptr + e0);
#pragma unroll
      for (int k = 0; k < 2; ++k)
        p[k] = ru4{__float_as_uint(v[4 * k]), __float_as_uint(v[4 * k + 1]), __float_as_uint(v[4 * k + 2]),
                   __float_as_uint(v[4 * k + 3])};
      return;
    }
    ru4 u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (DT == KTIR_F16)
        u[i] = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v[2 * i]) |
               ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v[2 * i + 1]) << 16);
      else
        u[i] = (__float_as_uint(round_bf16(v[2 * i])) >> 16) |
               (__float_as_uint(round_bf16(v[2 * i + 1])) & 0xffff0000u);
    }
    __builtin_nontemporal_store(u, (KTIR_G(ru4)*)((KTIR_G(uint16_t)*)L.ptr + e0));
    return;
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int64_t e = e0 + i;
    if (e >= L.lo && e < L.hi) store_elem(L.ptr, e, DT, v[i]);
  }
}

// element offset of the chunk at indices c of lane t; a wavefront that lies
// in one lane (`one`, t uniform) reads the lane's offset through the scalar cache
__device__ __forceinline__ int64_t rot_off(const ktir_leaf_t& L, int nd, uint32_t t, bool one, const uint32_t* c,
                                           int64_t col) {
  int64_t o;
  if (L.lane_base == 0) o = L.base + (int64_t)t * L.lane_stride;
  else if (one) o = ((const __attribute__((address_space(4))) int64_t*)L.lane_base)[uni((int)t)];
  else o = ((const KTIR_G(int64_t)*)L.lane_base)[t];
#pragma unroll
  for (int d = 0; d < KTIR_MAX_DIMS - 1; ++d)
    if (d < nd - 1) o += (int64_t)c[d] * L.strides[d];
  return o + col;
}

// One chunk of 8 elements per thread: all loads are issued before anything is
// computed.
template <int DT, int NOUT>
__global__ __launch_bounds__(256) void prog_rot(const ktir_prog_t P, const FlatDivs D, uint32_t total,
                                                const RotPlan R) {
  const int nd = P.ndim;
  const uint32_t v = blockIdx.x * 256 + threadIdx.x;
  if (v >= total) return;
  const uint32_t row = fdiv(v, D.nvi);
  const int64_t col = (int64_t)(v - row * D.nvi.d) * 8;
  uint32_t c[KTIR_MAX_DIMS] = {0, 0, 0, 0}, t = row;
#pragma unroll
  for (int d = KTIR_MAX_DIMS - 2; d >= 0; --d) {
    if (d < nd - 1) {
      const uint32_t q = fdiv(t, D.dim[d]);
      c[d] = t - q * D.dim[d].d;
      t = q;
    }
  }
  const bool one = __all((int)t == uni((int)t));
  const ktir_leaf_t &L0 = P.leaves[R.leaf[0]], &L1 = P.leaves[R.leaf[1]], &L2 = P.leaves[R.leaf[2]],
                    &L3 = P.leaves[R.leaf[3]], &O0 = P.leaves[R.out[0]], &O1 = P.leaves[R.out[1]];
  const int64_t o0 = rot_off(L0, nd, t, one, c, col), o1 = rot_off(L1, nd, t, one, c, col),
                o2 = rot_off(L2, nd, t, one, c, col), o3 = rot_off(L3, nd, t, one, c, col);
  const int64_t s0 = rot_off(O0, nd, t, one, c, col);
  const int64_t s1 = NOUT == 2 ? rot_off(O1, nd, t, one, c, col) : 0;
  auto in = [](const ktir_leaf_t& L, int64_t o) { return o >= L.lo && o + 8 <= L.hi; };
  RotRaw<DT> a, b, cc, d;
  if (__all(in(L0, o0) && in(L1, o1) && in(L2, o2) && in(L3, o3))) {
    a = rot_load<DT>(L0, o0);
    b = rot_load<DT>(L1, o1);
    cc = rot_load<DT>(L2, o2);
    d = rot_load<DT>(L3, o3);
  } else {
    a = rot_load_edge<DT>(L0, o0);
    b = rot_load_edge<DT>(L1, o1);
    cc = rot_load_edge<DT>(L2, o2);
    d = rot_load_edge<DT>(L3, o3);
  }
  float y[8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
    y[i] = rot_sum<DT>(rot_elem<DT>(a, i), rot_elem<DT>(b, i), rot_elem<DT>(cc, i), rot_elem<DT>(d, i), R.neg[0],
                       R.neg[1]);
  rot_store<DT>(O0, s0, y);
  if (NOUT == 2) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      y[i] = rot_sum<DT>(rot_elem<DT>(a, i), rot_elem<DT>(d, i), rot_elem<DT>(cc, i), rot_elem<DT>(b, i), R.neg[2],
                         R.neg[3]);
    rot_store<DT>(O1, s1, y);
  }
}

// What each register of a program of this form holds: an input, a product of
// two inputs, or the signed sum of two products.
struct RotVal {
  int kind = 0;             // 0 nothing, 1 input, 2 product, 3 sum
  int in[4] = {0, 0, 0, 0};
  bool sub = false;
};

static bool match_rot(const ktir_prog_t& P, RotPlan& R, int& dt) {
  if (P.mode != 0 || P.n_pf < 3 || P.n_pf > 4) return false;
  RotVal r[KTIR_NREG];
  for (int k = 0; k < P.n_pf; ++k) {
    r[k].kind = 1;
    r[k].in[0] = P.pf_leaf[k];
  }
  dt = P.leaves[P.pf_leaf[0]].dtype;
  RotVal out[2];
  R.n_out = 0;
  for (int i = 0; i < P.n_instr; ++i) {
    const ktir_instr_t& x = P.instr[i];
    if (x.a < 0 || x.a >= KTIR_NREG || x.b < 0 || x.b >= KTIR_NREG || x.dst < 0 || x.dst >= KTIR_NREG) return false;
    const RotVal a = r[x.a], b = r[x.b];
    if (x.op == KTIR_OP_ST) {
      if (a.kind != 3 || R.n_out == 2) return false;
      R.out[R.n_out] = x.aux;
      out[R.n_out++] = a;
      continue;
    }
    if (x.dt != dt) return false;
    RotVal v;
    if (x.op == KTIR_OP_MULF && a.kind == 1 && b.kind == 1) {
      v.kind = 2;
      v.in[0] = a.in[0];
      v.in[1] = b.in[0];
    } else if ((x.op == KTIR_OP_ADDF || x.op == KTIR_OP_SUBF) && a.kind == 2 && b.kind == 2) {
      v.kind = 3;
      v.in[0] = a.in[0], v.in[1] = a.in[1], v.in[2] = b.in[0], v.in[3] = b.in[1];
      v.sub = x.op == KTIR_OP_SUBF;
    } else {
      return false;
    }
    r[x.dst] = v;
  }
  if (R.n_out == 0 || P.instr[P.n_instr - 1].op != KTIR_OP_ST) return false;
  for (int k = 0; k < 4; ++k) R.leaf[k] = out[0].in[k];
  const uint32_t S = 0x80000000u;
  R.neg[0] = R.neg[2] = R.neg[3] = 0;
  R.neg[1] = out[0].sub ? S : 0;
  if (R.n_out == 1) {
    R.out[1] = R.out[0];
    return true;
  }
  // the second sum's products each take one factor from each product of the
  // first: name the factors so that they are a*d and c*b
  const int *p = out[0].in, *q = out[1].in;
  for (int i = 0; i < 4; ++i)
    for (int j = 0; j < i; ++j)
      if (p[i] == p[j]) return false;
  for (int m = 0; m < 2; ++m)
    for (int n = 0; n < 2; ++n) {
      const int A = p[m], B = p[1 - m], Dd = p[2 + n], C = p[3 - n];
      const bool first = (q[0] == A && q[1] == Dd) || (q[0] == Dd && q[1] == A);
      const bool second = (q[2] == C && q[3] == B) || (q[2] == B && q[3] == C);
      if (first && second) {
        R.leaf[0] = A, R.leaf[1] = B, R.leaf[2] = C, R.leaf[3] = Dd;
        R.neg[3] = out[1].sub ? S : 0;
        return true;
      }
    }
  return false;
}

template <int DT>
static void launch_rot(const ktir_prog_t& P, const FlatDivs& D, uint32_t total, const RotPlan& R) {
  const dim3 g((total + 255) / 256), b(256);
  if (R.n_out == 2) hipLaunchKernelGGL((prog_rot<DT, 2>), g, b, 0, stream(), P, D, total, R);
  else hipLaunchKernelGGL((prog_rot<DT, 1>), g, b, 0, stream(), P, D, total, R);
}

// Launch `P` as a sum of two products (or a pair of them) when every leaf is
// one 16- or 32-bit float type, read and written in aligned groups of 8.
bool try_launch_rot(const ktir_prog_t& P, int64_t rows, int64_t inner) {
  RotPlan R;
  int dt;
  if (inner % 8 || !match_rot(P, R, dt)) return false;
  if (dt != KTIR_F16 && dt != KTIR_BF16 && dt != KTIR_F32) return false;
  auto ok = [&](const ktir_leaf_t& L) {
    return L.dtype == dt && L.offsets == 0 && L.winner == 0 && L.strides[P.ndim - 1] == 1 &&
           (L.flags & KTIR_LEAF_VEC8);
  };
  for (int k = 0; k < 4; ++k)
    if (!ok(P.leaves[R.leaf[k]])) return false;
  for (int k = 0; k < R.n_out; ++k)
    if (!ok(P.leaves[R.out[k]])) return false;
  const int64_t chunks = rows * (inner / 8);
  if (chunks >= (int64_t)0x7fffff00) return false;
  FlatDivs D;
  D.nvi = make_fastdiv((uint32_t)(inner / 8));
  for (int d = 0; d < KTIR_MAX_DIMS; ++d) D.dim[d] = make_fastdiv(d < P.ndim - 1 ? (uint32_t)P.shape[d] : 1);
  D.rows_per_lane = 0;
  const uint32_t total = (uint32_t)chunks;
  if (dt == KTIR_F16) launch_rot<KTIR_F16>(P, D, total, R);
  else if (dt == KTIR_BF16) launch_rot<KTIR_BF16>(P, D, total, R);
  else launch_rot<KTIR_F32>(P, D, total, R);
  return true;
}

}  // namespace ktir
