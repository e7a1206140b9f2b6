// Softmax and norm-scale row programs (the fixed forms of ktir_rows.hip, f32
// math on f16 / bf16 rows: dialects/linalg_ops.py:86-246 folds with their
// elementwise ops) for rows of any length up to KTIR_MAX_ROW and any alignment.
//
// W wavefronts own a row (one up to 3072 elements, norm rows up to 4096, then
// two and four) and
// read it once, each thread C chunks of 8 elements; a workgroup runs a stream
// of rows.  Few wavefronts per row: what a row costs besides its elements (the
// reductions, the row instructions between the folds) every one of them pays.
// Rows that do not start on 16-byte boundaries are read with unaligned 16-byte
// loads; the chunk that the row's end cuts is read from the last 8 elements
// and shifted.  The exponentials stay in f32 registers between the sum and the
// store.  The launch takes rows that lie one step apart and wholly inside
// their allocations, so the kernel has no other bounds to check.
// Memory bounds it from about 1000 elements on, the reductions below.
// Against the interpreter's row kernel (prog_rows), f16 unless said:
//   softmax  8192 x 3000 bf16 1191 -> 20 us (4.9 TB/s), 32768 x 1000 2148 -> 25 us,
//            2048 x 16384 1298 -> 26 us;
//   rmsnorm  8192 x 5120 1395 -> 43 us (3.9 TB/s), 32768 x 1000 1813 -> 47 us,
//            2048 x 16384 979 -> 27 us.
//   row max and the softmax sum: per thread, lane exchanges, then one exchange
//     between the wavefronts through LDS;
//   the norm's sum of squares: the reference's halving tree (element i with
//     i + n/2, an odd last element carried) in LDS, up to three levels per
//     pass, the last 64 values by shuffles.  Where both halves of a row are
//     whole chunks (P = 2) a thread holds the same chunks of both, and the
//     first level runs in registers.
#include "ktir_rowform.h"

namespace ktir {

constexpr float RA_LOG2E = 1.44269504088896341f, RA_LOG2E_LO = 1.92596299112661746887e-8f, RA_LN2 = 0.693147180559945309f;

typedef float ra_f2 __attribute__((ext_vector_type(2)));
typedef __bf16 ra_b2 __attribute__((ext_vector_type(2)));
typedef _Float16 ra_h2 __attribute__((ext_vector_type(2)));

// 16 bytes at any 2-byte aligned address
typedef uint32_t ra_u4 __attribute__((ext_vector_type(4), aligned(2)));

// e^x within about one ulp: the hardware exp2 of x log2 e, times the rest of
// that product; results below f32's normal range through a scaled exp2
__device__ __forceinline__ float ra_exp(float x) {
  const float t = x * RA_LOG2E;
  const bool tiny = t < -125.f;
  const float e = __builtin_amdgcn_exp2f(tiny ? t + 64.f : t);
  const float r = __builtin_fmaf(x, RA_LOG2E_LO, __builtin_fmaf(x, RA_LOG2E, -t));
  // 0, infinity and NaN stand as they are
  return ldexpf(fabsf(t) < 200.f ? __builtin_fmaf(e, r * RA_LN2, e) : e, tiny ? -64 : 0);
}

// the same for x <= 0 or NaN, with 0 for results below f32's normal range
__device__ __forceinline__ float ra_exp_neg(float x) {
  x = __builtin_elementwise_maximum(x, -200.f);
  const float t = x * RA_LOG2E;
  const float e = __builtin_amdgcn_exp2f(t);
  const float r = __builtin_fmaf(x, RA_LOG2E_LO, __builtin_fmaf(x, RA_LOG2E, -t));
  return __builtin_fmaf(e, r * RA_LN2, e);
}

// eight values rounded to nearest-even in DT, packed
template <int DT>
__device__ __forceinline__ gu4 ra_pack(const float (&v)[8]) {
  gu4 c;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const ra_f2 x = {v[2 * k], v[2 * k + 1]};
    if constexpr (DT == KTIR_BF16) c[k] = __builtin_bit_cast(uint32_t, __builtin_convertvector(x, ra_b2));
    else c[k] = __builtin_bit_cast(uint32_t, __builtin_convertvector(x, ra_h2));
  }
  return c;
}

// the last `cnt` (1 .. 7) of the eight elements of c, moved to the front
__device__ __forceinline__ gu4 ra_shift(gu4 c, int cnt) {
  uint64_t lo = (uint64_t)c[0] | ((uint64_t)c[1] << 32), hi = (uint64_t)c[2] | ((uint64_t)c[3] << 32);
  int s = 8 - cnt;
  if (s >= 4) {
    lo = hi;
    hi = 0;
    s -= 4;
  }
  if (s) {
    lo = (lo >> (16 * s)) | (hi << (64 - 16 * s));
    hi >>= 16 * s;
  }
  return gu4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
}

// What the kernel needs of a plan: leaves as the address of row 0 and the
// step between rows (elements), and the row instructions.
struct RaPlan {
  uint64_t x, w, y;
  int64_t x_step, y_step;
  uint64_t lane_scalars;
  int64_t n_lane_scalars;
  int32_t n, rows, rows_per_lane, has_w, w_first, n_row0, n_row1;
  int8_t fold0, fold1, m, s;
  ktir_instr_t row0[RF_MAX_ROW], row1[RF_MAX_ROW];
};

// Where a thread's chunks lie in the row: chunk i = p (C / P) + q is chunk
// t + q T of part p of P equal parts.  Every chunk but a part's last (q =
// C / P - 1) lies whole inside the row: the launch picks C so.
template <int C, int P>
struct RaMap {
  static constexpr int Q = C / P;
  int t, T, part;                              // part: elements of one part
  __device__ __forceinline__ int off(int i) const { return (i / Q) * part + 8 * (t + (i % Q) * T); }
  // elements of a part's last chunk (below 1: none, above 7: all eight)
  __device__ __forceinline__ int last() const { return part - 8 * (t + (Q - 1) * T); }
};

template <int C, int P>
__device__ __forceinline__ gu4 ra_chunk(uint64_t row, const RaMap<C, P>& M, int i) {
  const int end = M.part * P - 8;
  int o = M.off(i);
  if (i % M.Q == M.Q - 1) o = o < end ? o : end;
  return *(const KTIR_G(ra_u4)*)((const KTIR_G(uint16_t)*)row + o);
}

template <int C, int P>
__device__ __forceinline__ void ra_load(uint64_t row, const RaMap<C, P>& M, gu4 (&c)[C]) {
  const KTIR_G(uint16_t)* p = (const KTIR_G(uint16_t)*)row;
  const int end = M.part * P - 8;
#pragma unroll
  for (int i = 0; i < C; ++i) {
    int o = M.off(i);
    if (i % M.Q == M.Q - 1) o = o < end ? o : end;
    c[i] = *(const KTIR_G(ra_u4)*)(p + o);
  }
}

// the cut chunk's elements to its front, `pad` (a packed pair) in the place
// of elements past the row's end (P = 2: parts are whole chunks)
template <int C, int P>
__device__ __forceinline__ void ra_trim(const RaMap<C, P>& M, gu4 (&c)[C], uint32_t pad) {
  const int k = M.last();
  if (k >= 8) return;
  if constexpr (P == 1) {
    if (k > 0) c[C - 1] = ra_shift(c[C - 1], k);
  }
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t u = c[(p + 1) * M.Q - 1][j];
      c[(p + 1) * M.Q - 1][j] = 2 * j >= k ? pad : (2 * j + 1 >= k ? (u & 0xffffu) | (pad & 0xffff0000u) : u);
    }
}

template <int C, int P>
__device__ __forceinline__ void ra_store(uint64_t row, const RaMap<C, P>& M, int i, const gu4 c) {
  KTIR_G(uint16_t)* p = (KTIR_G(uint16_t)*)row + M.off(i);
  const int k = i % M.Q == M.Q - 1 ? M.last() : 8;
  if (k >= 8) {
    *(KTIR_G(ra_u4)*)p = c;
  } else if (P == 1 && k > 0) {
#pragma unroll
    for (int j = 0; j < 7; ++j)
      if (j < k) p[j] = (uint16_t)(c[j >> 1] >> (16 * (j & 1)));
  }
}

// LDS written by this workgroup (W = 1: by this wavefront) is visible after it
template <int W>
__device__ __forceinline__ void ra_sync() {
  if constexpr (W == 1) {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  } else {
    __syncthreads();
  }
}

template <int CTRL>
__device__ __forceinline__ float ra_dpp(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false));
}

// v combined by the commutative f over the row's wavefronts, the same in every
// thread: lanes 32 and 16 apart trade places, then rotations inside the 16
// lanes of a row; lane 0's result goes to all
template <int W, typename F>
__device__ __forceinline__ float ra_all(float v, float* lds, F f) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(b[0]), __uint_as_float(b[1]));
  v = f(v, ra_dpp<0x128>(v));                  // row_ror:8
  v = f(v, ra_dpp<0x124>(v));                  // row_ror:4
  v = f(v, ra_dpp<0x122>(v));                  // row_ror:2
  v = f(v, ra_dpp<0x121>(v));                  // row_ror:1
  v = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
  if constexpr (W > 1) {
    lds[threadIdx.x >> 6] = v;                 // every lane of a wavefront the same value
    __syncthreads();
    v = lds[0];
#pragma unroll
    for (int w = 1; w < W; ++w) v = f(v, lds[w]);
  }
  return v;
}

// The reference's halving sum of the `cur` values in buf (T threads, thread t),
// the same in every thread.  A level writes value i over buf[i], which only the
// thread of i reads; the carried last value lands on buf[half], which thread 0
// has read by then.
template <int W>
__device__ __forceinline__ float ra_tree(float* buf, int cur, int t, int T) {
  ra_sync<W>();
  while (cur > 64) {
    if (!(cur & 7)) {
      const int s = cur >> 3;
      for (int i = t; i < s; i += T) {
        const float a = __fadd_rn(__fadd_rn(buf[i], buf[i + 4 * s]), __fadd_rn(buf[i + 2 * s], buf[i + 6 * s]));
        const float b = __fadd_rn(__fadd_rn(buf[i + s], buf[i + 5 * s]), __fadd_rn(buf[i + 3 * s], buf[i + 7 * s]));
        buf[i] = __fadd_rn(a, b);
      }
      cur = s;
    } else if (!(cur & 3)) {
      const int s = cur >> 2;
      for (int i = t; i < s; i += T)
        buf[i] = __fadd_rn(__fadd_rn(buf[i], buf[i + 2 * s]), __fadd_rn(buf[i + s], buf[i + 3 * s]));
      cur = s;
    } else {
      const int s = cur >> 1;
      for (int i = t; i < s; i += T) buf[i] = __fadd_rn(buf[i], buf[i + s]);
      if (cur & 1) {
        if (t == 0) buf[s] = buf[cur - 1];
        cur = s + 1;
      } else {
        cur = s;
      }
    }
    ra_sync<W>();
  }
  const int l = t & 63;
  float v = l < cur ? buf[l] : 0.f;
  while (cur > 1) {
    const int s = cur >> 1;
    const float y = __shfl(v, l + s);          // lane s of an odd level takes the carried value
    v = l < s ? __fadd_rn(v, y) : y;
    cur = s + (cur & 1);
  }
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

template <int C, int DT, int W>
__device__ __forceinline__ void ra_softmax(const RaPlan& F, gu4 (&c)[C], const RaMap<C, 1>& M, uint64_t y_row, int64_t lane,
                                           RowLanes& rr, float* lds) {
  auto maxf = [](float a, float b) { return __builtin_elementwise_maximum(a, b); };   // NaN-propagating
  float mx = -__builtin_inff();
  float lo = __builtin_inff();                // smallest element above -inf (bf16: its exponential may be subnormal)
#pragma unroll
  for (int i = 0; i < C; ++i) {
    float v[8];
    rf_unpack<DT>(c[i], v);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      mx = maxf(mx, v[j]);
      if constexpr (DT == KTIR_BF16) lo = fminf(lo, v[j] > -__builtin_inff() ? v[j] : __builtin_inff());
    }
    if constexpr (DT == KTIR_BF16) asm volatile("" : "+v"(lo));   // here, not after the exchange
  }
  mx = ra_all<W>(mx, lds, maxf);
  rr.set(F.fold0, mx);
  for (int k = 0; k < F.n_row0; ++k) rw_row_exec(F, F.row0[k], rr, lane);
  const float m = rr.get(F.m);
  // the row max itself subtracted, and no result below f32's normal range
  // that the output type could hold: the short exponential
  bool plain = m == mx;
  if constexpr (DT == KTIR_BF16) plain = plain && !__any(__fsub_rn(lo, m) < -87.f);
  float e[C][8], part[C];
  auto exps = [&](auto ex) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < C; ++i) {
      float v[8];
      rf_unpack<DT>(c[i], v);
#pragma unroll
      for (int j = 0; j < 8; ++j) e[i][j] = ex(__fsub_rn(v[j], m));
      part[i] = __fadd_rn(__fadd_rn(__fadd_rn(e[i][0], e[i][4]), __fadd_rn(e[i][2], e[i][6])),
                          __fadd_rn(__fadd_rn(e[i][1], e[i][5]), __fadd_rn(e[i][3], e[i][7])));
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if (plain) exps([](float x) { return ra_exp_neg(x); });
  else exps([](float x) { return ra_exp(x); });
  float sum = part[0];
#pragma unroll
  for (int i = 1; i < C; ++i) sum = __fadd_rn(sum, part[i]);
  rr.set(F.fold1, ra_all<W>(sum, lds + 4, [](float a, float b) { return __fadd_rn(a, b); }));
  for (int k = 0; k < F.n_row1; ++k) rw_row_exec(F, F.row1[k], rr, lane);
  const float s = rr.get(F.s);
  const float q = __fdiv_rn(1.f, s), as = fabsf(s);
  auto out = [&](auto div) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < C; ++i) {
      float y[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = div(e[i][j]);
      ra_store<C, 1>(y_row, M, i, ra_pack<DT>(y));
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if (as > 1e-30f && as < 1e30f) {
    out([&](float x) { return div_by(x, s, q); });
  } else {
    // rare: one quotient at a time, so that this branch does not set the register count
    out([&](float x) {
      const float v = __fdiv_rn(x, s);
      __builtin_amdgcn_sched_barrier(0);
      return v;
    });
  }
}

template <int C, int DT, int P, int W, bool KEEP>
__device__ __forceinline__ void ra_norm(const RaPlan& F, gu4 (&c)[C], const gu4 (&w)[KEEP ? C : 1], const RaMap<C, P>& M,
                                        uint64_t y_row, int64_t lane, RowLanes& rr, float* lds) {
  // squares into LDS, the two halves of the row combined first (P = 2)
#pragma unroll
  for (int i = 0; i < M.Q; ++i) {
    float q[8];
    rf_unpack<DT>(c[i], q);
#pragma unroll
    for (int j = 0; j < 8; ++j) q[j] = __fmul_rn(q[j], q[j]);
    if constexpr (P == 2) {
      float u[8];
      rf_unpack<DT>(c[i + M.Q], u);
#pragma unroll
      for (int j = 0; j < 8; ++j) q[j] = __fadd_rn(q[j], __fmul_rn(u[j], u[j]));
    }
    const int k = i == M.Q - 1 ? M.last() : 8;
    float* d = lds + 8 * (M.t + i * M.T);
    if (k >= 8) {
      *(float4*)d = make_float4(q[0], q[1], q[2], q[3]);
      *(float4*)(d + 4) = make_float4(q[4], q[5], q[6], q[7]);
    } else if (P == 1 && k > 0) {
#pragma unroll
      for (int j = 0; j < 7; ++j)
        if (j < k) d[j] = q[j];
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  rr.set(F.fold0, ra_tree<W>(lds, M.part, M.t, M.T));
  for (int k = 0; k < F.n_row0; ++k) rw_row_exec(F, F.row0[k], rr, lane);
  const float s = rr.get(F.s);
  gu4 wn = {0u, 0u, 0u, 0u};
  if (!KEEP && F.has_w) wn = ra_chunk<C, P>(F.w, M, 0);
#pragma unroll
  for (int i = 0; i < C; ++i) {
    float y[8];
    gu4 wi = wn;
    if (!KEEP && F.has_w && i + 1 < C) wn = ra_chunk<C, P>(F.w, M, i + 1);
    rf_unpack<DT>(c[i], y);
    if (F.has_w) {
      float wv[8];
      if constexpr (KEEP) {
        wi = w[i];
      } else if (P == 1 && i == C - 1) {
        const int k = M.last();
        if (k > 0 && k < 8) wi = ra_shift(wi, k);
      }
      rf_unpack<DT>(wi, wv);
      if (F.w_first) {
#pragma unroll
        for (int j = 0; j < 8; ++j) y[j] = mul_keep(__fmul_rn(y[j], wv[j]), s);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) y[j] = mul_keep(__fmul_rn(y[j], s), wv[j]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = mul_keep(y[j], s);
    }
    ra_store<C, P>(y_row, M, i, ra_pack<DT>(y));
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Whether a workgroup holds the weights and has the next row's loads in flight
// while it computes a row.  Those registers pay only where they cost no
// wavefront: rows of one chunk per thread, and the longest norm rows that keep
// all their squares in LDS (two workgroups per CU at most).  Elsewhere more
// wavefronts hide the loads better: rmsnorm 8192 x 5120 40.6 -> 34.7 us, softmax
// 10752 x 3072 21.4 -> 18.2 us (replayed on the same buffers).
constexpr bool ra_keep(int recipe, int C, int P, int W) {
  return C == 1 || (recipe == RF_NORM && W == 4 && P == 1 && C >= 7);
}

// wavefronts per SIMD to fit the registers to: the most that spills nothing
constexpr int ra_waves(int recipe, int C, int P, int W) {
  if (ra_keep(recipe, C, P, W)) return C == 1 ? 5 : 2;
  return C <= 3 ? 6 : (C == 4 ? 5 : (C <= 6 || recipe == RF_NORM ? 4 : 3));
}

template <int RECIPE, int DT, int C, int P, int W>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(ra_waves(RECIPE, C, P, W)))) void prog_rowany(const RaPlan F) {
  extern __shared__ __align__(16) float ra_lds[];
  const RaMap<C, P> M{(int)threadIdx.x, 64 * W, P == 1 ? F.n : F.n / P};
  constexpr uint32_t PAD = RECIPE == RF_SOFTMAX ? (DT == KTIR_BF16 ? 0xff80ff80u : 0xfc00fc00u) : 0u;   // -inf, or 0
  RowLanes rr{0, (int)(threadIdx.x & 63)};
  int r = blockIdx.x;
  constexpr bool KEEP = ra_keep(RECIPE, C, P, W);
  gu4 c[C], w[RECIPE == RF_NORM && KEEP ? C : 1];
  if constexpr (RECIPE == RF_NORM && KEEP)
    if (F.has_w) ra_load<C, P>(F.w, M, w);
  ra_load<C, P>(F.x + 2 * (uint64_t)(r * F.x_step), M, c);
  while (true) {
    const int rn = r + (int)gridDim.x;
    gu4 nx[KEEP ? C : 1];
    if constexpr (KEEP)
      if (rn < F.rows) ra_load<C, P>(F.x + 2 * (uint64_t)(rn * F.x_step), M, nx);
    ra_trim<C, P>(M, c, PAD);
    if constexpr (RECIPE == RF_NORM && P == 1 && KEEP) {
      if (r == (int)blockIdx.x && F.has_w) ra_trim<C, P>(M, w, 0u);
    }
    const uint64_t y_row = F.y + 2 * (uint64_t)(r * F.y_step);
    const int64_t lane = F.rows_per_lane == 1 ? r : r / F.rows_per_lane;
    if constexpr (RECIPE == RF_SOFTMAX) ra_softmax<C, DT, W>(F, c, M, y_row, lane, rr, ra_lds);
    else ra_norm<C, DT, P, W, KEEP>(F, c, w, M, y_row, lane, rr, ra_lds);
    if (rn >= F.rows) break;
    if constexpr (KEEP) {
#pragma unroll
      for (int i = 0; i < C; ++i) c[i] = nx[i];
    } else {
      ra_load<C, P>(F.x + 2 * (uint64_t)(rn * F.x_step), M, c);
    }
    r = rn;
    ra_sync<W>();                              // the next row's folds reuse the LDS
  }
}

int64_t row_grid_limit(int64_t blocks);

// as many workgroups as the device holds at once, each an equal share of the rows
template <int RECIPE, int DT, int C, int P, int W>
static void rowany_go(const RaPlan& F) {
  const int lds = RECIPE == RF_NORM ? 4 * ((F.n / P + 3) & ~3) : 32;
  int per_cu = 0, cus = 0, dev = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, prog_rowany<RECIPE, DT, C, P, W>, 64 * W, lds) != hipSuccess ||
      hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || per_cu < 1 || cus < 1) {
    per_cu = 1;
    cus = 256;
  }
  const int64_t resident = (int64_t)per_cu * cus, per_block = (F.rows + resident - 1) / resident;
  const int64_t blocks = row_grid_limit((F.rows + per_block - 1) / per_block);
  hipLaunchKernelGGL((prog_rowany<RECIPE, DT, C, P, W>), dim3((unsigned)blocks), dim3(64 * W), (size_t)lds, stream(), F);
}

template <int RECIPE, int DT, int C, int W>
static void rowany_p(const RaPlan& F) {
  // both halves whole chunks that a thread's even number of chunks covers
  if constexpr (RECIPE == RF_NORM && C % 2 == 0) {
    if (F.n % 16 == 0) return rowany_go<RECIPE, DT, C, 2, W>(F);
  }
  rowany_go<RECIPE, DT, C, 1, W>(F);
}

// C = the chunks per thread that the row fills to the last: up to six on one
// wavefront (norm rows, which hold no exponentials, up to eight: 8192 x 4000 26
// us, on two wavefronts 31), then two, then four (up to eight each)
template <int RECIPE, int DT>
static void rowany_c(const RaPlan& F) {
  const int q = (F.n + 7) / 8;
  switch ((q + 63) / 64) {
    case 1: return rowany_p<RECIPE, DT, 1, 1>(F);
    case 2: return rowany_p<RECIPE, DT, 2, 1>(F);
    case 3: return rowany_p<RECIPE, DT, 3, 1>(F);
    case 4: return rowany_p<RECIPE, DT, 4, 1>(F);
    case 5: return rowany_p<RECIPE, DT, 5, 1>(F);
    case 6: return rowany_p<RECIPE, DT, 6, 1>(F);
  }
  if constexpr (RECIPE == RF_NORM) {
    switch ((q + 63) / 64) {
      case 7: return rowany_p<RECIPE, DT, 7, 1>(F);
      case 8: return rowany_p<RECIPE, DT, 8, 1>(F);
    }
  }
  if (q <= 6 * 128) {
    switch ((q + 127) / 128) {
      case 4: return rowany_p<RECIPE, DT, 4, 2>(F);
      case 5: return rowany_p<RECIPE, DT, 5, 2>(F);
      default: return rowany_p<RECIPE, DT, 6, 2>(F);
    }
  }
  switch ((q + 255) / 256) {
    case 4: return rowany_p<RECIPE, DT, 4, 4>(F);
    case 5: return rowany_p<RECIPE, DT, 5, 4>(F);
    case 6: return rowany_p<RECIPE, DT, 6, 4>(F);
    case 7: return rowany_p<RECIPE, DT, 7, 4>(F);
    default: return rowany_p<RECIPE, DT, 8, 4>(F);
  }
}

// Row instructions that leave a value as it is: the maximum with the -inf
// that the fold's outs holds, and the sum of a fold of squares or exponentials
// (never -0) with 0.  Their result's readers take the value itself; constants
// that nothing reads any more go too.
static void ra_simplify(RfPlan& F) {
  RfPlan S = F;
  int alias[KTIR_NREG];
  bool known[KTIR_NREG] = {}, sum[KTIR_NREG] = {};
  int32_t imm[KTIR_NREG] = {};
  for (int i = 0; i < KTIR_NREG; ++i) alias[i] = i;
  auto write = [&](int r) {                   // false: a value read under another name would be lost
    for (int i = 0; i < KTIR_NREG; ++i)
      if (i != r && alias[i] == r) return false;
    alias[r] = r;
    known[r] = sum[r] = false;
    return true;
  };
  auto run = [&](ktir_instr_t* x, int n) -> int {
    int kept = 0;
    for (int k = 0; k < n; ++k) {
      ktir_instr_t in = x[k];
      const bool bin = in.op >= KTIR_OP_ADDF;
      if (in.op != KTIR_OP_CONST && in.op != KTIR_OP_LANE) {
        in.a = (int8_t)alias[in.a];
        if (bin || in.op == KTIR_OP_SELECT || in.op == KTIR_OP_FMA || in.op == KTIR_OP_CMPF || in.op == KTIR_OP_CMPI)
          in.b = (int8_t)alias[in.b];
        if (in.op == KTIR_OP_SELECT || in.op == KTIR_OP_FMA) in.c = (int8_t)alias[in.c];
      }
      int same = -1;
      if (bin && in.dt == KTIR_F32 && in.a != in.b) {
        for (int o = 0; o < 2 && same < 0; ++o) {
          const int c = o ? in.a : in.b, v = o ? in.b : in.a;
          if (!known[c] || known[v]) continue;
          if (in.op == KTIR_OP_MAXIMUMF && imm[c] == (int32_t)0xff800000) same = v;
          if (in.op == KTIR_OP_ADDF && imm[c] == 0 && sum[v]) same = v;
        }
      }
      const bool was_sum = same >= 0 && sum[same];
      if (same != in.dst && !write(in.dst)) return -1;
      if (same >= 0) {
        alias[in.dst] = same;
        if (same == in.dst) sum[same] = was_sum;
        continue;
      }
      if (in.op == KTIR_OP_CONST) {
        known[in.dst] = true;
        imm[in.dst] = in.imm;
      }
      x[kept++] = in;
    }
    return kept;
  };
  const bool softmax = S.fold1 >= 0;
  if (!write(S.fold0)) return;
  sum[S.fold0] = !softmax;
  if ((S.n_row0 = run(S.row0, S.n_row0)) < 0) return;
  if (softmax) {
    S.m = (int8_t)alias[S.m];
    if (!write(S.fold1)) return;
    sum[S.fold1] = true;
    if ((S.n_row1 = run(S.row1, S.n_row1)) < 0) return;
  }
  S.s = (int8_t)alias[S.s];
  // constants nothing reads
  auto reads = [](const ktir_instr_t& x, int r) {
    if (x.op == KTIR_OP_CONST || x.op == KTIR_OP_LANE) return false;
    return x.a == r || x.b == r || x.c == r;
  };
  auto drop = [&](ktir_instr_t* x, int n, const ktir_instr_t* after, int n_after, bool m_after) -> int {
    int kept = 0;
    for (int k = 0; k < n; ++k) {
      bool used = x[k].op != KTIR_OP_CONST || x[k].dst == S.s || (m_after && x[k].dst == S.m);
      for (int q = k + 1; q < n && !used; ++q) used = reads(x[q], x[k].dst);
      for (int q = 0; q < n_after && !used; ++q) used = reads(after[q], x[k].dst);
      if (used) x[kept++] = x[k];
    }
    return kept;
  };
  if (softmax) S.n_row1 = drop(S.row1, S.n_row1, nullptr, 0, false);
  S.n_row0 = drop(S.row0, S.n_row0, S.row1, softmax ? S.n_row1 : 0, softmax);
  F = S;
}

// The step between a leaf's rows, or false where they do not lie one step
// apart or leave their allocation.
static bool ra_step(const RfPlan& F, const RwLeaf& L, int64_t rows, int64_t n, int64_t& step) {
  if (L.lane_base) return false;
  step = 0;
  int64_t ext = 1;
  bool first = true;
  for (int d = F.nd - 2; d >= 0; --d) {
    if (F.shape[d] == 1) continue;
    if (first) step = L.strides[d];
    else if (L.strides[d] != step * ext) return false;
    first = false;
    ext *= F.shape[d];
  }
  if (rows > ext) {
    if (first) step = L.lane_stride;
    else if (L.lane_stride != step * ext) return false;
  }
  const int64_t last = L.base + (rows - 1) * step;
  return (step < 0 ? last : L.base) >= L.lo && (step < 0 ? L.base : last) + n <= L.hi;
}

// True when launched: the f32-math forms, rows of at least one chunk that lie
// one step apart inside their allocations.
bool launch_rowany(const RfPlan& plan, int recipe, int dt, int64_t rows, int64_t n) {
  static_assert(KTIR_MAX_ROW <= 8 * 8 * 256, "the longest row fits four wavefronts");
  if ((recipe != RF_SOFTMAX && recipe != RF_NORM) || n < 8 || n > KTIR_MAX_ROW || rows > (1 << 30)) return false;
  RfPlan F = plan;
  RaPlan R{};
  int64_t w_step = 0;
  if (!ra_step(F, F.x, rows, n, R.x_step) || !ra_step(F, F.y, rows, n, R.y_step) ||
      (F.has_w && (!ra_step(F, F.w, rows, n, w_step) || w_step != 0)))
    return false;
  if (recipe != RF_SOFTMAX) {
    F.fold1 = -1;
    F.n_row1 = 0;
  }
  ra_simplify(F);
  R.x = F.x.ptr + 2 * F.x.base;
  R.y = F.y.ptr + 2 * F.y.base;
  R.w = F.w.ptr + 2 * F.w.base;
  R.lane_scalars = F.lane_scalars;
  R.n_lane_scalars = F.n_lane_scalars;
  R.n = (int32_t)n;
  R.rows = (int32_t)rows;
  R.rows_per_lane = 1;
  for (int d = 0; d < F.nd - 1; ++d) R.rows_per_lane *= (int32_t)F.shape[d];
  R.has_w = F.has_w;
  R.w_first = F.w_first;
  R.n_row0 = F.n_row0;
  R.n_row1 = F.n_row1;
  R.fold0 = F.fold0;
  R.fold1 = F.fold1;
  R.m = F.m;
  R.s = F.s;
  for (int k = 0; k < RF_MAX_ROW; ++k) {
    R.row0[k] = F.row0[k];
    R.row1[k] = F.row1[k];
  }
  if (recipe == RF_SOFTMAX) {
    if (dt == KTIR_F16) rowany_c<RF_SOFTMAX, KTIR_F16>(R);
    else rowany_c<RF_SOFTMAX, KTIR_BF16>(R);
  } else {
    if (dt == KTIR_F16) rowany_c<RF_NORM, KTIR_F16>(R);
    else rowany_c<RF_NORM, KTIR_BF16>(R);
  }
  return true;
}

}  // namespace ktir
