// Fused online-softmax attention loop for tiles of 64 or 128 rows and keys
// and heads of 64 or 128 columns (other than 128 x 128 x 128, which
// ktir_attn.hip runs): the KV loop of the reference's attention kernels
// (notebooks/demo_gen_mlir.py:471-567, examples/triton-ktir/paged_attention.mlir:191-396)
// as one launch.
//
// A workgroup is four wavefronts of 32 query rows each: one lane (simulated
// core) of 128 rows, or two lanes of 64 rows that read one K/V stream (the
// host pairs them).  Per KV tile of N keys, as in ktir_attn.hip:
//   S^T = K Q^T     A = K rows from LDS, B = Q^T in registers, so a query row's
//                   scores lie in lanes l and l ^ 32;
//   softmax         row max and sum in the lane and one exchange, P, l and O kept
//                   relative to a base 2^b that moves when e^m passes it by e^P_LAG;
//   O^T += V^T P^T  V^T by transposing LDS reads, the keys in the order in which
//                   a lane's own scores are its P fragment.
// P, f32 in the op-by-op loop, enters P V as three bf16 terms (24 bits) or, in
// f16, as two terms (23 bits) and, in a step with a P below 2^-15, the rest
// of them too (ktir_attn_common.h): results from float64 by no more than one
// rounding of their type and f32's of the exponentials, as the loop's are.
// P = 2^(S log2 e - b) rounds once, for scores far from 0 too, as 2^b is the base
// itself.  Beyond 2^19 the rounding of b would pass 1, so b ends at -2^20 below (the
// P of a row that a mask of -1e9 or of the type's lowest value has filled so far are
// 0, as any later score makes them), and a workgroup with a row that ends up out there,
// or with a NaN in its result, runs its loop again in the general form: e^(S - mr)
// with a base mr, and V's infinities kept from the later terms of P.
//
// K and V tiles are double-buffered in LDS: tile j + 1 streams in (buffer_load
// ... lds, no registers) while tile j is computed, one barrier per tile.  A
// 64 x 64 x 64 step stages 16 KB for 24 MFMAs and about 300 vector
// instructions per wavefront and takes 32 KB of LDS, so several workgroups
// share a CU and one's softmax runs under another's MFMAs.  The vector
// instructions bound it (the split of P takes as many as the exponentials, the
// test for small P 3 to 4 % of the time).  Where no CU has a second workgroup,
// the key tiles go to two groups of four wavefronts, whose states meet in LDS at
// the end.  Full attention of 2048 x 64, f16, 64 x 64 tiles: 16 heads 37 us
// (465 TFLOP/s; 34 us, and 40 with one group, while f16 lost small P), and 43.4 ms
// for the loop's about 450 launches; 32 heads (two workgroups per CU) 68 us.
#include <type_traits>

#include "ktir_attn_common.h"

namespace ktir {

// Wavefront w (uniform, 0..3) copies rows N/4 w .. + N/4 of an N x D tile into
// LDS in 1 KB blocks of 512 / D rows: lane l fills slot l % (D / 8) of its row.
template <int N, int D>
__device__ __forceinline__ void att_stage(const uint16_t* src, int64_t row_stride, uint16_t* lds, int w, int l) {
  constexpr int CH = D / 8, RB = 512 / D, RW = N / 4;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(src + (int64_t)(RW * w) * row_stride), (short)0, (int)(((RW - 1) * row_stride + D) * 2), 0x00020000);
  const int r = l / CH, c = l % CH;
#pragma unroll
  for (int i = 0; i < RW / RB; ++i) {
    // a wavefront's rows start at a multiple of 16, so row % 16 is known here
    const int x = c ^ kv_swz<D>((RB * i + r) & 15);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(lds + D * (RW * w + RB * i)),
                                             16, (int)((r * row_stride + 8 * x) * 2), (int)(i * RB * row_stride * 2), 0, 0);
  }
}

// the lowest b, and whether a final row maximum asks for the general form
constexpr float AT_LOW = -0x1p20f;
__device__ __forceinline__ bool at_far(float m) { return fabsf(m) > 0x1p19f && fabsf(m) < __builtin_inff(); }

// The position mask keeps score (row, key) iff ((lo <= kpos - qpos <= hi) != inv).
// G groups of four wavefronts take every G-th key tile of the same lanes, each
// with tile buffers of its own.  Two wavefronts per SIMD, also where 256
// registers spill up to 17: one, with 512, takes 156 us for 122 (32 heads of 2048
// x 128, tiles of 64) and 55 for 43 (64 heads of 1024 x 64, tiles of 128); three,
// in 64 x 64 x 64 tiles, as long as two (77 us, 32 heads of 2048 x 64).
template <bool BF16, int M, int N, int D, int G>
__global__ __launch_bounds__(256 * G, 2) void attn_tile(const ktir_attn_t d, int mlo, int mhi, int minv) {
  constexpr int KT = N / 32, DS = D / 16, DT = D / 32, PARTS = BF16 ? 3 : 2;
  __shared__ __align__(16) uint16_t K0a[G][N * D];  // K tiles of a group's even / odd steps
  __shared__ __align__(16) uint16_t K1a[G][N * D];
  __shared__ __align__(16) uint16_t V0a[G][N * D];  // V tiles of a group's even / odd steps
  __shared__ __align__(16) uint16_t V1a[G][N * D];
  const int tid = threadIdx.x & 255, l = tid & 63, h = l >> 5, r32 = l & 31;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = G == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8);
  uint16_t *K0s = K0a[grp], *K1s = K1a[grp], *V0s = V0a[grp], *V1s = V1a[grp];
  const int32_t* trips = (const int32_t*)d.trips;
  // the workgroup's lanes: wavefronts 0, 1 run la, wavefronts 2, 3 lb
  int la, lb;
  if (M == 64 && d.pairs) {
    la = uni(((const int32_t*)d.pairs)[2 * blockIdx.x]);
    lb = uni(((const int32_t*)d.pairs)[2 * blockIdx.x + 1]);
  } else {
    la = uni(d.order ? ((const int32_t*)d.order)[blockIdx.x] : (int)blockIdx.x);
    lb = M == 64 ? -1 : la;
  }
  const int ta = la >= 0 ? uni(trips[la]) : 0, tb = lb >= 0 ? uni(trips[lb]) : 0;
  const int lane = w >> 1 ? lb : la, T = w >> 1 ? tb : ta, Tmax = ta > tb ? ta : tb;
  const int lk = la >= 0 ? la : lb;                 // whose K/V stream (both share it)
  if (lk < 0) return;
  const uint16_t* K = (const uint16_t*)d.k_ptr + uni(((const int64_t*)d.k_base)[lk]);
  const uint16_t* V = (const uint16_t*)d.v_ptr + uni(((const int64_t*)d.v_base)[lk]);
  const int row = (M == 64 ? (w & 1) : w) * 32 + r32;   // query row inside the lane's tile
  uint4 qf[DS];                                     // Q^T fragments: Q[row][16 s + 8 h .. + 8]
  int64_t qpos = 0;
  if (T > 0) {
    const uint16_t* qr = (const uint16_t*)d.q_ptr + uni(((const int64_t*)d.q_base)[lane]) + (int64_t)row * d.q_row + 8 * h;
#pragma unroll
    for (int s = 0; s < DS; ++s) qf[s] = *(const uint4*)(qr + 16 * s);
    qpos = uni(((const int64_t*)d.qpos0)[lane]) + row;
  }
  const int64_t kpos00 = uni(((const int64_t*)d.kpos0)[lk]);
  const bool pos_scale = d.scale > 0.f;
  const float c1 = __fmul_rn(d.scale, LOG2E);
  const f32x16_t z16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  f32x16_t o[DT];                                   // O^T tiles: d = 32 dt + 8 g + 4 h + t, row r32
  float m, b, lsum;                                 // b: the base's exponent (general form: mr)
  const int k_off = r32 * D, k_x = kv_swz<D>(r32 & 15);
  // V^T fragment: member tj of 16-lane group tg addresses key 4 (tg / 2) + tj / 4
  // (+ 8) of the 16-key step, columns 16 (tg % 2) + 4 (tj % 4) of a 32-column tile
  const int tg = l >> 4, tj = l & 15;
  const int v_row0 = 4 * (tg >> 1) + (tj >> 2);
  const int v_c = 2 * (tg & 1) + ((tj >> 1) & 1), v_in = 4 * (tj & 1);
  const int v_b0 = v_row0 * D + v_in, v_x0 = v_c ^ kv_swz<D>(v_row0), v_x1 = v_c ^ kv_swz<D>(v_row0 + 8);

  // GEN: the general form
  auto step = [&](auto gen, int j, const uint16_t* Kc, const uint16_t* Vc, uint16_t* Kn,
                  uint16_t* Vn) __attribute__((always_inline)) {
    constexpr bool GEN = decltype(gen)::value;
    if (j + G < Tmax) {
      att_stage<N, D>(K + (int64_t)(j + G) * d.k_step, d.k_row, Kn, w, l);
      att_stage<N, D>(V + (int64_t)(j + G) * d.v_step, d.v_row, Vn, w, l);
    }
    if (j < T) {
      f32x16_t sc[KT];
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) sc[kt] = z16;
#pragma unroll
      for (int s = 0; s < DS; ++s) {
        const uint16_t* kp = &Kc[k_off + 8 * ((2 * s + h) ^ k_x)];
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) sc[kt] = mfma_at<BF16>(*(const uint4*)(kp + kt * 32 * D), qf[s], sc[kt]);
      }
      // lane value (kt, i) is key kt * 32 + 8 (i / 4) + 4 h + i % 4 of row `row`
      const int dbase = (int)(kpos00 + (int64_t)j * d.kpos_step - qpos);
      const bool all_keep = !d.causal ||
          (minv ? (dbase + N - 1 < mlo || dbase > mhi) : (dbase >= mlo && dbase + N - 1 <= mhi));
      // no masked score in the wavefront and scale > 0: row max of S = scale *
      // row max of Q K^T, and P = 2^(QK scale log2e - b)
      const bool fast = pos_scale && __all(all_keep);
      if (!fast) {
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            float s = __fmul_rn(d.scale, sc[kt][i]);
            if (d.causal) {
              const int df = dbase + kt * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
              if ((df >= mlo && df <= mhi) == (bool)minv) s = d.neg;
            }
            sc[kt][i] = s;
          }
      }
      float x[KT];
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        x[kt] = sc[kt][0];
#pragma unroll
        for (int i = 1; i < 15; i += 2) x[kt] = fmax3_nan(x[kt], sc[kt][i], sc[kt][i + 1]);
        x[kt] = fmax_nan(x[kt], sc[kt][15]);
      }
      float xm = x[0];
#pragma unroll
      for (int kt = 1; kt < KT; ++kt) xm = fmax_nan(xm, x[kt]);
      xm = pair_max(xm);
      const float mn = fmax_nan(m, fast ? __fmul_rn(d.scale, xm) : xm);
      // -inf (tile 0 masked whole) stays: P is then the loop's NaN
      const float bn = GEN ? mn : fmax_nan(__fmul_rn(mn, LOG2E), mn == -__builtin_inff() ? mn : AT_LOW);
      const bool up = bn > __fadd_rn(b, GEN ? P_LAG<BF16> : P_LAG<BF16> * LOG2E);
      if (__any(up)) {
        const float db = __fsub_rn(b, bn), al = up ? (GEN ? exp_f(db) : __builtin_amdgcn_exp2f(db)) : 1.f;
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[t][i] = __fmul_rn(o[t][i], al);
        lsum = __fmul_rn(lsum, al);
        b = up ? bn : b;
      }
      // a group without tile 0 whose scores have all been -inf: P is 0 against
      // any base (with tile 0 it is the loop's exp(-inf - (-inf)), NaN)
      const float pb = G > 1 && grp && mn == -__builtin_inff() ? 0.f : b;
      if constexpr (GEN) {
        const float to_s = fast ? d.scale : 1.f;
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
          for (int i = 0; i < 16; ++i) sc[kt][i] = exp_f(__builtin_fmaf(sc[kt][i], to_s, -pb));
      } else {
        const float to_2 = fast ? c1 : LOG2E;
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
          for (int i = 0; i < 16; ++i) sc[kt][i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[kt][i], to_2, -pb));
      }
      // whether a P of this tile is too small for two f16 terms
      bool small = false;
      if constexpr (!BF16 && !GEN) {
        float least = 1.f;
        if (fast) {
#pragma unroll
          for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int i = 0; i < 16; i += 2)
              least = fmin3_nan(least, sc[kt][i], sc[kt][i + 1]);
        } else {
#pragma unroll
          for (int kt = 0; kt < KT; ++kt) {
            float p[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) p[i] = sc[kt][i];
            least = fminf(least, least_positive<16>(p));
          }
        }
        small = __any(least < P_SMALL);
      }
      float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int i = 0; i < 16; i += 4) {
          a0 = __fadd_rn(a0, sc[kt][i]);
          a1 = __fadd_rn(a1, sc[kt][i + 1]);
          a2 = __fadd_rn(a2, sc[kt][i + 2]);
          a3 = __fadd_rn(a3, sc[kt][i + 3]);
        }
      lsum = __fadd_rn(lsum, pair_sum(__fadd_rn(__fadd_rn(a0, a1), __fadd_rn(a2, a3))));
      m = mn;
      // P V: by the terms of the operand type, by the rest they leave (f16) or by
      // bf16 terms of the whole P (f16, general form)
      enum { TERMS, REST, WHOLE };
      auto pv = [&](auto how) __attribute__((always_inline)) {
        constexpr int HOW = decltype(how)::value;
#pragma unroll
        for (int ks = 0; ks < N / 16; ++ks) {
          const int kt = ks >> 1, g0 = 2 * (ks & 1);
          const uint16_t* vt = &Vc[16 * ks * D];
          float p[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            p[i] = sc[kt][4 * g0 + i];
            if constexpr (HOW == REST) asm volatile("" : "+v"(p[i]));   // nothing kept for it from the terms
            if constexpr (HOW == WHOLE) p[i] = __fmul_rn(p[i], P_SCALE<BF16>);
          }
          uint32_t t0[PARTS][2], t1[PARTS][2];
          uint4 tb[3];
          if constexpr (HOW != WHOLE) {
            p_split<BF16, PARTS, HOW == REST>(p, t0);
            p_split<BF16, PARTS, HOW == REST>(p + 4, t1);
          }
          if constexpr (HOW != TERMS) p_split_bf(p, tb);
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            const uint2 lo = ds_tr16(vt + v_b0 + 8 * ((4 * dt) ^ v_x0));
            const uint2 hi = ds_tr16(vt + v_b0 + 8 * D + 8 * ((4 * dt) ^ v_x1));
            const uint4 a = make_uint4(lo.x, lo.y, hi.x, hi.y);
            if constexpr (HOW == TERMS) {
              o[dt] = pv_mfma<BF16, PARTS, GEN>(a, t0, t1, o[dt]);
            } else {
              o[dt] = pv_mfma_bf<GEN>(a, tb, o[dt]);
              __builtin_amdgcn_sched_barrier(0);   // rare: must not set the register count
            }
          }
        }
      };
      if constexpr (!BF16 && GEN) {
        pv(std::integral_constant<int, WHOLE>{});
      } else {
        pv(std::integral_constant<int, TERMS>{});
        if (small) pv(std::integral_constant<int, REST>{});
      }
    }
    __builtin_amdgcn_s_waitcnt(0);                  // this wavefront's part of the next tile has landed
    __syncthreads();                                // every wavefront: done with tile j, the next one whole
  };
  auto loop = [&](auto gen) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < DT; ++t) o[t] = z16;
    m = b = -__builtin_inff();
    lsum = 0.f;
    if (grp < Tmax) {
      att_stage<N, D>(K + (int64_t)grp * d.k_step, d.k_row, K0s, w, l);
      att_stage<N, D>(V + (int64_t)grp * d.v_step, d.v_row, V0s, w, l);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    // as many steps in every group (one past the end computes nothing)
    for (int j = 0; j < Tmax; j += 2 * G) {
      step(gen, j + grp, K0s, V0s, K1s, V1s);
      if (j + G < Tmax) step(gen, j + G + grp, K1s, V1s, K0s, V0s);
    }
  };
  loop(std::false_type{});
  // An infinite V times the terms of P after the first (0, or of the other
  // sign) is NaN where P V is infinite, so a NaN anywhere in the workgroup's
  // result asks for the general form too.
  bool again = at_far(m);
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) again |= o[t][i] != o[t][i];
  const bool gen = __syncthreads_or(again);
  if (gen) loop(std::true_type{});
  // what brings l and O to e^m
  float fin = gen ? exp_f(__fsub_rn(b, m)) : __builtin_amdgcn_exp2f(__builtin_fmaf(-m, LOG2E, b));
  if constexpr (G == 2) {
    // group 1's state, through the tiles (read by now: the barrier above), to
    // the thread of group 0 with the same row and columns
    constexpr int ROWS = G * N * D * 2 / 4096;      // 256 x 16 bytes
    static_assert(4 * DT <= 2 * ROWS && ROWS >= 1, "state exchange");
    auto ex = [&](int k) -> float4* { return (float4*)(k < ROWS ? K0a[0] : K1a[0]) + (k < ROWS ? k : k - ROWS) * 256 + tid; };
    float* exs = (float*)V0a[0] + tid;
    if (grp == 1) {
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *ex(4 * t + g) = make_float4(o[t][4 * g], o[t][4 * g + 1], o[t][4 * g + 2], o[t][4 * g + 3]);
      exs[0] = m;
      exs[256] = fin;
      exs[512] = lsum;
    }
    __syncthreads();
    if (grp == 1) return;
    if (T > 0) {
      const float m1 = exs[0], mm = fmax_nan(m, m1);
      const float w0 = __fmul_rn(fin, exp_f(__fsub_rn(m, mm)));
      const float w1 = m1 == -__builtin_inff() ? 0.f : __fmul_rn(exs[256], exp_f(__fsub_rn(m1, mm)));
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const float4 x = *ex(4 * t + g);
          o[t][4 * g] = __fadd_rn(__fmul_rn(o[t][4 * g], w0), __fmul_rn(x.x, w1));
          o[t][4 * g + 1] = __fadd_rn(__fmul_rn(o[t][4 * g + 1], w0), __fmul_rn(x.y, w1));
          o[t][4 * g + 2] = __fadd_rn(__fmul_rn(o[t][4 * g + 2], w0), __fmul_rn(x.z, w1));
          o[t][4 * g + 3] = __fadd_rn(__fmul_rn(o[t][4 * g + 3], w0), __fmul_rn(x.w, w1));
        }
      lsum = __fadd_rn(__fmul_rn(lsum, w0), __fmul_rn(exs[512], w1));
      m = mm;
      fin = 1.f;
    }
  }
  if (lane < 0) return;
  if (T > 0) {
    // l and O to e^m, and O from P's scale
    if (!BF16 || !__all(fin == 1.f)) {
      const float f = __fmul_rn(fin, 1.f / P_SCALE<BF16>);
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[t][i] = __fmul_rn(o[t][i], f);
      lsum = __fmul_rn(lsum, fin);
    }
  }
  if (h == 0) {
    ((float*)d.m_out)[(int64_t)lane * M + row] = m;
    ((float*)d.l_out)[(int64_t)lane * M + row] = lsum;
  }
  if (d.acc_out) {
    float* orow = (float*)d.acc_out + ((int64_t)lane * M + row) * D + 4 * h;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *(float4*)(orow + 32 * t + 8 * g) = make_float4(o[t][4 * g], o[t][4 * g + 1], o[t][4 * g + 2], o[t][4 * g + 3]);
  }
  if (d.o_ptr) {
    // O = acc / l (f32, correctly rounded), then rounded to the output type
    const int64_t ob = uni(((const int64_t*)d.o_base)[lane]) + (int64_t)row * d.o_row + 4 * h;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float q0 = __fdiv_rn(o[t][4 * g], lsum), q1 = __fdiv_rn(o[t][4 * g + 1], lsum);
        const float q2 = __fdiv_rn(o[t][4 * g + 2], lsum), q3 = __fdiv_rn(o[t][4 * g + 3], lsum);
        const int64_t e = ob + 32 * t + 8 * g;
        if (d.o_dtype == KTIR_F32)
          *(float4*)((float*)d.o_ptr + e) = make_float4(q0, q1, q2, q3);
        else if (d.o_dtype == KTIR_BF16)
          *(uint2*)((uint16_t*)d.o_ptr + e) = make_uint2(cvt2<true>(q0, q1), cvt2<true>(q2, q3));
        else
          *(uint2*)((uint16_t*)d.o_ptr + e) = make_uint2(cvt2<false>(q0, q1), cvt2<false>(q2, q3));
      }
  }
}

bool attn_tile_shape(int64_t M, int64_t N, int64_t D) {
  return (M == 64 || M == 128) && (N == 64 || N == 128) && (D == 64 || D == 128) && !(M == 128 && N == 128 && D == 128);
}

// `lo`, `hi`, `inv`: the mask predicate as a range test on kpos - qpos
void launch_attn_tile(const ktir_attn_t& d, int lo, int hi, int inv) {
  const bool paired = d.M == 64 && d.pairs && d.n_pairs > 0;
  const dim3 grid((unsigned)(paired ? d.n_pairs : d.lanes));
  ktir_attn_t a = d;
  if (!paired) a.pairs = 0;
  const std::integral_constant<int, 64> c64;
  const std::integral_constant<int, 128> c128;
  // Two groups where every workgroup has a CU of its own (and the tiles fit): a
  // second wavefront per SIMD runs its softmax under the first one's MFMAs.  With
  // more workgroups those that share a CU do that, and the exchange costs.
  int cus = 0, dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    cus = 0;
  const bool two = (int)grid.x <= cus;
  auto go = [&](auto cm, auto cn, auto cd) {
    constexpr int M = decltype(cm)::value, N = decltype(cn)::value, D = decltype(cd)::value;
    auto run = [&](auto kern, int groups) {
      hipLaunchKernelGGL(kern, grid, dim3(256 * groups), 0, stream(), a, lo, hi, inv);
    };
    const bool bf = d.dtype == KTIR_BF16;
    if constexpr (N * D <= 64 * 128)
      if (two) return bf ? run(attn_tile<true, M, N, D, 2>, 2) : run(attn_tile<false, M, N, D, 2>, 2);
    bf ? run(attn_tile<true, M, N, D, 1>, 1) : run(attn_tile<false, M, N, D, 1>, 1);
  };
  switch ((d.M == 128) * 4 + (d.N == 128) * 2 + (d.D == 128)) {
    case 0: go(c64, c64, c64); break;
    case 1: go(c64, c64, c128); break;
    case 2: go(c64, c128, c64); break;
    case 3: go(c64, c128, c128); break;
    case 4: go(c128, c64, c64); break;
    case 5: go(c128, c64, c128); break;
    default: go(c128, c128, c64); break;
  }
}

}  // namespace ktir
