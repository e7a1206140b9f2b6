// Paged attention (the loop that ktir_pattn.hip describes: the KV loop of
// examples/triton-ktir/paged_attention.mlir:194-392) for lanes that read one
// sequence of pages: query rows gathered over lanes, keys split over
// wavefronts and workgroups.
//
// A lane has few rows (block_q tokens x the query heads of one KV head), and
// every lane of a KV head reads the same pages.  The host groups lanes with
// equal K and V offsets, table position, trip count and key positions into
// items of at most 32 rows.  A workgroup is W = 4 or 8 wavefronts on one item, each
// with the item's 32 rows and its own pages: pairs of pages (32 keys) k, k + W S,
// k + 2 W S, ... of the S workgroups that share the item.  So the wavefronts share
// nothing until the end, run without barriers, and a single query row of a
// decode step keeps the whole chip busy.  Per pair, as in ktir_attn_tile.hip:
//   S^T = K Q^T (32 x 32 x 16 MFMA), masked and scaled in f32,
//   m, l and O of the wavefront's keys (online softmax, O relative to mr <= m),
//   O^T += V^T P^T.
// P enters P V as PARTS terms of the operand type: one f16 / two bf16 terms for
// lanes of at most 16 rows (as the one-wavefront kernel), one more for others,
// whose f32 kernel holds P exactly: 24 bits in bf16, 23 in f16, and the rest of
// them too in a step with a P below 2^-15 (ktir_attn_common.h; the test for it
// takes 2 % of 256 tokens of 32 rows a lane after 1024, 40 us).
// Pages move HBM -> LDS (buffer_load ... lds) into the wavefront's own 16 KB
// (128 columns): the next pair's K while this pair's softmax and P V run, its V
// while the next scores are computed; two workgroups of four (or one of eight) share a CU.
// At the end the W states are merged through LDS; with S > 1 the merged
// state goes to a workspace and a second kernel merges the S of them.  A merge
// weighs each state by exp(m_i - m), 0 for keys that were all masked.
//
// Bound: latency.  A token after 8191 with 8 KV heads of 128 f16 columns reads 34 MB
// (6 us at a large copy's rate) in 11.6 us, of which about 4 are the chain item ->
// table -> first page, and 5.4 us go to the merge: 18.0 us in all, 343 us on one
// wavefront per lane; 256 tokens after 1024: 23.7 us with the copy of Q, 58.5 us.
//
// The loop's step is a page, so a row whose first page is masked whole is NaN
// (exp(-inf - (-inf))) whatever follows; the wavefront that has page 0 makes it so.
#include <climits>
#include <type_traits>

#include "ktir_attn_common.h"

namespace ktir {

constexpr int PS_ROWS = 32, PS_KEYS = 32;

__device__ __forceinline__ int64_t ps_index(uint64_t ptr, int64_t e, int dt) {
  switch (dt) {
    case KTIR_I64: return ((const KTIR_G(int64_t)*)ptr)[e];
    case KTIR_I16: return ((const KTIR_G(int16_t)*)ptr)[e];
    case KTIR_I8: return ((const KTIR_G(int8_t)*)ptr)[e];
  }
  return ((const KTIR_G(int32_t)*)ptr)[e];
}

// whether the page whose K or V tile starts at element e0 lies 16-byte
// aligned inside its window
template <int D>
__device__ __forceinline__ bool ps_fast(int64_t e0, int64_t row, int64_t lo, int64_t hi) {
  return !(e0 & 7) && e0 >= lo && e0 + 15 * row + D <= hi;
}

// N loads of 1 KB into successive KB of LDS in one asm statement (no result
// registers) that ps_wait alone waits for: the compiler, which does not tell the
// two buffers of a wavefront apart in a loop, would wait for both wherever one is
// read.  The hazards inside are not the compiler's either: a vector instruction
// (readfirstlane, a reload of a spilled register) may have written the
// descriptor just before, which a load may read five wait states later (M0 to
// the first load: move and s_nop 4), and M0, which holds the LDS address, is
// what it was afterwards.
template <int N>
__device__ __forceinline__ void ps_load(u32x4_t rsrc, const uint32_t (&off)[N], uint32_t lds) {
  static_assert(N == 2 || N == 4, "16 rows of 64 or 128 columns");
  uint32_t m0;
  if constexpr (N == 4)
    asm volatile(
        "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %6\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %5, 0 offen lds\n\t"
        "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %5, 0 offen lds\n\t"
        "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tbuffer_load_dwordx4 %3, %5, 0 offen lds\n\t"
        "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tbuffer_load_dwordx4 %4, %5, 0 offen lds\n\t"
        "s_mov_b32 m0, %0\n\ts_nop 0"
        : "=&s"(m0)
        : "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(rsrc), "s"(lds)
        : "memory", "scc");
  else
    asm volatile(
        "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %4\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %3, 0 offen lds\n\t"
        "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, 0 offen lds\n\t"
        "s_mov_b32 m0, %0\n\ts_nop 0"
        : "=&s"(m0)
        : "v"(off[0]), "v"(off[1]), "s"(rsrc), "s"(lds)
        : "memory", "scc");
}

// until at most N of this wavefront's loads are in flight; no memory access
// moves across
template <int N>
__device__ __forceinline__ void ps_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// 16 keys x D columns of such a page into LDS rows row0 .. + 16; zeros (loads
// past the end of a buffer of no bytes) if it is not `there`
template <int D>
__device__ __forceinline__ void ps_dma(uint64_t ptr, int64_t e0, int64_t row, bool there, uint32_t lds, int row0, int l) {
  constexpr int CH = D / 8, RB = 512 / D;      // chunks per row, rows per 1 KB
  const uint64_t a = ptr + 2 * (uint64_t)e0;
  const u32x4_t rs = {(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)a),
                      (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(a >> 32) & 0xffffu),
                      (uint32_t)__builtin_amdgcn_readfirstlane(there ? (uint32_t)((15 * row + D) * 2) : 0u), 0x00020000u};
  const int r = l / CH, c = l % CH;
  uint32_t off[16 / RB];
#pragma unroll
  for (int i = 0; i < 16 / RB; ++i) off[i] = (uint32_t)(((RB * i + r) * row + 8 * (c ^ kv_swz<D>((RB * i + r) & 15))) * 2);
  ps_load<16 / RB>(rs, off, lds + 2 * D * row0);
}

// the same of any page: zeros outside [lo, hi)
template <int D>
__device__ __forceinline__ void ps_copy(uint64_t ptr, int64_t e0, int64_t row, int64_t lo, int64_t hi, uint16_t* lds, int row0,
                                        int l) {
  const KTIR_G(uint16_t)* p = (const KTIR_G(uint16_t)*)ptr;
  for (int i = l; i < 16 * D; i += 64) {
    const int r = i / D, c = i % D;
    const int64_t e = e0 + r * row + c;
    lds[D * (row0 + r) + 8 * ((c >> 3) ^ kv_swz<D>(r)) + (c & 7)] = (e >= lo && e < hi) ? p[e] : (uint16_t)0;
  }
}

// the weight of a state with maximum mi in one with maximum m >= mi
__device__ __forceinline__ float ps_weight(float mi, float m) { return mi == -__builtin_inff() ? 0.f : exp_f(__fsub_rn(mi, m)); }

// where row `row` of an item goes (read before the work that ps_out waits for)
struct PsDst {
  int64_t lane, out;
  int r, trips;
  bool live;
};

__device__ __forceinline__ PsDst ps_dst(const ktir_pattn_t& d, const int32_t* lanes, int nl, int row) {
  const int M = (int)d.M, li = row / M;
  PsDst t;
  t.r = row - li * M;
  t.live = li < nl;
  t.lane = lanes[t.live ? li : 0];
  t.trips = ((const int32_t*)d.trips)[t.lane];
  t.out = d.out_ptr ? ((const int64_t*)d.out_base)[t.lane] + (int64_t)(t.r / d.out_grp) * d.out_gstride +
                          (int64_t)(t.r % d.out_grp) * d.out_row
                    : 0;
  return t;
}

// columns 16 q .. + 16 of such a row: acc (relative to m), l and m
// into the launch's outputs, and acc / l into the fused store
template <int D>
__device__ __forceinline__ void ps_out(const ktir_pattn_t& d, const PsDst& t, int q, const float (&acc)[16], float l, float m) {
  if (!t.live) return;
  const int64_t row = t.lane * d.M + t.r;
  if (t.trips > 0) l = __fadd_rn(l, __fmul_rn(d.l0, ps_weight(d.m0, m)));
  else l = d.l0, m = d.m0;
  if (q == 0) {
    ((float*)d.m_out)[row] = m;
    ((float*)d.l_out)[row] = l;
  }
  if (d.acc_out) {
    float4* a = (float4*)((float*)d.acc_out + row * D + 16 * q);
#pragma unroll
    for (int k = 0; k < 4; ++k) a[k] = make_float4(acc[4 * k], acc[4 * k + 1], acc[4 * k + 2], acc[4 * k + 3]);
  }
  if (!d.out_ptr) return;
  // the loop's finalisation: acc / l rounded to the output's dtype
  const int64_t e0 = t.out + 16 * q;
  float v[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) v[k] = __fdiv_rn(acc[k], l);
  if (d.out_dtype != KTIR_F32 && !(d.out_ptr & 15) && !(e0 & 7) && e0 >= d.out_lo && e0 + 16 <= d.out_hi) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      uint32_t w[4];
#pragma unroll
      for (int p = 0; p < 4; ++p)
        w[p] = d.out_dtype == KTIR_BF16 ? cvt2<true>(v[8 * k + 2 * p], v[8 * k + 2 * p + 1])
                                        : cvt2<false>(v[8 * k + 2 * p], v[8 * k + 2 * p + 1]);
      *(KTIR_G(u32x4_t)*)((KTIR_G(uint16_t)*)d.out_ptr + e0 + 8 * k) = u32x4_t{w[0], w[1], w[2], w[3]};
    }
    return;
  }
#pragma unroll
  for (int k = 0; k < 16; ++k)
    if (e0 + k >= d.out_lo && e0 + k < d.out_hi) store_elem(d.out_ptr, e0 + k, d.out_dtype, v[k]);
}

// one item, as the host lays it out
struct __attribute__((packed, aligned(64))) PsItem {
  int32_t first, count;                        // its lanes: item_lanes[first ..]
  int64_t trips, k_base, v_base, tbl_pos, kpos0;
};

template <bool BF16, int D, int PARTS, int W>
__global__ __launch_bounds__(64 * W, 2) void pattn_split(const ktir_pattn_t d, int vec, int* err) {
  constexpr int DS = D / 16, DT = D / 32;
  // per wavefront K then V, 32 keys x D each; at the end its O^T
  __shared__ __align__(16) uint16_t Ks[W][PS_KEYS * D];
  __shared__ __align__(16) uint16_t Vs[W][PS_KEYS * D];
  __shared__ float ms[W][PS_ROWS], ls[W][PS_ROWS];
  const int tid = threadIdx.x, l = tid & 63, h = l >> 5, r32 = l & 31;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int S = d.splits;
  const int item = blockIdx.x / S, part = blockIdx.x - item * S;
  const PsItem* it = (const PsItem*)d.items + item;
  const int first = uni(it->first), nl = uni(it->count), trips = uni((int)it->trips);
  const int64_t kb = uni(it->k_base), vb = uni(it->v_base), tp = uni(it->tbl_pos), kp0 = uni(it->kpos0);
  const int32_t* lanes = (const int32_t*)d.item_lanes + first;
  uint16_t* K = Ks[w];
  uint16_t* V = Vs[w];
  const uint32_t k_lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t*)K);
  const uint32_t v_lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t*)V);
  // this lane's query row
  const int M = (int)d.M, li = r32 / M, qr = r32 - li * M;
  const bool live = li < nl;
  const int64_t lane = lanes[live ? li : 0];
  const int64_t qpos = ((const int64_t*)d.qpos0)[lane] + qr / d.row_div;
  uint4 qf[DS];                                // Q^T fragments: Q[row][16 s + 8 h .. + 8]
  {
    const int64_t qe = ((const int64_t*)d.q_base)[lane] + (int64_t)qr * d.q_row + 8 * h;
    const KTIR_G(uint16_t)* Q = (const KTIR_G(uint16_t)*)d.q_ptr;
    if (vec && !(qe & 7) && qe >= d.q_lo && qe + D - 8 <= d.q_hi) {
#pragma unroll
      for (int s = 0; s < DS; ++s) qf[s] = __builtin_bit_cast(uint4, *(const KTIR_G(u32x4_t)*)(Q + qe + 16 * s));
    } else {
#pragma unroll
      for (int s = 0; s < DS; ++s) {
        uint32_t u[4];
        for (int k = 0; k < 4; ++k) {
          const int64_t e = qe + 16 * s + 2 * k;
          u[k] = ((e >= d.q_lo && e < d.q_hi) ? (uint32_t)Q[e] : 0u) |
                 (((e + 1 >= d.q_lo && e + 1 < d.q_hi) ? (uint32_t)Q[e + 1] : 0u) << 16);
        }
        qf[s] = make_uint4(u[0], u[1], u[2], u[3]);
      }
    }
  }
  // the position mask keeps key and row iff ((mlo <= kpos - qpos <= mhi) != inv)
  int mlo = INT_MIN, mhi = INT_MAX;
  bool inv = false;
  if (d.causal) {
    switch (d.pred) {
      case KTIR_CMP_EQ: mlo = mhi = 0; break;
      case KTIR_CMP_NE: mlo = mhi = 0; inv = true; break;
      case KTIR_CMP_SLT: case KTIR_CMP_ULTI: mhi = -1; break;
      case KTIR_CMP_SLE: case KTIR_CMP_ULEI: mhi = 0; break;
      case KTIR_CMP_SGT: case KTIR_CMP_UGTI: mlo = 1; break;
      default: mlo = 0; break;                 // SGE / UGE (the launcher rejects others)
    }
  }
  // pairs of pages first_pair, first_pair + stride, ...; the table's entries of
  // 32 of them at a time, entry 2 k + p of pair k in lane 2 k + p
  const int first_pair = part * W + w, stride = S * W, n_pairs = (trips + 1) >> 1;
  bool bad = false;
  auto entries = [&](int k0) -> int64_t {
    const int j = 2 * (first_pair + (k0 + (l >> 1)) * stride) + (l & 1);
    const int64_t te = tp + (int64_t)j * d.tbl_step;
    int64_t page = 0;
    if (j >= 0 && j < trips && te >= d.tbl_lo && te < d.tbl_hi) page = ps_index(d.tbl_ptr, te, d.tbl_dtype);
    bad |= page < 0;
    return page < 0 ? 0 : page;
  };
  int64_t table = entries(0);
  auto page_of = [&](int k, int p) -> int64_t {
    const int src = 2 * (k & 31) + p;
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)table, src), hi = __builtin_amdgcn_readlane((uint32_t)(table >> 32), src);
    return (int64_t)(((uint64_t)hi << 32) | lo);
  };
  // K or V of pair k, both pages by DMA (pages known to lie in their windows;
  // the second one of an odd loop's last pair is missing: zeros)
  auto dma = [&](int k, bool v) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const bool there = p == 0 || 2 * (first_pair + k * stride) + 1 < trips;
      if (!v) ps_dma<D>(d.k_ptr, kb + page_of(k, p) * d.k_page, d.k_row, there, k_lds, 16 * p, l);
      else ps_dma<D>(d.v_ptr, vb + page_of(k, p) * d.v_page, d.v_row, there, v_lds, 16 * p, l);
    }
  };
  // element by element, zeros outside the windows and for the missing second
  // page of an odd loop's last pair (whose scores are -inf)
  auto copy = [&](int k) {
    for (int p = 0; p < 2; ++p) {
      const bool in = 2 * (first_pair + k * stride) + p < trips;
      ps_copy<D>(d.k_ptr, kb + page_of(k, p) * d.k_page, d.k_row, d.k_lo, in ? d.k_hi : d.k_lo, K, 16 * p, l);
      ps_copy<D>(d.v_ptr, vb + page_of(k, p) * d.v_page, d.v_row, d.v_lo, in ? d.v_hi : d.v_lo, V, 16 * p, l);
    }
  };
  const f32x16_t z16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  f32x16_t o[DT];                              // O^T tiles: column 32 dt + 8 g + 4 h + t of row r32
  float m, mr, lsum;
  const int k_off = r32 * D, k_x = kv_swz<D>(r32 & 15);
  const int tg = l >> 4, tj = l & 15;
  const int v_row0 = 4 * (tg >> 1) + (tj >> 2);
  const int v_c = 2 * (tg & 1) + ((tj >> 1) & 1), v_in = 4 * (tj & 1);
  const int v_b0 = v_row0 * D + v_in, v_x0 = v_c ^ kv_swz<D>(v_row0), v_x1 = v_c ^ kv_swz<D>(v_row0 + 8);
  const int mine = first_pair < n_pairs ? (n_pairs - first_pair + stride - 1) / stride : 0;
  constexpr int LOADS = 32 * D / 512;          // a pair's K (or V) loads
  // One pair.  FAST: its K and V are in flight, K first; those of pair `next`
  // (the last pair again at the end, so that the count in flight is the same)
  // follow as each buffer falls free.  INF_V: V may hold infinities.
  auto step = [&](auto fast, auto inf_v, int k, int next) __attribute__((always_inline)) {
    constexpr bool FAST = decltype(fast)::value, INF_V = decltype(inf_v)::value;
    const int j0 = 2 * (first_pair + k * stride);
    if constexpr (FAST) ps_wait<LOADS>();
    f32x16_t sc = z16;
#pragma unroll
    for (int s = 0; s < DS; ++s) sc = mfma_at<BF16>(*(const uint4*)&K[k_off + 8 * ((2 * s + h) ^ k_x)], qf[s], sc);
    __builtin_amdgcn_sched_barrier(0);
    // every read of K has been used: the next pair's K streams in
    if constexpr (FAST) dma(next, false);
    // lane value i is key 8 (i / 4) + 4 h + i % 4 (i < 8: the first page)
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = __fmul_rn(d.scale, sc[i]);
    const bool two = j0 + 1 < trips;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      if (p && !two) {
#pragma unroll
        for (int i = 8; i < 16; ++i) x[i] = -__builtin_inff();
      } else if (d.causal) {
        int64_t d64 = kp0 + (int64_t)(j0 + p) * d.kpos_step - qpos;
        d64 = d64 < -(1 << 30) ? -(1 << 30) : (d64 > (1 << 30) ? (1 << 30) : d64);
        const int db = (int)d64;
        if (!__all(inv ? (db + 15 < mlo || db > mhi) : (db >= mlo && db + 15 <= mhi))) {
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const int df = db + 8 * (i >> 2) + 4 * h + (i & 3);
            if ((df >= mlo && df <= mhi) == inv) x[8 * p + i] = d.neg;
          }
        }
      }
    }
    float x0 = fmax3_nan(x[0], x[1], x[2]), x1 = fmax3_nan(x[8], x[9], x[10]);
#pragma unroll
    for (int i = 3; i < 7; i += 2) {
      x0 = fmax3_nan(x0, x[i], x[i + 1]);
      x1 = fmax3_nan(x1, x[8 + i], x[9 + i]);
    }
    x0 = fmax_nan(x0, x[7]);
    x1 = fmax_nan(x1, x[15]);
    bool poison = false;
    if (j0 == 0) poison = pair_max(x0) == -__builtin_inff();
    const float mn = fmax_nan(m, pair_max(fmax_nan(x0, x1)));
    const bool up = mn > __fadd_rn(mr, P_LAG<BF16>);
    if (__any(up)) {
      const float al = up ? exp_f(__fsub_rn(mr, mn)) : 1.f;
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[t][i] = __fmul_rn(o[t][i], al);
      lsum = __fmul_rn(lsum, al);
      mr = up ? mn : mr;
    }
    m = mn;
    // all keys so far masked: P = 0 against any base.  The exponent is (S - mr)
    // log2 e, not S log2 e - mr log2 e: the rounding of the second product would
    // stand between wavefronts of other bases, and passes 1 where a mask's fill
    // (-1e9, the type's lowest value) is the maximum so far.
    const float mb = mn == -__builtin_inff() ? 0.f : (mn != mn ? mn : mr);
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = exp_f(__fsub_rn(x[i], mb));
    // whether a P is too small for two f16 terms
    bool small = false;
    if constexpr (!BF16 && PARTS == 2 && !INF_V) small = __any(least_positive<16>(x) < P_SMALL);
    float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
      a0 = __fadd_rn(a0, x[i]);
      a1 = __fadd_rn(a1, x[i + 1]);
      a2 = __fadd_rn(a2, x[i + 2]);
      a3 = __fadd_rn(a3, x[i + 3]);
    }
    lsum = __fadd_rn(lsum, pair_sum(__fadd_rn(__fadd_rn(a0, a1), __fadd_rn(a2, a3))));
    // V of this pair has landed: only the next pair's K is in flight
    if constexpr (FAST) ps_wait<LOADS>();
    // P V: by the terms of the operand type, by the rest they leave (two f16
    // terms) or by bf16 terms of the whole P (the same with infinities in V)
    enum { TERMS, REST, WHOLE };
    auto pv = [&](auto how) __attribute__((always_inline)) {
      constexpr int HOW = decltype(how)::value;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const uint16_t* vt = &V[16 * ks * D];
        float p[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          p[i] = x[8 * ks + i];
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
            o[dt] = pv_mfma<BF16, PARTS, INF_V>(a, t0, t1, o[dt]);
          } else {
            o[dt] = pv_mfma_bf<INF_V>(a, tb, o[dt]);
            __builtin_amdgcn_sched_barrier(0);     // rare: must not set the register count
          }
        }
      }
      if constexpr (FAST && HOW == TERMS) {
        // the V reads of the second 16 keys between the MFMAs of the first
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * DT, 0);
#pragma unroll
        for (int q = 0; q < DT; ++q) {
          __builtin_amdgcn_sched_group_barrier(0x008, PARTS, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, DT * PARTS, 0);
      }
    };
    if constexpr (!BF16 && PARTS == 2 && INF_V) {
      pv(std::integral_constant<int, WHOLE>{});
    } else {
      pv(std::integral_constant<int, TERMS>{});
      if (small) pv(std::integral_constant<int, REST>{});
    }
    if (j0 == 0 && __any(poison)) {
      const float nan = __builtin_nanf("");
      if (poison) {
        lsum = nan;
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[t][i] = nan;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (FAST) dma(next, true);
  };
  auto pages = [&](auto inf_v) __attribute__((always_inline)) {
    constexpr bool INF_V = decltype(inf_v)::value;
#pragma unroll
    for (int t = 0; t < DT; ++t) o[t] = z16;
    m = mr = -__builtin_inff();
    lsum = 0.f;
    for (int c0 = 0; c0 < mine; c0 += 32) {
      if (INF_V || c0) table = entries(c0);
      const int c1 = c0 + 32 < mine ? c0 + 32 : mine;
      int k = c0;
      if constexpr (!INF_V) {
        // pages of these pairs that are wholly in their windows, or missing
        const int my_pair = c0 + (l >> 1);
        const int64_t ke = kb + table * d.k_page, ve = vb + table * d.v_page;
        const bool ok = my_pair >= c1 || (vec && (2 * (first_pair + my_pair * stride) + (l & 1) >= trips ||
                                                  (ps_fast<D>(ke, d.k_row, d.k_lo, d.k_hi) && ps_fast<D>(ve, d.v_row, d.v_lo, d.v_hi))));
        const uint64_t ballot = __builtin_amdgcn_ballot_w64(!ok);
        // the pairs before the first that is not
        const int nf = ballot ? __builtin_ctzll(ballot) >> 1 : c1 - c0;
        if (nf > 0) {
          dma(c0, false);
          dma(c0, true);
          for (; k < c0 + nf; ++k) step(std::true_type{}, inf_v, k, k + 1 < c0 + nf ? k + 1 : k);
          ps_wait<0>();
        }
      }
      for (; k < c1; ++k) {
        copy(k);
        step(std::false_type{}, inf_v, k, k);
      }
    }
  };
  pages(std::false_type{});
  // An infinite V times the terms of P after the first (0, or of the other
  // sign) is NaN where P V is infinite.  So a NaN anywhere in the wavefront's
  // result runs its pages again with only the first term meeting such values.
  if constexpr (PARTS > 1) {
    bool nan = false;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) nan |= o[t][i] != o[t][i];
    if (__any(nan)) pages(std::true_type{});
  }
  if (bad) *err = 1;
  // bring l and O from mr to m, and O from P's scale
  if (mine > 0 && m != -__builtin_inff()) {
    const float fin = exp_f(__fsub_rn(mr, m)), f = __fmul_rn(fin, 1.f / P_SCALE<BF16>);
    lsum = __fmul_rn(lsum, fin);
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[t][i] = __fmul_rn(o[t][i], f);
  }
  // the wavefront's state into its LDS: 4-column groups of a row, rows side by side
  __builtin_amdgcn_s_waitcnt(0);
  constexpr int HALF = D / 8;                  // 4-column groups in K's part
  auto grp = [&](int wv, int g) -> float4* {
    return (float4*)(g < HALF ? (uint8_t*)Ks[wv] + 512 * g : (uint8_t*)Vs[wv] + 512 * (g - HALF));
  };
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      grp(w, 8 * t + 2 * g + h)[r32] = make_float4(o[t][4 * g], o[t][4 * g + 1], o[t][4 * g + 2], o[t][4 * g + 3]);
  if (h == 0) {
    ms[w][r32] = m;
    ls[w][r32] = lsum;
  }
  // row tid % 32, columns 16 q .. + 16
  const int row = tid & 31;
  const PsDst dst = ps_dst(d, lanes, nl, row);
  __syncthreads();
  float mm = ms[0][row];
#pragma unroll
  for (int v = 1; v < W; ++v) mm = fmax_nan(mm, ms[v][row]);
  float wt[W], lm = 0.f;
#pragma unroll
  for (int v = 0; v < W; ++v) {
    wt[v] = ps_weight(ms[v][row], mm);
    lm = __fadd_rn(lm, __fmul_rn(ls[v][row], wt[v]));
  }
  for (int q = tid >> 5; q < D / 16; q += 2 * W) {
    float acc[16];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int v = 0; v < W; ++v) {
        const float4 x = grp(v, 4 * q + k)[row];
        a.x = __fadd_rn(a.x, __fmul_rn(x.x, wt[v]));
        a.y = __fadd_rn(a.y, __fmul_rn(x.y, wt[v]));
        a.z = __fadd_rn(a.z, __fmul_rn(x.z, wt[v]));
        a.w = __fadd_rn(a.w, __fmul_rn(x.w, wt[v]));
      }
      acc[4 * k] = a.x;
      acc[4 * k + 1] = a.y;
      acc[4 * k + 2] = a.z;
      acc[4 * k + 3] = a.w;
    }
    if (S == 1) {
      ps_out<D>(d, dst, q, acc, lm, mm);
    } else if (dst.live) {
      // workspace: per workgroup m [32], l [32], then O as the LDS holds it
      float* ws = (float*)d.ws + (int64_t)blockIdx.x * (64 + PS_ROWS * D);
      if (q == 0) {
        ws[row] = mm;
        ws[32 + row] = lm;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)
        *(float4*)(ws + 64 + ((4 * q + k) * 32 + row) * 4) = make_float4(acc[4 * k], acc[4 * k + 1], acc[4 * k + 2], acc[4 * k + 3]);
    }
  }
}

// The S states of an item, one workgroup per item and 16 columns.  Bound: a
// chain of memory latencies, so as many states as there are threads for are
// loaded at once: the item's live rows (to a power of two) side by side, G
// threads with a state each on every row, PM_U states per thread before anything
// waits for one.
constexpr int PM_THREADS = 256, PM_U = 4;

template <int D>
__global__ __launch_bounds__(PM_THREADS) void pattn_merge(const ktir_pattn_t d) {
  constexpr int SZ = 64 + PS_ROWS * D;
  const int S = d.splits;
  const int item = blockIdx.x / (D / 16), q = blockIdx.x % (D / 16);
  const PsItem* it = (const PsItem*)d.items + item;
  const int first = uni(it->first), nl = uni(it->count);
  const int32_t* lanes = (const int32_t*)d.item_lanes + first;
  const float* ws = (const float*)d.ws + (int64_t)item * S * SZ;
  __shared__ float4 part[4][PM_THREADS];
  __shared__ float lpart[PM_THREADS], mpart[PM_THREADS];
  const int tid = threadIdx.x, rows = nl * (int)d.M;        // 1 .. 32
  const int lg = rows > 1 ? 32 - __builtin_clz(rows - 1) : 0;
  const int row = tid & ((1 << lg) - 1), t = tid >> lg, G = PM_THREADS >> lg;   // states t, t + G, ...
  const bool live = row < rows;
  const float ninf = -__builtin_inff();
  float mu[PM_U], lu[PM_U];
  float4 x[PM_U][4];
#pragma unroll
  for (int u = 0; u < PM_U; ++u) {
    const int s = t + u * G;
    const bool on = live && s < S;
    const float* p = ws + (int64_t)(on ? s : 0) * SZ;
    mu[u] = on ? p[row] : ninf;
    lu[u] = on ? p[32 + row] : 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      x[u][k] = on ? *(const float4*)(p + 64 + ((4 * q + k) * 32 + row) * 4) : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  const PsDst dst = ps_dst(d, lanes, nl, row);
  float m = mu[0];
#pragma unroll
  for (int u = 1; u < PM_U; ++u) m = fmax_nan(m, mu[u]);
  if (live)
    for (int s = t + PM_U * G; s < S; s += G) m = fmax_nan(m, ws[(int64_t)s * SZ + row]);
  mpart[tid] = m;
  for (int off = G >> 1; off; off >>= 1) {
    __syncthreads();
    if (t < off) mpart[tid] = fmax_nan(mpart[tid], mpart[tid + (off << lg)]);
  }
  __syncthreads();
  m = mpart[row];
  float l = 0.f;
  float4 a[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) a[k] = make_float4(0.f, 0.f, 0.f, 0.f);
  auto add = [&](float ms, float ls, const float4 (&v)[4]) __attribute__((always_inline)) {
    const float w = ps_weight(ms, m);
    l = __fadd_rn(l, __fmul_rn(ls, w));
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      a[k].x = __fadd_rn(a[k].x, __fmul_rn(v[k].x, w));
      a[k].y = __fadd_rn(a[k].y, __fmul_rn(v[k].y, w));
      a[k].z = __fadd_rn(a[k].z, __fmul_rn(v[k].z, w));
      a[k].w = __fadd_rn(a[k].w, __fmul_rn(v[k].w, w));
    }
  };
#pragma unroll
  for (int u = 0; u < PM_U; ++u) add(mu[u], lu[u], x[u]);
  if (live)
    for (int s = t + PM_U * G; s < S; s += G) {
      const float* p = ws + (int64_t)s * SZ;
      float4 v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = *(const float4*)(p + 64 + ((4 * q + k) * 32 + row) * 4);
      add(p[row], p[32 + row], v);
    }
  lpart[tid] = l;
#pragma unroll
  for (int k = 0; k < 4; ++k) part[k][tid] = a[k];
  for (int off = G >> 1; off; off >>= 1) {
    __syncthreads();
    if (t < off) {
      const int o = tid + (off << lg);
      l = __fadd_rn(l, lpart[o]);
      lpart[tid] = l;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float4 y = part[k][o];
        a[k] = make_float4(__fadd_rn(a[k].x, y.x), __fadd_rn(a[k].y, y.y), __fadd_rn(a[k].z, y.z), __fadd_rn(a[k].w, y.w));
        part[k][tid] = a[k];
      }
    }
  }
  if (t != 0) return;
  float acc[16];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    acc[4 * k] = a[k].x;
    acc[4 * k + 1] = a[k].y;
    acc[4 * k + 2] = a[k].z;
    acc[4 * k + 3] = a[k].w;
  }
  ps_out<D>(d, dst, q, acc, l, m);
}

// True when launched: the caller gave items (at most 32 rows of lanes that read
// the same pages), pages of 16 keys, one 16-bit operand type, 64 or 128 columns,
// row maxima that start at -inf.
bool launch_pattn_split(const ktir_pattn_t* d) {
  if (!d->items || !d->item_lanes || d->n_items < 1 || d->splits < 1 || (d->splits > 1 && !d->ws)) return false;
  if (d->waves != 4 && d->waves != 8) return false;
  if (d->n_items * d->splits > INT_MAX || d->n_items * (d->D / 16) > INT_MAX) return false;
  if (d->q_dtype != d->kv_dtype || (d->kv_dtype != KTIR_F16 && d->kv_dtype != KTIR_BF16)) return false;
  if (d->N != 16 || d->M > PS_ROWS || (d->D != 64 && d->D != 128) || d->m0 != -__builtin_inff()) return false;
  if (d->k_row < d->D || d->v_row < d->D || d->k_row >= (1 << 24) || d->v_row >= (1 << 24)) return false;
  // vector loads: 16-byte aligned operands, rows and pages a multiple of 8 elements
  const int vec = !((d->q_ptr | d->k_ptr | d->v_ptr) & 15) && !((d->q_row | d->k_row | d->v_row | d->k_page | d->v_page) & 7);
  const bool bf = d->kv_dtype == KTIR_BF16, more = d->M > 16;
  const dim3 grid((unsigned)(d->n_items * d->splits));
  auto go = [&](auto kern, int waves) {
    hipLaunchKernelGGL(kern, grid, dim3(64 * waves), 0, stream(), *d, vec, device_error_flag());
  };
  auto by = [&](auto dim, auto waves) {
    constexpr int D = decltype(dim)::value, W = decltype(waves)::value;
    if (bf) more ? go(pattn_split<true, D, 3, W>, W) : go(pattn_split<true, D, 2, W>, W);
    else more ? go(pattn_split<false, D, 2, W>, W) : go(pattn_split<false, D, 1, W>, W);
  };
  const std::integral_constant<int, 64> d64;
  const std::integral_constant<int, 128> d128;
  const std::integral_constant<int, 4> w4;
  const std::integral_constant<int, 8> w8;
  if (d->D == 64) d->waves == 8 ? by(d64, w8) : by(d64, w4);
  else d->waves == 8 ? by(d128, w8) : by(d128, w4);
  if (d->splits > 1) {
    const dim3 mg((unsigned)(d->n_items * (d->D / 16)));
    if (d->D == 64) hipLaunchKernelGGL(pattn_merge<64>, mg, dim3(PM_THREADS), 0, stream(), *d);
    else hipLaunchKernelGGL(pattn_merge<128>, mg, dim3(PM_THREADS), 0, stream(), *d);
  }
  return true;
}

}  // namespace ktir
