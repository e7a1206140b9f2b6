// gfx950 MFMA matmul over planes of lanes: f16 / bf16 operands, f32
// accumulation (dialects/linalg_ops.py:325-347 fused over the K loop).
//
// The lanes (simulated cores and loop iterations) of one product are tiles of
// one result plane: the lane in row r, column c of the plane reads A r M rows
// and B c N columns after the first lane.  The plane is cut into BM x BN blocks
// without regard to the lanes' own tiles, one workgroup each, so small tiles
// (64 x 64) share operands as large ones do and the block can be chosen for
// the chip: the smaller blocks where the larger ones leave CUs idle.
//
// Four wavefronts, wavefront (wr, wc) a BM/2 x BN/2 quarter in 32 x 32 MFMA
// tiles.  K advances 64 at a time through NS (two or four) LDS stages filled by
// buffer_load ... lds (no registers) with one barrier a step; a step's
// 256 to 512 MFMA cycles are far less than a load's latency, so where one
// workgroup has a CU to itself three stages stay in flight (launches of
// 512 x 4096 x 4096, f16, one after another: 49 us with two stages, 29 with four).
// Then the LDS reads bound it: a 64 x 64 quarter reads 16 KB for 16 MFMAs.
// 512 x 4096 x 4096 in 64 x 64 tiles, as a pass between others: 1009 us
// (mm_generic, f32 FMA) -> 26 us (660 TFLOP/s); 2048^3 in 128 x 128 tiles: 30 us
// (mm_mfma_dma) -> 26 us.  Where those tiles fill the chip they stay the better
// blocks (plane_wins in ktir_mfma.hip).
// Layouts: A as 128-byte rows (16-byte chunk c of row
// r at slot c ^ swz_a(r), read by ds_read_b128), B row-major as in HBM (chunk c
// at c ^ mp_swz(r), read by ds_read_b64_tr_b16); both layouts are free of bank
// conflicts.  Rows and columns past the plane's end repeat the last one (their
// results are not written); k past the end (a last step of fewer than 64)
// repeats the first and is zeroed in LDS before use.
#include <climits>
#include <type_traits>

#include "ktir_mfma_common.h"

namespace ktir {

constexpr int MP_BK = 64;

// slot permutation of a B row's 16-byte chunks: 16 chunks (BN = 128) or 8
template <int BN>
__device__ __forceinline__ int mp_swz(int r) {
  if constexpr (BN == 128) return swz16(r);
  else return ((r & 1) << 1) ^ ((r & 2) << 1) ^ ((r >> 2) & 1) ^ (((r >> 3) & 1) << 1);
}

// wait until at most N of this wavefront's vector memory loads are in flight
template <int N>
__device__ __forceinline__ void mp_wait() {
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Workgroup barrier that leaves later stages' loads in flight
// (__syncthreads waits for all of them).  Nothing moves across it.
__device__ __forceinline__ void mp_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

struct MpShape {
  int64_t rows, cols, K;                       // the plane's extent and the whole K
  int64_t a_row, b_row;
  int32_t M, N;                                // a lane's tile
  int32_t lanes_n;                             // lanes in a plane row
  int32_t blocks_m, blocks_n;
  int32_t group;                               // block rows that run side by side
  int32_t planes;
};

template <bool BF16, int BM, int BN, int NS>
__global__ __launch_bounds__(256, 2) void mm_plane(const ktir_mm_t d, const MpShape S) {
  constexpr int MI = BM / 64, NI = BN / 64;    // 32 x 32 tiles of a wavefront
  constexpr int AB = BM / 32, BB = BN / 32;    // 1 KB blocks a wavefront stages: 8 rows of A, 512 / BN rows of B
  // distinct arrays, so that the compiler sees that a stage being filled is
  // not the one being read
  __shared__ __align__(16) uint16_t As0[BM * MP_BK], As1[BM * MP_BK];
  __shared__ __align__(16) uint16_t Bs0[MP_BK * BN], Bs1[MP_BK * BN];
  __shared__ __align__(16) uint16_t As2[NS > 2 ? BM * MP_BK : 8], As3[NS > 2 ? BM * MP_BK : 8];
  __shared__ __align__(16) uint16_t Bs2[NS > 2 ? MP_BK * BN : 8], Bs3[NS > 2 ? MP_BK * BN : 8];
  const int tid = threadIdx.x, l = tid & 63, h = l >> 5, r32 = l & 31;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wr = w >> 1, wc = w & 1;
  // XCD x runs the x-th eighth of the blocks; in that order `group` block rows
  // are swept column by column, so an XCD's L2 holds what its blocks share
  const int nblk = gridDim.x;
  int bid = blockIdx.x;
  if ((nblk & 7) == 0) bid = (bid & 7) * (nblk >> 3) + (bid >> 3);
  const int per = S.blocks_m * S.blocks_n, plane = bid / per;
  bid -= plane * per;
  const int gsz = S.group * S.blocks_n, g0 = bid / gsz * S.group;
  const int gm = S.blocks_m - g0 < S.group ? S.blocks_m - g0 : S.group;
  const int in_g = bid % gsz;
  const int bm = g0 + in_g % gm, bn = in_g / gm;
  const int lanes_m = (int)(S.rows / S.M);
  const int32_t* table = (const int32_t*)d.plane + (int64_t)plane * lanes_m * S.lanes_n;
  const int64_t l0 = uni(d.plane ? table[0] : plane);
  const int64_t m0 = (int64_t)bm * BM, n0 = (int64_t)bn * BN;
  const uint16_t* A = (const uint16_t*)d.a.ptr + uni(lane_offset(d.a, l0)) + m0 * S.a_row;
  const uint16_t* B = (const uint16_t*)d.b.ptr + uni(lane_offset(d.b, l0)) + n0;
  // valid rows / columns of this block, and per staged block the lane's byte
  // offset from A (row, chunk 0) and B (row 0, chunk), its chunk / row of the step
  const int vm = (int)(S.rows - m0 < BM ? S.rows - m0 : BM), vn = (int)(S.cols - n0 < BN ? S.cols - n0 : BN);
  uint32_t ao[AB], bo[BB];
  const int ac = (l & 7);                      // A slot
  constexpr int CB = BN / 8, RB = 512 / BN;    // B: chunks per row, rows per 1 KB
#pragma unroll
  for (int i = 0; i < AB; ++i) {
    const int r = (BM / 4) * w + 8 * i + (l >> 3);
    const int rr = r < vm ? r : vm - 1;
    ao[i] = (uint32_t)((rr * S.a_row + 8 * (ac ^ swz_a(r & 15))) * 2);
  }
#pragma unroll
  for (int i = 0; i < BB; ++i) {
    const int r = 16 * w + RB * i + l / CB;
    int c = (l % CB) ^ mp_swz<BN>(r & 15);
    c = 8 * c < vn ? c : 0;
    bo[i] = (uint32_t)((r * S.b_row + 8 * c) * 2);
  }
  const int64_t nk = (S.K + MP_BK - 1) / MP_BK;
  const int rem = (int)(S.K - (nk - 1) * MP_BK);   // k of the last step
  // A and B of k step kt into a stage
  auto issue = [&](int64_t kt, uint16_t* as, uint16_t* bs) __attribute__((always_inline)) {
    const uint16_t* a = A + kt * MP_BK;
    const uint16_t* b = B + kt * MP_BK * S.b_row;
    // every offset below lies inside the operand (the launch checked the
    // plane's extent); the buffer's range is the 2 GB the offsets can span
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)a, (short)0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void*)b, (short)0, 0x7fffffff, 0x00020000);
    const bool cut = kt == nk - 1 && rem < MP_BK;
#pragma unroll
    for (int i = 0; i < AB; ++i) {
      uint32_t o = ao[i];
      if (cut) {
        const int r = (BM / 4) * w + 8 * i + (l >> 3), c = ac ^ swz_a(r & 15);
        if (8 * c >= rem) o -= 16 * c;
      }
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (__attribute__((address_space(3))) void*)(as + MP_BK * ((BM / 4) * w + 8 * i)),
                                               16, o, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < BB; ++i) {
      uint32_t o = bo[i];
      if (cut) {
        const int r = 16 * w + RB * i + l / CB;
        if (r >= rem) o -= (uint32_t)(r * S.b_row * 2);
      }
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (__attribute__((address_space(3))) void*)(bs + BN * (16 * w + RB * i)), 16, o,
                                               0, 0, 0);
    }
  };
  // zeros over the k of a cut last step (the DMA has landed, nobody reads yet)
  auto zero_tail = [&](uint16_t* as, uint16_t* bs) {
    const uint4 z = make_uint4(0, 0, 0, 0);
    for (int i = tid; i < BM * 8; i += 256) {
      const int r = i >> 3, c = i & 7;
      if (8 * c >= rem) *(uint4*)&as[r * MP_BK + 8 * (c ^ swz_a(r & 15))] = z;
    }
    for (int i = tid; i < MP_BK * CB; i += 256) {
      const int r = i / CB;
      if (r >= rem) *(uint4*)&bs[r * BN + 8 * (i % CB)] = z;
    }
    __syncthreads();
  };
  // B fragment (column l % 32 of a 32-column tile, k 8 h .. + 8) as two
  // transposing reads: member tj of 16-lane group tg reads k-row 8 (tg / 2) +
  // tj / 4 (+ 4), columns 16 (tg % 2) + 4 (tj % 4)
  const int tg = l >> 4, tj = l & 15;
  const int br0 = 8 * (tg >> 1) + (tj >> 2);
  const int bc = 2 * (tg & 1) + ((tj >> 1) & 1), bin = 4 * (tj & 1);
  int b_off[2][NI];
#pragma unroll
  for (int hi = 0; hi < 2; ++hi)
#pragma unroll
    for (int j = 0; j < NI; ++j)
      b_off[hi][j] = (br0 + 4 * hi) * BN + 8 * ((4 * (NI * wc + j) + bc) ^ mp_swz<BN>(br0 + 4 * hi)) + bin;
  const f32x16 z16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  f32x16 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = z16;
  auto step = [&](const uint16_t* as, const uint16_t* bs) __attribute__((always_inline)) {
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int ch = 2 * kk + h;
      uint4 a[MI], b[NI];
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const int ar = wr * (BM / 2) + 32 * i + r32;
        a[i] = *(const uint4*)&as[ar * MP_BK + 8 * (ch ^ swz_a(ar & 15))];
      }
      const uint16_t* bt = bs + 16 * kk * BN;
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const uint2 lo = mm_tr16(bt + b_off[0][j]), hi = mm_tr16(bt + b_off[1][j]);
        b[j] = make_uint4(lo.x, lo.y, hi.x, hi.y);
      }
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = mfma32<BF16>(a[i], b[j], acc[i][j]);
    }
  };
  // Step kt: its stage has landed when at most the NS - 2 later stages' loads
  // are in flight; after the barrier every wavefront is also done with step
  // kt - 1, whose stage then takes step kt + NS - 1 (past the end the last
  // step again, which nobody reads, so that the count in flight is the same).
  auto run = [&](int64_t kt, const uint16_t* as, const uint16_t* bs, uint16_t* asf, uint16_t* bsf) __attribute__((always_inline)) {
    mp_wait<(NS - 2) * (AB + BB)>();
    mp_barrier();
    issue(kt + NS - 1 < nk ? kt + NS - 1 : nk - 1, asf, bsf);
    // two stages: the loads have one step to land, so they go first
    if constexpr (NS == 2) __builtin_amdgcn_sched_barrier(0);
    step(as, bs);
  };
  const int64_t whole = rem < MP_BK ? nk - 1 : nk;   // steps of 64
  issue(0, As0, Bs0);
  if constexpr (NS == 2) {
    int64_t kt = 0;
    for (; kt + 2 <= whole; kt += 2) {
      run(kt, As0, Bs0, As1, Bs1);
      run(kt + 1, As1, Bs1, As0, Bs0);
    }
    if (kt < whole) run(kt, As0, Bs0, As1, Bs1);
  } else {
    issue(nk > 1 ? 1 : 0, As1, Bs1);
    issue(nk > 2 ? 2 : nk - 1, As2, Bs2);
    int64_t kt = 0;
    for (; kt + 4 <= whole; kt += 4) {
      run(kt, As0, Bs0, As3, Bs3);
      run(kt + 1, As1, Bs1, As0, Bs0);
      run(kt + 2, As2, Bs2, As1, Bs1);
      run(kt + 3, As3, Bs3, As2, Bs2);
    }
    if (kt < whole) run(kt, As0, Bs0, As3, Bs3);
    if (kt + 1 < whole) run(kt + 1, As1, Bs1, As0, Bs0);
    if (kt + 2 < whole) run(kt + 2, As2, Bs2, As1, Bs1);
  }
  mp_wait<0>();
  if (whole < nk) {
    __syncthreads();
    const int q = (int)(whole % NS);
    uint16_t* as = q == 0 ? As0 : (q == 1 ? As1 : (q == 2 ? As2 : As3));
    uint16_t* bs = q == 0 ? Bs0 : (q == 1 ? Bs1 : (q == 2 ? Bs2 : Bs3));
    zero_tail(as, bs);
    step(as, bs);
  }
  // outs absent or a zero splat (accumulate == 2: x + 0.0), rounded to the
  // result dtype (the only forms launched here)
  const float z = d.accumulate == 2 ? 0.f : -0.f;
  const int64_t cs = d.c.strides[0];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int tr = wr * (BM / 2) + 32 * i, tc = wc * (BN / 2) + 32 * j;
      if (tr >= vm || tc >= vn) continue;
      const int64_t row = m0 + tr, col = n0 + tc;
      const int lr = (int)(row / S.M), lc = (int)(col / S.N);
      const int64_t ln = d.plane ? uni(table[lr * S.lanes_n + lc]) : plane;
      const int64_t o = uni(lane_offset(d.c, ln)) + (row - (int64_t)lr * S.M + 4 * h) * cs + (col - (int64_t)lc * S.N) + r32;
      auto put = [&](auto dt) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 16; ++e) mm_put<decltype(dt)::value>(d.c.ptr, o + (8 * (e >> 2) + (e & 3)) * cs, __fadd_rn(acc[i][j][e], z));
      };
      if (d.c.dtype == KTIR_F32) put(std::integral_constant<int, KTIR_F32>{});
      else if (d.c.dtype == KTIR_F16) put(std::integral_constant<int, KTIR_F16>{});
      else put(std::integral_constant<int, KTIR_BF16>{});
    }
}

// True when launched: f16 or bf16 operands, unit inner strides, 16-byte
// aligned rows, every lane's reads checked by the caller; M and N multiples
// of 32, the whole K (the fused loop's steps lie end to end) of 8; a result
// without an accumulator input.
bool launch_mm_plane(const ktir_mm_t* d) {
  const bool f16 = d->a.dtype == KTIR_F16 && d->b.dtype == KTIR_F16;
  const bool bf16 = d->a.dtype == KTIR_BF16 && d->b.dtype == KTIR_BF16;
  if (!(f16 || bf16) || d->M % 32 || d->N % 32 || d->K < 8 || d->K % 8) return false;
  if (!(d->a.flags & d->b.flags & KTIR_LEAF_CHECKED) || d->a.offsets || d->b.offsets) return false;
  if (d->a.strides[1] != 1 || d->b.strides[1] != 1 || d->c.strides[1] != 1 || d->c.offsets || d->c.winner) return false;
  if ((d->a.strides[0] | d->b.strides[0] | d->a_kstep | d->b_kstep) & 7 || (d->a.ptr | d->b.ptr) & 15) return false;
  if (d->accumulate == 1 || d->round_dt != KTIR_F32) return false;
  if (d->c.dtype != KTIR_F32 && d->c.dtype != KTIR_F16 && d->c.dtype != KTIR_BF16) return false;
  MpShape S{};
  S.a_row = d->a.strides[0];
  S.b_row = d->b.strides[0];
  if (S.a_row < 0 || S.b_row < 0) return false;
  if (d->ksteps > 1 && (d->a_kstep != d->K || d->b_kstep != d->K * S.b_row)) return false;
  S.K = d->K * d->ksteps;
  const int64_t lm = d->plane ? d->plane_m : 1, ln = d->plane ? d->plane_n : 1;
  if (lm < 1 || ln < 1 || d->lanes % (lm * ln) || d->M > (1 << 20) || d->N > (1 << 20) || lm * ln > INT32_MAX) return false;
  S.planes = (int32_t)(d->lanes / (lm * ln));
  if (d->lanes > INT32_MAX) return false;
  S.rows = lm * d->M;
  S.cols = ln * d->N;
  S.M = (int32_t)d->M;
  S.N = (int32_t)d->N;
  S.lanes_n = (int32_t)ln;
  // 32-bit byte offsets inside a block's rows of A and a step's rows of B
  if ((127 * S.a_row + 64) * 2 >= 0x7fffffff || (63 * S.b_row + 128) * 2 >= 0x7fffffff) return false;
  auto blocks = [&](int bm, int bn) { return (int64_t)S.planes * ((S.rows + bm - 1) / bm) * ((S.cols + bn - 1) / bn); };
  auto go = [&](auto kern16, auto kernbf, int bm, int bn) {
    S.blocks_m = (int32_t)((S.rows + bm - 1) / bm);
    S.blocks_n = (int32_t)((S.cols + bn - 1) / bn);
    S.group = 8;
    const dim3 grid((unsigned)blocks(bm, bn));
    if (f16) hipLaunchKernelGGL(kern16, grid, dim3(256), 0, stream(), *d, S);
    else hipLaunchKernelGGL(kernbf, grid, dim3(256), 0, stream(), *d, S);
  };
  if (blocks(64, 64) > INT32_MAX) return false;
  // The largest block that still gives every CU work (256 CUs; 128 x 128 with
  // two stages runs two workgroups per CU, with four one).  f16, us:
  //   3072 x 2048 x 4096 (384 blocks of 128 x 128): 68 two stages, 83 four;
  //   2048^3 (256): 27 four stages, 33 two, 33 as 64 x 128;
  //   512 x 4096 x 4096 (128, 256 of 64 x 128): 39 / 29 / 31 as 128 x 128 / 64 x 128 / 64 x 64;
  //   1024^3 (64, 128, 256): 15 / 11 / 8.6.
  const int64_t b = blocks(128, 128);
  if (b > 256) go(mm_plane<false, 128, 128, 2>, mm_plane<true, 128, 128, 2>, 128, 128);
  else if (b > 128) go(mm_plane<false, 128, 128, 4>, mm_plane<true, 128, 128, 4>, 128, 128);
  else if (blocks(64, 128) > 160) go(mm_plane<false, 64, 128, 4>, mm_plane<true, 64, 128, 4>, 64, 128);
  else go(mm_plane<false, 64, 64, 4>, mm_plane<true, 64, 64, 4>, 64, 64);
  return true;
}

}  // namespace ktir
