// Streaming kernel for launches of few product rows or few tiles (decode
// steps, short prompts, small squares): packed operands, small tiles, no LDS
// in the main loop.
//
// The 128 x 128 product tiles of the split and cubic kernels leave most CUs
// idle (or need many K shares) when a launch has few of them, and compute
// 128 product rows whatever M is. Here a workgroup owns 32 RB x 32 CB of
// product space, and each of its waves one product of the algorithm (seven
// for Strassen, eight for the cubic) over its share of K: no operand
// fragment is needed by two waves of the Strassen kernel, so fragments go
// straight from memory into registers (the packed layout is in lane order:
// one 1 KB load each), kDepth stages ahead, with no barrier before the last
// stage. The products are then combined and finished row by row from LDS
// (finish.hpp), or, when K is also divided among workgroups (p.ksplit),
// stored as FP32 [M, N] shares that stream_sum adds and finishes.
#pragma once

#include "common.hpp"
#include "finish.hpp"
#include "kernel_packed.hpp"

namespace smx {
namespace stream {

using packed::kBlocks;
using packed::kFrag;

// Operands of wave role r. A Strassen role is one product, operand r of A
// with operand r of B. A cubic role is one operand of B with the two of A
// that meet it, so that B is read once: B0, B1 with A0, A2 and B2, B3 with
// A1, A3. Role r's products are sets kProducts r ..; the cubic's quadrant q
// (row half q / 2, column half q % 2) is set 2 (q % 2) + q / 2 plus the same
// set of the roles two further on.
template <int kAlgo>
struct Roles {
  static constexpr int kCount = kAlgo == 7 ? 7 : 4;
  static constexpr int kProducts = kAlgo == 7 ? 1 : 2;
  static constexpr int kSets = kCount * kProducts;
  static constexpr int kOps = packed::nops_of(kAlgo);
  static __device__ __forceinline__ int op_a(int r, int product) {
    return kAlgo == 7 ? r : 2 * product + (r >> 1);
  }
};

// Threads of a workgroup, and the LDS its product sets take: kRG row blocks
// at a time (all of them when they fit), rows padded by 32 bytes so that the
// two half-waves of an accumulator store fall 32 banks apart.
template <int kAlgo, int RB, int CB>
struct Shape {
  static constexpr int kThreads = 64 * Roles<kAlgo>::kCount;
  static constexpr int kStride = CB * 128 + 32;  // bytes of one product row
  static constexpr int kRG = RB * CB > 4 ? 4 / CB : RB;
  static constexpr int kSet = 32 * kRG * kStride;
  static constexpr int kLds = Roles<kAlgo>::kSets * kSet;
  static_assert(RB % kRG == 0 && kLds <= 160 * 1024 && kThreads <= 1024, "workgroup limits");
  static_assert(4 % RB == 0 && 4 % CB == 0, "a tile stays inside one packed 128-row tile");
};

// A fragment of a panel; kNt: with the streaming cache policy.
template <bool kNt>
__device__ __forceinline__ bf16x8 load_frag(__amdgpu_buffer_rsrc_t rsrc, uint32_t voffset, uint32_t soffset) {
  return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rsrc, voffset, soffset, kNt ? 2 : 0));
}

// The two quadrants (left, right) of logical row half `half` for eight
// consecutive columns of one product row, from the product sets at `at`
// (kSet bytes apart), in the combinations and orders of quadrant_value
// (common.hpp).
template <int kAlgo, int kSet>
__device__ __forceinline__ void combine(const uint8_t* at, int formula, int half, F8& left, F8& right) {
  auto product = [&](int i) __attribute__((always_inline)) {
    const f32x4 lo = *reinterpret_cast<const f32x4*>(at + i * kSet);
    const f32x4 hi = *reinterpret_cast<const f32x4*>(at + i * kSet + 16);
    return F8{{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}};
  };
  if constexpr (kAlgo == 8) {
    left = add8<false>(product(half), product(half + 4));
    right = add8<false>(product(half + 2), product(half + 6));
  } else if (formula == kFormulaPowers) {
    const F8 z0 = add8<false>(product(2), product(4));  // R3 + R5
    // R1 - R3 + R4 + R7
    const F8 z3 = add8<false>(add8<false>(add8<true>(product(3), product(2)), product(6)), product(0));
    if (half) {
#pragma unroll
      for (int e = 0; e < 8; ++e) left.v[e] = z3.v[e] + z0.v[e] * 0.5f;
      right = z0;
      return;
    }
    const F8 z1 = add8<false>(product(5), product(6)), z2 = add8<true>(product(1), product(3));
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      left.v[e] = (z1.v[e] + z2.v[e]) * 0.5f + z0.v[e] * 0.25f;
      right.v[e] = ((z2.v[e] - z1.v[e]) + z3.v[e]) + z0.v[e] * 0.5f;
    }
  } else {
    const bool dual = formula == kFormulaDual;
    const F8 p1 = product(0);
    if (half == 0) {
      const F8 p4 = product(3), p5 = product(4);
      left = add8<false>(add8<false>(add8<true>(p4, p5), product(6)), p1);
      right = dual ? add8<false>(p4, product(1)) : add8<false>(p5, product(2));
    } else {
      const F8 p2 = product(1), p3 = product(2), p6 = product(5);
      left = dual ? add8<false>(product(4), p3) : add8<false>(product(3), p2);
      right = dual ? add8<false>(add8<true>(add8<false>(p6, p3), p2), p1)
                   : add8<false>(add8<false>(add8<true>(p6, p2), p3), p1);
    }
  }
}

// p.tiles_m x p.tiles_n tiles of 32 RB x 32 CB, in p.ksplit shares: workgroups
// take the tiles of share 0 first, in column groups of p.group_m tile rows,
// each XCD a contiguous eighth of that order (tiles that run together on
// an XCD share A's rows of one K range and, over several tile rows, B).
//
// kNt: B's fragments are loaded with the streaming cache policy, for launches
// of one tile row, which read every B fragment once: 141 against 154 us on
// 16 x 5120 x 51200 (6.5 against 6.0 TB/s of packed weight; 205 us and
// 4.5 TB/s for 128-row tiles). A fragment that a second workgroup or wave
// reads again must stay in the L2 instead.
template <int kAlgo, int RB, int CB, int kDepth, bool kNt>
__global__ __launch_bounds__((Shape<kAlgo, RB, CB>::kThreads)) void gemm_stream(Params p) {
  using R = Roles<kAlgo>;
  using S = Shape<kAlgo, RB, CB>;
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const int tid = (int)threadIdx.x, lane = tid & 63;
  const int role = __builtin_amdgcn_readfirstlane(tid >> 6);

  const int tiles = p.tiles_m * p.tiles_n;
  const int logical = xcd_order((int)blockIdx.x, tiles * p.ksplit, kRasterSpread);
  const int share = logical / tiles, at = logical - share * tiles;
  const int group = at / (p.group_m * p.tiles_n), first_m = group * p.group_m;
  const int rows_in_group = min(p.tiles_m - first_m, p.group_m);
  const int in_group = at - first_m * p.tiles_n;
  const int tile_m = __builtin_amdgcn_readfirstlane(first_m + in_group % rows_in_group);
  const int tile_n = __builtin_amdgcn_readfirstlane(in_group / rows_in_group);

  const int nstages_all = (int)(p.k / 32);
  const int stage0 = __builtin_amdgcn_readfirstlane((int)((int64_t)share * nstages_all / p.ksplit));
  const int nstages =
      __builtin_amdgcn_readfirstlane((int)((int64_t)(share + 1) * nstages_all / p.ksplit)) - stage0;

  // This wave's operands as buffers that end with the share's last stage:
  // loads of later stages return zeros, which add nothing.
  constexpr uint32_t kStage = R::kOps * kBlocks * kFrag;
  auto panel = [&](const void* base, int block, int op) __attribute__((always_inline)) {
    const uint32_t in_stage = (uint32_t)(op * kBlocks + block % kBlocks) * kFrag;
    return packed::panel_rsrc(reinterpret_cast<const uint8_t*>(base) +
                                  ((int64_t)(block / kBlocks) * nstages_all + stage0) * kStage + in_stage,
                              (uint32_t)nstages * kStage - in_stage);
  };
  constexpr int kP = R::kProducts;
  __amdgpu_buffer_rsrc_t a_src[kP];
#pragma unroll
  for (int x = 0; x < kP; ++x) a_src[x] = panel(p.a, tile_m * RB, R::op_a(role, x));
  const __amdgpu_buffer_rsrc_t b_src = panel(p.b, tile_n * CB, role);
  const uint32_t lane16 = lane * 16;

  struct Frags {
    bf16x8 a[kP][RB], b[CB];
  };
  auto load = [&](Frags& f, int stage) __attribute__((always_inline)) {
    const uint32_t at_stage = (uint32_t)stage * kStage;
#pragma unroll
    for (int c = 0; c < CB; ++c) f.b[c] = load_frag<kNt>(b_src, lane16 + c * kFrag, at_stage);
#pragma unroll
    for (int x = 0; x < kP; ++x)
#pragma unroll
      for (int r = 0; r < RB; ++r) f.a[x][r] = load_frag<false>(a_src[x], lane16 + r * kFrag, at_stage);
  };

  f32x16 acc[kP][RB][CB];
#pragma unroll
  for (int x = 0; x < kP; ++x)
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int c = 0; c < CB; ++c)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[x][r][c][e] = 0.0f;

  Frags f[kDepth];
#pragma unroll
  for (int d = 0; d < kDepth; ++d) load(f[d], d);
  for (int t = 0; t < nstages; t += kDepth) {
#pragma unroll
    for (int d = 0; d < kDepth; ++d) {
#pragma unroll
      for (int x = 0; x < kP; ++x)
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
          for (int c = 0; c < CB; ++c)
            acc[x][r][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[d].a[x][r], f[d].b[c], acc[x][r][c], 0, 0, 0);
      load(f[d], t + d + kDepth);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // Products to LDS (kRG row blocks at a time), then the rows' quadrants and
  // epilogue.
  const ThinRows rows{(uint32_t)(p.bm / 2), (uint32_t)p.bm, (uint32_t)(p.m / 2)};
  const uint32_t hn = (uint32_t)(p.bn / 2);
  const int swap_m = p.perm & 1, swap_n = (p.perm >> 2) & 1;
  uint8_t* const mine = lds + role * kP * S::kSet + (lane >> 5) * 4 * S::kStride + (lane & 31) * 4;
#pragma unroll
  for (int rg = 0; rg < RB / S::kRG; ++rg) {
    if (rg) __syncthreads();
#pragma unroll
    for (int x = 0; x < kP; ++x)
#pragma unroll
      for (int r = 0; r < S::kRG; ++r)
#pragma unroll
        for (int c = 0; c < CB; ++c)
#pragma unroll
          for (int e = 0; e < 16; ++e)
            *reinterpret_cast<float*>(mine + x * S::kSet + (r * 32 + 8 * (e >> 2) + (e & 3)) * S::kStride + c * 128) =
                acc[x][rg * S::kRG + r][c][e];
    __syncthreads();
    // One item per row half, row and eight columns.
    constexpr int kChunks = 4 * CB, kItems = 32 * S::kRG * kChunks;
    for (int item = tid; item < 2 * kItems; item += S::kThreads) {
      const int lr = item / kItems, row = item % kItems / kChunks, ch = item % kChunks;
      const uint32_t prow = (uint32_t)((tile_m * RB + rg * S::kRG) * 32 + row);
      if (!rows.valid(prow)) continue;  // uniform over the lanes of a row
      F8 left, right;
      combine<kAlgo, S::kSet>(lds + row * S::kStride + ch * 32, p.formula, lr, left, right);
      const uint32_t pcol = (uint32_t)(tile_n * CB * 32 + ch * 8);
      const uint32_t tj = pcol / hn, cin = pcol - tj * hn;
      // logical quadrant (row half, column half) is stored at (row half ^
      // swap_m, column half ^ swap_n)
      const int64_t out_row = rows.row(prow, lr ^ swap_m);
      if (p.ksplit > 1) {
        float* const to = reinterpret_cast<float*>(p.park) + (int64_t)share * p.split_stride + out_row * p.n +
                          (int64_t)tj * p.bn + cin;
        store8(to, 1, swap_n ? hn : 0, left);
        store8(to, 1, swap_n ? 0 : hn, right);
      } else if (swap_n) {
        finish_pair(p, p.epilogue, out_row, tj, cin, right, left);
      } else {
        finish_pair(p, p.epilogue, out_row, tj, cin, left, right);
      }
    }
  }
}

// Sums the FP32 [M, N] shares of a K-divided gemm_stream launch in share
// order and finishes the rows: one thread per output row and eight columns
// of both column halves.
__global__ __launch_bounds__(256) void stream_sum(Params p) {
  const uint32_t per_row = (uint32_t)(p.n / 16), hn = (uint32_t)(p.bn / 2);
  const int64_t item = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (item >= p.m * per_row) return;  // whole rows: uniform over a head's lanes
  const int64_t row = item / per_row;
  const uint32_t pcol = (uint32_t)(item - row * per_row) * 8;
  const int64_t tj = pcol / hn, cin = pcol - (uint32_t)tj * hn;
  const float* const from = reinterpret_cast<const float*>(p.park) + row * p.n + tj * p.bn + cin;
  F8 a = load8(from, 1, 0), b = load8(from, 1, hn);
#pragma unroll 4
  for (int h = 1; h < p.ksplit; ++h) {
    const F8 ah = load8(from + h * p.split_stride, 1, 0), bh = load8(from + h * p.split_stride, 1, hn);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      a.v[e] += ah.v[e];
      b.v[e] += bh.v[e];
    }
  }
  finish_pair(p, p.epilogue, row, tj, cin, a, b);
}

}  // namespace stream
}  // namespace smx
