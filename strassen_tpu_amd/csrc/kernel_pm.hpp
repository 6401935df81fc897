// Product-major Strassen kernel (gfx950): the seven products of a
// 128 x 256 product-space tile run one after another, each over the whole K
// range, into three FP32 accumulator sets instead of seven.
//
// Why: gemm_split keeps the seven products of a 128 x 128 product tile in
// registers for the whole K loop (448 registers per lane), so each 1 KB
// operand fragment it streams from L2 into LDS feeds four MFMAs (of 32 x 32 x
// 16): 512 bytes per MFMA, twice the matched cubic's, which keeps the texture
// address unit (TA, 16 cycles per 64-lane 16-byte load) as busy as the MFMAs.
// Three sets of a 128 x 256 tile are 384 registers per lane; each fragment of
// the tile's four row blocks meets eight column blocks and the other way
// round, 384 bytes for the same work.
//
// The products contribute to the four output quadrants as
//   C0 = P1 + P4 - P5 + P7,  C1 = P3 + P5,  C2 = P2 + P4,  C3 = P1 - P2 + P3 + P6
// (strassen_pallas.py:324-379). No VALU instruction touches an accumulator
// between two products: every combination comes from the MFMA itself, whose
// first instruction of a product may read its C operand from another set of
// the same register file (D = A B + C), and from two FP32 partial sets
// parked in global memory. Sets: V (VGPRs), A1 and A2 (AGPRs); parks q1, q3.
//   P5 -> V          park q1 = V = P5
//   P3 -> V (chain)  V = P3 + P5 = C1
//   P4 -> A1         A1 = P4
//   P1 -> A2 from A1 A2 = P1 + P4;   park q3 = A2 + V = P1 + P3 + P4 + P5
//   P7 -> A2 (chain) A2 = P1 + P4 + P7; row half 0: C0 = A2 - q1, C1 = V
//   P6 -> A2         A2 = P6
//   P2 -> A1 (chain) A1 = P2 + P4 = C2; row half 1: C2 = A1,
//                    C3 = q3 + A2 - q1 - A1 = P1 + P3 + P6 - P2
// V is dead after row half 0, so the second half's epilogue has the VGPRs
// for its parked blocks.
// Each row half's two quadrants (gate | up for SwiGLU / GeGLU) are complete
// together. The parks cost 256 KB written and 384 KB read per tile, against
// about 14 MB of operand fragments at the gate|up shape; each row half's
// epilogue reads its parked blocks two blocks ahead (kParkAhead).
//
// The packed operands are those of gemm_split (packed::Lay<7>): the tile
// reads packed A tile tile_m and packed B tiles 2 tile_n and 2 tile_n + 1,
// one operand (the current product's) per stage.
//
// Waves: wave w owns all 128 product rows and columns 64 w .. + 63 of the
// tile, 8 x 4 blocks of 16 x 16 per set; per 32 k it uses 8 A and 4 B
// fragments (16 x 32) for 32 MFMAs of 16 x 16 x 32, so an A fragment feeds 4 of
// its MFMAs and a B fragment 8. A's fragments are shared by the four waves and
// go through LDS; B's belong to one wave each and go straight into its
// registers. LDS then carries 64 KB of reads and 16 KB of DMA writes per
// 1024 cycles of MFMAs; with both operands in LDS and 64 x 128 waves it was
// 96 and 48 KB, more than its 128 bytes a cycle. Gate|up call (8192 x 5120 x
// 51200, SwiGLU): 3.488 -> 3.364 ms; with the stage addresses kept
// incrementally (Stream) and one wait per half step 3.30. What bounds it now is
// the operand path: on that call's head the data return unit (TD) is busy or
// waiting 98% of the cycles, half of them stalled on the L1, the MFMA pipe busy
// 61% (the cubic 70% and 69%), at a clock of about 1.8 of 2.4 GHz.
//
// Pipeline: a stage is kQ 16-k steps of one product. B is loaded one stage
// ahead (kQ = 8: 2048 cycles of MFMAs), A's ring is refilled kSlots - 1
// stages ahead, and both streams run on across product boundaries, except
// that no B is loaded ahead of an epilogue, which needs its registers. One
// barrier per stage, before its last step's MFMAs: it sees A's next stage
// landed and every wave done reading the stage, whose slot the refill then
// starts on. Each step issues one A DMA and two B loads, each between two
// MFMAs: VMEM operations issued back to back hold back the next MFMA's issue
// (4% on the gate|up launch).
#pragma once

#include "kernel_packed.hpp"

namespace smx {
namespace pm {

using packed::kBlocks;
using packed::kFrag;

constexpr int TM = 128;  // product rows of a tile (one packed A tile)
constexpr int TN = 256;  // product columns (two packed B tiles)
constexpr int kOps = 7;
// One packed 16-k stage of one operand of one packed tile: 4 KB; of all
// seven operands: 28 KB.
constexpr int kOpStage = kBlocks * kFrag;
constexpr int kPackedStage = kOps * kOpStage;
// Pipeline stage: kQ packed 16-k stages ("steps") of one product, 8 (K a
// multiple of 256) or 4. A's steps go through a ring of kSlots stages in
// LDS, refilled kSlots - 1 stages ahead; B's fragments, each read by one
// wave only, go straight into that wave's registers, one stage ahead.
constexpr int kMinSteps = 4;
constexpr int kRingBytes = 128 * 1024;
template <int kQ>
struct Ring {
  static constexpr int kStageBytes = kQ * kOpStage;
  static constexpr int kSlots = kRingBytes / kStageBytes;
  // VMEM operations of one wave and stage: one A DMA and two B loads a step.
  // What a wave may leave in flight at the barrier of stage g, which needs
  // A's stage g + 1: that was issued kSlots - 2 >= 2 stages before g.
  static constexpr int kPending = 3 * kQ;
  static_assert(kSlots >= 4 && kPending < 64, "ring depth and vmcnt range");
};
// Epilogue staging tile of a wave: 32 x 32 floats, each row padded by 16 bytes
// so that the four row groups of an accumulator store (4 rows apart) fall 16
// banks apart. Element e of the 16 x 16 block (i, j) of it, lane part excluded.
struct Tile {
  static constexpr int kRows = 32, kCols = 32;
  static constexpr int kStride = kCols * 4 + 16;
  static constexpr int kBytes = kRows * kStride;
  static constexpr int at(int i, int j, int e) { return (i * 16 + e) * kStride + j * 64; }
  static __device__ __forceinline__ int lane_part(int lane) { return (lane >> 4) * 4 * kStride + (lane & 15) * 4; }
};
constexpr int kLds = kRingBytes + 4 * Tile::kBytes;
static_assert(kLds <= 160 * 1024, "LDS budget");
// One parked set of one workgroup (FP32, 128 x 256), in the registers' lane
// order: [wave][32 blocks of 16 x 16][64 lanes][4 floats]; a workgroup parks
// two.
constexpr int64_t kParkSet = (int64_t)TM * TN * 4;
constexpr int64_t kParkBytes = 2 * kParkSet;

// Product (0-based: P1 = 0) of phase ph, four bits per phase:
// P5 P3 P4 P1 P7 P6 P2.
constexpr uint32_t kOrder = 4u | 2u << 4 | 3u << 8 | 0u << 12 | 6u << 16 | 5u << 20 | 1u << 24;
__host__ __device__ constexpr int product_of(int ph) { return (int)((kOrder >> (4 * ph)) & 15u); }

// A wave's accumulators of one set, 128 rows x 64 columns in 16 x 16 blocks,
// and the operands of half a step: 64 rows and 64 columns of 32 k.
constexpr int kRowBlocks = 8, kColBlocks = 4;
typedef f32x4 Set[kRowBlocks][kColBlocks];

struct FragsA {
  bf16x8 v[kRowBlocks / 2];
};
struct FragsB {
  bf16x8 v[kColBlocks];
};

// File of a set's accumulators: V in VGPRs, A1 and A2 in AGPRs.
constexpr int kV = 0, kA1 = 1, kA2 = 2;
__host__ __device__ constexpr bool in_agprs(int set) { return set != kV; }

// The MFMAs of one 32-k step on row half kHalf of a set, column by column,
// with hook(k) after MFMA k (k = 0..15) between scheduling barriers. kStart 0:
// chain (D = A B + D); 1: the product's first step from zero (D = A B); 2:
// its first step from set `from` of the same file (D = A B + from).
template <int kSet, int kStart, int kHalf, class Hook>
__device__ __forceinline__ void mfma16(Set& acc, const Set& from, const FragsA& a, const FragsB& b, Hook hook) {
#pragma unroll
  for (int j = 0; j < kColBlocks; ++j)
#pragma unroll
    for (int x = 0; x < kRowBlocks / 2; ++x) {
      const int i = kHalf * (kRowBlocks / 2) + x;
      if constexpr (kStart == 0) {
        if constexpr (in_agprs(kSet))
          packed::mfma16_agpr(acc[i][j], a.v[x], b.v[j]);
        else
          packed::mfma16_vgpr(acc[i][j], a.v[x], b.v[j]);
      } else if constexpr (kStart == 1) {
        if constexpr (in_agprs(kSet))
          asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&a"(acc[i][j]) : "v"(a.v[x]), "v"(b.v[j]));
        else
          asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(acc[i][j]) : "v"(a.v[x]), "v"(b.v[j]));
      } else {
        static_assert(in_agprs(kSet), "only the AGPR sets start from another set");
        asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %3"
            : "=&a"(acc[i][j])
            : "v"(a.v[x]), "v"(b.v[j]), "a"(from[i][j]));
      }
      __builtin_amdgcn_sched_barrier(0);
      hook((kRowBlocks / 2) * j + x);
      __builtin_amdgcn_sched_barrier(0);
    }
}

// Wait states past the MFMA result latency, then every accumulator of the
// set is bound (volatile asm, in program order after the s_nops), so no
// read of it moves above them.
template <int kSet>
__device__ __forceinline__ void drain(Set& acc) {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
#pragma unroll
  for (int i = 0; i < kRowBlocks; ++i)
#pragma unroll
    for (int j = 0; j < kColBlocks; ++j) {
      if constexpr (in_agprs(kSet))
        asm volatile("" : "+a"(acc[i][j]));
      else
        asm volatile("" : "+v"(acc[i][j]));
    }
  __builtin_amdgcn_sched_barrier(0);
}

// Parked sets go through a buffer resource over the workgroup's park
// region: a uniform base, the lane's 32-bit byte offset (derived where it is
// used, so no per-lane 64-bit address is held across the main loops) and a
// compile-time offset. Lane l of the 16 x 16 block (i, j) of set x of wave w sits
// at x kParkSet + w kParkSet / 4 + (4 i + j) KB + 16 l.
__device__ __forceinline__ uint32_t park_offset(int set, int wave, int i, int j) {
  return (uint32_t)(set * kParkSet + wave * (kParkSet / 4) + (kColBlocks * i + j) * 1024);
}

// Stores x (plus y, when kAdd) as parked set kSetIdx.
template <int kSetIdx, bool kAdd>
__device__ __forceinline__ void park_store(__amdgpu_buffer_rsrc_t park, int wave, const Set& x, const Set& y) {
  const uint32_t lane16 = opaque_lane_id() * 16;
#pragma unroll
  for (int i = 0; i < kRowBlocks; ++i)
#pragma unroll
    for (int j = 0; j < kColBlocks; ++j) {
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = kAdd ? x[i][j][e] + y[i][j][e] : x[i][j][e];
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), park, lane16,
                                             park_offset(kSetIdx, wave, i, j), 0);
    }
}

// 32 x 32 block (bi, bj) of parked set kSetIdx, as 2 x 2 blocks.
struct Block {
  f32x4 v[2][2];
};
template <int kSetIdx>
__device__ __forceinline__ Block park_block(__amdgpu_buffer_rsrc_t park, int wave, uint32_t lane16, int bi, int bj) {
  Block r;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      r.v[i][j] = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(park, lane16,
                                                       park_offset(kSetIdx, wave, 2 * bi + i, 2 * bj + j), 0));
  return r;
}

// Parked blocks are loaded this many blocks ahead of their use: the parks
// were written long before and come back from beyond the L2. Two ahead
// measured 0.7% faster than one on the gate|up site; three gained nothing
// more, and more spill.
constexpr int kParkAhead = 2;

// Epilogue of logical row half lr. quads(i, j, q1, q3, left, right) yields the
// FP32 values of quadrants (lr, 0) and (lr, 1) of the wave's 16 x 16 block
// (i, j), given that block of the parked sets (q3 only when kParks is 2),
// loaded kParkAhead 32 x 32 blocks ahead. One 32 x 32 block at a time passes
// through the wave's staging tile (strassen_pallas.py:739-792, :867-874):
// SwiGLU / GeGLU store gate(left) * right into [M, N/2]; residual_add and
// bias_add (and no epilogue) store each quadrant. Logical quadrant (row, col)
// is stored at physical (row ^ swap_m, col ^ swap_n) for the block
// permutation (strassen_pallas.py:205-226).
template <int kEpi, int kParks, class Quads>
__device__ __forceinline__ void emit_half(const Params& p, const TileOrigin& o, int wave, int lr,
                                          __amdgpu_buffer_rsrc_t park, Quads quads, uint8_t* tile) {
  using T = Tile;
  constexpr int kBlocksM = kRowBlocks / 2, kBlocksN = kColBlocks / 2, kCount = kBlocksM * kBlocksN;
  const int lane = opaque_lane_id();
  const int64_t hm = p.bm / 2, hn = p.bn / 2;
  const int swap_m = p.perm & 1, swap_n = (p.perm >> 2) & 1;
  const int64_t half = lr ^ swap_m;
  const int es = p.out_f32 ? 4 : 2;
  uint8_t* const te = tile + T::lane_part(lane);
  auto fence = []() __attribute__((always_inline)) { asm volatile("" ::: "memory"); };
  auto at = [&](int i, int j, int e) __attribute__((always_inline)) {
    return reinterpret_cast<float*>(te + T::at(i, j, e));
  };
  const uint32_t lane16 = lane * 16;
  Block pk[kParkAhead + 1][kParks];
  auto fetch = [&](Block (&to)[kParks], int b) __attribute__((always_inline)) {
    to[0] = park_block<0>(park, wave, lane16, b / kBlocksN, b % kBlocksN);
    if constexpr (kParks > 1) to[kParks - 1] = park_block<kParks - 1>(park, wave, lane16, b / kBlocksN, b % kBlocksN);
  };
#pragma unroll
  for (int f = 0; f < kParkAhead; ++f) fetch(pk[f], f);
#pragma unroll
  for (int b = 0; b < kCount; ++b) {
    const int bi = b / kBlocksN, bj = b % kBlocksN;
    if (b + kParkAhead < kCount) fetch(pk[(b + kParkAhead) % (kParkAhead + 1)], b + kParkAhead);
    const Block(&q)[kParks] = pk[b % (kParkAhead + 1)];
    const int64_t row = o.ti * p.bm + o.tr + bi * 32 + half * hm;
    const int64_t cc = o.tc + wave * 64 + bj * 32;  // column inside a column half
    Block left, right;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        quads(2 * bi + i, 2 * bj + j, q[0].v[i][j], q[kParks - 1].v[i][j], left.v[i][j], right.v[i][j]);
    if constexpr (kEpi == SMX_EPI_SWIGLU || kEpi == SMX_EPI_GEGLU) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float gate = swap_n ? right.v[i][j][e] : left.v[i][j][e];
            const float up = swap_n ? left.v[i][j][e] : right.v[i][j][e];
            *at(i, j, e) = gate_f32<kEpi>(gate) * up;
          }
      fence();
      tile_store<T>(tile, reinterpret_cast<char*>(p.c) + (row * p.ldc + o.tj * hn + cc) * es, p.ldc, p.out_f32,
                    lane);
      fence();
    } else {
#pragma unroll
      for (int lc = 0; lc < 2; ++lc) {
        const int64_t col = o.tj * p.bn + cc + (lc ^ swap_n) * hn;
        if constexpr (kEpi == SMX_EPI_RESIDUAL_ADD) {
          const int res = p.residual_f32 ? 4 : 2;
          tile_load<T>(tile, reinterpret_cast<const char*>(p.residual) + (row * p.ldr + col) * res, p.ldr,
                       p.residual_f32, lane);
          fence();
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          float bv = 0.f;
          if constexpr (kEpi == SMX_EPI_BIAS_ADD) bv = load_vec(p.bias, p.bias_f32, col + j * 16 + (lane & 15));
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              float v = lc ? right.v[i][j][e] : left.v[i][j][e];
              if constexpr (kEpi == SMX_EPI_RESIDUAL_ADD) v += *at(i, j, e);
              if constexpr (kEpi == SMX_EPI_BIAS_ADD) v += bv;
              *at(i, j, e) = v;
            }
        }
        fence();
        tile_store<T>(tile, reinterpret_cast<char*>(p.c) + (row * p.ldc + col) * es, p.ldc, p.out_f32, lane);
        fence();
      }
    }
  }
}

template <int kEpi, int kQ>
__global__ __launch_bounds__(kThreads, 1) void gemm_pm(Params p) {
  using R = Ring<kQ>;
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  int tile_m, tile_n;
  tile_of((int)blockIdx.x, p.tiles_m, p.tiles_n, p.group_m, p.raster, tile_m, tile_n);
  tile_m = __builtin_amdgcn_readfirstlane(tile_m);
  tile_n = __builtin_amdgcn_readfirstlane(tile_n);
  const TileOrigin o = tile_origin<false>(p, (int64_t)tile_m * TM, (int64_t)tile_n * TN);

  // Packed 16-k stages over K, and pipeline stages per product (the host
  // takes K a multiple of 32 kQ).
  const int nst16 = (int)(p.k / 32);
  const int nstages = nst16 / kQ;
  // One packed tile's panel (all stages, all operands); B's second tile
  // follows its first. Wave w moves block w of A's steps into LDS and loads
  // its own 64 columns of B: blocks 2 (w % 2) and the next of tile w / 2.
  const uint32_t panel = (uint32_t)nst16 * kPackedStage;
  const __amdgpu_buffer_rsrc_t a_src = packed::panel_rsrc(
      reinterpret_cast<const uint8_t*>(p.a) + (int64_t)tile_m * panel + wave * kFrag, panel - wave * kFrag);
  const uint32_t b_block = (wave & 1) * 2 * kFrag;
  const __amdgpu_buffer_rsrc_t b_src = packed::panel_rsrc(
      reinterpret_cast<const uint8_t*>(p.b) + (int64_t)(2 * tile_n + (wave >> 1)) * panel + b_block, panel - b_block);
  // The workgroup's parked sets q1 and q3.
  const __amdgpu_buffer_rsrc_t park = packed::panel_rsrc(
      reinterpret_cast<const uint8_t*>(p.park) + (int64_t)blockIdx.x * kParkBytes, (uint32_t)kParkBytes);
  uint8_t* const tile = lds + kRingBytes + wave * Tile::kBytes;

  // A stream of stages through the products: `at` is the byte offset of the
  // current stage's first step in a panel. Kept incrementally, so that a VMEM
  // operation between two MFMAs costs one scalar addition and not the
  // address of its step: the wave's other instructions only issue for free in
  // the 12 cycles that an MFMA leaves. Past the last stage it stays there
  // (in bounds, loaded again and never used).
  constexpr uint32_t kStageStep = kQ * kPackedStage;  // to the product's next stage
  struct Stream {
    int ph = 0, s = 0;
    uint32_t at = product_of(0) * kOpStage;
  };
  auto advance = [&](Stream& x) __attribute__((always_inline)) {
    // selects, not branches: the loop stays one block
    const int s1 = x.s + 1;
    const bool wraps = s1 == nstages, ends = x.ph == kOps - 1;
    const int ph = wraps && !ends ? x.ph + 1 : x.ph;
    x.at = wraps ? (ends ? x.at : (uint32_t)product_of(ph) * kOpStage) : x.at + kStageStep;
    x.s = wraps ? (ends ? x.s : 0) : s1;
    x.ph = ph;
  };
  auto dma_a = [&](uint32_t at, int q, int slot, uint32_t lane16) __attribute__((always_inline)) {
    packed::dma_frag(a_src, lane16, at + q * kPackedStage, lds + slot * R::kStageBytes + q * kOpStage + wave * kFrag);
  };
  // Columns 16 j .. of the wave's 64 in 32-k step t of the stage at `at`, and
  // rows 64 h + 16 x .. of A's step q / 2, h = q % 2.
  auto load_b = [&](uint32_t at, int t, int j, uint32_t lane_b) __attribute__((always_inline)) {
    return __builtin_bit_cast(
        bf16x8, __builtin_amdgcn_raw_buffer_load_b128(b_src, lane_b + (j >> 1) * kFrag + (j & 1) * (kFrag / 4),
                                                      at + 2 * t * kPackedStage, 0));
  };
  auto a_base = [&](int slot, uint32_t lane) __attribute__((always_inline)) {
    return lds + slot * R::kStageBytes + packed::half_frag_lane(lane, kOpStage);
  };
  auto read_a = [&](const uint8_t* base, int q, int x) __attribute__((always_inline)) {
    return packed::ld_frag(base + (q & ~1) * kOpStage + (q & 1) * 2 * kFrag + (x >> 1) * kFrag +
                           (x & 1) * (kFrag / 4));
  };
  auto read_a_half = [&](const uint8_t* base, int q) __attribute__((always_inline)) {
    FragsA f;
#pragma unroll
    for (int x = 0; x < kRowBlocks / 2; ++x) f.v[x] = read_a(base, q, x);
    return f;
  };

  Stream da, db;  // A's refill, B's loads
  FragsB b[kQ / 2];
  auto load_stage_b = [&]() __attribute__((always_inline)) {
    const uint32_t lane_b = packed::half_frag_lane(opaque_lane_id(), kPackedStage);
#pragma unroll
    for (int t = 0; t < kQ / 2; ++t)
#pragma unroll
      for (int j = 0; j < kColBlocks; ++j) b[t].v[j] = load_b(db.at, t, j, lane_b);
    advance(db);
  };
  // Prologue: A's stage 0, B's stage 0, A's stages 1 .. kSlots - 2, and the
  // first step of the refill that the stage loop goes on with.
  {
    const uint32_t lane16 = opaque_lane_id() * 16;
#pragma unroll
    for (int st = 0; st < R::kSlots - 1; ++st) {
#pragma unroll
      for (int q = 0; q < kQ; ++q) dma_a(da.at, q, st, lane16);
      advance(da);
      if (st == 0) load_stage_b();
    }
    dma_a(da.at, 0, R::kSlots - 1, lane16);
  }
  packed::stage_barrier<0>();

  Set V, A1, A2;
  int slot = 0;
  FragsA cur = read_a_half(a_base(0, opaque_lane_id()), 0);

  // One pipeline stage of kQ half steps (32 k of 64 rows each): every half's A
  // fragments are read under the half before; behind its MFMAs goes one A DMA
  // of the refill of the slot read at the previous stage (its 16-k steps 1 ..
  // kQ - 1 during the first kQ - 1 halves) and, in a step's second half, as each
  // column's last MFMA has gone, its B fragment of the next stage. Before the
  // last half the barrier: every wave has then read all of this stage's
  // slot, whose refill starts behind it, and A's next stage has landed. kStart
  // applies to the first step (the product's first stage). kLast: an epilogue
  // follows, which needs the registers: nothing is loaded ahead.
  auto stage = [&](auto setc, auto startc, auto lastc, Set& acc, const Set& from) __attribute__((always_inline)) {
    constexpr int kSet = decltype(setc)::value, kStart = decltype(startc)::value;
    constexpr bool kLast = decltype(lastc)::value != 0;
    const int next = slot == R::kSlots - 1 ? 0 : slot + 1;
    const int fill = slot == 0 ? R::kSlots - 1 : slot - 1;
    const uint32_t lane = opaque_lane_id();
    const uint32_t lane16 = lane * 16, lane_b = packed::half_frag_lane(lane, kPackedStage);
    const uint8_t* const base = a_base(slot, lane);
    const uint8_t* const next_base = a_base(next, lane);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      FragsA nxt{};
      // One wait per half for its fragments, in place of one per fragment: A's
      // were read under the last half; a step's B loads have all but the
      // newest stage's operations less its own six behind them (fewer before
      // an epilogue, where the compiler adds what is missing).
      if (q % 2 == 0)
        __builtin_amdgcn_s_waitcnt(packed::waitcnt_imm(3 * kQ - 6, 0));
      else
        __builtin_amdgcn_s_waitcnt(packed::waitcnt_imm(63, 0));
      if (q == kQ - 1) packed::stage_barrier<R::kPending>();
      __builtin_amdgcn_sched_barrier(0);
      FragsB& bt = b[q / 2];
      auto hook = [&](int k) __attribute__((always_inline)) {
        if (k == 1) dma_a(da.at, q < kQ - 1 ? q + 1 : 0, q < kQ - 1 ? fill : slot, lane16);
        if (k >= 4 && k % 2 == 0 && k < 12) {
          const int x = (k - 4) / 2;
          if (q < kQ - 1)
            nxt.v[x] = read_a(base, q + 1, x);
          else if (!kLast)
            nxt.v[x] = read_a(next_base, 0, x);  // past the last stage: a re-loaded copy, unused
        }
        if constexpr (!kLast) {
          if (q % 2 == 1 && k % 4 == 3) bt.v[k / 4] = load_b(db.at, q / 2, k / 4, lane_b);
          if (q == kQ - 1 && k == 15) advance(db);
        }
        if (q == kQ - 2 && k == 14) advance(da);
      };
      if (q == 0)
        mfma16<kSet, kStart, 0>(acc, from, cur, bt, hook);
      else if (q == 1)
        mfma16<kSet, kStart, 1>(acc, from, cur, bt, hook);
      else if (q % 2 == 0)
        mfma16<kSet, 0, 0>(acc, from, cur, bt, hook);
      else
        mfma16<kSet, 0, 1>(acc, from, cur, bt, hook);
      cur = nxt;
    }
    slot = next;
  };
  // One product over all stages into set kSet, its first stage started as
  // kStart says. The products before an epilogue (kLast) are chained ones.
  auto run = [&](auto setc, auto startc, auto lastc, Set& acc, const Set& from) __attribute__((always_inline)) {
    constexpr bool kLast = decltype(lastc)::value != 0;
    if constexpr (kLast) {
      static_assert(decltype(startc)::value == 0, "a product before an epilogue is chained");
      for (int s = 0; s < nstages - 1; ++s) stage(setc, startc, QuadC<0>{}, acc, from);
      stage(setc, startc, QuadC<1>{}, acc, from);
    } else {
      stage(setc, startc, QuadC<0>{}, acc, from);
      for (int s = 1; s < nstages; ++s) stage(setc, QuadC<0>{}, QuadC<0>{}, acc, from);
    }
  };
  using SV = QuadC<kV>;
  using SA1 = QuadC<kA1>;
  using SA2 = QuadC<kA2>;
  using Zero = QuadC<1>;
  using From = QuadC<2>;
  using Chain = QuadC<0>;
  using On = QuadC<0>;
  using Last = QuadC<1>;

  // P5 -> V, parked as q1.
  run(SV{}, Zero{}, On{}, V, V);
  drain<kV>(V);
  park_store<0, false>(park, wave, V, V);
  // The parked stores leave the VMEM count before the next barrier counts
  // refills again.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // P3 chained into V: V = C1.
  run(SV{}, Chain{}, On{}, V, V);
  drain<kV>(V);
  // P4 -> A1.
  run(SA1{}, Zero{}, On{}, A1, A1);
  // P1 -> A2 from A1: A2 = P1 + P4; q3 = A2 + V parked.
  run(SA2{}, From{}, On{}, A2, A1);
  drain<kA2>(A2);
  park_store<1, true>(park, wave, A2, V);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // P7 chained into A2: row half 0, C0 = A2 - q1, C1 = V.
  run(SA2{}, Chain{}, Last{}, A2, A2);
  drain<kA2>(A2);
  emit_half<kEpi, 1>(p, o, wave, 0, park, [&](int i, int j, const f32x4& q1, const f32x4&, f32x4& left, f32x4& right)
                                              __attribute__((always_inline)) {
    left = A2[i][j] - q1;
    right = V[i][j];
  }, tile);
  load_stage_b();
  cur = read_a_half(a_base(slot, opaque_lane_id()), 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // P6 -> A2.
  run(SA2{}, Zero{}, On{}, A2, A2);
  // P2 chained into A1: row half 1, C2 = A1, C3 = q3 + A2 - q1 - A1.
  run(SA1{}, Chain{}, Last{}, A1, A1);
  drain<kA1>(A1);
  drain<kA2>(A2);
  emit_half<kEpi, 2>(p, o, wave, 1, park, [&](int i, int j, const f32x4& q1, const f32x4& q3, f32x4& left, f32x4& right)
                                              __attribute__((always_inline)) {
    left = A1[i][j];
    right = ((q3 + A2[i][j]) - q1) - A1[i][j];
  }, tile);
  // Every wave's DMA (the unread re-loads past the last stage) has landed
  // before the workgroup ends.
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
}

}  // namespace pm
}  // namespace smx
