// Second pass of a K-split launch (smx_gemm with a workspace): some tiles
// of a packed launch ran as p.ksplit shares of their K stages, each share
// writing its FP32 result into the workspace as one dense 256 x 256 block per
// split tile (dense_share_output). This pass sums the shares in share order
// and applies the epilogue the fused kernels apply
// (strassen_pallas.py:739-879), on the physical output positions.
#pragma once

#include "common.hpp"
#include "finish.hpp"
#include "kernel_packed.hpp"

namespace smx {

// Workgroups per split tile: each takes 32 of the tile's 256 output rows, so
// a pass over r tiles runs 8 r workgroups and keeps enough loads in flight
// to stream at HBM speed.
constexpr int kFixupSlices = 8;

// Workgroup w serves split tile u = w / kFixupSlices (tile tile_base + u of
// the launch's grid): its 128 x 128 product-space block is 128 product rows
// in each output row half by 128 columns of each column half. Thread t takes
// columns 8 (t % 16) .. + 7 of both column halves (the a | b or gate | up
// pair of the epilogues) on rows 32 (w % kFixupSlices) + t / 16 + 16 i,
// i < 2, of the 256. Product row P is output row (P / hm) bm + half hm +
// P % hm (one row tile per product tile unless the tiling is thin); rows
// past M/2 (a thin tiling's padding) are neither read nor written. `ws`
// holds the p.ksplit shares, split_stride floats apart; in a share, split
// tile u's block starts at u * kSplitTileFloats and holds the tile's row
// lr (row half lr / 128) and column half c at lr * 256 + 128 c. p is the
// fused call's Params.
template <int kEpi>
__global__ __launch_bounds__(256) void split_fixup(Params p, const float* __restrict__ ws) {
  const int u = (int)blockIdx.x / kFixupSlices, slice = (int)blockIdx.x % kFixupSlices;
  int tile_m, tile_n;
  tile_of(p.tile_base + u, p.tiles_m, p.tiles_n, p.group_m, p.raster, tile_m, tile_n);
  const TileOrigin o = tile_origin<false>(p, (int64_t)tile_m * packed::TM, (int64_t)tile_n * packed::TN);
  const ThinRows rows{(uint32_t)(p.bm / 2), (uint32_t)p.bm, (uint32_t)(p.m / 2)};
  const uint32_t prow0 = (uint32_t)tile_m * packed::TM;
  const int t = (int)threadIdx.x;
  const int64_t cin = o.tc + (t & 15) * 8;  // column inside a column half
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int lr = 32 * slice + (t >> 4) + 16 * i;  // row half lr / 128, row lr % 128 of the tile
    const uint32_t prow = prow0 + (uint32_t)(lr & 127);
    if (!rows.valid(prow)) continue;  // uniform over the 16 lanes of a row
    const int64_t row = rows.row(prow, lr >> 7);
    const int64_t at = (int64_t)u * kSplitTileFloats + lr * 256 + (t & 15) * 8;
    F8 a = load8(ws, 1, at), b = load8(ws, 1, at + 128);
    for (int h = 1; h < p.ksplit; ++h) {
      const float* const wh = ws + h * p.split_stride;
      const F8 ah = load8(wh, 1, at), bh = load8(wh, 1, at + 128);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        a.v[e] += ah.v[e];
        b.v[e] += bh.v[e];
      }
    }
    finish_pair<kEpi>(p, row, o.tj, cin, a, b);
  }
}

}  // namespace smx
