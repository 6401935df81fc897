// The fused epilogues (strassen_pallas.py:739-879) on FP32 results that a
// thread holds as eight consecutive columns of both column halves of one
// output row: the form in which the K split's summing pass and the streaming
// kernel finish their rows.
#pragma once

#include "common.hpp"

namespace smx {

// Applies the epilogue to output row `row`, column tile tj, columns cin ..
// cin + 7 of both column halves (a: the first half, b: the second) and
// stores the result. kEpi and p are the fused call's. For qk_norm_rope the
// eight threads of a head (64 columns of each half, cin 64-aligned on the
// first) are neighbouring lanes, all active.
template <int kEpi>
__device__ __forceinline__ void finish_pair(const Params& p, int64_t row, int64_t tj, int64_t cin, F8 a, F8 b) {
  const int64_t hn = p.bn / 2;
  const int64_t col_a = tj * p.bn + cin, col_b = col_a + hn;
  if constexpr (kEpi == SMX_EPI_SWIGLU || kEpi == SMX_EPI_GEGLU) {
    // gate | up: the tile's first and second column halves
    F8 g;
#pragma unroll
    for (int e = 0; e < 8; ++e) g.v[e] = gate_f32<kEpi>(a.v[e]) * b.v[e];
    store8(p.c, p.out_f32, row * p.ldc + tj * hn + cin, g);
    return;
  }
  if constexpr (kEpi == SMX_EPI_RESIDUAL_ADD) {
    const F8 ra = load8(p.residual, p.residual_f32, row * p.ldr + col_a);
    const F8 rb = load8(p.residual, p.residual_f32, row * p.ldr + col_b);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      a.v[e] += ra.v[e];
      b.v[e] += rb.v[e];
    }
  }
  if constexpr (kEpi == SMX_EPI_BIAS_ADD) {
    // the bias has no alignment requirement: element loads
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      a.v[e] += load_vec(p.bias, p.bias_f32, col_a + e);
      b.v[e] += load_vec(p.bias, p.bias_f32, col_b + e);
    }
  }
  if constexpr (kEpi == SMX_EPI_QK_NORM_ROPE) {
    // A head is 64 columns of each half: eight lanes of a row. recip =
    // rsqrt((sum a^2 + sum b^2) / head_dim + eps) (v_rsq_f32, as in the
    // fused epilogue); a' = (a recip) gamma_a, b' = (b recip) gamma_b; out_a =
    // a' cos - b' sin, out_b = b' cos + a' sin (cos, sin at the output row
    // and the column inside the half).
    const F8 ga = load8(p.rope_scale, p.scale_f32, cin), gb = load8(p.rope_scale, p.scale_f32, hn + cin);
    const float inv_width = 1.0f / (float)p.head_dim;
    float ssa = 0.f, ssb = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      ssa += a.v[e] * a.v[e];
      ssb += b.v[e] * b.v[e];
    }
#pragma unroll
    for (int x = 1; x < 8; x <<= 1) {
      ssa += __shfl_xor(ssa, x);
      ssb += __shfl_xor(ssb, x);
    }
    const float recip = __builtin_amdgcn_rsqf((ssa + ssb) * inv_width + p.eps);
    const F8 cs = unpack8(*reinterpret_cast<const u32x4*>(p.rope_cos + row * hn + cin));
    const F8 sn = unpack8(*reinterpret_cast<const u32x4*>(p.rope_sin + row * hn + cin));
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float na = (a.v[e] * recip) * ga.v[e], nb = (b.v[e] * recip) * gb.v[e];
      a.v[e] = na * cs.v[e] - nb * sn.v[e];
      b.v[e] = nb * cs.v[e] + na * sn.v[e];
    }
  }
  store8(p.c, p.out_f32, row * p.ldc + col_a, a);
  store8(p.c, p.out_f32, row * p.ldc + col_b, b);
}

// The same with the epilogue chosen at run time (uniform over the launch).
__device__ __forceinline__ void finish_pair(const Params& p, int epilogue, int64_t row, int64_t tj, int64_t cin,
                                            const F8& a, const F8& b) {
  switch (epilogue) {
    case SMX_EPI_SWIGLU: return finish_pair<SMX_EPI_SWIGLU>(p, row, tj, cin, a, b);
    case SMX_EPI_GEGLU: return finish_pair<SMX_EPI_GEGLU>(p, row, tj, cin, a, b);
    case SMX_EPI_RESIDUAL_ADD: return finish_pair<SMX_EPI_RESIDUAL_ADD>(p, row, tj, cin, a, b);
    case SMX_EPI_BIAS_ADD: return finish_pair<SMX_EPI_BIAS_ADD>(p, row, tj, cin, a, b);
    case SMX_EPI_QK_NORM_ROPE: return finish_pair<SMX_EPI_QK_NORM_ROPE>(p, row, tj, cin, a, b);
    default: return finish_pair<SMX_EPI_NONE>(p, row, tj, cin, a, b);
  }
}

}  // namespace smx
