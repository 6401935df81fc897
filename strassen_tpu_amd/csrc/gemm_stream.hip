// Instantiates and launches the streaming kernels (kernel_stream.hpp).
#include <utility>

#include "kernel_stream.hpp"
#include "launch.hpp"

namespace smx {

// Stages loaded ahead per wave: six or eight measured the same as four.
constexpr int kDepth = 4;

template <int kShape>
static int launch_shape(const Params& p, hipStream_t stream) {
  constexpr StreamShape t = kStreamShape[kShape];
  using S = stream::Shape<t.algo, t.rb, t.cb>;
  auto kern = stream::gemm_stream<t.algo, t.rb, t.cb, kDepth, t.one_row>;
  hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, S::kLds);
  if (e != hipSuccess) return fail(SMX_ERR_LAUNCH, "hipFuncSetAttribute: %s", hipGetErrorString(e));
  hipLaunchKernelGGL(kern, dim3((unsigned)(p.tiles_m * p.tiles_n * p.ksplit)), dim3(S::kThreads), S::kLds, stream, p);
  return check_launch();
}

template <int... kShape>
static int launch_one(const Params& p, int shape, hipStream_t s, std::integer_sequence<int, kShape...>) {
  int rc = SMX_ERR_INVALID;
  ((shape == kShape ? (void)(rc = launch_shape<kShape>(p, s)) : (void)0), ...);
  return rc;
}

int launch_stream(const Params& p, int shape, hipStream_t s) {
  return launch_one(p, shape, s, std::make_integer_sequence<int, kStreamShapes>{});
}

int launch_stream_sum(const Params& p, hipStream_t s) {
  const int64_t items = p.m * (p.n / 16);
  hipLaunchKernelGGL(stream::stream_sum, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, s, p);
  return check_launch();
}

}  // namespace smx
