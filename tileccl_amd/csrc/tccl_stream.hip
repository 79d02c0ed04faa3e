// The streaming GEMM's kernels (tccl_stream.h), a translation unit of their own so that they compile beside the others.
#include <hip/hip_runtime.h>

#include "tccl_stream.h"

namespace tccl {

template <typename InT, int kMB, int kNB, int kWaves, bool kBKMajor>
__global__ __launch_bounds__(kWaves * 64, kWaves >= 16 ? 4 : 2) void stream_kernel(StreamArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef StreamGemm<InT, kMB, kNB, kWaves, kBKMajor> Gemm;
  __shared__ __attribute__((aligned(16))) char lds[Gemm::kLdsBytes];
  warm_kernargs<(int)sizeof(StreamArgs)>();
  Gemm(a, lds).run((int)blockIdx.x);
#endif
}

namespace {

template <typename InT, int kShape, bool kBKMajor>
int launch_t(StreamArgs& a, hipStream_t stream) {
  constexpr StreamShape s = kStreamShapes[kShape];
  a.tiles_m = (a.seg_rows + 16 * s.mb - 1) / (16 * s.mb);
  a.tiles_n = (a.N + 16 * s.nb - 1) / (16 * s.nb);
  a.segs = a.M / a.seg_rows;
  a.tiles_m_magic = 0xffffffffu / (uint32_t)a.tiles_m + 1u;
  const int xcds = 1 << a.xcd_shift;
  a.per_xcd = (a.tiles_m * a.tiles_n + xcds - 1) / xcds;
  const StreamGrid grid = stream_grid(a.segs * xcds * a.per_xcd, a.pull.active != 0, a.pull.cus, a.world);
  a.pull.first = grid.first;
  hipLaunchKernelGGL((stream_kernel<InT, s.mb, s.nb, s.waves, kBKMajor>), dim3(grid.wgs), dim3(s.waves * 64), 0, stream, a);
  return (int)hipGetLastError();
}

template <typename InT, bool kBKMajor>
int launch_shape(int shape, StreamArgs& a, hipStream_t stream) {
  static_assert(kStreamShapeCount == 5, "one case per shape");
  switch (shape) {
    case 0: return launch_t<InT, 0, kBKMajor>(a, stream);
    case 1: return launch_t<InT, 1, kBKMajor>(a, stream);
    case 2: return launch_t<InT, 2, kBKMajor>(a, stream);
    case 3: return launch_t<InT, 3, kBKMajor>(a, stream);
    default: return launch_t<InT, 4, kBKMajor>(a, stream);
  }
}

}  // namespace

int launch_stream(int in_dtype, bool b_kmajor, int shape, StreamArgs& a, hipStream_t stream) {
  if (in_dtype == kF8E4M3)
    return b_kmajor ? launch_shape<fp8e4m3, true>(shape, a, stream) : launch_shape<fp8e4m3, false>(shape, a, stream);
  if (in_dtype == kF16)
    return b_kmajor ? launch_shape<_Float16, true>(shape, a, stream) : launch_shape<_Float16, false>(shape, a, stream);
  return b_kmajor ? launch_shape<__bf16, true>(shape, a, stream) : launch_shape<__bf16, false>(shape, a, stream);
}

}  // namespace tccl
