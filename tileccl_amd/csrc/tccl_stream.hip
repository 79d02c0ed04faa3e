// The streaming GEMM's kernels (tccl_stream.h), a translation unit of their own so that they compile beside the others.
#include <hip/hip_runtime.h>

#include "tccl_stream.h"

namespace tccl {

// kPulls: launches with workgroups behind the tiles.  The others run code in which those have no part: with it the tiles'
// scalar registers ran short (they spilled 81 of them to vector lanes, 42 without; 1000 x 1000 x 1024: 9.8 us, 9.3 without).
template <typename InT, int kMB, int kNB, int kWaves, bool kBKMajor, bool kPulls>
__global__ __launch_bounds__(kWaves * 64, kWaves >= 16 ? 4 : 2) void stream_kernel(StreamArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef StreamGemm<InT, kMB, kNB, kWaves, kBKMajor> Gemm;
  __shared__ __attribute__((aligned(16))) char lds[Gemm::kLdsBytes];
  warm_kernargs<(int)sizeof(StreamArgs)>();
  const int slot = (int)blockIdx.x;
  Gemm gemm(a, lds);
  if (kPulls && slot >= a.pull.first)
    gemm.pull(slot);
  else
    gemm.tile(slot);
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
  const dim3 wgs(grid.wgs), threads(s.waves * 64);
  if (a.pull.active)
    hipLaunchKernelGGL((stream_kernel<InT, s.mb, s.nb, s.waves, kBKMajor, true>), wgs, threads, 0, stream, a);
  else
    hipLaunchKernelGGL((stream_kernel<InT, s.mb, s.nb, s.waves, kBKMajor, false>), wgs, threads, 0, stream, a);
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
