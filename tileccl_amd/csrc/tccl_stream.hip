// The streaming GEMM's kernels (tccl_stream.h), a translation unit of their own so that they compile beside the others.
#include <hip/hip_runtime.h>

#include "tccl_stream.h"

namespace tccl {

template <typename InT, int kMB, int kNB, int kWaves, bool kBKMajor>
__global__ __launch_bounds__(kWaves * 64, kWaves >= 16 ? 4 : 2) void stream_kernel(StreamArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef StreamGemm<InT, kMB, kNB, kWaves, kBKMajor> Gemm;
  __shared__ __attribute__((aligned(16))) char lds[Gemm::kLdsBytes];
  Gemm(a, lds).run((int)blockIdx.x);
#endif
}

// The same with communication workgroups behind the tiles' (no tile waits for them; they start once every tile
// has been started).
template <typename InT, int kMB, int kNB, int kWaves, bool kBKMajor>
__global__ __launch_bounds__(kWaves * 64, kWaves >= 16 ? 4 : 2) void stream_pull_kernel(StreamArgs a, CommArgs c, int tile_wgs) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef StreamGemm<InT, kMB, kNB, kWaves, kBKMajor> Gemm;
  __shared__ __attribute__((aligned(16))) char lds[Gemm::kLdsBytes];
  if ((int)blockIdx.x < tile_wgs)
    Gemm(a, lds).run((int)blockIdx.x);
  else
    comm_role<kWaves * 64>(c, (int)blockIdx.x - tile_wgs, (int)gridDim.x - tile_wgs, (int*)lds);
#endif
}

namespace {

template <typename InT, int kShape, bool kBKMajor>
int launch_t(StreamArgs& a, const CommArgs* comm, int comm_wgs, hipStream_t stream) {
  constexpr StreamShape s = kStreamShapes[kShape];
  a.tiles_m = (a.seg_rows + 16 * s.mb - 1) / (16 * s.mb);
  a.tiles_n = (a.N + 16 * s.nb - 1) / (16 * s.nb);
  a.segs = a.M / a.seg_rows;
  a.per_xcd = (a.tiles_m * a.tiles_n + a.xcds - 1) / a.xcds;
  const int tile_wgs = a.segs * a.xcds * a.per_xcd;
  const dim3 block(s.waves * 64);
  if (comm)
    hipLaunchKernelGGL((stream_pull_kernel<InT, s.mb, s.nb, s.waves, kBKMajor>), dim3(tile_wgs + comm_wgs), block, 0, stream, a, *comm, tile_wgs);
  else
    hipLaunchKernelGGL((stream_kernel<InT, s.mb, s.nb, s.waves, kBKMajor>), dim3(tile_wgs), block, 0, stream, a);
  return (int)hipGetLastError();
}

template <typename InT, bool kBKMajor>
int launch_shape(int shape, StreamArgs& a, const CommArgs* comm, int comm_wgs, hipStream_t stream) {
  static_assert(kStreamShapeCount == 5, "one case per shape");
  switch (shape) {
    case 0: return launch_t<InT, 0, kBKMajor>(a, comm, comm_wgs, stream);
    case 1: return launch_t<InT, 1, kBKMajor>(a, comm, comm_wgs, stream);
    case 2: return launch_t<InT, 2, kBKMajor>(a, comm, comm_wgs, stream);
    case 3: return launch_t<InT, 3, kBKMajor>(a, comm, comm_wgs, stream);
    default: return launch_t<InT, 4, kBKMajor>(a, comm, comm_wgs, stream);
  }
}

}  // namespace

int launch_stream(int in_dtype, bool b_kmajor, int shape, StreamArgs& a, const CommArgs* comm, int comm_wgs, hipStream_t stream) {
  if (in_dtype == kF8E4M3)
    return b_kmajor ? launch_shape<fp8e4m3, true>(shape, a, comm, comm_wgs, stream) : launch_shape<fp8e4m3, false>(shape, a, comm, comm_wgs, stream);
  if (in_dtype == kF16)
    return b_kmajor ? launch_shape<_Float16, true>(shape, a, comm, comm_wgs, stream) : launch_shape<_Float16, false>(shape, a, comm, comm_wgs, stream);
  return b_kmajor ? launch_shape<__bf16, true>(shape, a, comm, comm_wgs, stream) : launch_shape<__bf16, false>(shape, a, comm, comm_wgs, stream);
}

}  // namespace tccl
