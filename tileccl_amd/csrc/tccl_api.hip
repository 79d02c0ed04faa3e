// Host side of libtileccl_hip.so: argument checks, launch geometry, and the extern "C"
// entry points declared in include/tileccl_hip.h.  No Python, no torch types.
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <type_traits>

// The library is built with -fvisibility=hidden: only what the public header declares is exported.
#pragma GCC visibility push(default)
#include "../../include/tileccl_hip.h"
#pragma GCC visibility pop
#include "tccl_bulk.h"
#include "tccl_comm.h"
#include "tccl_gemm.h"
#include "tccl_gemm256.h"
#include "tccl_kernels256.h"
#include "tccl_probe.h"
#include "tccl_staged.h"
#include "tccl_stream.h"

namespace {

using tccl::Fused256Args;

thread_local char g_error[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof g_error, fmt, ap);
  va_end(ap);
  return code;
}

int hip_fail(hipError_t e, const char* what) {
  return fail((int)e, "HIP error in %s: %s (%d)", what, hipGetErrorString(e), (int)e);
}

static_assert(tccl::kArrivalStride == TCCL_ARRIVAL_STRIDE, "the kernel and the interface agree");
#define TCCL_HIP(call)                                  \
  do {                                                  \
    hipError_t e_ = (call);                             \
    if (e_ != hipSuccess) return hip_fail(e_, #call);   \
  } while (0)

struct DeviceCache {
  bool valid = false;
  int device = -1;
  tccl_device_info info;
};
thread_local DeviceCache g_dev;  // per host thread: no lock, no sharing

int query_device(int device, tccl_device_info* out) {
  if (device < 0) TCCL_HIP(hipGetDevice(&device));
  if (!g_dev.valid || g_dev.device != device) {
    hipDeviceProp_t p;
    TCCL_HIP(hipGetDeviceProperties(&p, device));
    tccl_device_info i;
    memset(&i, 0, sizeof i);
    i.compute_units = p.multiProcessorCount;
    i.clock_khz = p.clockRate;
    i.lds_bytes = (int)p.sharedMemPerBlock;
    i.wavefront = p.warpSize;
    strncpy(i.arch, p.gcnArchName, sizeof(i.arch) - 1);
    // MI300/MI350 class parts expose 8 accelerator dies; each owns compute_units / 8 CUs
    // and one L2.  Smaller parts are treated as one die.
    i.xcds = (i.compute_units >= 64 && i.compute_units % 8 == 0) ? 8 : 1;
    g_dev.info = i;
    g_dev.device = device;
    g_dev.valid = true;
  }
  *out = g_dev.info;
  return 0;
}

size_t dtype_size(int dt) {
  switch (dt) {
    case TCCL_F16:
    case TCCL_BF16: return 2;
    case TCCL_F32: return 4;
    case TCCL_F8E4M3: return 1;
    default: return 0;
  }
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// ------------------------------------------------------------------------------------------
// Kernels
// ------------------------------------------------------------------------------------------
// One launch holds both roles: workgroups [0, num_compute) run the GEMM, the rest move
// data.  Three waves per SIMD (two GEMM workgroups plus one communication workgroup per
// CU) bounds the register budget.
// kAColumns, here and below: A is given by columns.  Kernels of their own: the loop for it beside the others takes registers from
// them (10 here, 24 in the deep form; wide form, 1500 x 2240 x 1000 for eight ranks: 28.3 us with it, 28.0 without).
template <typename InT, typename OutT, bool kAColumns>
__global__ __launch_bounds__(256, 3) void fused_kernel(tccl::GemmArgs g, tccl::SignalArgs s, tccl::CommArgs c, tccl::PushArgs push,
                                                       int num_compute, int64_t* trace_start) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(1024))) char stage0[tccl::kStage128];
  __shared__ __attribute__((aligned(1024))) char stage1[tccl::kStage128];
  __shared__ __attribute__((aligned(1024))) char stage2[tccl::kStage128];
  if ((int)blockIdx.x < num_compute) {
    if (trace_start && blockIdx.x == 0 && threadIdx.x == 0) *trace_start = tccl::now_ticks();
    tccl::EpilogueReduce none;
    none.active = 0;
    tccl::GemmRole<InT, OutT>(g, push, none, stage0, stage1, stage2).template run<false, kAColumns>(s, (int)blockIdx.x, num_compute);
  } else {
    tccl::comm_role(c, (int)blockIdx.x - num_compute, (int)gridDim.x - num_compute, (int*)stage0);
  }
#endif
}

// Launches without communication workgroups: the GEMM alone, pushes from the epilogue, reductions in it
// (kReduce).  Nothing has to fit beside two of them on a CU, so they take five stages (80 KiB): a load then has three
// steps and a half to arrive instead of one and a half.  1000 x 2064 x 1008 with its push: 18.3 us with three stages,
// 16.4 with five (traced).
template <typename InT, typename OutT, bool kReduce, bool kAColumns>
__global__ __launch_bounds__(256, 2) void gemm128_kernel(tccl::GemmArgs g, tccl::SignalArgs s, tccl::PushArgs push, tccl::EpilogueReduce reduce) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(1024))) char stage0[tccl::kStage128];
  __shared__ __attribute__((aligned(1024))) char stage1[tccl::kStage128];
  __shared__ __attribute__((aligned(1024))) char stage2[tccl::kStage128];
  __shared__ __attribute__((aligned(1024))) char stage3[tccl::kStage128];
  __shared__ __attribute__((aligned(1024))) char stage4[tccl::kStage128];
  tccl::GemmRole<InT, OutT, 5> role(g, push, reduce, stage0, stage1, stage2, stage3, stage4);
  role.template run<kReduce, kAColumns>(s, (int)blockIdx.x, (int)gridDim.x);
#endif
}

// At most one tile per CU and a K of some length: K steps of 64, four stages of 32 KiB.  Twice the bytes in flight,
// half the barriers, and 128-byte pieces of the rows of A (of a k-major B), which cost less where rows start off a
// 64-byte boundary.  bf16, row-major / k-major B: 2573 x 968 x 3520 41.7 / 42.0 -> 34.3 / 31.8 us, 370 x 5280 x 1656
// 23.0 / 27.6 -> 21.1 / 22.7, 512 x 7168 x 2944 33.7 / 34.2 -> 29.0 / 28.2.
template <typename InT, typename OutT, bool kAColumns>
__global__ __launch_bounds__(256, 1) void gemm128_deep_kernel(tccl::GemmArgs g, tccl::SignalArgs s, tccl::PushArgs push) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(1024))) char stage0[tccl::kStageDeep];
  __shared__ __attribute__((aligned(1024))) char stage1[tccl::kStageDeep];
  __shared__ __attribute__((aligned(1024))) char stage2[tccl::kStageDeep];
  __shared__ __attribute__((aligned(1024))) char stage3[tccl::kStageDeep];
  tccl::EpilogueReduce none;
  none.active = 0;
  tccl::GemmRole<InT, OutT, 4, 4, 2> role(g, push, none, stage0, stage1, stage2, stage3);
  role.template run<false, kAColumns>(s, (int)blockIdx.x, (int)gridDim.x);
#endif
}

// A reduce-scatter of column shards whose peers' partials are there, at most one tile per CU.  A tile of one owner's columns
// leaves all of this rank's sums to the CUs that happen to have its tiles (a quarter of them on four ranks: 196 KiB of
// addends each, 36 us where a reduction of its own behind the GEMM takes 29), and that reduction waits for the whole GEMM, a
// launch and the memory's first answer.  So a sub-tile takes a run of every owner's columns: each CU has 1 / world of its sums
// to make, asks for their addends three K steps before its product is done, and publishes its part of `world` plan tiles.
// bf16, GEMM and reduction before, this after: k-major B 1024 x 4096 x 2048 on 2 / 4 / 8 ranks 31.3 / 30.5 / 30.7 -> 25.6 / 24.7
// / 26.5 us, 512 x 8192 x 1024 23.1 / 22.6 / 22.3 -> 16.8 / 17.1 / 18.8; row-major 1024 x 4096 x 2048 on 2 / 4 31.7 / 30.7 ->
// 26.1 / 27.8, 512 x 8192 x 1024 22.8 / 22.5 -> 17.3 / 19.2.  What bounds it is the operands' way from L2, as in the deep form.
template <typename InT, int kWorld, bool kBKMajor>
__global__ __launch_bounds__(256, 1) void gemm_across_kernel(tccl::GemmArgs g, tccl::SignalArgs s, tccl::EpilogueReduce reduce) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef tccl::GemmRole<InT, float, 4, 4, 2, kWorld, tccl::across_cols(kWorld, kBKMajor) / 64> Role;
  __shared__ __attribute__((aligned(1024))) char stage0[Role::kStage];
  __shared__ __attribute__((aligned(1024))) char stage1[Role::kStage];
  __shared__ __attribute__((aligned(1024))) char stage2[Role::kStage];
  __shared__ __attribute__((aligned(1024))) char stage3[Role::kStage];
  tccl::PushArgs none;
  none.world = 0;
  Role(g, none, reduce, stage0, stage1, stage2, stage3).template run_across<kBKMajor>(s, (int)blockIdx.x, (int)gridDim.x);
#endif
}

// 128 x 256 tiles, eight wavefronts, K steps of 64 in three stages of 48 KiB: a quarter less operand traffic per FLOP
// than two 128 x 128 workgroups on a CU, and half as many tiles to share out.  bf16, row-major / k-major B, against
// those two: 6854 x 520 x 2248 51.2 / 61.0 -> 32.1 / 37.7 us, 534 x 7088 x 2960 60.0 / 72.8 -> 38.8 / 45.7, 1956 x
// 2784 x 2096 43.2 / 51.9 -> 31.2 / 35.7, 1061 x 4432 x 1088 24.5 / 24.0 -> 19.1 / 18.1.
template <typename InT, typename OutT, bool kAColumns>
__global__ __launch_bounds__(512, 2) void gemm_wide_kernel(tccl::GemmArgs g, tccl::SignalArgs s, tccl::PushArgs push) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ __attribute__((aligned(1024))) char stage0[tccl::kStageWide];
  __shared__ __attribute__((aligned(1024))) char stage1[tccl::kStageWide];
  __shared__ __attribute__((aligned(1024))) char stage2[tccl::kStageWide];
  tccl::EpilogueReduce none;
  none.active = 0;
  tccl::GemmRole<InT, OutT, 3, 8, 2> role(g, push, none, stage0, stage1, stage2);
  role.template run<false, kAColumns>(s, (int)blockIdx.x, (int)gridDim.x);
#endif
}

// The transfers that wait for nothing (tccl_bulk.h): blockIdx.y is the rectangle.
__global__ __launch_bounds__(256) void copy_kernel(tccl::BulkCopyArgs a) {
  tccl::bulk_copy<tccl::kThreadsComm>(a, (int)blockIdx.y, (int)blockIdx.x, (int)gridDim.x);
}
template <typename PT, typename OT, int kRanks>
__global__ __launch_bounds__(256) void reduce_kernel(tccl::BulkReduceArgs a) {
  tccl::bulk_reduce<PT, OT, kRanks, tccl::kThreadsComm>(a, a.first_owner + (int)blockIdx.y, (int)blockIdx.x, (int)gridDim.x);
}

// Sums of partials that peers may still be writing.  A waiting workgroup holds what a peer's launch on the same device may need, so
// either at most half of the CUs wait and then add up (two ranks: the other one finds the other half), or one workgroup
// per owner waits in a launch of its own and the launch behind it, which fills the device, only looks at the words and leaves where
// the wait has expired (a fault is raised, nothing is summed): `patience` ticks of waiting, 0 to look.  Loads pass the caches.
constexpr int kThreadsReady = 512;
__global__ __launch_bounds__(kThreadsReady) void rows_wait_kernel(tccl::CommArgs c, int first_owner) {
#if defined(__HIP_DEVICE_COMPILE__)
  tccl::rows_published<kThreadsReady>(c, first_owner + (int)blockIdx.x, tccl::now_ticks() + c.spin_ticks);
#endif
}
template <typename PT, typename OT, int kRanks>
__global__ __launch_bounds__(kThreadsReady) void ready_reduce_kernel(tccl::BulkReduceArgs a, tccl::CommArgs c, int64_t patience) {
#if defined(__HIP_DEVICE_COMPILE__)
  const int owner = a.first_owner + (int)blockIdx.y;
  if (tccl::rows_published<kThreadsReady>(c, owner, tccl::now_ticks() + patience))
    tccl::bulk_reduce<PT, OT, kRanks, kThreadsReady, tccl::kCoherent>(a, owner, (int)blockIdx.x, (int)gridDim.x);
#endif
}

// Staged collectives: workgroup w carries slot w % slots of the (w / slots)-th rank named in a.ranks.
__global__ __launch_bounds__(256) void staged_kernel(tccl::StagedArgs a) {
  __shared__ int word;
  int which = (int)blockIdx.x / a.slots, r = 0;
  for (; r < a.world; ++r)
    if (((a.ranks >> r) & 1u) && which-- == 0) break;
  if (r >= a.world) return;
  const int slot = (int)blockIdx.x % a.slots;
  if (a.dtype == tccl::kF16)
    tccl::staged_role<_Float16>(a, r, slot, &word);
  else if (a.dtype == tccl::kBF16)
    tccl::staged_role<__bf16>(a, r, slot, &word);
  else
    tccl::staged_role<float>(a, r, slot, &word);
}

__global__ void fill_kernel(int32_t* w, int64_t n, int32_t v) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) w[i] = v;
}

// Strided matrices -> dense rows, one 64 x 64 patch per workgroup through LDS: the patch is read along
// whichever source index is closer in memory and written along the destination's rows in 16-byte vectors, so
// both sides move whole lines whatever the source's strides are.  Elements outside the source are written as
// zero.  Both operands of a GEMM are one launch, and a thread's sixteen reads are all requested before the first is
// used: 1000 x 1003 transposed and 1003 x 2064 took 9.8 and 10.4 us one after the other, 5.8 us together.
struct PackJobs {
  tccl_pack_desc job[2];
  int first[2];  // first workgroup of each job
};
template <typename T>
__global__ __launch_bounds__(256) void pack_kernel(PackJobs jobs, int n) {
  constexpr int kVec = 16 / (int)sizeof(T), kPitch = 64 + kVec;
  __shared__ __attribute__((aligned(16))) T patch[64 * kPitch];
  const int which = n > 1 && (int)blockIdx.x >= jobs.first[1] ? 1 : 0;
  const tccl_pack_desc& p = jobs.job[which];
  const int wg = (int)blockIdx.x - jobs.first[which];
  const int across = (p.dst_cols + 63) / 64;
  const int r0 = wg / across * 64, c0 = wg % across * 64;
  const int fast = (int)threadIdx.x & 63, slow = (int)threadIdx.x >> 6;
  const bool along_cols = p.stride_col <= p.stride_row;
  const T* src = (const T*)p.src;
  T v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = along_cols ? slow + 4 * i : fast, c = along_cols ? fast : slow + 4 * i;
    const bool live = r0 + r < p.rows && c0 + c < p.cols;
    v[i] = live ? src[(int64_t)(r0 + r) * p.stride_row + (int64_t)(c0 + c) * p.stride_col] : (T)0;
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = along_cols ? slow + 4 * i : fast, c = along_cols ? fast : slow + 4 * i;
    patch[r * kPitch + c] = v[i];
  }
  __syncthreads();
  T* dst = (T*)p.dst;
  const bool vectors = (((uintptr_t)p.dst | (uint64_t)(p.ld_dst * (int64_t)sizeof(T))) & 15) == 0;
  for (int u = (int)threadIdx.x; u < 64 * (64 / kVec); u += 256) {
    const int r = u / (64 / kVec), c = u % (64 / kVec) * kVec;
    if (r0 + r >= p.dst_rows || c0 + c >= p.dst_cols) continue;
    T* to = dst + (int64_t)(r0 + r) * p.ld_dst + c0 + c;
    if (vectors && c0 + c + kVec <= p.dst_cols) {
      *(tccl::u32x4*)to = *(const tccl::u32x4*)&patch[r * kPitch + c];
    } else {
      for (int e = 0; e < kVec && c0 + c + e < p.dst_cols; ++e) to[e] = patch[r * kPitch + c + e];
    }
  }
}

__global__ void prim_signal_kernel(int32_t* locks, int i) { tccl::tile_signal(locks, i); }
__global__ void prim_signal_add_kernel(int32_t* w, int i, int v, int32_t* res) { *res = tccl::tile_signal_add(w, i, v); }
__global__ void prim_try_wait_kernel(int32_t* locks, int i, int spins, int consume, int32_t* res) {
  *res = tccl::tile_try_wait(locks, i, spins, consume != 0) ? 1 : 0;
}
__global__ void prim_wait_ge_kernel(int32_t* w, int i, int thr, int64_t ticks, int32_t* res) {
  *res = tccl::tile_wait_ge(w, i, thr, tccl::now_ticks() + ticks) ? 1 : 0;
}

// ------------------------------------------------------------------------------------------
// Argument translation
// ------------------------------------------------------------------------------------------
constexpr int64_t kDefaultSpinNs = 2000000000ll;

bool plan_tile_fits_macro(const tccl_gemm_desc* d) {
  return (d->block_m == 128 || d->block_m == 256) && (d->block_n == 128 || d->block_n == 256);
}

// ragged_shards: row blocks of column_shards need not be whole plan tiles.
int check_gemm(const tccl_gemm_desc* d, bool ragged_shards = false) {
  if (!d) return fail(TCCL_ERR_INVALID, "gemm descriptor is NULL");
  if (!d->A || !d->B || !d->C) return fail(TCCL_ERR_INVALID, "gemm: A, B and C must be non-NULL");
  if (d->M <= 0 || d->N <= 0 || d->K <= 0) return fail(TCCL_ERR_INVALID, "gemm: M, N, K must be positive (got %d, %d, %d)", d->M, d->N, d->K);
  if (d->block_m <= 0 || d->block_n <= 0 || d->group_m <= 0) return fail(TCCL_ERR_INVALID, "gemm: block_m, block_n, group_m must be positive");
  if (d->block_m % tccl::kTile || d->block_n % tccl::kTile)
    return fail(TCCL_ERR_UNSUPPORTED, "gemm: plan tile %dx%d must be a multiple of 128x128", d->block_m, d->block_n);
  if (d->macro_tile != 0 && d->macro_tile != 128 && d->macro_tile != 256)
    return fail(TCCL_ERR_INVALID, "gemm: macro_tile=%d must be 0, 128 or 256", d->macro_tile);
  const size_t isz = dtype_size(d->in_dtype), osz = dtype_size(d->out_dtype);
  if (!isz || !osz) return fail(TCCL_ERR_INVALID, "gemm: unknown dtype");
  if (d->in_dtype == TCCL_F32) return fail(TCCL_ERR_UNSUPPORTED, "gemm: fp32 inputs have no MFMA kernel here");
  if (d->in_dtype == TCCL_F8E4M3 && (d->macro_tile == 128 || !plan_tile_fits_macro(d)))
    return fail(TCCL_ERR_UNSUPPORTED, "gemm: fp8 inputs need the 256x256 kernel (macro_tile 0 or 256, plan tile edges 128 or 256)");
  if (d->out_dtype == TCCL_F8E4M3) return fail(TCCL_ERR_UNSUPPORTED, "gemm: fp8 output is not supported");
  const int shards = d->column_shards > 1 ? d->column_shards : 1;
  if (d->column_shards < 0 || d->M % shards || (shards > 1 && !ragged_shards && (d->M / shards) % d->block_m))
    return fail(TCCL_ERR_INVALID, "gemm: column_shards=%d must split M=%d into blocks of whole %d-row plan tiles", d->column_shards, d->M, d->block_m);
  if (d->in_dtype == TCCL_F8E4M3 && shards > 1 && (d->M / shards) % 256)
    return fail(TCCL_ERR_UNSUPPORTED, "gemm: fp8 inputs with column_shards need row blocks of whole 256-row tiles");
  const int in_vec = (int)(16 / isz), out_vec = (int)(16 / osz);
  if (d->K % in_vec) return fail(TCCL_ERR_UNSUPPORTED, "gemm: K=%d must be a multiple of %d", d->K, in_vec);
  if (d->N % 8) return fail(TCCL_ERR_UNSUPPORTED, "gemm: N=%d must be a multiple of 8", d->N);
  const bool b_kmajor = (d->flags & TCCL_GEMM_B_KMAJOR) != 0;
  const int b_short = (d->flags >> TCCL_GEMM_B_SHORT_SHIFT) & 15;
  if (b_short >= in_vec || b_short >= d->K || (b_short && b_kmajor))
    return fail(TCCL_ERR_INVALID, "gemm: B can lack fewer than %d rows of K, and only row-major (%d)", in_vec, b_short);
  const bool a_columns = (d->flags & TCCL_GEMM_A_COLUMNS) != 0;
  const int a_short = (d->flags >> TCCL_GEMM_A_SHORT_SHIFT) & 15;
  if (a_columns && (a_short >= in_vec || a_short >= d->K))
    return fail(TCCL_ERR_INVALID, "gemm: A can lack fewer than %d columns of K where it is given by columns (%d)", in_vec, a_short);
  if (a_columns && (isz != 2 || b_kmajor || shards > 1 || d->macro_tile == 256 || d->M % in_vec))
    return fail(TCCL_ERR_UNSUPPORTED, "gemm: A by columns takes 16-bit inputs, M=%d in whole vectors, a row-major B, no column shards and 128x128 tiles", d->M);
  if (d->lda < (a_columns ? d->M : d->K) || d->ldb < (b_kmajor ? (int64_t)d->K : (int64_t)d->N * shards) || d->ldc < d->N)
    return fail(TCCL_ERR_INVALID, "gemm: leading dimension smaller than the row length");
  if (d->lda % in_vec || d->ldb % in_vec || d->ldc % out_vec || !aligned16(d->A) || !aligned16(d->B) || !aligned16(d->C))
    return fail(TCCL_ERR_UNSUPPORTED, "gemm: A, B, C rows must start on 16-byte boundaries");
  // The kernels address an operand with 32-bit byte offsets from a per-tile base: B from its
  // first row down to row K-1 (k-major B: over the 256 columns of a tile), A and C over the 256 rows of a tile.
  // Offsets from 0xfffffff0 on mean "reads as zero" there; A, a k-major B and 16-bit ones are whole 16-byte vectors and never
  // that long unless they are longer.  An A by columns has nothing but its end to make the columns of the last K step (of 64) zero,
  // so these have to be within reach as well: an offset that goes past 2^32 is one of the first columns'.
  const int64_t limit = 0xffffffffll, operand_limit = 0xfffffff0ll;
  const int64_t b_span = (b_kmajor ? 255 * d->ldb + d->K : (int64_t)(d->K - 1) * d->ldb + (int64_t)d->N * shards) * (int64_t)isz;
  const int64_t a_span = (a_columns ? (((int64_t)d->K + 63) / 64 * 64 - 1) * d->lda + d->M : 255 * d->lda + d->K) * (int64_t)isz;
  const int64_t c_span = (255 * d->ldc + d->N) * (int64_t)osz;
  if (b_span > operand_limit || a_span > operand_limit || c_span > limit)
    return fail(TCCL_ERR_UNSUPPORTED, "gemm: an operand spans more than 4 GiB from a tile's base (B %lld, A %lld, C %lld bytes)",
                (long long)b_span, (long long)a_span, (long long)c_span);
  return 0;
}

int gemm_span(int in_flight, int group_m, int xcds) {
  // Tile ids an XCD takes from each block of xcds * span ids: its share of the tiles in flight, in whole
  // columns of a band (ids run down the group_m rows of a band column, then to the next column), so that
  // the tiles resident on an XCD at one time form a compact patch and share their operand panels in its
  // L2.  What an XCD's L2 misses comes over the fabric, which is what bounds the 128 x 128-tile kernel:
  // with 32 tiles in flight per XCD a patch of 8 x 4 tiles reads 12 panels, one of 8 x 2 twice over 20.
  if (xcds <= 1) return 1;
  int span = in_flight / xcds;
  if (span >= group_m) span = span / group_m * group_m;
  return span > 0 ? span : 1;
}

int build_gemm_args(const tccl_gemm_desc* d, const tccl_device_info& dev, tccl::GemmArgs* g) {
  g->A = d->A;
  g->B = d->B;
  g->C = d->C;
  g->M = d->M;
  g->N = d->N;
  g->K = d->K;
  g->lda = d->lda;
  g->ldb = d->ldb;
  g->ldc = d->ldc;
  g->alpha = d->alpha;
  g->block_m = d->block_m;
  g->block_n = d->block_n;
  g->group_m = d->group_m;
  g->tile_rows = (d->M + d->block_m - 1) / d->block_m;
  g->tile_cols = (d->N + d->block_n - 1) / d->block_n;
  g->xcds = dev.xcds;
  {
    const int total = g->tile_rows * g->tile_cols;
    int wgs = d->num_wgs > 0 ? d->num_wgs : 2 * dev.compute_units;  // default_gemm_wgs()
    g->span = gemm_span(wgs < total ? wgs : total, d->group_m, dev.xcds);
  }
  g->wrap_rows = d->column_shards > 1 ? d->M / d->column_shards : 0;
  g->ragged = 0;
  g->b_kmajor = (d->flags & TCCL_GEMM_B_KMAJOR) ? 1 : 0;
  g->b_short = (d->flags >> TCCL_GEMM_B_SHORT_SHIFT) & 15;
  return 0;
}

int default_gemm_wgs(const tccl_gemm_desc* d, const tccl_device_info& dev, int total_tiles) {
  int n = d->num_wgs > 0 ? d->num_wgs : 2 * dev.compute_units;
  if (n > total_tiles) n = total_tiles;
  return n < 1 ? 1 : n;
}

void fill_comm_common(tccl::CommArgs* c, const tccl::GemmArgs& g, int esize, const tccl_heap_view* heap,
                      const tccl_sync_desc* sync, const tccl_transport_desc* tr) {
  memset(c, 0, sizeof *c);
  c->heap_bases = heap->heap_bases;
  c->rank = heap->rank;
  c->world = heap->world_size;
  c->C = (char*)g.C;
  c->ldc_bytes = g.ldc * esize;
  c->M = g.M;
  c->N = g.N;
  c->esize = esize;
  c->block_m = g.block_m;
  c->block_n = g.block_n;
  c->group_m = g.group_m;
  c->tile_rows = g.tile_rows;
  c->tile_cols = g.tile_cols;
  c->xcds = g.xcds;
  c->span = g.span;
  c->directions = tr ? tr->directions : TCCL_DIR_PUSH;
  c->n_groups = 1;
  c->epoch = 1;
  c->spin_ticks = kDefaultSpinNs / 10;
  if (sync) {
    c->locks = sync->locks;
    c->counter = sync->counter;
    c->barrier = sync->barrier;
    c->row_starts = sync->row_starts;
    c->row_ends = sync->row_ends;
    c->tile_counts = sync->tile_counts;
    if (sync->row_starts && sync->n_groups > 0) c->n_groups = sync->n_groups;
    c->epoch = sync->epoch > 0 ? sync->epoch : 1;
    c->trace_comm_counter = sync->trace_comm_counter;
    c->trace_ready_clock = sync->trace_ready_clock;
    c->trace_done_clock = sync->trace_done_clock;
    c->fault = sync->fault;
    if (sync->spin_limit_ns > 0) c->spin_ticks = sync->spin_limit_ns / 10 + 1;
  }
}

int check_heap(const tccl_heap_view* h) {
  if (!h || !h->heap_bases) return fail(TCCL_ERR_INVALID, "heap view / heap_bases is NULL");
  if (h->world_size < 1 || h->world_size > TCCL_MAX_WORLD) return fail(TCCL_ERR_INVALID, "world_size=%d outside [1, %d]", h->world_size, TCCL_MAX_WORLD);
  if (h->rank < 0 || h->rank >= h->world_size) return fail(TCCL_ERR_INVALID, "rank=%d out of range for world_size=%d", h->rank, h->world_size);
  return 0;
}

// Elements per task of a transport descriptor, checked: whole 16-byte units (reductions: 8 elements).
int task_elems(const tccl_transport_desc* tr, bool reduce) {
  const int elems = tr ? (reduce && tr->reduce_elems > 0 ? tr->reduce_elems : tr->copy_elems) : 0;
  return elems > 0 ? elems : 16384;
}

int check_task_elems(const tccl_transport_desc* tr, bool reduce, int esize) {
  const int elems = task_elems(tr, reduce), unit_elems = reduce ? 8 : 16 / esize;
  if (elems % unit_elems) return fail(TCCL_ERR_UNSUPPORTED, "task size %d elements is not a multiple of %d", elems, unit_elems);
  return 0;
}

int set_task_units(tccl::CommArgs* c, const tccl_transport_desc* tr, bool reduce) {
  const int rc = check_task_elems(tr, reduce, c->esize);
  if (rc) return rc;
  c->copy_units = c->reduce_units = task_elems(tr, reduce) / (reduce ? 8 : 16 / c->esize);
  return 0;
}

int check_sync(const tccl_sync_desc* s, int variant) {
  if (variant == TCCL_S0_BULK) return 0;
  if (!s) return fail(TCCL_ERR_INVALID, "variant S%d needs a sync descriptor", variant);
  if (variant == TCCL_S1_TILE && !s->locks) return fail(TCCL_ERR_INVALID, "S1 needs locks");
  if (s->epoch < 1) return fail(TCCL_ERR_INVALID, "S%d epoch must be >= 1", variant);
  if (variant == TCCL_S2_TILEGROUP) {
    if (!s->counter || !s->group_table || !s->row_starts || !s->row_ends || !s->tile_counts || s->n_groups <= 0)
      return fail(TCCL_ERR_INVALID, "S2 needs counter, group_table, row_starts, row_ends, tile_counts and n_groups > 0");
  }
  return 0;
}

// ------------------------------------------------------------------------------------------
// Launchers
// ------------------------------------------------------------------------------------------
// Kernels for 16-bit inputs, beside the streaming one (tccl_stream.h).  They add products up in the same order: the
// same bits.
enum TileKernel { kTiles128, kTiles128Deep, kTilesWide, kTiles256 };

template <typename InT, typename OutT, bool kAColumns>
void launch_tiles(const tccl::GemmArgs& g, const tccl::SignalArgs& s, const tccl::CommArgs& c, const tccl::PushArgs& push,
                  const tccl::EpilogueReduce& reduce, TileKernel kernel, int compute, int comm, int64_t* trace_start, hipStream_t stream) {
  const dim3 block(tccl::kThreads);
  if (comm > 0 || trace_start)
    hipLaunchKernelGGL((fused_kernel<InT, OutT, kAColumns>), dim3(compute + comm), block, 0, stream, g, s, c, push, compute, trace_start);
  else if (kernel == kTilesWide)
    hipLaunchKernelGGL((gemm_wide_kernel<InT, OutT, kAColumns>), dim3(compute), dim3(tccl::kThreadsWide), 0, stream, g, s, push);
  else if (kernel == kTiles128Deep)
    hipLaunchKernelGGL((gemm128_deep_kernel<InT, OutT, kAColumns>), dim3(compute), block, 0, stream, g, s, push);
  else
    hipLaunchKernelGGL((gemm128_kernel<InT, OutT, false, kAColumns>), dim3(compute), block, 0, stream, g, s, push, reduce);
}

template <typename InT, typename OutT>
int launch_fused_t(const tccl::GemmArgs& g, bool a_columns, const tccl::SignalArgs& s, const tccl::CommArgs& c, const tccl::PushArgs& push,
                   const tccl::EpilogueReduce& reduce, TileKernel kernel, int compute, int comm, int64_t* trace_start, hipStream_t stream) {
  if (reduce.active)  // (A by rows: tccl_gemm_reducescatter)
    hipLaunchKernelGGL((gemm128_kernel<InT, OutT, true, false>), dim3(compute), dim3(tccl::kThreads), 0, stream, g, s, push, reduce);
  else if (a_columns)
    launch_tiles<InT, OutT, true>(g, s, c, push, reduce, kernel, compute, comm, trace_start, stream);
  else
    launch_tiles<InT, OutT, false>(g, s, c, push, reduce, kernel, compute, comm, trace_start, stream);
  TCCL_HIP(hipGetLastError());
  return 0;
}

// `compute` workgroups for the tiles of 128 x 128; the other kernels take what is left of them.
int launch_fused(const tccl_gemm_desc* d, const tccl::GemmArgs& gemm, const tccl::SignalArgs& s, const tccl::CommArgs& c,
                 TileKernel kernel, int compute, int comm, int64_t* trace_start, hipStream_t stream, const tccl::PushArgs* push_args = nullptr,
                 const tccl::EpilogueReduce* reduce_args = nullptr) {
  tccl::PushArgs push;
  memset(&push, 0, sizeof push);
  if (push_args) push = *push_args;
  tccl::EpilogueReduce reduce;
  memset(&reduce, 0, sizeof reduce);
  if (reduce_args) reduce = *reduce_args;
  tccl::GemmArgs g = gemm;
  if (kernel == kTilesWide) {
    const int per = 256 / g.block_n, total = g.tile_rows * ((g.tile_cols + per - 1) / per);
    if (compute > total) compute = total;
    g.span = gemm_span(compute, g.group_m, g.xcds);
  }
  const bool a_columns = (d->flags & TCCL_GEMM_A_COLUMNS) != 0;
  if (a_columns) g.a_short = (d->flags >> TCCL_GEMM_A_SHORT_SHIFT) & 15;
  const int in_dtype = d->in_dtype, out_dtype = d->out_dtype;
  if (in_dtype == TCCL_F16 && out_dtype == TCCL_F16) return launch_fused_t<_Float16, _Float16>(g, a_columns, s, c, push, reduce, kernel, compute, comm, trace_start, stream);
  if (in_dtype == TCCL_F16 && out_dtype == TCCL_F32) return launch_fused_t<_Float16, float>(g, a_columns, s, c, push, reduce, kernel, compute, comm, trace_start, stream);
  if (in_dtype == TCCL_BF16 && out_dtype == TCCL_BF16) return launch_fused_t<__bf16, __bf16>(g, a_columns, s, c, push, reduce, kernel, compute, comm, trace_start, stream);
  if (in_dtype == TCCL_BF16 && out_dtype == TCCL_F32) return launch_fused_t<__bf16, float>(g, a_columns, s, c, push, reduce, kernel, compute, comm, trace_start, stream);
  return fail(TCCL_ERR_UNSUPPORTED, "gemm: no kernel for in_dtype=%d, out_dtype=%d", in_dtype, out_dtype);
}

// ---- large-tile path ----------------------------------------------------------------------------

// 256 x 256 tiles pay off once there are enough of them to occupy most CUs; below that
// the 128 x 128 kernel spreads the work over more workgroups.  With large tiles on exactly half of the CUs
// the GEMM alone is 5-6 % faster on small tiles (2048 x 4096 x 1024: 22.3 against 23.3 us; 4096 x 2048 x 2048:
// 38.1 against 40.6; 96 large tiles: 63.3 against 73.8), from 144 large tiles on it is slower (3072^3: 76.6
// against 58.5 us); the fused launches keep the large tiles there (their transfers ride on the K loops).
bool use_macro(const tccl_gemm_desc* d, const tccl_device_info& dev, bool fused = true) {
  if (d->in_dtype == TCCL_F8E4M3) return true;  // fp8 exists only as the large-tile kernel (check_gemm vets the plan tile)
  if (!plan_tile_fits_macro(d) || (d->flags & TCCL_GEMM_A_COLUMNS)) return false;
  if (d->column_shards > 1 && (d->M / d->column_shards) % 256) return false;  // a tile must not straddle two row blocks
  if (d->macro_tile == 128) return false;
  if (d->macro_tile == 256) return true;
  const int64_t tiles = (int64_t)((d->M + 255) / 256) * ((d->N + 255) / 256);
  return fused ? tiles * 2 >= dev.compute_units : tiles * 2 > dev.compute_units;
}

tccl::Macro build_macro(const tccl_gemm_desc* d, const tccl_device_info& dev, int num_wgs) {
  tccl::Macro m;
  m.rows = (d->M + 255) / 256;
  m.cols = (d->N + 255) / 256;
  const int band_rows = d->group_m * d->block_m / 256;
  m.rows_per_band = band_rows > 0 ? band_rows : 1;
  m.xcds = dev.xcds;
  // Ids an XCD takes from each block: its share of the tiles in flight, in whole band columns.
  const int total = m.rows * m.cols;
  const int in_flight = total < num_wgs ? total : num_wgs;
  int span = in_flight / (dev.xcds > 0 ? dev.xcds : 1);
  span = span / m.rows_per_band * m.rows_per_band;
  m.span = span > 0 ? span : 1;
  m.row_shift = 0;
  return m;
}

int default_macro_wgs(const tccl_gemm_desc* d, const tccl_device_info& dev) {
  const int total = ((d->M + 255) / 256) * ((d->N + 255) / 256);
  int n = d->num_wgs > 0 ? d->num_wgs : dev.compute_units;
  // One workgroup fills a CU, and workgroups of a fused launch wait on each other's tiles
  // after their own: every workgroup must be resident, so the grid never exceeds the CUs.
  if (n > dev.compute_units) n = dev.compute_units;
  if (n > total) n = total;
  return n < 1 ? 1 : n;
}

// ---- the choice among the tiled kernels ------------------------------------------------------------
// Estimated time of a launch, in us beside the launch itself: workgroups take tiles in rounds, a round takes a K
// step's time per 64 k (more of it the more CUs are busy: they share the XCDs' L2s and the part's power) and the
// stores at its end, and rows off a 64-byte boundary cost each step something.
struct TileCost {
  double idle, busy;          // K step with few and with all workgroups at work: idle, idle + busy
  double misaligned;          // added to a step where rows of A or of a k-major B start off 64-byte boundaries
  double stores, stores_busy; // end of a tile
  double pushes;              // and for each tile that goes to peers as well
};
constexpr TileCost kCost256 = {1.05, 0.28, 0.08, 3.0, 4.0, 3.5};   // fitted to its loop of one barrier per step; full launches are up to 12 % quicker now
constexpr TileCost kCostWide = {0.60, 0.25, 0.12, 2.5, 1.5, 3.0};
constexpr TileCost kCostDeep = {0.42, 0.13, 0.12, 2.0, 0.0, 1.5};
constexpr TileCost kCost128 = {0.50, 0.15, 0.12, 0.5, 0.0, 1.5};   // one workgroup per CU
constexpr TileCost kCost128Two = {1.25, 0.0, 0.10, 1.5, 0.0, 1.5}; // two: as soon as some CU has two

double rounds_us(const TileCost& c, int64_t tiles, int slots, const tccl_gemm_desc* d, bool pushes) {
  // (An A given by columns is judged by its pitch as well: the costs were fitted on rows.)
  const bool aligned = d->lda % 32 == 0 && (!(d->flags & TCCL_GEMM_B_KMAJOR) || d->ldb % 32 == 0);
  const double steps = (d->K + 63) / 64, step = c.idle + (aligned ? 0.0 : c.misaligned), end = c.stores + (pushes ? c.pushes : 0.0);
  const double rest = (double)(tiles % slots) / slots;
  double us = (double)(tiles / slots) * (steps * (step + c.busy) + end + c.stores_busy);
  if (rest > 0) us += steps * (step + c.busy * rest) + end + c.stores_busy * rest;
  return us;
}

struct TileChoice {
  TileKernel kernel;
  double us;
};

// The kernel for `segs` row blocks of `seg_rows` rows in a launch that carries nothing but pushes.  Measured, bf16, on 40
// seeded shapes of 100 .. 2200 tiles of 128 x 128, row-major and k-major B: the choice is the quickest kernel or within
// 10 % of it for 73 of the 80, within 25 % for all, 2.6 % off on average; the 128-tile kernel alone would be 25 % off.
// What keeps to the old rule: tiles named by the caller, plan tiles other than 128 x 128, workgroup counts.
TileChoice choose_tiles(const tccl_gemm_desc* d, int64_t seg_rows, int64_t segs, bool allow256, bool pushes, const tccl_device_info& dev) {
  if (d->in_dtype == TCCL_F8E4M3) return {kTiles256, 0};
  if (d->macro_tile != 0 || d->num_wgs > 0 || d->block_m != 128 || d->block_n != 128)
    return {allow256 && use_macro(d, dev, false) ? kTiles256 : kTiles128, 0};
  const int cus = dev.compute_units;
  const int64_t rows = (seg_rows + 127) / 128 * segs, small = rows * ((d->N + 127) / 128), wide = rows * ((d->N + 255) / 256);
  TileChoice best = {kTiles128, small <= cus ? rounds_us(kCost128, small, cus, d, pushes) : rounds_us(kCost128Two, small, 2 * cus, d, pushes)};
  const auto offer = [&](TileKernel kernel, double us) {
    if (us < best.us) best = {kernel, us};
  };
  if (small <= cus) offer(kTiles128Deep, rounds_us(kCostDeep, small, cus, d, pushes));
  if (small > cus) offer(kTilesWide, rounds_us(kCostWide, wide, cus, d, pushes));
  if (allow256 && !(d->flags & TCCL_GEMM_A_COLUMNS) && (segs == 1 || seg_rows % 256 == 0))
    offer(kTiles256, rounds_us(kCost256, (seg_rows + 255) / 256 * segs * ((d->N + 255) / 256), cus, d, pushes));
  return best;
}

int tile_wgs(TileKernel kernel, const tccl_gemm_desc* d, const tccl_device_info& dev, int total_tiles) {
  const int n = default_gemm_wgs(d, dev, total_tiles);
  return kernel != kTiles128 && n > dev.compute_units ? dev.compute_units : n;
}

// Large-tile kernels: B row-major ones are instantiated here, the k-major ones in tccl_kmajor.hip.
int launch_status(int rc, int in_dtype, int out_dtype) {
  if (rc == 0) return 0;
  if (rc == tccl::kNoKernel) return fail(TCCL_ERR_UNSUPPORTED, "gemm: no kernel for in_dtype=%d, out_dtype=%d", in_dtype, out_dtype);
  if (rc == tccl::kGatherTypes) return fail(TCCL_ERR_UNSUPPORTED, "gathered input read in place: output type must equal the input type, B row-major");
  return hip_fail((hipError_t)rc, "large-tile kernel launch");
}

int launch_gemm256(int in_dtype, int out_dtype, const tccl::GemmArgs& g, const tccl::Macro& m, int wgs, hipStream_t stream) {
  const int rc = g.b_kmajor ? tccl::launch_gemm256_kmajor(in_dtype, out_dtype, g, m, wgs, stream)
                            : tccl::launch_gemm256_table<false>(in_dtype, out_dtype, g, m, wgs, stream);
  return launch_status(rc, in_dtype, out_dtype);
}

int launch_fused256(int in_dtype, int out_dtype, const Fused256Args& f, int wgs, hipStream_t stream) {
  const int rc = f.g.b_kmajor ? tccl::launch_fused256_kmajor(in_dtype, out_dtype, f, wgs, stream)
                              : tccl::launch_fused256_table<false>(in_dtype, out_dtype, f, wgs, stream);
  return launch_status(rc, in_dtype, out_dtype);
}

// How the background transfer addresses the 16-byte units of a block (PullArgs::row_units and what follows):
// rows of `upr` units, `pitch` bytes apart on the destination side and `src_pitch` on the source side.  Rows that
// follow each other without gaps on both sides are one long row.  The kernel divides by multiplying:
// u / d = mulhi(u, magic) >> shift with shift = floor(log2 d), magic = ceil(2^(32 + shift) / d), which fits 32
// bits for every d that is not a power of two and is exact for u < 2^31 (the error term u * (magic * d -
// 2^(32 + shift)) stays below 2^(32 + shift)); a power of two is magic = 0 and a plain shift.
void set_row_divider(tccl::PullArgs* p, uint32_t upr, uint32_t pitch, uint32_t src_pitch) {
  const bool flat = pitch == upr * 16u && src_pitch == upr * 16u;
  const uint32_t d = flat ? (p->units > 0 ? p->units : 1u) : upr;
  p->row_units = d;
  p->row_pitch = pitch;
  p->src_row_pitch = src_pitch;
  uint32_t shift = 0;
  while ((2ull << shift) <= d) ++shift;  // floor(log2 d)
  p->row_shift = shift;
  p->row_magic = (d & (d - 1)) == 0 ? 0u : (uint32_t)((((uint64_t)1 << (32 + shift)) + d - 1) / d);
}

// The pull half of a TileGroup all-gather, as the large-tile K loop performs it in the
// background.  Returns false when there is nothing of the kind to do (the communication role
// after the last tile then does it).
bool build_background(const tccl::CommArgs& c, tccl::PullArgs* p) {
  memset(p, 0, sizeof *p);
  if (c.op != tccl::kOpAllGather || !(c.directions & tccl::kDirPull) || c.world <= 1) return false;
  const bool by_tile = c.granularity == tccl::kPerTile;
  int band_shift = 0;
  if (by_tile) {
    // One probe looks at the locks of two plan-tile rows, 32 lanes each; the lock index needs
    // the swizzle band as a shift.
    while ((1 << band_shift) < c.group_m) ++band_shift;
    if (!c.locks || c.tile_cols > 32 || (1 << band_shift) != c.group_m) return false;
  } else if (!c.row_ends || !c.tile_counts || !c.counter) {
    return false;
  }
  const int64_t row_bytes = (int64_t)c.N * c.esize;
  const int64_t block_bytes = (int64_t)c.M * c.ld_out_bytes;
  if (row_bytes % 16 || c.ld_out_bytes % 16 || block_bytes >= (int64_t)1 << 32) return false;
  p->mode = tccl::kBgGather;
  p->slots = c.world - 1;
  p->rank = c.rank;
  p->world = c.world;
  p->heap_bases = c.heap_bases;
  p->src0 = c.out;
  p->block_bytes = block_bytes;
  p->block_rows = c.M;
  p->pitch = (uint32_t)c.ld_out_bytes;
  p->upr = (uint32_t)(row_bytes / 16);
  p->units = (uint32_t)p->block_rows * p->upr;
  p->pieces = (int)((p->units + tccl::kPieceUnits - 1) / tccl::kPieceUnits);
  set_row_divider(p, p->upr, p->pitch, p->pitch);
  p->counter = by_tile ? c.locks : c.counter;
  p->row_ends = c.row_ends;
  p->tile_counts = c.tile_counts;
  p->n_groups = by_tile ? (c.tile_rows + 1) / 2 : c.n_groups;
  p->tile_mode = by_tile ? 1 : 0;
  p->group_m_shift = band_shift;
  p->epoch = c.epoch;
  p->barrier = c.barrier;
  p->trace_done_clock = c.trace_done_clock;
  p->fault = c.fault;
  p->spin_ticks = c.spin_ticks;
  p->word_stride = c.word_stride;
  return true;
}

// Can the large-tile kernel perform the reduction tile by tile?  A tile must not straddle two owners.
bool reduces_in_tiles(const tccl::CommArgs& c) {
  return c.op == tccl::kOpReduceScatter && c.world > 1 && c.M % c.world == 0 && c.M / c.world % tccl::kMacro == 0 &&
         (c.out_dtype == tccl::kF16 || c.out_dtype == tccl::kBF16) && c.ld_rs_out_bytes % 8 == 0;
}

bool build_reduce(const tccl::CommArgs& c, const tccl_sync_desc* sync, int flags, tccl::ReduceArgs* r, tccl::Macro* m) {
  memset(r, 0, sizeof *r);
  if (!reduces_in_tiles(c)) return false;
  const int shard = c.M / c.world;
  r->active = 1;
  r->rank = c.rank;
  r->world = c.world;
  r->emulate_peer = c.emulate_peer;
  r->peers_resident = c.peers_resident;
  r->shard_rows = shard;
  r->out_bf16 = c.out_dtype == tccl::kBF16;
  r->own_in_registers = (flags & TCCL_GEMM_OWN_ROWS_IN_REGISTERS) != 0;
  r->heap_bases = c.heap_bases;
  r->out = c.rs_out;
  r->ld_out = c.ld_rs_out_bytes / 2;
  r->locks = sync->locks;
  r->counter = sync->counter;
  r->tile_counts = sync->tile_counts;
  r->epoch = c.epoch;
  r->fault = c.fault;
  r->spin_ticks = c.spin_ticks;
  m->row_shift = ((c.rank + 1) % c.world) * (shard / tccl::kMacro);  // this rank's own rows come last
  return true;
}

// The push half of an all-scatter / all-gather, as the large-tile epilogue performs it.
// Returns false when the operation has no push to fold (reduce-scatter, push not asked for).
bool build_push(const tccl::CommArgs& c, const tccl::GemmArgs& g, tccl::PushArgs* p) {
  memset(p, 0, sizeof *p);
  if (!(c.directions & tccl::kDirPush) || c.world <= 1) return false;
  if (c.op != tccl::kOpAllScatter && c.op != tccl::kOpAllGather) return false;
  p->world = c.world;
  p->rank = c.rank;
  p->heap_bases = c.heap_bases;  // device memory: only the kernel reads it
  if (c.op == tccl::kOpAllScatter) {
    p->col_lo = c.src_col_off;
    p->col_hi = c.src_col_off + c.cols;
    p->col_shift = c.dst_col_off - c.src_col_off;
    p->ld = c.dst_ld;
  } else {
    p->col_lo = 0;
    p->col_hi = g.N;
    p->col_shift = 0;
    p->ld = g.ldc;
  }
  return true;
}

// The communication code addresses a rectangle (at most all M rows of one block) with 32-bit
// byte offsets from the rectangle's base.
int check_rows_span(int64_t rows, int64_t pitch_bytes) {
  if (rows * pitch_bytes > 0xffffffffll)
    return fail(TCCL_ERR_UNSUPPORTED, "a block of %lld rows of %lld bytes spans more than 4 GiB", (long long)rows,
                (long long)pitch_bytes);
  return 0;
}

int check_comm_span(const tccl::CommArgs& c) {
  int64_t pitch = c.ldc_bytes;
  if (c.ld_out_bytes > pitch) pitch = c.ld_out_bytes;
  if (c.ld_rs_out_bytes > pitch) pitch = c.ld_rs_out_bytes;
  if ((int64_t)c.dst_ld * c.esize > pitch) pitch = (int64_t)c.dst_ld * c.esize;
  return check_rows_span(c.M, pitch);
}

// ---- stand-alone transfers -------------------------------------------------------------------
// Workgroups of a stand-alone kernel, per CU.  Copies: swept on the 128 MiB exchange of the 4096 x 4096 x 1024
// all-gather (2 / 4 / 8 per CU: 20.7 / 20.3 / 19.7 us).
#ifndef TCCL_BULK_COPY_WGS
#define TCCL_BULK_COPY_WGS 8
#endif
#ifndef TCCL_BULK_REDUCE_WGS
#define TCCL_BULK_REDUCE_WGS 8
#endif
constexpr int kReadyReduceWgs = 2;  // of the reductions behind a wait, 512 threads each
// Up to this many bytes read and written half of the CUs are quicker than a launch more (two ranks, whole operation, us, on half of
// the CUs / behind a wait of their own: 1792 x 1200 x 1520 30.7 / 32.0, 1792 x 3408 x 2144 (58 MiB) 49.6 / 51.6, 9472 x 736 x 1120
// (66 MiB) 45.6 / 43.7, 12544 x 3072 x 1024 215.7 / 175.8; with all CUs waiting, which leaves a peer none, 28.5, 47.8, 40.0, 171.7).
constexpr int64_t kWaitInsideBytes = 64ll << 20;
// Units a copying workgroup takes at a time: one 16-byte access per thread while that does not fill the
// device, then more, up to 32 KiB (tasks of 128 KiB took 21.7 us instead of 19.7 on that exchange).
constexpr int kBulkTaskUnits = 2048;

uint32_t all_but(int world, int rank) { return ((1u << world) - 1u) & ~(1u << rank); }

int launch_bulk_copy(tccl::BulkCopyArgs& a, int transfers, int64_t rows, const tccl_device_info& dev, hipStream_t stream) {
  a.units = (int)(rows * a.upr);
  if (a.units <= 0 || transfers <= 0) return 0;
  const int64_t wgs = (int64_t)dev.compute_units * TCCL_BULK_COPY_WGS;
  int64_t task = ((int64_t)a.units * transfers + wgs - 1) / wgs;
  task = (task + tccl::kThreadsComm - 1) / tccl::kThreadsComm * tccl::kThreadsComm;
  if (task > kBulkTaskUnits) task = kBulkTaskUnits;
  a.task_units = (int)task;
  int64_t x = (a.units + task - 1) / task;
  if (x > wgs / transfers) x = wgs / transfers;
  hipLaunchKernelGGL(copy_kernel, dim3((unsigned)x, (unsigned)transfers), dim3(tccl::kThreadsComm), 0, stream, a);
  TCCL_HIP(hipGetLastError());
  return 0;
}

template <typename PT, typename OT>
void launch_reduce_t(const tccl::BulkReduceArgs& a, dim3 grid, int ranks, hipStream_t stream, const tccl::CommArgs* waits, int64_t patience) {
  if (waits) {
    const dim3 block(kThreadsReady);
    if (ranks == 2)
      hipLaunchKernelGGL((ready_reduce_kernel<PT, OT, 2>), grid, block, 0, stream, a, *waits, patience);
    else if (ranks == 4)
      hipLaunchKernelGGL((ready_reduce_kernel<PT, OT, 4>), grid, block, 0, stream, a, *waits, patience);
    else
      hipLaunchKernelGGL((ready_reduce_kernel<PT, OT, 8>), grid, block, 0, stream, a, *waits, patience);
    return;
  }
  const dim3 block(tccl::kThreadsComm);
  if (ranks == 2)
    hipLaunchKernelGGL((reduce_kernel<PT, OT, 2>), grid, block, 0, stream, a);
  else if (ranks == 4)
    hipLaunchKernelGGL((reduce_kernel<PT, OT, 4>), grid, block, 0, stream, a);
  else
    hipLaunchKernelGGL((reduce_kernel<PT, OT, 8>), grid, block, 0, stream, a);
}

int launch_bulk_reduce(tccl::BulkReduceArgs& a, int owners, int64_t rows, int partial_dtype, int out_dtype, const tccl_device_info& dev,
                       hipStream_t stream, const tccl::CommArgs* waits = nullptr, int most_wgs = 0) {
  a.units = (int)(rows * a.upr);
  if (a.units <= 0 || owners <= 0) return 0;
  const int ranks = a.world <= 2 ? 2 : (a.world <= 4 ? 4 : 8);
  const int64_t per_wg = (int64_t)(waits ? kThreadsReady : tccl::kThreadsComm) * (8 / ranks);
  int64_t x = (a.units + per_wg - 1) / per_wg;
  // Two ranks and little to add: half of the CUs wait themselves.
  const int64_t bytes = (int64_t)a.units * 8 * owners * (a.world * (int64_t)dtype_size(partial_dtype) + (int64_t)dtype_size(out_dtype));
  const bool wait_inside = waits && a.world == 2 && bytes <= kWaitInsideBytes;
  int64_t most = !waits ? (int64_t)dev.compute_units * TCCL_BULK_REDUCE_WGS : wait_inside ? dev.compute_units / 2 : (int64_t)dev.compute_units * kReadyReduceWgs;
  if (most_wgs > 0 && most_wgs < most) most = most_wgs;
  most /= owners;
  if (x > most) x = most > 0 ? most : 1;
  const int64_t patience = wait_inside ? waits->spin_ticks : 0;
  if (waits && !wait_inside) hipLaunchKernelGGL(rows_wait_kernel, dim3((unsigned)owners), dim3(kThreadsReady), 0, stream, *waits, a.first_owner);
  const dim3 grid((unsigned)x, (unsigned)owners);
  const int key = partial_dtype * 4 + out_dtype;
  switch (key) {
    case TCCL_F32 * 4 + TCCL_F32: launch_reduce_t<float, float>(a, grid, ranks, stream, waits, patience); break;
    case TCCL_F32 * 4 + TCCL_F16: launch_reduce_t<float, _Float16>(a, grid, ranks, stream, waits, patience); break;
    case TCCL_F32 * 4 + TCCL_BF16: launch_reduce_t<float, __bf16>(a, grid, ranks, stream, waits, patience); break;
    case TCCL_F16 * 4 + TCCL_F16: launch_reduce_t<_Float16, _Float16>(a, grid, ranks, stream, waits, patience); break;
    case TCCL_F16 * 4 + TCCL_BF16: launch_reduce_t<_Float16, __bf16>(a, grid, ranks, stream, waits, patience); break;
    case TCCL_BF16 * 4 + TCCL_BF16: launch_reduce_t<__bf16, __bf16>(a, grid, ranks, stream, waits, patience); break;
    case TCCL_BF16 * 4 + TCCL_F16: launch_reduce_t<__bf16, _Float16>(a, grid, ranks, stream, waits, patience); break;
    default: return fail(TCCL_ERR_UNSUPPORTED, "reduce: no kernel for partial dtype %d, output dtype %d", partial_dtype, out_dtype);
  }
  TCCL_HIP(hipGetLastError());
  return 0;
}

// The transfer of a GEMM + collective operation as a launch of its own (the second kernel of S0).
// waits: the reductions wait for the peers' words.  most_wgs > 0: with at most that many workgroups.
int launch_bulk(const tccl::CommArgs& c, const tccl_device_info& dev, hipStream_t stream, bool waits = false, int most_wgs = 0) {
  const int span = check_comm_span(c);
  if (span) return span;
  if (c.op == tccl::kOpReduceScatter) {
    const int shard = c.M / c.world;
    tccl::BulkReduceArgs a;
    memset(&a, 0, sizeof a);
    a.heap_bases = c.heap_bases;
    a.rank = c.rank;
    a.world = c.world;
    a.src = (int64_t)(uintptr_t)c.C;
    a.dst = (int64_t)(uintptr_t)c.rs_out;
    a.src_shift = shard * c.ldc_bytes;
    a.src_pitch = (uint32_t)c.ldc_bytes;
    a.dst_pitch = (uint32_t)c.ld_rs_out_bytes;
    a.upr = c.N / 8;
    a.first_owner = c.emulate_peer ? 0 : c.rank;
    return launch_bulk_reduce(a, c.emulate_peer ? c.world : 1, shard, c.partial_dtype, c.out_dtype, dev, stream, waits ? &c : nullptr, waits ? most_wgs : 0);
  }
  tccl::BulkCopyArgs a;
  memset(&a, 0, sizeof a);
  a.heap_bases = c.heap_bases;
  a.rank = c.rank;
  a.world = c.world;
  int n = 0;
  if (c.op == tccl::kOpAllScatter) {
    a.src = (int64_t)(uintptr_t)c.C + (int64_t)c.src_col_off * c.esize;
    a.dst = (int64_t)(uintptr_t)c.C + (int64_t)c.dst_col_off * c.esize;
    a.src_pitch = (uint32_t)c.ldc_bytes;
    a.dst_pitch = (uint32_t)((int64_t)c.dst_ld * c.esize);
    a.upr = c.cols * c.esize / 16;
    a.t[n++] = {0, 0, c.rank, all_but(c.world, c.rank)};
  } else {
    a.src = a.dst = (int64_t)(uintptr_t)c.out;
    a.src_pitch = a.dst_pitch = (uint32_t)c.ld_out_bytes;
    a.upr = c.N * c.esize / 16;
    const int64_t block = c.M * c.ld_out_bytes;
    if (c.directions & tccl::kDirPull)
      for (int p = 0; p < c.world; ++p)
        if (p != c.rank) a.t[n++] = {p * block, p * block, p, 1u << c.rank};
    if (c.directions & tccl::kDirPush) a.t[n++] = {c.rank * block, c.rank * block, c.rank, all_but(c.world, c.rank)};
  }
  return launch_bulk_copy(a, n, c.M, dev, stream);
}

// The shards that make up the GEMM's A operand, when the chained operation reads them in place.
struct GatherSpec {
  const void* shard;
  int64_t ld_shard;
  int k_shard;
};

// Can the one-launch variants of the chained operation read the gathered input in place?
// Large-tile kernel, 16-bit inputs and an output of the same type, shards of whole K steps.
bool gather_in_place(const tccl_gemm_desc* d, const tccl_device_info& dev, int k_shard, int variant);

// The background transfer that fills the gathered workspace (gemm->A) while the K loops run.
void build_gather_background(const tccl_gemm_desc* d, const GatherSpec& gs, const tccl_heap_view* heap, const tccl::CommArgs& c,
                             tccl::PullArgs* p, tccl::GatherArgs* ga) {
  const int esz = (int)dtype_size(d->in_dtype);
  memset(ga, 0, sizeof *ga);
  ga->active = 1;
  ga->rank = heap->rank;
  ga->world = heap->world_size;
  ga->heap_bases = heap->heap_bases;
  ga->shard = gs.shard;
  ga->ld_shard = gs.ld_shard;
  ga->k_shard = gs.k_shard;
  memset(p, 0, sizeof *p);
  p->mode = tccl::kBgGatherCols;
  p->slots = heap->world_size;  // every rank's shard, the own one included
  p->rank = heap->rank;
  p->world = heap->world_size;
  p->heap_bases = heap->heap_bases;
  p->block_rows = d->M;
  p->pitch = (uint32_t)(d->lda * esz);
  p->src_pitch = (uint32_t)(gs.ld_shard * esz);
  p->upr = (uint32_t)((int64_t)gs.k_shard * esz / 16);
  p->units = (uint32_t)d->M * p->upr;
  p->pieces = (int)((p->units + tccl::kPieceUnits - 1) / tccl::kPieceUnits);
  set_row_divider(p, p->upr, p->pitch, p->src_pitch);
  p->epoch = 1;
  p->fault = c.fault;
  p->spin_ticks = c.spin_ticks;
}

bool gather_in_place(const tccl_gemm_desc* d, const tccl_device_info& dev, int k_shard, int variant) {
  if (variant == TCCL_S0_BULK || !use_macro(d, dev)) return false;
  if (d->in_dtype != d->out_dtype || (d->in_dtype != TCCL_F16 && d->in_dtype != TCCL_BF16)) return false;
  return k_shard % 64 == 0 && d->column_shards <= 1 && !(d->flags & TCCL_GEMM_B_KMAJOR);
}

// ---- streaming path (tccl_stream.h) -------------------------------------------------------------
// Estimated time of a launch, in us.  A tile's operands pass its CU's vector memory path once, at a rate (KB/us) that
// depends on its shape; a tile's sums take the last term.  The rates measured with 256 tiles, k-major and row-major B, are 72
// and 33, 97 and 73, 97 and 78, 99 and 89, 73 and 50; the constants are those of the kernel's first form and lower, and as only
// their ratios matter among the shapes, they choose the quickest shape or kernel, or one within 10 %, for 39 of 40 forms
// measured (20 shapes of 1 .. 1024 rows, both layouts of B; 32 x 2048 x 4096 row-major: 18 % off) and 19 of 20 of e4m3
// (64 x 4096 x 4096 row-major: 14 % off).  Neither the layout of B nor the variant enters, so that all
// of them add the products up in the same order: the same bits.
struct StreamCost {
  double rate, sums;
};
constexpr StreamCost kStreamCost[tccl::kStreamShapeCount] = {{46, 0.0}, {60, 0.1}, {70, 0.3}, {80, 0.5}, {54, 1.2}};
constexpr double kLaunchUs = 3.7;

int64_t stream_tiles(int shape, int64_t seg_rows, int64_t segs, int64_t N) {
  const int64_t bm = 16 * tccl::kStreamShapes[shape].mb, bn = 16 * tccl::kStreamShapes[shape].nb;
  return (seg_rows + bm - 1) / bm * segs * ((N + bn - 1) / bn);
}

double stream_cost(int shape, int64_t k_bytes, int64_t rounds) {
  const tccl::StreamShape& s = tccl::kStreamShapes[shape];
  return kLaunchUs + (double)rounds * ((double)(16 * (s.mb + s.nb) * k_bytes) / 1024.0 / kStreamCost[shape].rate + kStreamCost[shape].sums);
}

// The 256 x 256-tile kernel with e4m3 inputs: K steps of 128, 1.05 us each, and 1 us (half the CUs storing: 4.5 us) of
// epilogue per tile.  16 .. 2048 x 2048 x 4096 .. 512: within 10 %.
double tile256_f8_cost(int64_t M, int64_t N, int64_t K, int cus) {
  const int64_t tiles = (M + 255) / 256 * ((N + 255) / 256);
  const double load = tiles >= cus / 2 ? 1.0 : (double)tiles / (cus / 2);
  return kLaunchUs + (double)((tiles + cus - 1) / cus) * ((double)((K + 127) / 128) * 1.05 + 1.0 + 3.5 * load);
}

// The 128 x 128-tile kernel: K steps of 32, 0.19 us each with a few tiles and 0.3 us once every CU has one; its fused
// form (three stages instead of five) takes half as long again.  In between, for both.
double tile128_cost(int64_t M, int64_t N, int64_t K, int cus) {
  const int64_t tiles = (M + 127) / 128 * ((N + 127) / 128);
  const double load = tiles >= cus / 2 ? 1.0 : (double)tiles / (cus / 2);
  const double rounds = (double)((tiles + 2 * cus - 1) / (2 * cus));
  return kLaunchUs + rounds * ((double)((K + 31) / 32) * (0.19 + 0.11 * load) * 1.25 + 1.0);
}

// The caller's arrival words, if it has brought any.
uint32_t* arrival_words(const tccl_gemm_desc* d, const tccl_sync_desc* sync) {
  if (!sync || !(d->flags & TCCL_GEMM_ARRIVALS)) return nullptr;
  return (uint32_t*)((const tccl_sync_desc_arrivals*)sync)->arrivals;
}

// The streaming shape to use for this problem, or -1: another kernel is quicker, or the call names things the
// streaming kernel does not have (a tile, workgroup counts, clock stamps).  Signals need the caller's arrival words.
// At most one tile per CU: beyond that the larger tiles are about as quick (1000 x 2064 x 1000 in 528 tiles: 17.5 against
// 13 .. 18 us), and the workgroups of a reduce-scatter that wait for a peer's partials are all resident beside the peer's.
// e4m3 inputs have no 128 x 128-tile kernel to turn to: up to four 64 x 64 tiles per CU (two are resident).
int stream_shape(const tccl_gemm_desc* d, const tccl_sync_desc* sync, const tccl_transport_desc* tr, int variant, int64_t seg_rows,
                 const tccl_device_info& dev) {
  const bool f8 = d->in_dtype == TCCL_F8E4M3;
  if (!f8 && d->out_dtype != TCCL_F32 && d->out_dtype != d->in_dtype) return -1;
  if (d->flags & TCCL_GEMM_A_COLUMNS) return -1;
  if (d->macro_tile != 0 || d->num_wgs > 0 || (tr && tr->num_comm_wgs > 0)) return -1;
  const bool fused = variant != TCCL_S0_BULK;
  if (fused) {
    if (!arrival_words(d, sync)) return -1;
    if (sync->trace_start_clock || sync->trace_ready_clock || sync->trace_done_clock || sync->trace_comm_counter) return -1;
  }
  if (!f8 && use_macro(d, dev, fused)) return -1;
  const int cus = dev.compute_units;
  int best = -1;
  double least = f8 ? tile256_f8_cost(d->M, d->N, d->K, cus) : tile128_cost(d->M, d->N, d->K, cus);
  for (int i = 0; i < tccl::kStreamShapeCount; ++i) {
    const int64_t tiles = stream_tiles(i, seg_rows, d->M / seg_rows, d->N);
    if (tiles > (f8 && i == tccl::kStreamShapeCount - 1 ? 4 * cus : cus)) continue;
    const double us = stream_cost(i, d->K * (f8 ? 1 : 2), (tiles + cus - 1) / cus);
    if (us < least) {
      least = us;
      best = i;
    }
  }
  return best;
}

void build_stream(const tccl_gemm_desc* d, const tccl::GemmArgs& g, int64_t seg_rows, const tccl_device_info& dev, tccl::StreamArgs* a) {
  memset(a, 0, sizeof *a);
  a->A = d->A;
  a->B = d->B;
  a->C = (char*)d->C;
  a->lda = d->lda;
  a->ldb = d->ldb;
  a->ldc = d->ldc;
  a->M = d->M;
  a->N = d->N;
  a->K = d->K;
  a->b_short = g.b_short;
  a->alpha = d->alpha;
  a->out_dtype = d->out_dtype;
  a->seg_rows = (int)seg_rows;
  a->wrapped = g.wrap_rows > 0;
  a->xcd_shift = dev.xcds == 8 ? 3 : 0;  // query_device() knows no others
  a->block_m = g.block_m;
  a->block_n = g.block_n;
  a->group_m = g.group_m;
  a->plan_rows = g.tile_rows;
  a->plan_cols = g.tile_cols;
  a->world = 1;
}

int stream_status(int rc) { return rc == 0 ? 0 : hip_fail((hipError_t)rc, "streaming GEMM launch"); }

// A reduce-scatter carried out in the epilogue.
tccl::EpilogueReduce build_epilogue_reduce(const tccl::CommArgs& c, const tccl_gemm_desc* d) {
  tccl::EpilogueReduce r;
  memset(&r, 0, sizeof r);
  r.active = 1;
  r.emulate_peer = c.emulate_peer;
  r.peers_resident = c.peers_resident;
  r.own_in_registers = (d->flags & TCCL_GEMM_OWN_ROWS_IN_REGISTERS) != 0;
  r.out_dtype = c.out_dtype;
  r.rank = c.rank;
  r.world = c.world;
  r.shard_rows = c.M / c.world;
  r.heap_bases = c.heap_bases;
  r.out = c.rs_out;
  r.ld_out_bytes = c.ld_rs_out_bytes;
  r.locks = c.locks;
  r.counter = c.counter;
  r.tile_counts = c.tile_counts;
  r.fault = c.fault;
  r.spin_ticks = c.spin_ticks;
  return r;
}

bool overlap(const void* a, int64_t a_bytes, const void* b, int64_t b_bytes) {
  const uintptr_t x = (uintptr_t)a, y = (uintptr_t)b;
  return x < y + (uint64_t)b_bytes && y < x + (uint64_t)a_bytes;
}

// May a reduce-scatter of column shards run on sub-tiles across the owners?  Where the 128 x 128-tile kernel of one tile per CU
// would precede a reduction of its own, the peers' partials are there and only this rank's columns are summed.
// Either kernel of one tile per CU: where the costs name the five-stage one, the two are within a tenth of each other, and the
// launch that goes is a fifth to a third of the time.  bf16, K = 200 / 360 / 744, before -> after: row-major 1024 x 4096 on two
// ranks 17.0 / 19.4 / 22.0 -> 11.7 / 12.9 / 15.8 us, on four 16.1 / 17.0 / 20.1 -> 11.5 / 12.5 / 15.8; k-major 1920 x 1504 on two
// 15.1 / 17.4 / 20.7 -> 11.1 / 12.1 / 16.7, 1920 x 1472 on eight 14.7 / 16.6 / 22.6 -> 12.5 / 13.8 / 18.4.
bool sums_across(const tccl_gemm_desc* d, const tccl::CommArgs& c, TileKernel kernel, int tiles, int cus) {
  const bool named = d->macro_tile != 0 || d->num_wgs > 0 || d->block_m != 128 || d->block_n != 128;  // by the caller
  if (kernel != kTiles128Deep && (kernel != kTiles128 || tiles > cus || named)) return false;
  if (d->out_dtype != TCCL_F32 || !c.peers_resident || c.emulate_peer || d->column_shards != c.world) return false;
  if (c.out_dtype != tccl::kF16 && c.out_dtype != tccl::kBF16) return false;
  if (c.ld_rs_out_bytes % 16 || ((uintptr_t)c.rs_out & 15)) return false;
  if (d->K <= 3 * 64) return false;  // the last three K steps are apart, and one goes before them
  const bool kmajor = (d->flags & TCCL_GEMM_B_KMAJOR) != 0;
  // A k-major B costs the same in runs.  A row-major one costs more per K step, on two ranks a tenth, on four (64 x 256) a third, and
  // twice that where its runs of 64 columns start off 64-byte boundaries and take a line more each (less of it where the tiles beside
  // them lose as much by A's rows): up to here the reduction's time pays for it (at the line itself some shapes gain and others lose 3 %).  bf16, GEMM and
  // reduction -> this:
  //   four ranks, whole lines: 1024 x 4096 x 2048 30.5 -> 27.7 us, 2048 x 2048 x 2560 33.1 -> 32.2, 1024 x 4096 x 3072 36.1 -> 36.2
  //   64-byte boundaries: 1920 x 1920 x 1600 27.2 -> 25.7, x 1800 30.5 -> 29.9, x 2048 30.2 -> 30.2; 768 x 2944 x 1600 / 2048 24.0 / 26.9 -> 23.8 / 27.8
  //   off them: 1500 x 2208 x 1024 / 1280 / 1600 22.3 / 24.7 / 26.9 -> 21.4 / 24.3 / 28.0, 1000 x 2592 20.8 / 22.9 / 25.0 -> 20.6 / 23.3 / 26.7
  //   and A's rows too: 1500 x 2208 x 1304 / 1528 / 1800 26.8 / 28.3 / 31.3 -> 25.7 / 28.2 / 31.8, 1000 x 2592 24.8 / 26.4 / 29.0 -> 24.6 / 27.4 / 30.5
  //   two ranks off them: 1500 x 2208 x 4096 / 6144 / 8192 / 16384 44.3 / 60.2 / 75.4 / 136 -> 42.3 / 59.3 / 75.6 / 143; on them x 16384 no loss
  //   four ranks, a device less than half full: 512 x 2048 x 2048 16.9 -> 17.2; eight: 1024 x 4096 x 2048 30.4 -> 43.7
  const bool on64 = ((uintptr_t)d->B & 63) == 0 && d->ldb % 32 == 0 && d->N % 32 == 0;
  int longest = 0;  // K
  if (kmajor ? c.world == 2 || c.world == 4 || c.world == 8 : c.world == 2 && on64)
    longest = INT32_MAX;
  else if (c.world == 2)
    longest = 6144;
  else if (c.world == 4 && 2 * tiles >= cus)
    longest = on64 ? (d->N % 64 == 0 ? 2048 : 1792) : (d->lda % 32 ? 1536 : 1280);
  if (d->K > longest) return false;
  // The first sums are stored while other workgroups still read A and B and store partials: an output that shares memory with them (a
  // square layer in place) is written by a launch behind the GEMM.
  const int64_t rows = d->M / c.world, cols = (int64_t)c.world * d->N, k_rows = d->K - ((d->flags >> TCCL_GEMM_B_SHORT_SHIFT) & 15);
  const int64_t out_bytes = (rows - 1) * c.ld_rs_out_bytes + (int64_t)d->N * 2;
  if (overlap(c.rs_out, out_bytes, d->C, ((int64_t)(d->M - 1) * d->ldc + d->N) * 4)) return false;
  if (overlap(c.rs_out, out_bytes, d->A, ((rows - 1) * d->lda + d->K) * 2)) return false;
  if (overlap(c.rs_out, out_bytes, d->B, (kmajor ? (cols - 1) * d->ldb + d->K : (k_rows - 1) * d->ldb + cols) * 2)) return false;
  // 32-bit offsets that now run over all shards.
  const int64_t limit = 0xfffffff0ll;
  return (kmajor ? (int64_t)c.world * d->N : (int64_t)d->K) * d->ldb * 2 <= limit && (int64_t)d->M * d->ldc * 4 <= limit;
}

template <typename InT>
void launch_across_t(const tccl::GemmArgs& g, const tccl::SignalArgs& s, const tccl::EpilogueReduce& r, int wgs, hipStream_t stream) {
  const dim3 grid(wgs), block(tccl::kThreads);
  if (r.world == 2 && !g.b_kmajor)
    hipLaunchKernelGGL((gemm_across_kernel<InT, 2, false>), grid, block, 0, stream, g, s, r);
  else if (r.world == 2)
    hipLaunchKernelGGL((gemm_across_kernel<InT, 2, true>), grid, block, 0, stream, g, s, r);
  else if (r.world == 4 && !g.b_kmajor)
    hipLaunchKernelGGL((gemm_across_kernel<InT, 4, false>), grid, block, 0, stream, g, s, r);
  else if (r.world == 4)
    hipLaunchKernelGGL((gemm_across_kernel<InT, 4, true>), grid, block, 0, stream, g, s, r);
  else
    hipLaunchKernelGGL((gemm_across_kernel<InT, 8, true>), grid, block, 0, stream, g, s, r);
}

int launch_across(const tccl_gemm_desc* d, const tccl::GemmArgs& gemm, const tccl::SignalArgs& s, const tccl::CommArgs& c, uint32_t* arrivals,
                  hipStream_t stream) {
  tccl::EpilogueReduce r = build_epilogue_reduce(c, d);
  r.arrivals = arrivals;
  tccl::GemmArgs g = gemm;
  const int cols = tccl::across_cols(r.world, g.b_kmajor), rows = 128 * 128 / cols;  // of a sub-tile
  const int total = (g.wrap_rows + rows - 1) / rows * g.tile_cols * (128 * r.world / cols);
  // A patch as high in rows as the other kernels': the XCD that has fewer columns of B fetches less of what costs more (64 x 256,
  // 1024 x 4096 x 2048: bands of 2 / 4 / 8 / 16 sub-tiles 33.6 / 30.2 / 28.9 / 27.5 us).
  r.band = cols == 256 ? 2 * g.group_m : g.group_m;
  g.span = gemm_span(total, r.band, g.xcds);
  if (d->in_dtype == TCCL_F16)
    launch_across_t<_Float16>(g, s, r, total, stream);
  else
    launch_across_t<__bf16>(g, s, r, total, stream);
  TCCL_HIP(hipGetLastError());
  return 0;
}

void add_stream_reduce(const tccl::CommArgs& c, const tccl_gemm_desc* d, tccl::StreamArgs* a) {
  a->heap_bases = c.heap_bases;
  a->rank = c.rank;
  a->world = c.world;
  a->first_seg = (c.rank + 1) % c.world;  // this rank's own rows come last: what its peers wait for comes first
  a->reduce = build_epilogue_reduce(c, d);
}

int run_stream(const tccl_gemm_desc* d, tccl::CommArgs& c, const tccl_sync_desc* sync, int variant, int shape, int64_t seg_rows,
               const tccl_device_info& dev, const tccl::GemmArgs& g, hipStream_t stream) {
  tccl::StreamArgs a;
  build_stream(d, g, seg_rows, dev, &a);
  const bool kmajor = (d->flags & TCCL_GEMM_B_KMAJOR) != 0;
  if (variant == TCCL_S0_BULK) {
    const int rc = stream_status(tccl::launch_stream(d->in_dtype, kmajor, shape, a, stream));
    if (rc || (c.world <= 1 && c.op != tccl::kOpReduceScatter)) return rc;
    return launch_bulk(c, dev, stream);
  }
  a.heap_bases = c.heap_bases;
  a.rank = c.rank;
  a.world = c.world;
  a.arrivals = arrival_words(d, sync);
  a.s.epoch = sync->epoch > 0 ? sync->epoch : 1;
  if (variant == TCCL_S1_TILE) {
    a.s.mode = tccl::kSignalTile;
    a.s.locks = sync->locks;
    c.granularity = tccl::kPerTile;
  } else {
    a.s.mode = tccl::kSignalGroup;
    a.s.counter = sync->counter;
    a.s.group_table = sync->group_table;
    c.granularity = tccl::kPerGroup;
  }
  if (c.op == tccl::kOpReduceScatter) {
    add_stream_reduce(c, d, &a);
    return stream_status(tccl::launch_stream(d->in_dtype, kmajor, shape, a, stream));
  }
  if (build_push(c, g, &a.push)) c.directions &= ~tccl::kDirPush;
  if (c.op != tccl::kOpAllGather || !(c.directions & tccl::kDirPull) || c.world <= 1)
    return stream_status(tccl::launch_stream(d->in_dtype, kmajor, shape, a, stream));
  a.pull.active = 1;
  a.pull.cus = dev.compute_units;
  a.pull.rows = c.M;
  a.pull.pitch = (uint32_t)c.ld_out_bytes;
  a.pull.upr = (uint32_t)((int64_t)c.N * c.esize / 16);
  a.pull.block_bytes = c.M * c.ld_out_bytes;
  a.pull.out = c.out;
  a.pull.words = variant == TCCL_S1_TILE ? c.locks : c.counter;
  a.pull.row_starts = c.row_starts;
  a.pull.row_ends = c.row_ends;
  a.pull.tile_counts = c.tile_counts;
  a.pull.n_groups = c.n_groups;
  a.pull.word_stride = c.word_stride;
  a.pull.fault = c.fault;
  a.pull.spin_ticks = c.spin_ticks;
  return stream_status(tccl::launch_stream(d->in_dtype, kmajor, shape, a, stream));
}

// GEMM (+ optional communication role) for one of the three operations.
int run_variant(const tccl_gemm_desc* d, tccl::CommArgs& c, const tccl_sync_desc* sync, const tccl_transport_desc* tr,
                int variant, const tccl_device_info& dev, const tccl::GemmArgs& g, hipStream_t stream,
                const GatherSpec* gather = nullptr, const tccl_heap_view* heap = nullptr) {
  const int span = c.op != tccl::kOpNone ? check_comm_span(c) : 0;
  if (span) return span;
  const bool traced = sync && (sync->trace_start_clock || sync->trace_ready_clock || sync->trace_done_clock || sync->trace_comm_counter);
  // Reduce-scatter: may the sums be a launch of their own, behind a GEMM that stores and publishes partials?  They are wherever
  // tiles cannot sum themselves (own rows in whole 256-row tiles, or one streaming tile per CU): communication workgroups
  // beside a three-stage GEMM and a large-tile kernel's workgroups turning to the reductions after their tiles, which this
  // launch replaced, took longer.  bf16 1792 x 3408 x 2144 on two ranks 85 -> 48 us, e4m3 13824 x 736 x 2496 on four 86 -> 50,
  // e4m3 512 x 7056 x 1888 on four 75 -> 35 (before the wait made room for a peer on the same device: launch_bulk_reduce()).
  // Measured with all partials in one memory: where a peer's come over a link this gives up the overlap with the GEMM, and the
  // rule has to be measured again.
  const bool apart = c.op == tccl::kOpReduceScatter && variant != TCCL_S0_BULK && c.world > 1 && !traced && !(tr && tr->num_comm_wgs > 0);
  // Own rows that the caller keeps out of memory (a promise of the header) stay in the epilogue of 128-row tiles that wait for their
  // peers, at most one per CU.  (Calls without that flag take the quicker of the two: below.)
  const bool keeps_own = apart && !c.peers_resident && (d->flags & TCCL_GEMM_OWN_ROWS_IN_REGISTERS) && !use_macro(d, dev, true) &&
                         default_gemm_wgs(d, dev, g.tile_rows * g.tile_cols) <= dev.compute_units;
  const auto sums_apart = [&] { return launch_bulk(c, dev, stream, !c.peers_resident, d->num_wgs); };
  if (!gather) {
    // Tiles of a reduce-scatter must not straddle two owners' rows.
    const int64_t seg = g.wrap_rows > 0 ? g.wrap_rows : (c.op == tccl::kOpReduceScatter ? d->M / c.world : d->M);
    const int shape = stream_shape(d, sync, tr, variant, seg, dev);
    // Tiles that wait for a peer (the own rows', the last ones) leave every CU room for the peer's launch.
    const bool waits = c.op == tccl::kOpReduceScatter && variant != TCCL_S0_BULK && !c.peers_resident && c.world > 1;
    if (shape >= 0 && !(waits && stream_tiles(shape, seg, 1, d->N) > dev.compute_units))
      return run_stream(d, c, sync, variant, shape, seg, dev, g, stream);
    if (shape >= 0 && apart) {  // (e4m3: 16-bit inputs take no more streaming tiles than one per CU)
      tccl::CommArgs none = c;
      none.op = tccl::kOpNone;
      const int rc = run_stream(d, none, sync, variant, shape, seg, dev, g, stream);
      c.granularity = none.granularity;
      return rc ? rc : sums_apart();
    }
  }
  // Does the launch carry nothing but pushes?
  const bool lone = !gather && (variant == TCCL_S0_BULK ||
                                (!traced && !(tr && tr->num_comm_wgs > 0) &&
                                 (c.op == tccl::kOpReduceScatter ? apart
                                                                 : c.world <= 1 || c.op != tccl::kOpAllGather || !(c.directions & tccl::kDirPull))));
  // A reduce-scatter on large tiles sums in their epilogue: the rule for launches that carry more decides there.
  const bool sums_inside = variant != TCCL_S0_BULK && use_macro(d, dev, true) && reduces_in_tiles(c) &&
                           !(apart && c.world > 2 && !(d->flags & TCCL_GEMM_OWN_ROWS_IN_REGISTERS));
  TileKernel kernel = use_macro(d, dev, variant != TCCL_S0_BULK) ? kTiles256 : kTiles128;
  if (lone && !sums_inside && !keeps_own) {
    const int segs = d->column_shards > 1 ? d->column_shards : 1;
    kernel = choose_tiles(d, d->M / segs, segs, plan_tile_fits_macro(d), variant != TCCL_S0_BULK && c.op != tccl::kOpReduceScatter && c.world > 1, dev).kernel;
  }
  const int total_tiles = g.tile_rows * g.tile_cols;
  const int compute = tile_wgs(kernel, d, dev, total_tiles);
  tccl::SignalArgs s;
  memset(&s, 0, sizeof s);
  int64_t* trace_start = sync ? sync->trace_start_clock : nullptr;
  if (kernel == kTiles256) {
    const int wgs = default_macro_wgs(d, dev);
    const tccl::Macro m = build_macro(d, dev, wgs);
    if (variant == TCCL_S0_BULK) {
      int rc = launch_gemm256(d->in_dtype, d->out_dtype, g, m, wgs, stream);
      if (rc) return rc;
      if (c.world <= 1 && c.op != tccl::kOpReduceScatter) return 0;
      return launch_bulk(c, dev, stream);
    }
    Fused256Args f;
    f.g = g;
    f.m = m;
    f.trace_start = trace_start;
    s.epoch = sync->epoch > 0 ? sync->epoch : 1;
    if (variant == TCCL_S1_TILE) {
      s.mode = tccl::kSignalTile;
      s.locks = sync->locks;
      c.granularity = tccl::kPerTile;
    } else {
      s.mode = tccl::kSignalGroup;
      s.counter = sync->counter;
      s.group_table = sync->group_table;
      s.tile_counts = sync->tile_counts;
      s.trace_ready_clock = sync->trace_ready_clock;
      c.granularity = tccl::kPerGroup;
    }
    f.s = s;
    // Pushes leave from the epilogue; what remains for the communication role are the
    // pulls (and, for a reduce-scatter, the reductions).
    if (build_push(c, g, &f.push)) c.directions &= ~tccl::kDirPush;
    memset(&f.reduce, 0, sizeof f.reduce);
    memset(&f.gather, 0, sizeof f.gather);
    if (gather) {
      build_gather_background(d, *gather, heap, c, &f.pull, &f.gather);
    } else if (!(apart && !sums_inside) && build_reduce(c, sync, d->flags, &f.reduce, &f.m)) {
      memset(&f.pull, 0, sizeof f.pull);
      c.op = tccl::kOpNone;
    } else if (apart) {
      const int rc = [&] {
        tccl::CommArgs none = c;
        none.op = tccl::kOpNone;
        memset(&f.pull, 0, sizeof f.pull);
        f.comm = none;
        return launch_fused256(d->in_dtype, d->out_dtype, f, wgs, stream);
      }();
      return rc ? rc : sums_apart();
    } else if (build_background(c, &f.pull)) {
      c.directions &= ~tccl::kDirPull;
    }
    if (c.op != tccl::kOpReduceScatter && !(c.directions & (tccl::kDirPush | tccl::kDirPull))) c.op = tccl::kOpNone;
    f.comm = c;
    return launch_fused256(d->in_dtype, d->out_dtype, f, wgs, stream);
  }
  if (variant == TCCL_S0_BULK) {
    tccl::CommArgs none;
    memset(&none, 0, sizeof none);
    int rc = launch_fused(d, g, s, none, kernel, compute, 0, trace_start, stream);
    if (rc) return rc;
    if (c.world <= 1 && c.op != tccl::kOpReduceScatter) return 0;
    return launch_bulk(c, dev, stream);
  }
  int comm = tr && tr->num_comm_wgs > 0 ? tr->num_comm_wgs : dev.compute_units;
  s.epoch = sync->epoch > 0 ? sync->epoch : 1;
  if (variant == TCCL_S1_TILE) {
    s.mode = tccl::kSignalTile;
    s.locks = sync->locks;
    c.granularity = tccl::kPerTile;
  } else {
    s.mode = tccl::kSignalGroup;
    s.counter = sync->counter;
    s.group_table = sync->group_table;
    c.granularity = tccl::kPerGroup;
  }
  // Pushes leave from the GEMM's epilogue (the tile goes to the peers from the registers it is stored from and
  // is never read back); what remains for the communication workgroups are pulls and reductions.  A traced
  // launch keeps the pushes in the communication role, whose tasks carry the per-group clock stamps.
  tccl::PushArgs push;
  memset(&push, 0, sizeof push);
  // Two ranks, at most a tile per CU, few K steps: the second launch costs more than 128-row tiles lose that sum in their
  // epilogue (bf16, us, in the epilogue and apart: 4352 x 752 x 336 21.3 / 22.9, 3328 x 800 x 640 22.9 / 24.6, 2560 x 1536 x
  // 1024 27.0 / 28.3; 2048 x 1408 x 1280 29.0 / 28.1, 1792 x 1200 x 1520 31.4 / 30.5, 1280 x 3136 x 3968 51.7 / 49.4).
  if (keeps_own || (apart && !c.peers_resident && c.world == 2 && compute <= dev.compute_units && kernel != kTilesWide && d->K <= 1024)) {
    const tccl::EpilogueReduce r = build_epilogue_reduce(c, d);
    return launch_fused(d, g, s, c, kTiles128, compute, 0, nullptr, stream, nullptr, &r);
  }
  if (apart && arrival_words(d, sync) && sums_across(d, c, kernel, total_tiles, dev.compute_units))
    return launch_across(d, g, s, c, arrival_words(d, sync), stream);
  if (apart) {
    const int rc = launch_fused(d, g, s, c, kernel, compute, 0, nullptr, stream);
    return rc ? rc : sums_apart();
  }
  if (!traced && build_push(c, g, &push)) {
    c.directions &= ~tccl::kDirPush;
    if (c.op != tccl::kOpReduceScatter && !(c.directions & tccl::kDirPull)) comm = 0;
  }
  return launch_fused(d, g, s, c, kernel, compute, comm, trace_start, stream, &push);
}


// GEMM-output AllGather.  word_stride: 0 when the ranks' signal words live in the heap (a
// peer's at the same slice offset), else the distance between consecutive ranks' words.
int allgather_impl(const tccl_gemm_desc* d, void* out, int64_t ld_out, const tccl_heap_view* heap, const tccl_sync_desc* sync,
                   const tccl_transport_desc* tr, int32_t variant, int64_t word_stride, hipStream_t stream) {
  int rc = check_gemm(d);
  if (rc) return rc;
  if ((rc = check_heap(heap))) return rc;
  if (variant < TCCL_S0_BULK || variant > TCCL_S2_TILEGROUP) return fail(TCCL_ERR_INVALID, "unknown variant %d", variant);
  if ((rc = check_sync(sync, variant))) return rc;
  if (!out) return fail(TCCL_ERR_INVALID, "allgather: out is NULL");
  const int esize = (int)dtype_size(d->out_dtype);
  if (ld_out != d->ldc) return fail(TCCL_ERR_INVALID, "allgather: ld_out must equal the GEMM's ldc");
  const char* want = (const char*)out + (int64_t)heap->rank * d->M * ld_out * esize;
  if ((const char*)d->C != want) return fail(TCCL_ERR_INVALID, "allgather: gemm C must point at row rank*M of out");
  if ((d->N * esize) % 16 || (ld_out * esize) % 16) return fail(TCCL_ERR_UNSUPPORTED, "allgather: rows must be multiples of 16 bytes");
  if (tr && !(tr->directions & (TCCL_DIR_PUSH | TCCL_DIR_PULL))) return fail(TCCL_ERR_INVALID, "allgather: no transfer direction selected");
  tccl_device_info dev;
  if ((rc = query_device(-1, &dev))) return rc;
  tccl::GemmArgs g;
  build_gemm_args(d, dev, &g);
  tccl::CommArgs c;
  fill_comm_common(&c, g, esize, heap, sync, tr);
  c.op = tccl::kOpAllGather;
  c.out = (char*)out;
  c.ld_out_bytes = ld_out * esize;
  c.word_stride = word_stride;
  if ((rc = set_task_units(&c, tr, false))) return rc;
  return run_variant(d, c, sync, tr, variant, dev, g, stream);
}

// ---- signal words that the library keeps itself (tccl_gemm_allgather_static) --------------------
// One rank's words, then the next rank's: a peer's words are a fixed distance away.
struct StaticWords {
  int32_t locks[TCCL_STATIC_MAX_TILES];
  int32_t counter[TCCL_STATIC_MAX_GROUPS];
  int32_t barrier[TCCL_STATIC_MAX_GROUPS];
};
struct StaticScratch {
  int32_t group_table[TCCL_STATIC_MAX_TILES];
  int32_t row_starts[TCCL_STATIC_MAX_GROUPS];
  int32_t row_ends[TCCL_STATIC_MAX_GROUPS];
  int32_t tile_counts[TCCL_STATIC_MAX_GROUPS];
  StaticWords words[TCCL_MAX_WORLD];
};
// Device memory that exists from the moment the library is loaded: about 581 KiB on every
// GPU the process uses.  In host code this name is only a handle for hipGetSymbolAddress; the
// address kernels and copies may use is the one static_scratch() returns.
static __device__ __align__(256) unsigned char scratch[sizeof(StaticScratch)];

constexpr int kMaxDevices = 64;
StaticScratch* g_scratch_ptr[kMaxDevices];  // per device, resolved on first use
// Calls of tccl_gemm_allgather_static so far, per device and rank (host memory: nothing is allocated).
// Call n of a rank stores n into its locks and brings each of its TileGroup counters to n * kStaticGroupUnit,
// so what call n - 1 left behind (or what a call with another plan left) never satisfies a peer that is in
// its own call n: the guarantee tccl_gemm_allgather gets from the caller's growing launch numbers.
uint32_t g_static_calls[kMaxDevices][TCCL_MAX_WORLD];
std::mutex g_scratch_mutex;
// What every TileGroup counter of the static words grows to per call, whatever the group's tile count (the
// set-up kernel starts the counter that many tiles short of the next multiple): more than any group can hold.
constexpr int32_t kStaticGroupUnit = 2 * TCCL_STATIC_MAX_TILES;

void static_call_words(uint32_t call, int32_t tile_count, int32_t* epoch, int32_t* counter_start, int32_t* counter_ready) {
  const uint32_t n = (call - 1u) % 0x7fffffffu + 1u;  // 1 .. 2^31 - 1, then 1 again: a lock value is a positive int32
  const uint32_t ready = n * (uint32_t)kStaticGroupUnit;  // modulo 2^32, compared as sequence numbers (word_reached)
  *epoch = (int32_t)n;
  *counter_ready = (int32_t)ready;
  *counter_start = (int32_t)(ready - (uint32_t)tile_count);
}

// The current device's copy of the scratch.  The first call on a device asks the runtime for
// the symbol's address on that device (no allocation); later calls read the cached pointer.
int static_scratch(StaticScratch** out) {
  int device = -1;
  TCCL_HIP(hipGetDevice(&device));
  if (device < 0 || device >= kMaxDevices) return fail(TCCL_ERR_NO_DEVICE, "device %d outside [0, %d)", device, kMaxDevices);
  std::lock_guard<std::mutex> hold(g_scratch_mutex);
  if (!g_scratch_ptr[device]) {
    void* p = nullptr;
    TCCL_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return fail(TCCL_ERR_NO_DEVICE, "the static scratch has no address on device %d", device);
    g_scratch_ptr[device] = (StaticScratch*)p;
  }
  *out = g_scratch_ptr[device];
  return 0;
}

// Prepares rank `rank`'s words for its call number `call` and writes the plan tables: group_table by the
// rule of build_group_table (tileccl_v2/tile_group.py:214-241: the first group whose rows contain the
// tile's first row, 0 if none), under the tile numbering of tile_coords.  A counter starts its tile count
// short of call * kStaticGroupUnit, the table of tile counts that the kernels multiply the launch number
// with holds kStaticGroupUnit for every group, and locks keep what the call before stored (a smaller
// launch number).  The other ranks' words are left as their own last call left them.
__global__ void static_setup_kernel(StaticScratch* s, tccl_static_plan plan, int rank, uint32_t call, int tile_rows, int tile_cols,
                                    int block_m, int group_m) {
  const int total = tile_rows * tile_cols;
  StaticWords* mine = &s->words[rank];
  const int first = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
  for (int t = first; t < total; t += stride) {
    const int row = tccl::tile_coords(t, tile_rows, tile_cols, group_m).m * block_m;
    int gid = 0;
    for (int g = plan.n_groups - 1; g >= 0; --g)
      if (plan.row_starts[g] <= row && row < plan.row_ends[g]) gid = g;
    s->group_table[t] = gid;
  }
  for (int g = first; g < plan.n_groups; g += stride) {
    s->row_starts[g] = plan.row_starts[g];
    s->row_ends[g] = plan.row_ends[g];
    s->tile_counts[g] = kStaticGroupUnit;
    const uint32_t n = (call - 1u) % 0x7fffffffu + 1u;
    mine->counter[g] = (int32_t)(n * (uint32_t)kStaticGroupUnit - (uint32_t)plan.tile_counts[g]);
    mine->barrier[g] = 0;
  }
}

}  // namespace

// ============================================================================================
// extern "C"
// ============================================================================================
extern "C" {

int tccl_abi_version(void) { return TCCL_ABI_VERSION; }

const char* tccl_last_error_string(void) { return g_error; }

int tccl_device_query(int device, tccl_device_info* out) {
  if (!out) return fail(TCCL_ERR_INVALID, "out is NULL");
  return query_device(device, out);
}

int tccl_tile_coords(int32_t tile_id, int32_t tile_rows, int32_t tile_cols, int32_t group_m, int32_t* tile_m, int32_t* tile_n) {
  if (tile_rows <= 0 || tile_cols <= 0 || group_m <= 0 || tile_id < 0 || tile_id >= tile_rows * tile_cols || !tile_m || !tile_n)
    return fail(TCCL_ERR_INVALID, "tile_coords: bad arguments");
  const tccl::TileCoord c = tccl::tile_coords(tile_id, tile_rows, tile_cols, group_m);
  *tile_m = c.m;
  *tile_n = c.n;
  return 0;
}

int tccl_tile_for_slot(int32_t slot, int32_t total_tiles, int32_t xcds, int32_t span, int32_t* tile_id) {
  if (slot < 0 || slot >= total_tiles || xcds <= 0 || span <= 0 || !tile_id) return fail(TCCL_ERR_INVALID, "tile_for_slot: bad arguments");
  *tile_id = tccl::tile_for_slot(slot, total_tiles, xcds, span);
  return 0;
}

int tccl_stream_grid(int32_t tiles, int32_t pulls, int32_t compute_units, int32_t world_size, int32_t* first_pull, int32_t* workgroups) {
  if (tiles <= 0 || compute_units <= 0 || world_size < 1 || world_size > TCCL_MAX_WORLD || !first_pull || !workgroups)
    return fail(TCCL_ERR_INVALID, "stream_grid: bad arguments");
  const tccl::StreamGrid g = tccl::stream_grid(tiles, pulls != 0, compute_units, world_size);
  *first_pull = g.first;
  *workgroups = g.wgs;
  return 0;
}

int tccl_heap_create(size_t slice_bytes, int world_size, void** arena_out, int64_t* bases_out) {
  if (!arena_out || !bases_out) return fail(TCCL_ERR_INVALID, "heap_create: NULL output");
  if (slice_bytes == 0) return fail(TCCL_ERR_INVALID, "heap_create: slice size must be positive");
  if (world_size < 1 || world_size > TCCL_MAX_WORLD) return fail(TCCL_ERR_INVALID, "heap_create: world_size=%d outside [1, %d]", world_size, TCCL_MAX_WORLD);
  // Slices start on 2 MiB boundaries so that symmetric offsets keep page alignment.
  const size_t align = 2u << 20;
  const size_t stride = (slice_bytes + align - 1) / align * align;
  void* p = nullptr;
  TCCL_HIP(hipMalloc(&p, stride * (size_t)world_size));
  *arena_out = p;
  for (int r = 0; r < world_size; ++r) bases_out[r] = (int64_t)(uintptr_t)p + (int64_t)(stride * (size_t)r);
  return 0;
}

int tccl_heap_destroy(void* arena) {
  if (!arena) return 0;
  TCCL_HIP(hipFree(arena));
  return 0;
}

int tccl_fill_i32(int32_t* words, int64_t n, int32_t value, void* stream) {
  if (n <= 0) return 0;
  if (!words) return fail(TCCL_ERR_INVALID, "fill: NULL pointer");
  int blocks = (int)((n + 255) / 256);
  if (blocks > 1024) blocks = 1024;
  hipLaunchKernelGGL(fill_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream, words, n, value);
  TCCL_HIP(hipGetLastError());
  return 0;
}

int tccl_pack_matrices(const tccl_pack_desc* descs, int32_t n, int32_t elem_bytes, void* stream) {
  if (n <= 0) return 0;
  if (!descs || n > 2) return fail(TCCL_ERR_INVALID, "pack_matrices: one or two matrices, got %d", n);
  PackJobs jobs;
  memset(&jobs, 0, sizeof jobs);
  int kept = 0;
  int64_t wgs = 0;
  for (int i = 0; i < n; ++i) {
    const tccl_pack_desc& p = descs[i];
    if (p.dst_rows <= 0 || p.dst_cols <= 0) continue;
    if (!p.src || !p.dst) return fail(TCCL_ERR_INVALID, "pack_matrix: NULL pointer");
    if (p.rows < 0 || p.cols < 0 || p.rows > p.dst_rows || p.cols > p.dst_cols || p.stride_row < 0 || p.stride_col < 0 || p.ld_dst < p.dst_cols)
      return fail(TCCL_ERR_INVALID, "pack_matrix: source %dx%d (strides %lld, %lld) does not fit a %dx%d destination of pitch %lld",
                  p.rows, p.cols, (long long)p.stride_row, (long long)p.stride_col, p.dst_rows, p.dst_cols, (long long)p.ld_dst);
    jobs.job[kept] = p;
    jobs.first[kept] = (int)wgs;
    ++kept;
    wgs += ((int64_t)p.dst_rows + 63) / 64 * (((int64_t)p.dst_cols + 63) / 64);
    if (wgs > 0x7fffffffll) return fail(TCCL_ERR_UNSUPPORTED, "pack_matrix: more than 2^31 patches of 64 x 64");
  }
  if (kept == 0) return 0;
  const hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)wgs), block(256);
  if (elem_bytes == 1)
    hipLaunchKernelGGL(pack_kernel<uint8_t>, grid, block, 0, st, jobs, kept);
  else if (elem_bytes == 2)
    hipLaunchKernelGGL(pack_kernel<uint16_t>, grid, block, 0, st, jobs, kept);
  else if (elem_bytes == 4)
    hipLaunchKernelGGL(pack_kernel<uint32_t>, grid, block, 0, st, jobs, kept);
  else
    return fail(TCCL_ERR_INVALID, "pack_matrix: elem_bytes=%d must be 1, 2 or 4", elem_bytes);
  TCCL_HIP(hipGetLastError());
  return 0;
}

int tccl_pack_matrix(const void* src, int64_t stride_row, int64_t stride_col, int32_t rows, int32_t cols, void* dst,
                     int64_t ld_dst, int32_t dst_rows, int32_t dst_cols, int32_t elem_bytes, void* stream) {
  const tccl_pack_desc p{src, dst, stride_row, stride_col, ld_dst, rows, cols, dst_rows, dst_cols};
  return tccl_pack_matrices(&p, 1, elem_bytes, stream);
}

int tccl_prim_signal(int32_t* locks, int32_t index, void* stream) {
  if (!locks || index < 0) return fail(TCCL_ERR_INVALID, "prim_signal: bad arguments");
  hipLaunchKernelGGL(prim_signal_kernel, dim3(1), dim3(1), 0, (hipStream_t)stream, locks, index);
  TCCL_HIP(hipGetLastError());
  return 0;
}

int tccl_prim_signal_add(int32_t* words, int32_t index, int32_t value, int32_t* result, void* stream) {
  if (!words || !result || index < 0) return fail(TCCL_ERR_INVALID, "prim_signal_add: bad arguments");
  hipLaunchKernelGGL(prim_signal_add_kernel, dim3(1), dim3(1), 0, (hipStream_t)stream, words, index, value, result);
  TCCL_HIP(hipGetLastError());
  return 0;
}

int tccl_prim_try_wait(int32_t* locks, int32_t index, int32_t max_spins, int32_t consume, int32_t* result, void* stream) {
  if (!locks || !result || index < 0 || max_spins < 0) return fail(TCCL_ERR_INVALID, "prim_try_wait: bad arguments");
  hipLaunchKernelGGL(prim_try_wait_kernel, dim3(1), dim3(1), 0, (hipStream_t)stream, locks, index, max_spins, consume, result);
  TCCL_HIP(hipGetLastError());
  return 0;
}

int tccl_prim_wait_ge(int32_t* words, int32_t index, int32_t threshold, int64_t spin_limit_ns, int32_t* result, void* stream) {
  if (!words || !result || index < 0) return fail(TCCL_ERR_INVALID, "prim_wait_ge: bad arguments");
  if (spin_limit_ns <= 0 || spin_limit_ns > kDefaultSpinNs) spin_limit_ns = kDefaultSpinNs;
  hipLaunchKernelGGL(prim_wait_ge_kernel, dim3(1), dim3(1), 0, (hipStream_t)stream, words, index, threshold, spin_limit_ns / 10 + 1, result);
  TCCL_HIP(hipGetLastError());
  return 0;
}

int tccl_gemm(const tccl_gemm_desc* d, void* stream) {
  int rc = check_gemm(d);
  if (rc) return rc;
  tccl_device_info dev;
  if ((rc = query_device(-1, &dev))) return rc;
  tccl::GemmArgs g;
  build_gemm_args(d, dev, &g);
  const int64_t seg = g.wrap_rows > 0 ? g.wrap_rows : d->M;
  const int shape = stream_shape(d, nullptr, nullptr, TCCL_S0_BULK, seg, dev);
  if (shape >= 0) {
    tccl::StreamArgs a;
    build_stream(d, g, seg, dev, &a);
    return stream_status(tccl::launch_stream(d->in_dtype, g.b_kmajor != 0, shape, a, (hipStream_t)stream));
  }
  tccl::SignalArgs s;
  memset(&s, 0, sizeof s);
  const int segs = d->column_shards > 1 ? d->column_shards : 1;
  const TileKernel kernel = choose_tiles(d, d->M / segs, segs, plan_tile_fits_macro(d), false, dev).kernel;
  if (kernel == kTiles256) {
    const int wgs = default_macro_wgs(d, dev);
    return launch_gemm256(d->in_dtype, d->out_dtype, g, build_macro(d, dev, wgs), wgs, (hipStream_t)stream);
  }
  tccl::CommArgs none;
  memset(&none, 0, sizeof none);
  return launch_fused(d, g, s, none, kernel, tile_wgs(kernel, d, dev, g.tile_rows * g.tile_cols), 0, nullptr,
                      (hipStream_t)stream);
}

// The 128-row tile kernels read an A given by columns in place; the streaming and the large-tile kernel do not, and where they would run a
// launch that turns A into rows comes first (as it does for what check_gemm() refuses).  From CUs / 2 large tiles on it always does, also where
// choose_tiles() would name a 128-row kernel for a launch of pushes.  bf16 pushed to one peer, with that launch -> in place: 1000 x 2064 x 1003
// 21.6 -> 15.3 us, 256 x 6144 x 72 11.7 -> 7.2, 2048 x 2048 x 2048 33.3 -> 24.7, 1544 x 4112 x 8192 119 -> 113 (60 shapes, K = 72 to 8192: 1.05 to 1.79
// times as fast).
int tccl_gemm_reads_columns(const tccl_gemm_desc* d) {
  if (!d || !(d->flags & TCCL_GEMM_A_COLUMNS) || d->macro_tile != 0 || d->block_m != 128 || d->block_n != 128 || check_gemm(d)) return 0;
  tccl_device_info dev;
  if (query_device(-1, &dev)) return 0;
  tccl_gemm_desc rows = *d;
  rows.flags &= ~TCCL_GEMM_A_COLUMNS;
  return !use_macro(&rows, dev, true) && stream_shape(&rows, nullptr, nullptr, TCCL_S0_BULK, d->M, dev) < 0;
}

static int check_scatter(const tccl_scatter_desc* sc, int M, int N, int esize, int64_t ldc, const void* C) {
  if (!sc) return fail(TCCL_ERR_INVALID, "scatter descriptor is NULL");
  if (sc->cols <= 0 || sc->src_col_offset < 0 || sc->dst_col_offset < 0 || sc->dst_ld <= 0)
    return fail(TCCL_ERR_INVALID, "scatter: bad placement (src_col_offset=%d cols=%d dst_ld=%d dst_col_offset=%d)", sc->src_col_offset, sc->cols, sc->dst_ld, sc->dst_col_offset);
  if (sc->src_col_offset + sc->cols > N) return fail(TCCL_ERR_INVALID, "scatter: source columns [%d, %d) exceed N=%d", sc->src_col_offset, sc->src_col_offset + sc->cols, N);
  if (sc->dst_col_offset + sc->cols > sc->dst_ld) return fail(TCCL_ERR_INVALID, "scatter: destination columns exceed dst_ld");
  const int v = 16 / esize;
  if (sc->src_col_offset % v || sc->cols % v || sc->dst_col_offset % v || sc->dst_ld % v || ldc % v || !aligned16(C))
    return fail(TCCL_ERR_UNSUPPORTED, "scatter: column offsets, widths and leading dimensions must be multiples of %d elements", v);
  (void)M;
  return 0;
}

int tccl_scatter_cols(const void* C, int32_t M, int64_t ldc, int32_t elem_bytes, const tccl_scatter_desc* sc,
                      const tccl_heap_view* heap, void* stream) {
  int rc = check_heap(heap);
  if (rc) return rc;
  if (!C || M <= 0 || (elem_bytes != 1 && elem_bytes != 2 && elem_bytes != 4)) return fail(TCCL_ERR_INVALID, "scatter_cols: bad arguments");
  if (!sc) return fail(TCCL_ERR_INVALID, "scatter descriptor is NULL");
  const int N = sc->src_col_offset + sc->cols;
  if ((rc = check_scatter(sc, M, N, elem_bytes, ldc, C))) return rc;
  if (heap->world_size == 1) return 0;
  if ((rc = check_rows_span(M, (ldc > sc->dst_ld ? ldc : (int64_t)sc->dst_ld) * elem_bytes))) return rc;
  tccl_device_info dev;
  if ((rc = query_device(-1, &dev))) return rc;
  tccl::BulkCopyArgs a;
  memset(&a, 0, sizeof a);
  a.heap_bases = heap->heap_bases;
  a.rank = heap->rank;
  a.world = heap->world_size;
  a.src = (int64_t)(uintptr_t)C + (int64_t)sc->src_col_offset * elem_bytes;
  a.dst = (int64_t)(uintptr_t)C + (int64_t)sc->dst_col_offset * elem_bytes;
  a.src_pitch = (uint32_t)(ldc * elem_bytes);
  a.dst_pitch = (uint32_t)((int64_t)sc->dst_ld * elem_bytes);
  a.upr = sc->cols * elem_bytes / 16;
  a.t[0] = {0, 0, heap->rank, all_but(heap->world_size, heap->rank)};
  return launch_bulk_copy(a, 1, M, dev, (hipStream_t)stream);
}

int tccl_exchange_rows(void* out, int32_t rows_per_rank, int32_t N, int64_t ld, int32_t elem_bytes,
                       const tccl_heap_view* heap, const tccl_transport_desc* tr, void* stream) {
  int rc = check_heap(heap);
  if (rc) return rc;
  if (!out || rows_per_rank <= 0 || N <= 0 || ld < N || (elem_bytes != 1 && elem_bytes != 2 && elem_bytes != 4))
    return fail(TCCL_ERR_INVALID, "exchange_rows: bad arguments");
  const int v = 16 / elem_bytes;
  if (N % v || ld % v || !aligned16(out)) return fail(TCCL_ERR_UNSUPPORTED, "exchange_rows: rows must be multiples of 16 bytes");
  if (heap->world_size == 1) return 0;
  if ((rc = check_rows_span(rows_per_rank, ld * elem_bytes))) return rc;
  tccl_device_info dev;
  if ((rc = query_device(-1, &dev))) return rc;
  if ((rc = check_task_elems(tr, false, elem_bytes))) return rc;
  const int64_t pitch = ld * elem_bytes, block = rows_per_rank * pitch;
  const int directions = tr ? tr->directions : TCCL_DIR_PUSH;
  tccl::BulkCopyArgs a;
  memset(&a, 0, sizeof a);
  a.heap_bases = heap->heap_bases;
  a.rank = heap->rank;
  a.world = heap->world_size;
  a.src = a.dst = (int64_t)(uintptr_t)out;
  a.src_pitch = a.dst_pitch = (uint32_t)pitch;
  a.upr = N * elem_bytes / 16;
  int n = 0;
  if (directions & TCCL_DIR_PULL)
    for (int p = 0; p < a.world; ++p)
      if (p != a.rank) a.t[n++] = {p * block, p * block, p, 1u << a.rank};
  if (directions & TCCL_DIR_PUSH) a.t[n++] = {a.rank * block, a.rank * block, a.rank, all_but(a.world, a.rank)};
  return launch_bulk_copy(a, n, rows_per_rank, dev, (hipStream_t)stream);
}

int tccl_copy_block(void* dst, uint32_t dst_ranks, const void* src, int32_t src_rank, int32_t rows, int64_t row_bytes,
                    int64_t src_pitch_bytes, int64_t dst_pitch_bytes, const tccl_heap_view* heap, void* stream) {
  int rc = check_heap(heap);
  if (rc) return rc;
  if (!dst || !src || rows <= 0 || row_bytes <= 0 || src_pitch_bytes < row_bytes || dst_pitch_bytes < row_bytes)
    return fail(TCCL_ERR_INVALID, "copy_block: bad arguments");
  if (src_rank < 0 || src_rank >= heap->world_size)
    return fail(TCCL_ERR_INVALID, "copy_block: src_rank=%d out of range for world_size=%d", src_rank, heap->world_size);
  if (heap->world_size < 32 && (dst_ranks >> heap->world_size))
    return fail(TCCL_ERR_INVALID, "copy_block: dst_ranks=0x%x names ranks beyond world_size=%d", dst_ranks, heap->world_size);
  if (row_bytes % 16 || src_pitch_bytes % 16 || dst_pitch_bytes % 16 || !aligned16(dst) || !aligned16(src))
    return fail(TCCL_ERR_UNSUPPORTED, "copy_block: rows must be multiples of 16 bytes and 16-byte aligned");
  if (row_bytes > 0x7fffffffll) return fail(TCCL_ERR_UNSUPPORTED, "copy_block: rows of %lld bytes (limit 2 GiB)", (long long)row_bytes);
  if ((rc = check_rows_span(rows, src_pitch_bytes > dst_pitch_bytes ? src_pitch_bytes : dst_pitch_bytes))) return rc;
  if (dst_ranks == 0) return 0;
  tccl_device_info dev;
  if ((rc = query_device(-1, &dev))) return rc;
  tccl::BulkCopyArgs a;
  memset(&a, 0, sizeof a);
  a.heap_bases = heap->heap_bases;
  a.rank = heap->rank;
  a.world = heap->world_size;
  a.src = (int64_t)(uintptr_t)src;
  a.dst = (int64_t)(uintptr_t)dst;
  a.src_pitch = (uint32_t)src_pitch_bytes;
  a.dst_pitch = (uint32_t)dst_pitch_bytes;
  a.upr = (int)(row_bytes / 16);
  a.t[0] = {0, 0, src_rank, dst_ranks};
  return launch_bulk_copy(a, 1, rows, dev, (hipStream_t)stream);
}

int tccl_gather_cols(void* gathered, int64_t ld_gathered, const void* shard, int64_t ld_shard, int32_t M,
                     int32_t cols, int32_t elem_bytes, const tccl_heap_view* heap, const tccl_transport_desc* tr,
                     void* stream) {
  int rc = check_heap(heap);
  if (rc) return rc;
  if (!gathered || !shard || M <= 0 || cols <= 0 || ld_shard < cols || (elem_bytes != 1 && elem_bytes != 2 && elem_bytes != 4))
    return fail(TCCL_ERR_INVALID, "gather_cols: bad arguments");
  if (ld_gathered < (int64_t)cols * heap->world_size)
    return fail(TCCL_ERR_INVALID, "gather_cols: gathered rows hold %lld elements, need %lld", (long long)ld_gathered,
                (long long)cols * heap->world_size);
  const int v = 16 / elem_bytes;
  if (cols % v || ld_shard % v || ld_gathered % v || !aligned16(gathered) || !aligned16(shard))
    return fail(TCCL_ERR_UNSUPPORTED, "gather_cols: shard rows must be multiples of 16 bytes and 16-byte aligned");
  if ((rc = check_rows_span(M, (ld_gathered > ld_shard ? ld_gathered : ld_shard) * elem_bytes))) return rc;
  tccl_device_info dev;
  if ((rc = query_device(-1, &dev))) return rc;
  if ((rc = check_task_elems(tr, false, elem_bytes))) return rc;
  tccl::BulkCopyArgs a;
  memset(&a, 0, sizeof a);
  a.heap_bases = heap->heap_bases;
  a.rank = heap->rank;
  a.world = heap->world_size;
  a.src = (int64_t)(uintptr_t)shard;
  a.dst = (int64_t)(uintptr_t)gathered;
  a.src_pitch = (uint32_t)(ld_shard * elem_bytes);
  a.dst_pitch = (uint32_t)(ld_gathered * elem_bytes);
  a.upr = cols * elem_bytes / 16;
  for (int p = 0; p < a.world; ++p) a.t[p] = {0, (int64_t)p * cols * elem_bytes, p, 1u << a.rank};
  return launch_bulk_copy(a, a.world, M, dev, (hipStream_t)stream);
}

static int fill_reduce(tccl::CommArgs* c, const void* partial, int partial_dtype, void* out, int out_dtype, int64_t ld_out,
                       int M, int N, int world, int emulate_peer, bool allow_f32_out = false) {
  if (partial_dtype != TCCL_F16 && partial_dtype != TCCL_BF16 && partial_dtype != TCCL_F32)
    return fail(TCCL_ERR_UNSUPPORTED, "reduce: partial dtype %d", partial_dtype);
  if (out_dtype == TCCL_F32 && !(allow_f32_out && partial_dtype == TCCL_F32))
    return fail(TCCL_ERR_UNSUPPORTED, "reduce: fp32 output only from fp32 partials in the stand-alone reduction");
  if (out_dtype != TCCL_F16 && out_dtype != TCCL_BF16 && out_dtype != TCCL_F32)
    return fail(TCCL_ERR_UNSUPPORTED, "reduce: output dtype must be fp16, bf16 or fp32");
  if (partial_dtype != TCCL_F32 && partial_dtype != out_dtype && !(partial_dtype == TCCL_BF16 || partial_dtype == TCCL_F16))
    return fail(TCCL_ERR_UNSUPPORTED, "reduce: dtype combination");
  if (M % world) return fail(TCCL_ERR_INVALID, "reduce: M=%d must be divisible by world_size=%d", M, world);
  if (N % 8 || ld_out % 8 || !aligned16(out) || !aligned16(partial)) return fail(TCCL_ERR_UNSUPPORTED, "reduce: rows must be multiples of 8 elements and 16-byte aligned");
  c->op = tccl::kOpReduceScatter;
  c->rs_out = (char*)out;
  c->ld_rs_out_bytes = ld_out * (out_dtype == TCCL_F32 ? 4 : 2);
  c->partial_dtype = partial_dtype;
  c->out_dtype = out_dtype;
  c->emulate_peer = (emulate_peer & TCCL_RS_EMULATE_PEERS) != 0;
  c->peers_resident = (emulate_peer & TCCL_RS_PEERS_RESIDENT) != 0;
  // Without a plan the kernel works shard by shard (one implicit group per owner).
  if (!c->row_starts) c->n_groups = world;
  return 0;
}

int tccl_reduce_rows(const void* partial, int32_t partial_dtype, int64_t ld_partial, void* out, int32_t out_dtype,
                     int64_t ld_out, int32_t M, int32_t N, const tccl_heap_view* heap, const tccl_transport_desc* tr,
                     int32_t emulate_peer, void* stream) {
  int rc = check_heap(heap);
  if (rc) return rc;
  if (!partial || !out || M <= 0 || N <= 0 || ld_partial < N || ld_out < N) return fail(TCCL_ERR_INVALID, "reduce_rows: bad arguments");
  const int esize = (int)dtype_size(partial_dtype);
  if (!esize || ld_partial % (16 / esize)) return fail(TCCL_ERR_UNSUPPORTED, "reduce_rows: partial rows must be 16-byte multiples");
  if ((rc = check_rows_span(M, ld_partial * esize)) || (rc = check_rows_span(M, ld_out * 4))) return rc;
  tccl_device_info dev;
  if ((rc = query_device(-1, &dev))) return rc;
  tccl::CommArgs c;
  memset(&c, 0, sizeof c);
  c.heap_bases = heap->heap_bases;
  c.rank = heap->rank;
  c.world = heap->world_size;
  c.C = (char*)partial;
  c.ldc_bytes = ld_partial * esize;
  c.M = M;
  c.N = N;
  if ((rc = fill_reduce(&c, partial, partial_dtype, out, out_dtype, ld_out, M, N, heap->world_size, emulate_peer, true))) return rc;
  if ((rc = check_task_elems(tr, true, esize))) return rc;
  return launch_bulk(c, dev, (hipStream_t)stream);
}

static int allscatter_impl(const tccl_gemm_desc* d, const tccl_scatter_desc* sc, const tccl_heap_view* heap,
                           const tccl_sync_desc* sync, const tccl_transport_desc* tr, int32_t variant, const GatherSpec* gather,
                           hipStream_t stream) {
  int rc = check_gemm(d);
  if (rc) return rc;
  if ((rc = check_heap(heap))) return rc;
  if (variant < TCCL_S0_BULK || variant > TCCL_S2_TILEGROUP) return fail(TCCL_ERR_INVALID, "unknown variant %d", variant);
  if ((rc = check_sync(sync, variant))) return rc;
  const int esize = (int)dtype_size(d->out_dtype);
  if ((rc = check_scatter(sc, d->M, d->N, esize, d->ldc, d->C))) return rc;
  tccl_device_info dev;
  if ((rc = query_device(-1, &dev))) return rc;
  tccl::GemmArgs g;
  build_gemm_args(d, dev, &g);
  tccl::CommArgs c;
  fill_comm_common(&c, g, esize, heap, sync, tr);
  c.op = tccl::kOpAllScatter;
  c.directions = TCCL_DIR_PUSH;
  c.src_col_off = sc->src_col_offset;
  c.cols = sc->cols;
  c.dst_ld = sc->dst_ld;
  c.dst_col_off = sc->dst_col_offset;
  if ((rc = set_task_units(&c, tr, false))) return rc;
  return run_variant(d, c, sync, tr, variant, dev, g, stream, gather, heap);
}

int tccl_collective_staged(int32_t op, const void* src, void* dst, int32_t dtype, int64_t block_elems, void* staging,
                           int32_t* published, int32_t* consumed, int32_t chunk_elems, int32_t slots, int32_t base_epoch,
                           uint32_t ranks, int32_t root, const tccl_heap_view* heap, int64_t* fault, int64_t spin_limit_ns,
                           void* stream) {
  static const char* const names[] = {"allreduce", "allgather", "reduce_scatter", "broadcast", "scatter"};
  int rc = check_heap(heap);
  if (rc) return rc;
  if (op < TCCL_STAGED_ALLREDUCE || op > TCCL_STAGED_SCATTER) return fail(TCCL_ERR_INVALID, "collective_staged: unknown op %d", op);
  const char* name = names[op];
  const bool reduces = op == TCCL_STAGED_ALLREDUCE || op == TCCL_STAGED_REDUCE_SCATTER;
  const bool in_place = op == TCCL_STAGED_ALLREDUCE || op == TCCL_STAGED_BROADCAST;
  const bool rooted = op == TCCL_STAGED_BROADCAST || op == TCCL_STAGED_SCATTER;
  const int esize = (int)dtype_size(dtype);
  if (!esize || (reduces && dtype != TCCL_F16 && dtype != TCCL_BF16 && dtype != TCCL_F32))
    return fail(TCCL_ERR_UNSUPPORTED, "%s_staged: dtype %d", name, dtype);
  if (!dst || (!in_place && !src) || !staging || !published || !consumed || block_elems <= 0 || chunk_elems <= 0 || slots <= 0 ||
      base_epoch < 1)
    return fail(TCCL_ERR_INVALID, "%s_staged: bad arguments", name);
  if (rooted && (root < 0 || root >= heap->world_size)) return fail(TCCL_ERR_INVALID, "%s_staged: root=%d out of range [0, %d)", name, root, heap->world_size);
  const int per_unit = 16 / esize;
  if (block_elems % per_unit || chunk_elems % per_unit || !aligned16(dst) || !aligned16(src) || !aligned16(staging))
    return fail(TCCL_ERR_UNSUPPORTED, "%s_staged: blocks and chunks must be whole 16-byte units (%d elements)", name, per_unit);
  if ((int64_t)chunk_elems * esize * heap->world_size > 0x7fffffffll) return fail(TCCL_ERR_UNSUPPORTED, "%s_staged: chunk too large", name);
  if (heap->world_size < 32 && (ranks >> heap->world_size))
    return fail(TCCL_ERR_INVALID, "%s_staged: ranks=0x%x names ranks beyond world_size=%d", name, ranks, heap->world_size);
  const int roles = __builtin_popcount(ranks);
  if (roles == 0) return 0;
  const int64_t chunks = (block_elems + chunk_elems - 1) / chunk_elems;
  if ((int64_t)base_epoch + chunks > 0x7fffffffll) return fail(TCCL_ERR_INVALID, "%s_staged: epoch range overflows int32", name);
  tccl_device_info dev;
  if ((rc = query_device(-1, &dev))) return rc;
  // Every (rank, slot) workgroup waits on others of the same launch: all must be resident.
  if ((int64_t)roles * slots > (int64_t)dev.compute_units * 4)
    return fail(TCCL_ERR_UNSUPPORTED, "%s_staged: %d roles x %d slots exceed what the device keeps resident (%d workgroups)", name, roles,
                slots, dev.compute_units * 4);
  tccl::StagedArgs a;
  memset(&a, 0, sizeof a);
  a.heap_bases = heap->heap_bases;
  a.rank = heap->rank;
  a.world = heap->world_size;
  a.ranks = ranks;
  a.op = op;
  a.root = root;
  a.src = (char*)src;
  a.dst = (char*)dst;
  a.staging = (char*)staging;
  a.published = published;
  a.consumed = consumed;
  a.units = block_elems / per_unit;
  a.chunk_units = chunk_elems / per_unit;
  a.slots = slots;
  a.base_epoch = base_epoch;
  a.dtype = reduces ? dtype : TCCL_F16;  // copies move bytes
  a.fault = fault;
  a.spin_ticks = (spin_limit_ns > 0 ? spin_limit_ns : kDefaultSpinNs) / 10 + 1;
  hipLaunchKernelGGL(staged_kernel, dim3(roles * slots), dim3(256), 0, (hipStream_t)stream, a);
  TCCL_HIP(hipGetLastError());
  return 0;
}

// A collective whose inputs are complete and whose roles are all carried by one launch needs no staging and
// no waits: each byte of a result is read from where it lies and written where it is wanted.
int tccl_collective_direct(int32_t op, const void* src, void* dst, int32_t dtype, int64_t block_elems, int32_t root,
                           const tccl_heap_view* heap, void* stream) {
  static const char* const names[] = {"allreduce", "allgather", "reduce_scatter", "broadcast", "scatter"};
  int rc = check_heap(heap);
  if (rc) return rc;
  if (op < TCCL_STAGED_ALLREDUCE || op > TCCL_STAGED_SCATTER) return fail(TCCL_ERR_INVALID, "collective_direct: unknown op %d", op);
  const char* name = names[op];
  const bool reduces = op == TCCL_STAGED_ALLREDUCE || op == TCCL_STAGED_REDUCE_SCATTER;
  const bool in_place = op == TCCL_STAGED_ALLREDUCE || op == TCCL_STAGED_BROADCAST;
  const int esize = (int)dtype_size(dtype), world = heap->world_size;
  if (!esize || (reduces && dtype != TCCL_F16 && dtype != TCCL_BF16 && dtype != TCCL_F32))
    return fail(TCCL_ERR_UNSUPPORTED, "%s_direct: dtype %d", name, dtype);
  if (!dst || (!in_place && !src) || block_elems <= 0) return fail(TCCL_ERR_INVALID, "%s_direct: bad arguments", name);
  if (root < 0 || root >= world) return fail(TCCL_ERR_INVALID, "%s_direct: root=%d out of range [0, %d)", name, root, world);
  const int per_unit = 16 / esize;
  if (block_elems % per_unit || !aligned16(dst) || (!in_place && !aligned16(src)))
    return fail(TCCL_ERR_UNSUPPORTED, "%s_direct: blocks must be whole 16-byte units (%d elements)", name, per_unit);
  if (reduces && block_elems % 8) return fail(TCCL_ERR_UNSUPPORTED, "%s_direct: blocks must be multiples of 8 elements", name);
  tccl_device_info dev;
  if ((rc = query_device(-1, &dev))) return rc;
  const int64_t block = block_elems * esize, piece = 1ll << 30;  // a launch addresses its rectangle with 32-bit offsets
  for (int64_t at = 0; at < block; at += piece) {
    const int64_t bytes = block - at < piece ? block - at : piece;
    if (reduces) {
      tccl::BulkReduceArgs a;
      memset(&a, 0, sizeof a);
      a.heap_bases = heap->heap_bases;
      a.rank = heap->rank;
      a.world = world;
      a.src = (int64_t)(uintptr_t)(in_place ? dst : src) + at;
      a.dst = (int64_t)(uintptr_t)dst + at;
      a.src_shift = in_place ? 0 : block;
      a.src_pitch = a.dst_pitch = (uint32_t)bytes;
      a.upr = (int)(bytes / esize / 8);
      a.ascending = a.to_all = in_place ? 1 : 0;
      rc = launch_bulk_reduce(a, in_place ? 1 : world, 1, dtype, dtype, dev, (hipStream_t)stream);
    } else {
      tccl::BulkCopyArgs a;
      memset(&a, 0, sizeof a);
      a.heap_bases = heap->heap_bases;
      a.rank = heap->rank;
      a.world = world;
      a.src = (int64_t)(uintptr_t)(in_place ? dst : src) + at;
      a.dst = (int64_t)(uintptr_t)dst + at;
      a.src_pitch = a.dst_pitch = (uint32_t)bytes;
      a.upr = (int)(bytes / 16);
      int n = 0;
      if (op == TCCL_STAGED_ALLGATHER)
        for (int r = 0; r < world; ++r) a.t[n++] = {0, r * block, r, (1u << world) - 1u};
      else if (op == TCCL_STAGED_BROADCAST)
        a.t[n++] = {0, 0, root, all_but(world, root)};
      else
        for (int q = 0; q < world; ++q) a.t[n++] = {q * block, 0, root, 1u << q};
      rc = launch_bulk_copy(a, n, 1, dev, (hipStream_t)stream);
    }
    if (rc) return rc;
  }
  return 0;
}

int tccl_allreduce_chunk(void* tensor, int32_t dtype, int64_t numel, const tccl_heap_view* heap, void* stream) {
  int rc = check_heap(heap);
  if (rc) return rc;
  const int esize = (int)dtype_size(dtype), world = heap->world_size;
  if (dtype != TCCL_F16 && dtype != TCCL_BF16 && dtype != TCCL_F32) return fail(TCCL_ERR_UNSUPPORTED, "allreduce_chunk: dtype %d", dtype);
  if (!tensor || numel <= 0 || numel % world) return fail(TCCL_ERR_INVALID, "allreduce_chunk: bad arguments");
  if ((numel / world) % 8 || !aligned16(tensor))
    return fail(TCCL_ERR_UNSUPPORTED, "allreduce_chunk: a rank's chunk must be a multiple of 8 elements and 16-byte aligned");
  tccl_device_info dev;
  if ((rc = query_device(-1, &dev))) return rc;
  const int64_t chunk = numel / world * esize, piece = 1ll << 30;
  for (int64_t at = 0; at < chunk; at += piece) {
    const int64_t bytes = chunk - at < piece ? chunk - at : piece;
    tccl::BulkReduceArgs a;
    memset(&a, 0, sizeof a);
    a.heap_bases = heap->heap_bases;
    a.rank = heap->rank;
    a.world = world;
    a.src = a.dst = (int64_t)(uintptr_t)tensor + at;
    a.src_shift = a.dst_shift = chunk;
    a.src_pitch = a.dst_pitch = (uint32_t)bytes;
    a.upr = (int)(bytes / esize / 8);
    a.first_owner = heap->rank;
    a.to_all = 1;
    if ((rc = launch_bulk_reduce(a, 1, 1, dtype, dtype, dev, (hipStream_t)stream))) return rc;
  }
  return 0;
}

int tccl_allreduce_staged(void* tensor, int32_t dtype, int64_t numel, void* staging, int32_t* published, int32_t* consumed,
                          int32_t chunk_elems, int32_t slots, int32_t base_epoch, uint32_t ranks, const tccl_heap_view* heap,
                          int64_t* fault, int64_t spin_limit_ns, void* stream) {
  return tccl_collective_staged(TCCL_STAGED_ALLREDUCE, nullptr, tensor, dtype, numel, staging, published, consumed, chunk_elems, slots,
                                base_epoch, ranks, 0, heap, fault, spin_limit_ns, stream);
}

int tccl_gemm_allscatter(const tccl_gemm_desc* d, const tccl_scatter_desc* sc, const tccl_heap_view* heap,
                         const tccl_sync_desc* sync, const tccl_transport_desc* tr, int32_t variant, void* stream) {
  return allscatter_impl(d, sc, heap, sync, tr, variant, nullptr, (hipStream_t)stream);
}

int tccl_chained_ag_gemm_rs(const tccl_gemm_desc* d, const void* shard, int64_t ld_shard, int32_t k_shard,
                            const tccl_heap_view* heap, const tccl_sync_desc* sync, const tccl_transport_desc* tr,
                            int32_t variant, void* stream) {
  int rc = check_gemm(d);
  if (rc) return rc;
  if ((rc = check_heap(heap))) return rc;
  if (d->flags & TCCL_GEMM_A_COLUMNS) return fail(TCCL_ERR_UNSUPPORTED, "chained: the gathered workspace has rows");
  if (k_shard <= 0 || (int64_t)k_shard * heap->world_size != d->K)
    return fail(TCCL_ERR_INVALID, "chained: input_shard columns (%d) * world_size (%d) != W rows (%d)", k_shard,
                heap->world_size, d->K);
  tccl_device_info dev;
  if ((rc = query_device(-1, &dev))) return rc;
  // Stages 2 and 3: the GEMM, whose whole output goes to every peer's output.
  tccl_scatter_desc sc;
  sc.src_col_offset = 0;
  sc.cols = d->N;
  sc.dst_ld = (int32_t)d->ldc;
  sc.dst_col_offset = 0;
  const int esz = (int)dtype_size(d->in_dtype);
  const bool shard_ok = shard && ld_shard >= k_shard && (ld_shard * esz) % 16 == 0 && ((int64_t)k_shard * esz) % 16 == 0 &&
                        aligned16(shard) && (255 * ld_shard + k_shard) * (int64_t)esz <= 0xffffffffll;
  if (shard_ok && gather_in_place(d, dev, k_shard, variant)) {
    // One launch: the K loops read every rank's shard where it lies, and the gathered
    // workspace (gemm->A) is filled on the side while they run.
    if ((rc = check_rows_span(d->M, (d->lda > ld_shard ? d->lda : ld_shard) * esz))) return rc;
    const GatherSpec gs{shard, ld_shard, k_shard};
    return allscatter_impl(d, &sc, heap, sync, tr, variant, &gs, (hipStream_t)stream);
  }
  // Stage 1 as a launch of its own: the gathered input (gemm->A) is filled from every rank's shard.
  if ((rc = tccl_gather_cols((void*)d->A, d->lda, shard, ld_shard, d->M, k_shard, (int32_t)esz, heap, tr, stream)))
    return rc;
  return allscatter_impl(d, &sc, heap, sync, tr, variant, nullptr, (hipStream_t)stream);
}

int tccl_gemm_allgather(const tccl_gemm_desc* d, void* out, int64_t ld_out, const tccl_heap_view* heap,
                        const tccl_sync_desc* sync, const tccl_transport_desc* tr, int32_t variant, void* stream) {
  return allgather_impl(d, out, ld_out, heap, sync, tr, variant, 0, (hipStream_t)stream);
}

int tccl_gemm_allgather_static(const tccl_gemm_desc* d, void* out, int64_t ld_out, const tccl_heap_view* heap,
                               const tccl_static_plan* plan, const tccl_transport_desc* tr, int32_t variant,
                               int64_t* fault, int64_t spin_limit_ns, void* stream) {
  int rc = check_gemm(d);
  if (rc) return rc;
  if ((rc = check_heap(heap))) return rc;
  if (variant != TCCL_S1_TILE && variant != TCCL_S2_TILEGROUP)
    return fail(TCCL_ERR_INVALID, "allgather_static: variant %d keeps no signal words; use tccl_gemm_allgather with sync = NULL", variant);
  if (!plan) return fail(TCCL_ERR_INVALID, "allgather_static: plan is NULL");
  if (plan->n_groups < 1 || plan->n_groups > TCCL_STATIC_MAX_GROUPS)
    return fail(TCCL_ERR_INVALID, "allgather_static: n_groups=%d outside [1, %d]", plan->n_groups, TCCL_STATIC_MAX_GROUPS);
  const int tile_rows = (d->M + d->block_m - 1) / d->block_m, tile_cols = (d->N + d->block_n - 1) / d->block_n;
  const int64_t tiles = (int64_t)tile_rows * tile_cols;
  if (tiles > TCCL_STATIC_MAX_TILES)
    return fail(TCCL_ERR_UNSUPPORTED, "allgather_static: %lld plan tiles exceed the static scratch (%d tiles)", (long long)tiles, TCCL_STATIC_MAX_TILES);
  for (int g = 0; g < plan->n_groups; ++g)
    if (plan->row_starts[g] < 0 || plan->row_ends[g] <= plan->row_starts[g] || plan->row_ends[g] > d->M || plan->tile_counts[g] <= 0 ||
        (g > 0 && plan->row_starts[g] < plan->row_ends[g - 1]))
      return fail(TCCL_ERR_INVALID, "allgather_static: group %d = rows [%d, %d), %d tiles is not an ascending cover of M=%d", g,
                  plan->row_starts[g], plan->row_ends[g], plan->tile_counts[g], d->M);
  StaticScratch* sc = nullptr;
  if ((rc = static_scratch(&sc))) return rc;
  int device = -1;
  TCCL_HIP(hipGetDevice(&device));
  uint32_t call;
  {
    std::lock_guard<std::mutex> hold(g_scratch_mutex);
    call = ++g_static_calls[device][heap->rank];
  }
  int32_t epoch, start, ready;
  static_call_words(call, 0, &epoch, &start, &ready);
  // One small kernel prepares this rank's words for this call and (re)writes the plan tables; it is
  // ordered before the fused launch by the stream.  Nothing is allocated and nothing is memset.
  const int threads = 256;
  int blocks = (int)((tiles + threads - 1) / threads);
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(static_setup_kernel, dim3(blocks), dim3(threads), 0, (hipStream_t)stream, sc, *plan, heap->rank, call, tile_rows,
                     tile_cols, d->block_m, d->group_m);
  TCCL_HIP(hipGetLastError());
  tccl_sync_desc sync;
  memset(&sync, 0, sizeof sync);
  StaticWords* mine = &sc->words[heap->rank];
  sync.locks = mine->locks;
  sync.counter = mine->counter;
  sync.barrier = mine->barrier;
  sync.group_table = sc->group_table;
  sync.row_starts = sc->row_starts;
  sync.row_ends = sc->row_ends;
  sync.tile_counts = sc->tile_counts;
  sync.n_groups = plan->n_groups;
  sync.epoch = epoch;
  sync.fault = fault;
  sync.spin_limit_ns = spin_limit_ns;
  tccl_gemm_desc own = *d;
  own.flags &= ~TCCL_GEMM_ARRIVALS;  // `sync` is this function's
  return allgather_impl(&own, out, ld_out, heap, &sync, tr, variant, (int64_t)sizeof(StaticWords), (hipStream_t)stream);
}

int tccl_static_call_words(uint32_t call, int32_t tile_count, int32_t* epoch, int32_t* counter_start, int32_t* counter_ready) {
  if (call == 0 || tile_count < 0 || tile_count > TCCL_STATIC_MAX_TILES || !epoch || !counter_start || !counter_ready)
    return fail(TCCL_ERR_INVALID, "static_call_words: call numbers start at 1, tile_count within [0, %d]", TCCL_STATIC_MAX_TILES);
  static_call_words(call, tile_count, epoch, counter_start, counter_ready);
  return 0;
}

int tccl_word_reached(int32_t word, int32_t need) { return tccl::word_reached(word, need) ? 1 : 0; }

int tccl_mfma_rate_probe(int32_t kind, const void* a_like, int64_t a_bytes, const void* b_like, int64_t b_bytes, float* sink,
                         int32_t steps, int32_t workgroups, void* stream) {
  if (!a_like || !b_like || !sink) return fail(TCCL_ERR_INVALID, "mfma_rate_probe: NULL buffer");
  if (a_bytes < 32 || b_bytes < 32 || a_bytes % 32 || b_bytes % 32 || a_bytes > 0x7fffffffll || b_bytes > 0x7fffffffll)
    return fail(TCCL_ERR_INVALID, "mfma_rate_probe: operand buffers must hold a multiple of 32 bytes, below 2 GiB (got %lld, %lld)",
                (long long)a_bytes, (long long)b_bytes);
  if (steps < 0 || workgroups < 1) return fail(TCCL_ERR_INVALID, "mfma_rate_probe: steps=%d, workgroups=%d", steps, workgroups);
  const dim3 grid(workgroups), block(tccl::kThreads256);
  const char* a = (const char*)a_like;
  const char* b = (const char*)b_like;
  const uint32_t an = (uint32_t)a_bytes, bn = (uint32_t)b_bytes;
  hipStream_t st = (hipStream_t)stream;
  switch (kind) {
    case TCCL_PROBE_F16_32X32X16: hipLaunchKernelGGL((tccl::mfma_rate_wide_kernel<_Float16>), grid, block, 0, st, a, an, b, bn, sink, steps); break;
    case TCCL_PROBE_F16_16X16X32: hipLaunchKernelGGL((tccl::mfma_rate_kernel<_Float16>), grid, block, 0, st, a, an, b, bn, sink, steps); break;
    case TCCL_PROBE_BF16_16X16X32: hipLaunchKernelGGL((tccl::mfma_rate_kernel<__bf16>), grid, block, 0, st, a, an, b, bn, sink, steps); break;
    case TCCL_PROBE_F8_16X16X128: hipLaunchKernelGGL((tccl::mfma_rate_kernel<tccl::fp8e4m3>), grid, block, 0, st, a, an, b, bn, sink, steps); break;
    case TCCL_PROBE_F8_32X32X64: hipLaunchKernelGGL((tccl::mfma_rate_wide_kernel<tccl::fp8e4m3>), grid, block, 0, st, a, an, b, bn, sink, steps); break;
    default: return fail(TCCL_ERR_INVALID, "mfma_rate_probe: unknown kind %d", kind);
  }
  TCCL_HIP(hipGetLastError());
  return 0;
}

int tccl_static_reset(void* stream) {
  StaticScratch* sc = nullptr;
  int rc = static_scratch(&sc);
  if (rc) return rc;
  int device = -1;
  TCCL_HIP(hipGetDevice(&device));
  {
    std::lock_guard<std::mutex> hold(g_scratch_mutex);
    for (int r = 0; r < TCCL_MAX_WORLD; ++r) g_static_calls[device][r] = 0;
  }
  return tccl_fill_i32((int32_t*)sc->words, (int64_t)(sizeof(sc->words) / sizeof(int32_t)), 0, stream);
}

// Column shards of M rows that are no whole plan tiles: no signals, so the peers' partials have to be there.
static int reduce_ragged_shards(const tccl_gemm_desc* d, void* out, int32_t out_dtype, int64_t ld_out, const tccl_heap_view* heap,
                                const tccl_sync_desc* sync, const tccl_transport_desc* tr, int32_t mode, hipStream_t stream) {
  if (!(mode & TCCL_RS_PEERS_RESIDENT))
    return fail(TCCL_ERR_INVALID, "reducescatter: column shards of %d rows carry no signals (plan tiles have %d rows): the peers must be resident",
                d->M / d->column_shards, d->block_m);
  tccl_device_info dev;
  int rc = query_device(-1, &dev);
  if (rc) return rc;
  tccl::GemmArgs g;
  build_gemm_args(d, dev, &g);
  tccl::CommArgs c;
  fill_comm_common(&c, g, (int)dtype_size(d->out_dtype), heap, sync, tr);
  if ((rc = fill_reduce(&c, d->C, d->out_dtype, out, out_dtype, ld_out, d->M, d->N, heap->world_size, mode))) return rc;
  if ((rc = check_task_elems(tr, true, c.esize)) || (rc = check_comm_span(c))) return rc;
  const int shape = stream_shape(d, nullptr, tr, TCCL_S0_BULK, g.wrap_rows, dev);
  if (shape >= 0) {
    tccl::StreamArgs a;
    build_stream(d, g, g.wrap_rows, dev, &a);
    add_stream_reduce(c, d, &a);
    return stream_status(tccl::launch_stream(d->in_dtype, g.b_kmajor != 0, shape, a, stream));
  }
  // All column blocks in one launch, each with tile rows of its own, or, where they are large enough to fill the device,
  // one GEMM per block (four blocks of 1956 x 696 x 2096: 42 us with the sums, 119 us one after the other); then the
  // reduction.
  tccl_gemm_desc one = *d;
  one.M = g.wrap_rows;
  one.column_shards = 0;
  const TileChoice together = choose_tiles(d, g.wrap_rows, d->column_shards, false, false, dev);
  const double apart = d->column_shards * (kLaunchUs + choose_tiles(&one, one.M, 1, plan_tile_fits_macro(&one), false, dev).us);
  if (d->block_m == 128 && d->block_n == 128 && d->macro_tile != 256 && together.us < apart) {
    g.ragged = 1;
    g.tile_rows = (g.wrap_rows + 127) / 128 * d->column_shards;
    tccl::SignalArgs s;
    memset(&s, 0, sizeof s);
    if (sums_across(d, c, together.kernel, g.tile_rows * g.tile_cols, dev.compute_units)) return launch_across(d, g, s, c, nullptr, stream);
    rc = launch_fused(d, g, s, c, together.kernel, tile_wgs(together.kernel, d, dev, g.tile_rows * g.tile_cols), 0,
                      nullptr, stream);
    return rc ? rc : launch_bulk(c, dev, stream);
  }
  const size_t isz = dtype_size(d->in_dtype);
  for (int q = 0; q < d->column_shards; ++q) {
    one.B = (const char*)d->B + (int64_t)q * d->N * (g.b_kmajor ? d->ldb : 1) * (int64_t)isz;
    one.C = (char*)d->C + (int64_t)q * g.wrap_rows * d->ldc * c.esize;
    if ((rc = tccl_gemm(&one, stream))) return rc;
  }
  return launch_bulk(c, dev, stream);
}

int tccl_gemm_reducescatter(const tccl_gemm_desc* d, void* out, int32_t out_dtype, int64_t ld_out,
                            const tccl_heap_view* heap, const tccl_sync_desc* sync, const tccl_transport_desc* tr,
                            int32_t emulate_peer, int32_t variant, void* stream) {
  int rc = check_gemm(d, true);
  if (rc) return rc;
  if ((rc = check_heap(heap))) return rc;
  if (variant < TCCL_S0_BULK || variant > TCCL_S2_TILEGROUP) return fail(TCCL_ERR_INVALID, "unknown variant %d", variant);
  if (!out || ld_out < d->N) return fail(TCCL_ERR_INVALID, "reducescatter: bad output");
  const int esize = (int)dtype_size(d->out_dtype);
  const int shard = d->M / heap->world_size;
  const bool ragged = d->column_shards > 1 && d->column_shards == heap->world_size && d->M % heap->world_size == 0 && shard % d->block_m;
  if (d->flags & TCCL_GEMM_A_COLUMNS) return fail(TCCL_ERR_UNSUPPORTED, "reducescatter: A given by columns");
  if (!ragged && (rc = check_sync(sync, variant))) return rc;
  if (ragged) {
    tccl_gemm_desc own = *d;
    if (variant == TCCL_S0_BULK) own.flags &= ~TCCL_GEMM_OWN_ROWS_IN_REGISTERS;  // S0 stores every partial
    return reduce_ragged_shards(&own, out, out_dtype, ld_out, heap, sync, tr, emulate_peer, (hipStream_t)stream);
  }
  if (d->M % heap->world_size || shard % d->block_m)
    return fail(TCCL_ERR_INVALID, "reducescatter: M=%d must split into world_size=%d shards of whole %d-row plan tiles", d->M, heap->world_size, d->block_m);
  tccl_device_info dev;
  if ((rc = query_device(-1, &dev))) return rc;
  tccl::GemmArgs g;
  build_gemm_args(d, dev, &g);
  tccl::CommArgs c;
  fill_comm_common(&c, g, esize, heap, sync, tr);
  if ((rc = fill_reduce(&c, d->C, d->out_dtype, out, out_dtype, ld_out, d->M, d->N, heap->world_size, emulate_peer))) return rc;
  if ((rc = set_task_units(&c, tr, true))) return rc;
  return run_variant(d, c, sync, tr, variant, dev, g, (hipStream_t)stream);
}

}  // extern "C"
