// Persistent MFMA GEMM role for gfx950 (CDNA4), 16-bit inputs, 128 x 128 tiles.
//
// One workgroup = 256 threads = 4 wavefronts (2 x 2, wave tile 64 x 64), producing 128 x 128
// output sub-tiles with K consumed 32 at a time through three (or five) LDS stages of 16 KiB.  A plan tile
// (block_m x block_n, multiples of 128) is a small loop of such sub-tiles; when the whole plan
// tile is in memory the workgroup publishes it (per-tile lock or per-TileGroup counter).
// 48 KiB of LDS and <= 168 registers per lane let three workgroups share a CU (two that multiply
// and one that moves data, in the fused launches), each with one wavefront per SIMD and barriers
// of its own, so that one workgroup's waits are covered by the others' MFMAs.  The GEMM alone runs
// a five-stage form (80 KiB, two workgroups per CU).
//
// Data path of one K step
//   global --buffer_load_dwordx4 ... lds--> LDS stage --ds_read--> operands of v_mfma_f32_16x16x32
//   A stage: 128 rows x 64 B (32 k); 16-byte chunk kc of row r sits in slot kc ^ ((r >> 1) & 3).  (Measured
//            with the LDS saturated by eight wavefronts: a ds_read_b128 of rows l % 16, chunk l / 16 takes
//            1.78 times as long with ((r >> 2) & 3) or with no swizzle at all, and no longer than a
//            conflict-free read with this term.)
//   B stage: 32 k rows x 256 B (128 columns); chunk c of row k in slot c ^ 4 (k & 3) ^ 2 ((k >> 3) & 1);
//            operands come out through ds_read_b64_tr_b16 (the transposing read: within 16 lanes,
//            lane i supplies 4 columns of k row i / 4, lane j receives 4 k of column j), two per operand.
//   The hardware writes lane l's 16 bytes at base + 16 l, so the swizzles are applied on the global
//   side, by the choice of the chunk a lane fetches.  Rows >= M, columns >= N and k >= K read as
//   zero through the buffer bounds (A chunks at k >= K are redirected past the buffer's end).
//   A k-major B (GemmArgs::b_kmajor: element (k, n) at B[n * ldb + k]) takes A's route and layout.
//   A given by columns (kAColumns: element (m, k) at A[k * lda + m]; the input of a weight gradient) takes a
//   row-major B's, 128 rows wide: its operands come out through the transposing reads as well.  1000 x 2064 x 1003 pushed to one
//   peer: 15.5 us, and 21.6 where a launch of its own turns A into rows first.
//
// Pipeline (S stages: 3 in the fused launches, 5 in the GEMM-only kernel): step t computes from stage
// t % S and issues the loads of K step t + S - 1 into stage (t - 1) % S, which every wavefront finished
// reading before the barrier of step t - 1; one load per item, four items per step (one 16-row block of A
// against the four 16-column blocks of B).  The step's one barrier sits before its last item and waits
// with vmcnt(4 (S - 2) - 1): the loads of the last S - 2 steps may stay in flight, those of K step t + 1
// have landed.  Behind it the last item already fetches the next step's first operands, and reloads each
// B operand in place once its MFMA is issued.
// What bounds the tile shape: per K step a CU's address unit takes in 16 KiB (256 clocks at 64 B/clk) and
// its LDS 16 KiB of writes and 32 KiB of reads, against 256 clocks of MFMAs: all three are level, where
// the 256 x 256 tile has half the traffic per FLOP.  Measured at 4096 x 4096 x 1024: 41 us as it is,
// 29 us without the global loads, 36 us without the LDS reads, 24 us with neither (and no barrier).
//
// MFMA orientation: the B operand is passed first, i.e. the instruction computes the transposed
// 16 x 16 block.  Each lane then owns 4 consecutive output columns of one output row, and the
// register -> LDS -> global epilogue moves 8 / 16 bytes per access.
//
// Reference semantics reproduced: C = A @ B with fp32 accumulation and one rounding to
// the output type (tileccl/kernels/gemm.py:139-167); rows/columns past M/N are not
// written (gemm.py:163-167); the K tail is zero-filled (gemm.py:153-160).
#pragma once

#include <type_traits>

#include "tccl_comm.h"
#include "tccl_device.h"

namespace tccl {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kTile = 128;                        // sub-tile edge
constexpr int kThreads = 256;                     // threads per workgroup
constexpr int kStage128 = 16384;                  // a K step of 32: A 128 x 64 B, B 32 x 256 B
constexpr int kStageDeep = 32768;                 // a K step of 64: A 128 x 128 B, B 64 x 256 B
constexpr int kThreadsWide = 512;                 // wide form
constexpr int kStageWide = 49152;                 // a K step of 64: A 128 x 128 B, B 64 x 512 B

enum SignalMode { kSignalNone = 0, kSignalTile = 1, kSignalGroup = 2 };

struct GemmArgs {
  const void* A;
  const void* B;
  void* C;
  int M, N, K;
  int64_t lda, ldb, ldc;
  float alpha;
  int block_m, block_n, group_m;  // plan tile and swizzle band
  int tile_rows, tile_cols;       // plan tiles
  int xcds, span;                 // slot -> tile remap
  // Column shards stacked as row blocks (0: plain GEMM): C row block q of wrap_rows rows is
  // A (wrap_rows x K) times columns [q * N, (q + 1) * N) of B; tiles never straddle two blocks.
  int wrap_rows;
  // The row blocks are no whole tiles: each starts a tile row of its own (tile_rows counts them all).
  int ragged;
  union {
    // B is k-major: element (k, n) at B[n * ldb + k] (the `.t()` view of an (N, K) tensor).
    int b_kmajor;
    // Kernels for an A given by columns (element (m, k) at A[k * lda + m]; B is row-major): of the K columns it lacks the last
    // a_short, which read as zero.  (No word of its own: with more fields here the compiler laid out the large-tile
    // kernels, which read none of them, another way; 4096 x 4096 x 1024 gathered by rows 45.7 -> 46.4 us.)
    int a_short;
  };
  // Row-major B lacks its last b_short of the K rows: they read as zero (A is zero there as well).
  int b_short;
};

// Where a tile whose first output row is row0 and first output column col0 reads its operands.
struct OperandOrigin {
  int a_row, a_rows;  // first row of A, rows A has
  int b_col, b_cols;  // first column of B, columns B has
};
TCCL_HD OperandOrigin operand_origin(const GemmArgs& g, int row0, int col0) {
  OperandOrigin o;
  if (g.wrap_rows > 0) {
    int wrap_rows = g.wrap_rows;
#if defined(__HIP_DEVICE_COMPILE__)
    // Hidden from the optimiser: it would otherwise prepare this division (a reciprocal and its
    // corrections) at the kernel's start for every launch, column shards or not.
    asm volatile("" : "+s"(wrap_rows));
#endif
    const int q = row0 / wrap_rows;
    o.a_row = row0 - q * wrap_rows;
    o.a_rows = wrap_rows;
    o.b_col = col0 + q * g.N;
    o.b_cols = (g.M / wrap_rows) * g.N;
  } else {
    o.a_row = row0;
    o.a_rows = g.M;
    o.b_col = col0;
    o.b_cols = g.N;
  }
  return o;
}

struct SignalArgs {
  int mode;
  int32_t* locks;
  const int32_t* group_table;
  int32_t* counter;
  const int32_t* tile_counts;
  int epoch;  // launch number: locks[tile] = epoch (tile mode); a group is complete at epoch * tile_counts[g]
  // optional device trace: the producer that completes a group stamps its clock
  int64_t* trace_ready_clock;
};

// all-scatter / all-gather folded into the GEMM: the tile goes out from the staging LDS it
// already sits in, instead of being written, signalled, re-read and copied by a second party
// (reference: the per-tile scatter of patterns/_helpers.py:86-199, tile_allgather of
// primitives/collectives.py:613-663).
struct PushArgs {
  int world;           // ranks; every rank but `rank` is a target.  0: the epilogue writes C only
  int rank;
  int col_lo, col_hi;  // columns of C that travel
  int col_shift;       // target column = C column + col_shift
  int64_t ld;          // target pitch in elements
  const int64_t* heap_bases;  // C's address inside target q is C + heap_bases[q] - heap_bases[rank]
};

// Counters of neighbouring plan tiles in one cache line take each other's time: 256 tiles of one launch counting into 16
// words of a line or two cost it 2.2 us (512 x 512 x 256, two ranks: 8.3 -> 6.0 us; 16 x 2048 x 4096 9.2 -> 8.5).
constexpr int kArrivalStride = 32;
// Of a plan tile's words a launch counts in one that no launch near it in number uses, and neither does the other kind of
// launch, which is numbered separately: launches of the same words that overlap (two streams), whatever their tile shapes, do not
// add to each other's counts, so each of them leaves zero behind and publishes a plan tile exactly when it is complete.
TCCL_HD int arrival_word(int plan_tile, int32_t epoch, bool by_tile) {
  constexpr int kHalf = kArrivalStride / 2;
  return kArrivalStride * plan_tile + (int)((uint32_t)epoch % kHalf) + (by_tile ? kHalf : 0);
}

// Reduce-scatter carried out in the epilogue of the GEMM: the tiles of rows this rank owns take the peers' partials
// and leave as output; under single-GPU emulation the other owners' rows are reduced as well.
struct EpilogueReduce {
  int active, emulate_peer;
  int peers_resident;    // the peers' partials are complete in memory: their words are not looked at
  int own_in_registers;  // own rows: no partial is stored
  int out_dtype;
  int rank, world, shard_rows;
  const int64_t* heap_bases;
  char* out;             // this rank's output shard (the partial is the GEMM's C)
  int64_t ld_out_bytes;
  const int32_t* locks;  // this rank's words; a peer's sit at the same slice offset
  const int32_t* counter;
  const int32_t* tile_counts;
  int64_t* fault;
  int64_t spin_ticks;
  int band;              // sub-tiles across the owners: rows of sub-tiles in a band (tile_coords())
  uint32_t* arrivals;    // kArrivalStride words per plan tile (arrival_word()), zero between launches
};

// Columns of a sub-tile across the owners (its rows: 16384 over that).  A row-major B is read in runs of an owner's columns:
// those of four ranks get 64, whole lines where a shard's rows start on them, in a sub-tile of 64 x 256.  With runs of 32 they take as long per K step,
// with a quarter less to read; the eight ranks' runs of 16 take half as long again (sums_across()).
TCCL_HD constexpr int across_cols(int world, bool b_kmajor) { return world == 4 && !b_kmajor ? 256 : 128; }

template <typename T>
struct Mfma;
template <>
struct Mfma<_Float16> {
  typedef f16x8 Vec;
  static TCCL_D f32x16 run(Vec a, Vec b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
  // 16 x 16 x 32: lane l holds 8 consecutive k (group l / 16) of row / column l % 16 and gets
  // D[4 * (l / 16) + e][l % 16], e = 0..3.
  static TCCL_D f32x4 run16(Vec a, Vec b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
};
template <>
struct Mfma<__bf16> {
  typedef bf16x8 Vec;
  static TCCL_D f32x16 run(Vec a, Vec b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
  static TCCL_D f32x4 run16(Vec a, Vec b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
};

// OCP fp8 e4m3 ("e4m3fn"), the 8-bit input type of gfx950's v_mfma_f32_32x32x64_f8f6f4.
struct fp8e4m3 {
  uint8_t bits;
};
typedef int i32x8 __attribute__((ext_vector_type(8)));
#if defined(__HIP_DEVICE_COMPILE__)
template <>
struct Mfma<fp8e4m3> {
  typedef i32x8 Vec;  // 32 consecutive k of one row / column
  // cbsz = blgp = 0 selects e4m3 for both operands; zero scale operands select the unscaled form.
  static TCCL_D f32x16 run(Vec a, Vec b, f32x16 c) { return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0); }
  // 16 x 16 x 128: lane l holds 32 consecutive k (group l / 16) of row / column l % 16 and gets
  // D[4 * (l / 16) + e][l % 16], e = 0..3.
  static TCCL_D f32x4 run16(Vec a, Vec b, f32x4 c) { return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0); }
};
#endif

// fp32 -> output element, round to nearest even (what a cast of the accumulator does in
// the reference, gemm.py:167 / bulk_sync.py:238).
template <typename OutT>
TCCL_D OutT to_out(float v);
template <>
TCCL_D _Float16 to_out<_Float16>(float v) { return (_Float16)v; }
template <>
TCCL_D __bf16 to_out<__bf16>(float v) { return (__bf16)v; }
template <>
TCCL_D float to_out<float>(float v) { return v; }

#if defined(__HIP_DEVICE_COMPILE__)
// Request every 64-byte line of the kernel arguments at once.  The compiler reads arguments
// where it first needs them, each group of reads followed by its own wait, so a kernel's
// start used to be a chain of a dozen dependent trips to memory before the first operand load
// could go out; after this the later reads hit in the scalar cache.
template <int kBytes>
TCCL_D void warm_kernargs() {
  typedef const __attribute__((address_space(4))) uint32_t* Words;
  Words p = (Words)__builtin_amdgcn_kernarg_segment_ptr();
  uint32_t any = 0;
#pragma unroll
  for (int o = 0; o < kBytes; o += 64) any |= p[o / 4];
  asm volatile("" ::"s"(any));
}

// kWorld: sub-tiles across the owners of a reduce-scatter of so many column shards (run_across()).
template <typename InT, typename OutT, int kStages = 3, int kWaves = 4, int kHalves = 1, int kWorld = 0, int kWn = kWaves / 2>
struct GemmRole {
  static constexpr int kCols = 64 * kWn, kRows = 64 * (kWaves / kWn);  // of a sub-tile (kWn: wavefronts across)
  // Column block cb of wavefront wn: columns 64 wn + 16 cb .. + 15, or, spread, 64 cb + 16 wn .. + 15: every wavefront has a
  // part of each owner's run of 64.
  static constexpr bool kSpread = kWorld == 4 && kWn == 4;
  static constexpr int kStepK = 32 * kHalves;
  static constexpr int kRowB = 2 * kStepK;                      // bytes of an A row in a stage
  static constexpr int kRowLanes = kRowB / 16;                  // lanes that fetch one
  static constexpr int kAStage = kRows * kRowB;
  static constexpr int kBPitch = kCols * 2;                     // bytes of a k row of B in a stage
  static constexpr int kStage = kAStage + kStepK * kBPitch;
  static constexpr int kBLanes = kBPitch / 16;                  // lanes that fetch a k row of B
  static constexpr int kAPitch = kRows * 2, kALanes = kAPitch / 16;  // of a k row of an A given by columns
  static constexpr int kALoads = kAStage / 1024 / kWaves;           // 1 KiB pieces per wavefront and step
  static constexpr int kBLoads = kStepK * kBPitch / 1024 / kWaves;
  static constexpr int kLoads = kALoads + kBLoads;
  typedef typename Mfma<InT>::Vec Vec;
  static_assert(sizeof(InT) == 2, "16-bit inputs");
  typedef __attribute__((address_space(3))) void LdsVoid;
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  typedef __attribute__((address_space(3))) s16x4 LdsQuad;

  const GemmArgs& g;
  const PushArgs& push;  // world == 0: nothing leaves from the epilogue
  const EpilogueReduce& reduce;
  char* st0;
  char* st1;
  char* st2;
  char* st3;  // (forms of four and five stages)
  char* st4;
  const int tid, lane, wave, wm, wn;

  // The wavefront's number lives in a scalar register: the LDS addresses its loads land at derive from it.
  TCCL_D GemmRole(const GemmArgs& args, const PushArgs& push_args, const EpilogueReduce& reduce_args, char* s0, char* s1, char* s2,
                  char* s3 = nullptr, char* s4 = nullptr)
      : g(args), push(push_args), reduce(reduce_args), st0(s0), st1(s1), st2(s2), st3(s3), st4(s4), tid(threadIdx.x), lane(threadIdx.x & 63),
        wave(__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6))), wm(wave / kWn), wn(wave % kWn) {}

  static TCCL_D int fresh(int v) {
    asm volatile("" : "+v"(v));
    return v;
  }
  static TCCL_D uint32_t clamp_u32(int64_t v) { return v > 0xffffffffll ? 0xffffffffu : (v < 0 ? 0u : (uint32_t)v); }

  // ---- global -> LDS ------------------------------------------------------------------------
  // Per K step a wavefront fetches two 1 KiB pieces of A and kBLoads of B (wide form in brackets):
  //   A piece i: rows 16 [8] (2 wave + i) .. + 15 [7]    (lane l: row + l / 4 [8], slot l % 4 [8])
  //   B piece j: k rows 4 (2 wave + j) .. + 3            (lane l: k row + l / 16, slot l % 16)
  //              [2 (4 wave + j), + 1                    (lane l: k row + l / 32, slot l % 32)]
  //   k-major B piece j: columns as A's rows.
  struct Source {
    __amdgpu_buffer_rsrc_t a, b;
    uint32_t off_a[kALoads], off_b[kBLoads];  // byte offsets of this lane's 16-byte loads, K step 0
    uint32_t step_a, step_b;            // byte advance per K step
    int k_lane[2];                      // first k of this lane's chunk of a row of piece 0 / 1 (even / odd pieces) within a step
  };
  // Swizzle of an A row (of a k-major B row) in a stage: 16-byte chunk c in slot c ^ swizzle(row).
  static TCCL_D int swizzle(int row) { return (row >> 1) & (kRowLanes - 1); }

  // Column `c` of a sub-tile, as one of B's counted from the sub-tile's first: across the owners, equal runs of every shard.
  TCCL_D int64_t across(int c) const {
    if constexpr (kWorld == 0) return c;
    return (int64_t)(c / kRun) * g.N + c % kRun;
  }

  template <bool kBKMajor, bool kAColumns>
  TCCL_D Source make_source(int row0, int col0) const {
    Source s;
    const int ln = fresh(lane);
    OperandOrigin o = operand_origin(g, kWorld ? 0 : row0, col0);
    if constexpr (kWorld != 0) o.a_row = row0;
    const InT* A = (const InT*)g.A + (kAColumns ? (int64_t)o.a_row : (int64_t)o.a_row * g.lda);
    const InT* B = (const InT*)g.B + (kBKMajor ? (int64_t)o.b_col * g.ldb : (int64_t)o.b_col);
    const int64_t a_elems = kAColumns ? (int64_t)(g.K - 1 - g.a_short) * g.lda + (o.a_rows - o.a_row) : (int64_t)(o.a_rows - 1 - o.a_row) * g.lda + g.K;
    s.a = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, clamp_u32(a_elems * 2), 0x00020000);
    const int64_t b_elems = kBKMajor ? (int64_t)(o.b_cols - 1 - o.b_col) * g.ldb + g.K : (int64_t)(g.K - 1 - g.b_short) * g.ldb + (o.b_cols - o.b_col);
    s.b = __builtin_amdgcn_make_buffer_rsrc((void*)B, 0, clamp_u32(b_elems * 2), 0x00020000);
    constexpr int kPiece = 64 / kRowLanes;  // rows of a piece
#pragma unroll
    for (int i = 0; i < 2; ++i) s.k_lane[i] = ((ln % kRowLanes) ^ swizzle(kPiece * i + ln / kRowLanes)) * 8;
#pragma unroll
    for (int i = 0; i < kALoads; ++i) {
      if constexpr (kAColumns) {
        const int k = 64 / kALanes * (kALoads * wave + i) + ln / kALanes;
        s.off_a[i] = (uint32_t)(k * g.lda * 2 + ((ln % kALanes) ^ (4 * (k & 3)) ^ (2 * ((k >> 3) & 1))) * 16);
      } else {
        s.off_a[i] = (uint32_t)((kPiece * (kALoads * wave + i) + ln / kRowLanes) * g.lda * 2 + s.k_lane[i & 1] * 2);
      }
    }
#pragma unroll
    for (int j = 0; j < kBLoads; ++j) {
      if constexpr (kBKMajor) {
        const int row = kPiece * (kBLoads * wave + j) + ln / kRowLanes;
        s.off_b[j] = (uint32_t)(across(row) * g.ldb * 2 + s.k_lane[j & 1] * 2);
      } else {
        const int k = 64 / kBLanes * (kBLoads * wave + j) + ln / kBLanes;
        const int c = (ln % kBLanes) ^ (4 * (k & 3)) ^ (2 * ((k >> 3) & 1));
        s.off_b[j] = (uint32_t)(k * g.ldb * 2 + across(c * 8) * 2);
      }
    }
    s.step_a = kAColumns ? (uint32_t)(kStepK * g.lda * 2) : (uint32_t)(kStepK * 2);
    s.step_b = kBKMajor ? (uint32_t)(kStepK * 2) : (uint32_t)(kStepK * g.ldb * 2);
    return s;
  }

  // Piece i of K step kt, straight into `stage`.
  template <bool kAColumns>
  TCCL_D void issue_a(char* stage, const Source& s, int kt, int i) const {
    const bool dead = !kAColumns && kt * kStepK + s.k_lane[i & 1] >= g.K;  // (by columns: those >= K lie past the end of the buffer)
    const uint32_t oa = dead ? 0xfffffff0u : s.off_a[i] + kt * s.step_a;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(s.a, (LdsVoid*)(stage + (kALoads * wave + i) * 1024), 16, oa, 0, 0, 0);
  }
  template <bool kBKMajor>
  TCCL_D void issue_b(char* stage, const Source& s, int kt, int i) const {
    uint32_t ob = s.off_b[i] + kt * s.step_b;  // row-major B: rows >= K lie past the end of the buffer
    if constexpr (kBKMajor) ob = (kt * kStepK + s.k_lane[i & 1] >= g.K) ? 0xfffffff0u : ob;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(s.b, (LdsVoid*)(stage + kAStage + (kBLoads * wave + i) * 1024), 16, ob, 0, 0, 0);
  }
  // Load number n of a K step: A 0, B 0, A 1, B 1, then the rest of B.
  template <bool kBKMajor, bool kAColumns>
  TCCL_D void issue(char* stage, const Source& s, int kt, int n) const {
    if (n < 2 * kALoads && !(n & 1))
      issue_a<kAColumns>(stage, s, kt, n >> 1);
    else
      issue_b<kBKMajor>(stage, s, kt, n < 2 * kALoads ? n >> 1 : n - kALoads);
  }
  template <bool kBKMajor, bool kAColumns>
  TCCL_D void issue_step(char* stage, const Source& s, int kt) const {
#pragma unroll
    for (int n = 0; n < kLoads; ++n) issue<kBKMajor, kAColumns>(stage, s, kt, n);
  }

  // ---- LDS -> MFMA operands -------------------------------------------------------------------
  // 16 x 16 x 32 operands: lane l holds the 8 consecutive k of group l / 16 for row (column) l % 16.
  // (the wide form's second 32-k half: A chunks 4 + group, i.e. bit 2 of the slot flipped; B k rows 32 further on)
  struct Reader {
    uint32_t a_base;   // this lane's row of A row block 0, slot applied
    uint32_t b_base0;  // this lane's address for column block 0
  };
  template <bool kBKMajor, bool kAColumns>
  TCCL_D Reader make_reader() const {
    const int i16 = lane & 15, kg = lane >> 4;
    Reader r;
    if constexpr (kAColumns) {
      const int t = i16 >> 2, cq = i16 & 3;
      r.a_base = (uint32_t)((8 * kg + t) * kAPitch + ((wm * 8 + (cq >> 1)) ^ (4 * t) ^ (2 * (kg & 1))) * 16 + (cq & 1) * 8);
    } else {
      r.a_base = (uint32_t)((wm * 64 + i16) * kRowB + ((kg ^ swizzle(i16)) << 4));
    }
    if constexpr (kBKMajor) {
      r.b_base0 = (uint32_t)(kAStage + (wn * 64 + i16) * kRowB + ((kg ^ swizzle(i16)) << 4));
    } else {
      // Lane group kg covers k rows 8 kg .. + 7 in two transposing reads (k + 0, k + 4).
      const int t = i16 >> 2, cq = i16 & 3;
      const int chunk = (wn * (kSpread ? 2 : 8) + (cq >> 1)) ^ (4 * t) ^ (2 * (kg & 1));
      r.b_base0 = (uint32_t)(kAStage + (8 * kg + t) * kBPitch + chunk * 16 + (cq & 1) * 8);
    }
    return r;
  }
  // Two transposing reads, at `p` and four k rows of `pitch` bytes further on.
  static TCCL_D Vec turned(const char* p, int pitch) {
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsQuad*)p);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsQuad*)(p + 4 * pitch));
    return __builtin_bit_cast(Vec, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  }
  template <bool kAColumns>
  TCCL_D Vec load_a(const char* stage, const Reader& r, int h, int rb) const {
    if constexpr (kAColumns) return turned(stage + (r.a_base ^ (uint32_t)(32 * rb)) + 32 * h * kAPitch, kAPitch);
    return *(const Vec*)(stage + (r.a_base ^ (uint32_t)(64 * h)) + rb * 16 * kRowB);
  }
  template <bool kBKMajor>
  TCCL_D Vec load_b(const char* stage, const Reader& r, int h, int cb) const {
    if constexpr (kBKMajor) return *(const Vec*)(stage + (r.b_base0 ^ (uint32_t)(64 * h)) + cb * 16 * kRowB);
    // column block cb: two chunks further on, spread eight (the XOR commutes with the swizzle terms)
    return turned(stage + (r.b_base0 ^ (uint32_t)((kSpread ? 128 : 32) * cb)) + 32 * h * kBPitch, kBPitch);
  }

  struct Frags {
    Vec fa[4], fb[4];
  };

  // One K step: four items per 32-k half (A row block rb against the four B column blocks).  On entry fa[0], fa[1]
  // and fb[0..3] hold this step's operands; items 0 and 1 of a half fetch fa[2] and fa[3]; its last item
  // fetches the next half's fa[0], fa[1] and reloads each fb in place, the step's last item, behind the
  // barrier, from `nxt`.  The loads of K step kt_load into `far` (the stage read during the step before) go out one per
  // item: a wavefront issues nothing else while the address unit accepts its load, and the wavefronts reach an item
  // together.  At the barrier the loads that may still be in flight are those of the kStages - 2 steps before
  // (four-wavefront form: less the fourth one, which goes out behind the barrier).
  static constexpr int kItems = 4 * kHalves;
  static constexpr int kInFlight = kLoads * (kStages - 2) - (kLoads >= kItems ? 1 : 0);
  // kLeft > 0: one of the last steps of a sub-tile across the owners, behind request_sums(): no loads go out any more and
  // `kLeft - 1` steps follow; what has been requested stays in flight.
  template <bool kBKMajor, bool kAColumns, int kLeft = 0>
  TCCL_D void k_step(const char* cur, const char* nxt, char* far, const Source& src, const Reader& rd, int kt_load,
                     f32x4 (&acc)[4][4], Frags& f) const {
#pragma unroll
    for (int it = 0; it < kItems; ++it) {
      const int rb = it & 3, h = it >> 2;
      const bool last = it == kItems - 1;
      const char* from = last ? nxt : cur;  // of the next half's operands
      const int hn = last ? 0 : h + 1;
      if (last && kLeft > 0) {
        if (kLeft == 1) {
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        } else {
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((kLeft == 3 ? kLoads : 0) + kAddends) : "memory");
        }
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      } else if (last) {
        // The loads of K step t + 1 (into `nxt`) have landed; this wavefront's reads of `cur` are done.
        // The barrier is the bare instruction (__syncthreads() carries a release fence); the empty asm
        // keeps LDS accesses from moving across it.
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kInFlight) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
      if (rb == 3 && last && kLeft == 1) {
      } else if (rb == 3) {
        f.fa[0] = load_a<kAColumns>(from, rd, hn, 0);
        f.fa[1] = load_a<kAColumns>(from, rd, hn, 1);
      } else if (rb < 2) {
        f.fa[rb + 2] = load_a<kAColumns>(cur, rd, h, rb + 2);
      }
      if (kLeft == 0 && it < kLoads) issue<kBKMajor, kAColumns>(far, src, kt_load, it);
      if (kLeft == 0 && it + kItems < kLoads) issue<kBKMajor, kAColumns>(far, src, kt_load, it + kItems);
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) {
        acc[rb][cb] = Mfma<InT>::run16(f.fb[cb], f.fa[rb], acc[rb][cb]);
        if (rb == 3) {
          __builtin_amdgcn_sched_barrier(0);
          if (!(last && kLeft == 1)) f.fb[cb] = load_b<kBKMajor>(from, rd, hn, cb);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // ---- accumulators -> LDS -> global -------------------------------------------------------
  // Block (rb, cb) of the wave tile: the lane holds row 16 rb + l % 16, columns 16 cb + 4 (l / 16) .. + 3.
  // Each wavefront stages a 32-row slab (two row blocks) in its own 8 KiB window and writes it out
  // with 16-byte stores that are contiguous along the row; a wavefront's LDS operations execute in
  // the order issued, so nothing inside the loop waits for another wavefront.
  // kReduce: the launch is a reduce-scatter that reduces here; `sums`: this sub-tile's rows are summed (its owner is this
  // rank, or emulated, and the peers' partials are there).
  template <int kPolicy, bool kReduce>
  TCCL_D void epilogue(int row0, int row_end, int col0, const f32x4 (&acc)[4][4], bool sums) const {
    constexpr int kEsz = sizeof(OutT);
    constexpr int kRowBytes = 64 * kEsz;       // one wave row: 64 columns
    constexpr int kChunks = kRowBytes / 16;    // 16-byte chunks per row (8 or 16)
    constexpr int kPerChunk = 16 / kEsz;       // elements per chunk
    constexpr int kWindows = kStage / 8192;  // 8 KiB per wavefront (fp32 worst case), in stages 0 and 1
    char* win = (wave < kWindows ? st0 : st1) + (wave % kWindows) * 8192;
    // The lane id is taken afresh: what the epilogue derives from it is invariant across tiles
    // and would otherwise be hoisted out of the tile loop and held in registers through the K loop.
    const int ln = fresh(lane);
    const int i16 = ln & 15, kg = ln >> 4;
    // Stores go through a buffer resource rooted at the sub-tile so that the cache policy
    // can be chosen: plain write-back when nobody waits for the tile, device-coherent
    // write-through when a communication workgroup will read it right after the signal.
    OutT* C = (OutT*)g.C + (int64_t)row0 * g.ldc + col0;
    const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc((void*)C, 0, 0xffffffffu, 0x00020000);
    const int owner = kReduce ? row0 / reduce.shard_rows : 0;
    const bool store = !(kReduce && sums && owner == reduce.rank && reduce.own_in_registers);
    __syncthreads();  // every wavefront has left the K loop's stages
#pragma unroll
    for (int bi = 0; bi < 2; ++bi) {
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
          const int row = 16 * r + i16;
          OutT v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = to_out<OutT>(acc[2 * bi + r][cb][e] * g.alpha);
          const int byte = (16 * cb + 4 * kg) * kEsz;
          const int chunk = (byte >> 4) ^ (row & 7);
          char* p = win + row * kRowBytes + chunk * 16 + (byte & 15);
          if constexpr (kEsz == 2) {
            uint2 u;
            __builtin_memcpy(&u, v, 8);
            *(uint2*)p = u;
          } else {
            u32x4 u;
            __builtin_memcpy(&u, v, 16);
            *(u32x4*)p = u;
          }
        }
      asm volatile("" ::: "memory");  // staged by this wavefront itself: LDS keeps the order
      constexpr int kRounds = (32 * kChunks) / 64;
      u32x4 v[kRounds];
      int lrow[kRounds], lcol[kRounds];
      bool live[kRounds];
#pragma unroll
      for (int r = 0; r < kRounds; ++r) {
        const int idx = ln + 64 * r;
        const int row = idx / kChunks, chunk = idx % kChunks;
        v[r] = *(const u32x4*)(win + row * kRowBytes + ((chunk ^ (row & 7)) * 16));
        lrow[r] = wm * 64 + bi * 32 + row;
        lcol[r] = wn * 64 + chunk * kPerChunk;
        live[r] = row0 + lrow[r] < row_end && col0 + lcol[r] < g.N;
        if (kReduce && !store) continue;
        if (live[r]) __builtin_amdgcn_raw_buffer_store_b128(v[r], rc, (uint32_t)((lrow[r] * g.ldc + lcol[r]) * kEsz), 0, kPolicy);
      }
      if (kReduce && sums) {
        // The owner's partial first, then the other ranks ascending; this rank's is the value as it would be stored.
        const int64_t my_base = reduce.heap_bases[reduce.rank];
        const __amdgpu_buffer_rsrc_t to = window((int64_t)(uintptr_t)reduce.out + (reduce.heap_bases[owner] - my_base) +
                                                 (int64_t)(row0 - owner * reduce.shard_rows) * reduce.ld_out_bytes + (int64_t)col0 * 2);
        // The addends of kBatch chunks from kPeers ranks are requested together.
        constexpr int kBatch = 4, kPeers = 4;
#pragma unroll
        for (int b = 0; b < kRounds; b += kBatch) {
          float sum[kBatch][kPerChunk];
          for (int i0 = 0; i0 < reduce.world; i0 += kPeers) {
            u32x4 w[kPeers][kBatch];
#pragma unroll
            for (int i = 0; i < kPeers; ++i) {
              const int n = i0 + i, p = n == 0 ? owner : (n <= owner ? n - 1 : n);
              if (n >= reduce.world) break;
              const __amdgpu_buffer_rsrc_t from = window((int64_t)(uintptr_t)C + (reduce.heap_bases[p] - my_base));
#pragma unroll
              for (int r = 0; r < kBatch; ++r)
                w[i][r] = p == reduce.rank ? v[b + r]
                                           : ld16<kCoherent>(from, live[b + r] ? (uint32_t)((lrow[b + r] * g.ldc + lcol[b + r]) * kEsz) : 0u);
            }
#pragma unroll
            for (int i = 0; i < kPeers; ++i) {
              if (i0 + i >= reduce.world) break;
#pragma unroll
              for (int r = 0; r < kBatch; ++r) {
                OutT e[kPerChunk];
                __builtin_memcpy(e, &w[i][r], 16);
#pragma unroll
                for (int j = 0; j < kPerChunk; ++j) sum[r][j] = i0 + i == 0 ? (float)e[j] : sum[r][j] + (float)e[j];
              }
            }
          }
#pragma unroll
          for (int r = 0; r < kBatch; ++r) {
            if (!live[b + r]) continue;
            const uint32_t off = (uint32_t)(lrow[b + r] * reduce.ld_out_bytes + lcol[b + r] * 2);
            uint16_t h[kPerChunk];
#pragma unroll
            for (int j = 0; j < kPerChunk; ++j)
              h[j] = reduce.out_dtype == kBF16 ? __builtin_bit_cast(uint16_t, (__bf16)sum[r][j])
                                               : __builtin_bit_cast(uint16_t, (_Float16)sum[r][j]);
            if constexpr (kPerChunk == 4) {
              typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
              u32x2 o;
              __builtin_memcpy(&o, h, 8);
              __builtin_amdgcn_raw_buffer_store_b64(o, to, off, 0, kStreaming);
            } else {
              u32x4 o;
              __builtin_memcpy(&o, h, 16);
              st16<kStreaming>(to, off, o);
            }
          }
        }
      }
      // Fused push: the same chunks go to every peer's slice from the registers they sit in; the tile is
      // never read back.  The signal that follows the tile's last store covers these stores as well.
      for (int t = 0; t < push.world; ++t) {
        if (t == push.rank) continue;
        const int64_t push_ld = push.ld;
        const int col_lo = push.col_lo, col_hi = push.col_hi;
        typedef const __attribute__((address_space(4))) int64_t* Bases;
        const int64_t delta = ((Bases)push.heap_bases)[t] - ((Bases)push.heap_bases)[push.rank];
        char* base = (char*)g.C + delta + ((int64_t)row0 * push_ld + col0 + push.col_shift) * kEsz;
        const __amdgpu_buffer_rsrc_t rt = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, 0xffffffffu, 0x00020000);
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
          const int col = col0 + lcol[r];
          if (live[r] && col >= col_lo && col < col_hi)
            __builtin_amdgcn_raw_buffer_store_b128(v[r], rt, (uint32_t)((lrow[r] * push_ld + lcol[r]) * kEsz), 0, kCoherent);
        }
      }
      asm volatile("" ::: "memory");
    }
  }

  // ---- sub-tiles across the owners: the sums -------------------------------------------------------------
  // Each owner has kRun of the columns.  The wavefronts that hold this rank's sum them; their addends are requested three K
  // steps before the last one ends.
  static constexpr int kRun = kWorld ? kCols / (kWorld ? kWorld : 1) : 16;
  static constexpr int kOwnCols = kSpread ? 16 : kRun, kOwners = 64 / kOwnCols;  // of an owner in a wavefront; owners there
  static constexpr int kOwnChunks = kOwnCols / 4, kOwnRounds = 32 * kOwnChunks / 64;  // 16 bytes of fp32; per 32-row slab
  static constexpr int kAddends = 2 * kOwnRounds * (kWorld - 1);                  // per lane
  struct Addends {
    f32x4 v[2][kOwnRounds][kWorld > 1 ? kWorld - 1 : 1];
  };
  TCCL_D bool sums_here() const { return kSpread || wn == reduce.rank / kOwners; }
  // This lane's chunk of round r: row of the slab, column of the run.
  static TCCL_D int own_row(int ln, int r) { return (ln + 64 * r) / kOwnChunks; }
  TCCL_D int own_col(int ln) const { return (kSpread ? wn * kOwnCols : 0) + ln % kOwnChunks * 4; }  // (64 is a multiple of kOwnChunks)
  // Every wavefront issues the same loads, so that the waits behind them count the same everywhere; where there is nothing to sum they
  // fetch nothing.  (Under a branch the compiler waits for all of them before the next step's first operand.)  The peers' bases
  // come through scalar loads: a vector load's answer is waited for together with the operands under way, and each addend's
  // descriptor has to be made uniform first.  bf16 1000 x 4032 x 256 / 1024 x 4096 x 1000 k-major on eight ranks 13.7 / 21.4 -> 12.5 / 20.2
  // us, 512 x 4096 x 1000 on four 16.0 -> 15.1, 1500 x 2208 x 2048 on two 23.8 -> 23.0.
  // Where every wavefront sums (row-major, four ranks) the branch is none and the vector loads stay: without them the compiler moves
  // operands between register files in the K loop (1920 x 2048 x 904 20.6, 20.9 us with scalar ones).
  TCCL_D void request_sums(int row0, int col0, Addends& w) const {
    const int ln = (int)((uint32_t)fresh(lane) & 63u), rows = g.wrap_rows - row0, col = own_col(ln);
    const bool live = sums_here() && col < g.N - col0;
    const int64_t first = (int64_t)(uintptr_t)((const float*)g.C + ((int64_t)reduce.rank * g.wrap_rows + row0) * g.ldc + col0);
    const uint32_t pitch = (uint32_t)(g.ldc * 4);
    // A window ends with this rank's block (below 0xfffffff0: sums_across()), so that the offset of what does not exist is past it.
    const uint32_t end = kSpread ? 0xffffffffu : (uint32_t)(rows - 1) * pitch + (uint32_t)(g.N - col0) * 4u;
    const uint32_t nowhere = kSpread ? 0u : 0xfffffff0u;  // (kSpread: the first chunk instead, inside every window)
    typedef typename std::conditional<kSpread, const int64_t*, const __attribute__((address_space(4))) int64_t*>::type Bases;
    const Bases bases = (Bases)reduce.heap_bases;
#pragma unroll
    for (int n = 0; n < kWorld - 1; ++n) {
      const int p = n + (n >= reduce.rank);
      const __amdgpu_buffer_rsrc_t from =
          __builtin_amdgcn_make_buffer_rsrc((void*)(uintptr_t)(first + (bases[p] - bases[reduce.rank])), 0, end, 0x00020000);
#pragma unroll
      for (int bi = 0; bi < 2; ++bi)
#pragma unroll
        for (int r = 0; r < kOwnRounds; ++r) {
          const uint32_t row = wm * 64 + bi * 32 + own_row(ln, r);
          w.v[bi][r][n] = __builtin_bit_cast(f32x4, ld16<kCoherent>(from, live && (int)row < rows ? row * pitch + col * 4 : nowhere));
        }
    }
  }
  template <bool kBKMajor>
  TCCL_D void last_steps(const char* s0, const char* s1, const char* s2, const char* s3, const Source& src, const Reader& rd,
                         f32x4 (&acc)[4][4], Frags& f) const {
    k_step<kBKMajor, false, 3>(s0, s1, nullptr, src, rd, 0, acc, f);
    k_step<kBKMajor, false, 2>(s1, s2, nullptr, src, rd, 0, acc, f);
    k_step<kBKMajor, false, 1>(s2, s3, nullptr, src, rd, 0, acc, f);
  }
  template <int kPolicy>
  TCCL_D void epilogue_across(int row0, int col0, const f32x4 (&acc)[4][4], const Addends& w) const {
    static_assert(sizeof(OutT) == 4 || kWorld == 0, "fp32 partials");
    static_assert(kStage >= 32768 || kWorld == 0, "a staging window per wavefront");
    constexpr int kRowBytes = 256, kChunks = 16, kRounds = 32 * kChunks / 64;
    char* win = st0 + wave * 8192;
    const int ln = (int)((uint32_t)fresh(lane) & 63u), i16 = ln & 15, kg = ln >> 4;
    const int rows = g.wrap_rows - row0, cols = g.N - col0;
    const bool mine = sums_here();
    const int first = reduce.rank % kOwners * kOwnChunks;  // this rank's first chunk in a row of the wavefront
    const __amdgpu_buffer_rsrc_t rc = window((int64_t)(uintptr_t)((float*)g.C + (int64_t)row0 * g.ldc + col0));
    const __amdgpu_buffer_rsrc_t to = window((int64_t)(uintptr_t)reduce.out + (int64_t)row0 * reduce.ld_out_bytes + (int64_t)col0 * 2);
#pragma unroll
    for (int bi = 0; bi < 2; ++bi) {
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
          const int row = 16 * r + i16;
          *(f32x4*)(win + row * kRowBytes + ((4 * cb + kg) ^ (row & 7)) * 16) = acc[2 * bi + r][cb] * g.alpha;
        }
      asm volatile("" ::: "memory");  // staged by this wavefront itself: LDS keeps the order
#pragma unroll
      for (int r = 0; r < kRounds; ++r) {
        const int row = (ln + 64 * r) / kChunks, chunk = ln % kChunks, lrow = wm * 64 + bi * 32 + row;
        const int q = (kSpread ? 0 : wn * kOwners) + chunk / kOwnChunks, col = own_col(chunk);
        const u32x4 v = *(const u32x4*)(win + row * kRowBytes + ((chunk ^ (row & 7)) * 16));
        if (lrow < rows && col < cols && !(q == reduce.rank && reduce.own_in_registers))
          __builtin_amdgcn_raw_buffer_store_b128(v, rc, (uint32_t)((((int64_t)q * g.wrap_rows + lrow) * g.ldc + col) * 4), 0, kPolicy);
      }
      if (mine) {
        const int col = own_col(ln), chunk = first + ln % kOwnChunks;
#pragma unroll
        for (int r = 0; r < kOwnRounds; ++r) {
          const int row = own_row(ln, r), lrow = wm * 64 + bi * 32 + row;
          f32x4 sum = *(const f32x4*)(win + row * kRowBytes + ((chunk ^ (row & 7)) * 16));  // the owner's first
#pragma unroll
          for (int n = 0; n < kWorld - 1; ++n) sum += w.v[bi][r][n];
          uint16_t h[4];
#pragma unroll
          for (int j = 0; j < 4; ++j)
            h[j] = reduce.out_dtype == kBF16 ? __builtin_bit_cast(uint16_t, (__bf16)sum[j]) : __builtin_bit_cast(uint16_t, (_Float16)sum[j]);
          typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
          u32x2 o;
          __builtin_memcpy(&o, h, 8);
          if (lrow < rows && col < cols)
            __builtin_amdgcn_raw_buffer_store_b64(o, to, (uint32_t)(lrow * reduce.ld_out_bytes + col * 2), 0, kStreaming);
        }
      }
      asm volatile("" ::: "memory");
    }
  }

  // ---- one 128 x kCols sub-tile -------------------------------------------------------------------
  template <int kPolicy, bool kBKMajor, bool kReduce, bool kAColumns = false>
  TCCL_D void subtile(int row0, int row_end, int col0, int tile_id, const SignalArgs& s) const {
    f32x4 acc[4][4];  // cleared two registers per instruction
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        typedef double f64x2 __attribute__((ext_vector_type(2)));
        f64x2 z;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          double d;
          asm volatile("v_mov_b64 %0, 0" : "=v"(d));
          z[e] = d;
        }
        acc[i][j] = __builtin_bit_cast(f32x4, z);
      }

    const Source src = make_source<kBKMajor, kAColumns>(row0, col0);
    const Reader rd = make_reader<kBKMajor, kAColumns>();
    const int ksteps = (g.K + kStepK - 1) / kStepK;
    __syncthreads();  // the previous sub-tile's epilogue has left LDS
    // K steps 0 .. kStages - 2 go out up front (past K: zeros, never consumed).
    issue_step<kBKMajor, kAColumns>(st0, src, 0);
    issue_step<kBKMajor, kAColumns>(st1, src, 1);
    if constexpr (kStages >= 4) issue_step<kBKMajor, kAColumns>(st2, src, 2);
    if constexpr (kStages == 5) issue_step<kBKMajor, kAColumns>(st3, src, 3);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoads * (kStages - 2)) : "memory");  // stage 0 has landed
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    Frags f;
    f.fa[0] = load_a<kAColumns>(st0, rd, 0, 0);
    f.fa[1] = load_a<kAColumns>(st0, rd, 0, 1);
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) f.fb[cb] = load_b<kBKMajor>(st0, rd, 0, cb);
    // Step t computes from stage t % kStages, fetches its last operands from the next one and loads K step
    // t + kStages - 1 into the one before.  Stages are named statically (the compiler tracks loads into LDS
    // per array), so the loop comes in rounds of kStages steps with an exit after every step.
    if constexpr (kWorld != 0) {
      Addends w;
      int left = 0;  // stage of the first of the last three steps
      for (int kt = 0, n = ksteps - 3;; kt += 4) {
        k_step<kBKMajor, kAColumns>(st0, st1, st3, src, rd, kt + 3, acc, f);
        left = 1;
        if (kt + 1 >= n) break;
        k_step<kBKMajor, kAColumns>(st1, st2, st0, src, rd, kt + 4, acc, f);
        left = 2;
        if (kt + 2 >= n) break;
        k_step<kBKMajor, kAColumns>(st2, st3, st1, src, rd, kt + 5, acc, f);
        left = 3;
        if (kt + 3 >= n) break;
        k_step<kBKMajor, kAColumns>(st3, st0, st2, src, rd, kt + 6, acc, f);
        left = 0;
        if (kt + 4 >= n) break;
      }
      request_sums(row0, col0, w);
      if (left == 0)
        last_steps<kBKMajor>(st0, st1, st2, st3, src, rd, acc, f);
      else if (left == 1)
        last_steps<kBKMajor>(st1, st2, st3, st0, src, rd, acc, f);
      else if (left == 2)
        last_steps<kBKMajor>(st2, st3, st0, st1, src, rd, acc, f);
      else
        last_steps<kBKMajor>(st3, st0, st1, st2, src, rd, acc, f);
      epilogue_across<kPolicy>(row0, col0, acc, w);
      return;
    } else if constexpr (kStages == 3) {
      for (int kt = 0;; kt += 3) {
        k_step<kBKMajor, kAColumns>(st0, st1, st2, src, rd, kt + 2, acc, f);
        if (kt + 1 >= ksteps) break;
        k_step<kBKMajor, kAColumns>(st1, st2, st0, src, rd, kt + 3, acc, f);
        if (kt + 2 >= ksteps) break;
        k_step<kBKMajor, kAColumns>(st2, st0, st1, src, rd, kt + 4, acc, f);
        if (kt + 3 >= ksteps) break;
      }
    } else if constexpr (kStages == 4) {
      for (int kt = 0;; kt += 4) {
        k_step<kBKMajor, kAColumns>(st0, st1, st3, src, rd, kt + 3, acc, f);
        if (kt + 1 >= ksteps) break;
        k_step<kBKMajor, kAColumns>(st1, st2, st0, src, rd, kt + 4, acc, f);
        if (kt + 2 >= ksteps) break;
        k_step<kBKMajor, kAColumns>(st2, st3, st1, src, rd, kt + 5, acc, f);
        if (kt + 3 >= ksteps) break;
        k_step<kBKMajor, kAColumns>(st3, st0, st2, src, rd, kt + 6, acc, f);
        if (kt + 4 >= ksteps) break;
      }
    } else {
      for (int kt = 0;; kt += 5) {
        k_step<kBKMajor, kAColumns>(st0, st1, st4, src, rd, kt + 4, acc, f);
        if (kt + 1 >= ksteps) break;
        k_step<kBKMajor, kAColumns>(st1, st2, st0, src, rd, kt + 5, acc, f);
        if (kt + 2 >= ksteps) break;
        k_step<kBKMajor, kAColumns>(st2, st3, st1, src, rd, kt + 6, acc, f);
        if (kt + 3 >= ksteps) break;
        k_step<kBKMajor, kAColumns>(st3, st4, st2, src, rd, kt + 7, acc, f);
        if (kt + 4 >= ksteps) break;
        k_step<kBKMajor, kAColumns>(st4, st0, st3, src, rd, kt + 8, acc, f);
        if (kt + 5 >= ksteps) break;
      }
    }
    wait_vmem();  // the look-ahead loads must not land on the epilogue's staging
    bool sums = false;
    if constexpr (kReduce) {
      const int owner = row0 / reduce.shard_rows;
      sums = (owner == reduce.rank || reduce.emulate_peer) && peers_there(tile_id, s);
    }
    epilogue<kPolicy, kReduce>(row0, row_end, col0, acc, sums);
  }

  // The peers' partials of plan tile `tile_id` are published (one lane waits, bounded).
  TCCL_D bool peers_there(int tile_id, const SignalArgs& s) const {
    if (reduce.peers_resident) return true;
    volatile int* verdict = (volatile int*)st2;  // the epilogue stages in st0 and st1
    __syncthreads();  // every wavefront has left the K loop's stages
    if (tid == 0) {
      const int64_t deadline = now_ticks() + reduce.spin_ticks;
      bool ok = true;
      for (int p = 0; p < reduce.world && ok; ++p) {
        if (p == reduce.rank) continue;
        if (s.mode == kSignalTile) {
          ok = tile_wait_ge<true>(translate_ptr(reduce.locks, reduce.rank, p, reduce.heap_bases), tile_id, s.epoch, deadline);
        } else {
          const int gid = s.group_table[tile_id];
          const int32_t need = (int32_t)((uint32_t)s.epoch * (uint32_t)reduce.tile_counts[gid]);
          ok = tile_wait_ge<true>(translate_ptr(reduce.counter, reduce.rank, p, reduce.heap_bases), gid, need, deadline);
        }
      }
      if (!ok && reduce.fault) *reduce.fault = 1;
      *verdict = ok ? 1 : 0;
    }
    __syncthreads();
    return *verdict != 0;
  }

  // ---- sub-tiles across the owners ----------------------------------------------------------------------
  // A sub-tile has kRows rows of A and kRun columns of every owner's shard; plan tiles of 128 x 128.
  template <bool kBKMajor>
  TCCL_D void run_across(const SignalArgs& s, int wg, int num_wgs) const {
    constexpr int kParts = 128 / kRun;  // runs of a plan tile
    const int tiles = (g.wrap_rows + kRows - 1) / kRows, cols = g.tile_cols * kParts, total = tiles * cols;
    for (int slot = wg; slot < total; slot += num_wgs) {
      const TileCoord tc = tile_coords(tile_for_slot(slot, total, g.xcds, g.span), tiles, cols, reduce.band);
      const int n = tc.n / kParts, col0 = n * 128 + tc.n % kParts * kRun;
      if (col0 >= g.N) continue;
      if (s.mode == kSignalNone) {
        subtile<0, kBKMajor, true>(tc.m * kRows, 0, col0, 0, s);
        continue;
      }
      subtile<kCoherent, kBKMajor, true>(tc.m * kRows, 0, col0, 0, s);
      wait_vmem();  // the write-through stores have landed
      __syncthreads();
      if (tid < kWorld) {  // one plan tile of each shard; the last sub-tile to cover a part of it publishes
        const int id = tile_id_of(tid * (g.tile_rows / kWorld) + tc.m * kRows / 128, n, g.tile_rows, g.tile_cols, g.group_m);
        const int left = (g.N - n * 128 + kRun - 1) / kRun;
        const uint32_t parts = (uint32_t)(128 / kRows * (left < kParts ? left : kParts));  // (with signals: whole plan tiles of rows)
        // Counts to parts - 1 and starts over by itself, so the word is zero again when the launch has ended.
        const uint32_t before = parts > 1 ? atomicInc(&reduce.arrivals[arrival_word(id, s.epoch, s.mode == kSignalTile)], parts - 1) : 0u;
        if (before == parts - 1) {
          if (s.mode == kSignalTile)
            tile_publish(s.locks, id, s.epoch);
          else
            tile_signal_add<true>(s.counter, s.group_table[id], 1);
        }
      }
    }
  }

  // ---- persistent loop over plan tiles ----------------------------------------------------------
  // A workgroup takes a plan tile at a time, as sub-tiles; in the wide form, where one is narrower than a sub-tile, the
  // one on its right with it.
  template <bool kReduce = false, bool kAColumns = false>
  TCCL_D void run(const SignalArgs& s, int wg, int num_wgs) const {
    const int per = kWn == 4 ? kCols / g.block_n : 1;  // plan tiles across
    const int cols = kWn == 4 ? (g.tile_cols + per - 1) / per : g.tile_cols;
    const int total = g.tile_rows * cols;
    for (int slot = wg; slot < total; slot += num_wgs) {
      TileCoord tc = tile_coords(tile_for_slot(slot, total, g.xcds, g.span), g.tile_rows, cols, g.group_m);
      if constexpr (kReduce) {  // this rank's own rows come last: what its peers wait for comes first
        tc.m += (reduce.rank + 1) % reduce.world * (g.tile_rows / reduce.world);
        if (tc.m >= g.tile_rows) tc.m -= g.tile_rows;
      }
      tc.n *= per;
      int first_row = tc.m * g.block_m, row_end = g.M;
      if (g.ragged) {
        const int tiles = (g.wrap_rows + g.block_m - 1) / g.block_m, q = tc.m / tiles;
        first_row = q * g.wrap_rows + (tc.m - q * tiles) * g.block_m;
        row_end = (q + 1) * g.wrap_rows;
      }
      const int tile_id = kReduce ? tile_id_of(tc.m, tc.n, g.tile_rows, g.tile_cols, g.group_m) : 0;
      for (int sm = 0; sm < g.block_m; sm += kTile)
        for (int sn = 0; sn < per * g.block_n; sn += kCols) {
          const int row0 = first_row + sm, col0 = tc.n * g.block_n + sn;
          if (row0 >= row_end || col0 >= g.N) continue;
          if constexpr (kAColumns) {  // (with a row-major B: check_gemm)
            static_assert(!kReduce, "an A given by columns is not reduced");
            if (s.mode == kSignalNone)
              subtile<0, false, false, true>(row0, row_end, col0, tile_id, s);
            else
              subtile<kCoherent, false, false, true>(row0, row_end, col0, tile_id, s);
          } else if (s.mode == kSignalNone) {
            if (g.b_kmajor)
              subtile<0, true, kReduce>(row0, row_end, col0, tile_id, s);
            else
              subtile<0, false, kReduce>(row0, row_end, col0, tile_id, s);
          } else {
            if (g.b_kmajor)
              subtile<kCoherent, true, kReduce>(row0, row_end, col0, tile_id, s);
            else
              subtile<kCoherent, false, kReduce>(row0, row_end, col0, tile_id, s);
          }
        }
      if (s.mode != kSignalNone) {
        // The tile was stored write-through; once every wave's stores have completed the
        // data is visible device-wide and one lane (per plan tile) may publish the signal.
        wait_vmem();
        __syncthreads();
        if (tid < per && tc.n + tid < g.tile_cols) {
          const int done = tile_id_of(tc.m, tc.n + tid, g.tile_rows, g.tile_cols, g.group_m);
          if (s.mode == kSignalTile)
            tile_publish(s.locks, done, s.epoch);
          else
            tile_signal_add<true>(s.counter, s.group_table[done], 1);
        }
      }
    }
  }
};
#endif  // __HIP_DEVICE_COMPILE__

}  // namespace tccl
