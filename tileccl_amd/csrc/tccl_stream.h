// Streaming MFMA GEMM for gfx950 (CDNA4), 16-bit and e4m3 inputs: small outputs, where the large-tile kernels leave
// most of the device idle (decoding rows, short prompts, ragged and narrow problems).
//
// One workgroup produces one output tile of (16 kMB) x (16 kNB); its kWaves wavefronts each take every
// kWaves-th K block of 64 (e4m3: 128) for the WHOLE tile and add their accumulators up through LDS at the end.  A
// wavefront loads its K blocks in whole lines and turns each to the operand order of v_mfma_f32_16x16x32 through LDS of
// its own, so there is no barrier in the K loop.  A tile of 16 rows of a 4096-deep product is then sixteen chains of four
// K blocks, all requested at once, instead of one chain of 128 K steps.  Measured, bf16, 16 x 2048 x 4096: 6.0 us with a
// k-major B and 7.6 us row-major against 29 us on the 128 x 128-tile kernel, whose 16 tiles keep 16 CUs busy;
// 1024 x 1024 x 2048: 11.9 and 15.4 against 19 us; an empty launch takes 3.7 us of that.
//
// What bounds it: the vector memory path of a CU delivers 70 to 110 KB/us of operands here, and each operand
// byte of a tile passes it once, (kMB + kNB) * 2 KiB per 64 k; tiles are as large as the output allows while
// every CU still gets one (stream_shape() in tccl_api.hip).  A row-major B is slower because a narrow tile reads
// 32 to 128 bytes of each k row.  The matrix pipes are busy 3 % (16 rows) to 15 % of the time.
#pragma once

#include "tccl_comm.h"
#include "tccl_gemm.h"

namespace tccl {

// The pull half of an all-gather: this rank's copy of every peer's row block.  Workgroups behind those of the tiles share it
// out and wait (bounded) for the peers; a workgroup with a tile never waits (stream_grid()).
struct StreamPull {
  int active;
  int cus;              // of the device
  int first;            // the first workgroup that pulls: all tiles are below it
  int rows;             // of a block
  uint32_t upr, pitch;  // 16-byte units and bytes per row
  int64_t block_bytes;  // from one block to the next
  char* out;            // block 0 of the gathered output in this rank's slice
  const int32_t* words;  // this rank's TileGroup counters or locks; a peer's: word_stride apart, or (0) at the same slice offset
  const int32_t* row_starts;
  const int32_t* row_ends;
  const int32_t* tile_counts;
  int n_groups;
  int64_t word_stride;
  int64_t* fault;
  int64_t spin_ticks;
};

struct StreamArgs {
  const void* A;
  const void* B;
  char* C;
  int64_t lda, ldb, ldc;  // elements
  int M, N, K;            // C is M x N
  int b_short;            // rows that a row-major B lacks at the end of K: they read as zero
  float alpha;
  int out_dtype;
  // Rows come in segments (the owners' shards of a reduce-scatter, stacked column shards); tiles do not straddle
  // them.  `wrapped`: segment q is A (seg_rows x K) times columns [q N, (q + 1) N) of B.
  int seg_rows, wrapped;
  int first_seg;                   // segments are visited from this one on, wrapping around
  int tiles_m, tiles_n, segs;      // tiles down and across a segment; segments
  uint32_t tiles_m_magic;          // 2^32 / tiles_m, rounded up: n / tiles_m is mulhi(n, magic) for the tile numbers there are
  int xcd_shift, per_xcd;          // of 2^xcd_shift XCDs, XCD x works on tiles [x per_xcd, (x + 1) per_xcd) of a segment: neighbours share a slab of B in its L2
  // Signals: a plan tile is published when the last of its tiles has been stored.
  SignalArgs s;
  uint32_t* arrivals;              // kArrivalStride words per plan tile (arrival_word()), zero between launches
  int block_m, block_n, group_m, plan_rows, plan_cols;
  const int64_t* heap_bases;
  int rank, world;
  PushArgs push;
  EpilogueReduce reduce;
  StreamPull pull;
};

#if defined(__HIP_DEVICE_COMPILE__)
template <typename InT, int kMB, int kNB, int kWaves, bool kBKMajor>
struct StreamGemm {
  typedef typename Mfma<InT>::Vec Vec;
  static constexpr int kEsz = sizeof(InT), kVec = 16 / kEsz;  // elements per 16-byte chunk
  static constexpr int kKB = 128 / kEsz;                      // K per block: 64, or 128 for e4m3
  static constexpr int kBM = 16 * kMB, kBN = 16 * kNB;
  // K blocks of 64 in flight per wavefront, within the registers that kWaves wavefronts leave each.
  static constexpr int kBudget = (kWaves >= 16 ? 64 : 128) / ((kMB + kNB) * 8);
  static constexpr int kDepth = kBudget < 1 ? 1 : (kBudget > 4 ? 4 : kBudget);
  static constexpr int kSlots = kMB * kNB;            // accumulator quads per lane
  // LDS of a wavefront: one K block on its way from load order to operand order, then its sums.
  static constexpr int kStagedBlocks = kMB + kNB;
  static constexpr int kWaveBytes = kStagedBlocks * 2048 > kSlots * 1024 ? kStagedBlocks * 2048 : kSlots * 1024;
  static constexpr int kPitch = kBN * 4 + 16;         // bytes of a row of sums
  static constexpr int kRowsBytes = kBM * kPitch;
  static constexpr int kLdsBytes = kWaves * kWaveBytes > kRowsBytes ? kWaves * kWaveBytes : kRowsBytes;

  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  // What a tile's end needs from memory and the divisions that its signal takes: done while the first operands are on
  // their way.  Behind the tile's stores, where they are used, they were a chain of trips to memory and of scalar
  // instructions with nothing to overlap them (176 x 1440 x 336, pushed to three peers: 8.5 -> 7.6 us).
  struct Signal {
    int tile;        // the plan tile under this tile
    int word;        // and where its tiles are counted
    uint32_t tiles;  // tiles of it
    int32_t group;   // its TileGroup (group mode)
    u32x2 base;      // lane p: rank p's heap base
  };

  const StreamArgs& a;
  char* lds;
  const int lane, wave;

  TCCL_D StreamGemm(const StreamArgs& args, char* l)
      : a(args), lds(l), lane(threadIdx.x & 63), wave(__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6))) {}

  static TCCL_D uint32_t clamp_u32(int64_t v) { return v > 0xfffffff0ll ? 0xfffffff0u : (v < 0 ? 0u : (uint32_t)v); }

  // One K block as it is loaded, 16 bytes per lane with neighbouring lanes on neighbouring addresses (a
  // load whose lanes 0..3 lie in four rows takes in a third of the bytes per clock: 34 against 104 KB/us per CU).
  //   A, k-major B: rows of 128 bytes; instruction h of a 16-row block covers its rows 8 h + l / 8, chunk l % 8.
  //   Row-major B: 64 k rows of 32 kNB bytes (e4m3: 128 of 16 kNB); instruction h covers kRowsPerLoad of them.
  struct Block {
    u32x4 a[2 * kMB], b[2 * kNB];
  };
  static constexpr int kRowBytes = 16 * kNB * kEsz, kRowLanes = kRowBytes / 16;  // of a k row of row-major B in a tile
  static constexpr int kRowsPerLoad = 64 / kRowLanes;
  static constexpr uint32_t kOutside = 0xffffff00u;  // beyond every buffer: reads as zero

  __amdgpu_buffer_rsrc_t ra, rb;
  uint32_t off_a, off_b, pitch_a, pitch_b;  // this lane's offset in K block 0; bytes per row
  int kg, i16;

  // kTail: the block may reach past K; a chunk, or a row of B, at k >= K reads as zero.
  template <bool kTail>
  TCCL_D void load(Block& v, int kb) const {
    const bool past = kTail && kb * kKB + kVec * (lane & 7) >= a.K;
#pragma unroll
    for (int h = 0; h < 2 * kMB; ++h) {
      const uint32_t o = off_a + (uint32_t)(8 * h) * pitch_a + (uint32_t)kb * 128u;
      v.a[h] = __builtin_amdgcn_raw_buffer_load_b128(ra, past ? kOutside : o, 0, 0);
    }
#pragma unroll
    for (int h = 0; h < 2 * kNB; ++h) {
      if constexpr (kBKMajor) {
        const uint32_t o = off_b + (uint32_t)(8 * h) * pitch_b + (uint32_t)kb * 128u;
        v.b[h] = __builtin_amdgcn_raw_buffer_load_b128(rb, past ? kOutside : o, 0, 0);
      } else {
        const int k = kb * kKB + h * kRowsPerLoad;  // and the lane's row
        const bool none = off_b == kOutside || (kTail && k + lane / kRowLanes >= a.K);
        v.b[h] = __builtin_amdgcn_raw_buffer_load_b128(rb, none ? kOutside : off_b + (uint32_t)k * pitch_b, 0, 0);
      }
    }
  }

  // Load order -> operand order through this wavefront's own LDS (a wavefront's LDS operations execute in the
  // order issued: no barrier).
  //   Rows of 128 bytes: chunk c of row r in slot c ^ ((r >> 1) & 7), read with ds_read_b128.
  //   Row-major B: the 32-byte units (e4m3: 16-byte chunks) of k row k permuted by swizzle(k), so that the rows that
  //   32 lanes of a transposing read (ds_read_b64_tr_b16, _tr_b8) touch at a time lie in different banks.
  static TCCL_D int swizzle(int k) {
    if constexpr (kEsz == 1) return kNB == 4 ? ((k >> 2) & 1) | (((k >> 4) & 1) << 1) : (kNB == 2 ? (k >> 4) & 1 : 0);
    if constexpr (kNB == 4) return (k & 2) ^ ((k >> 3) & 1);
    return kNB == 2 ? (k >> 3) & 1 : 0;
  }
  static TCCL_D int row_at(int k) { return kNB == 1 && kEsz == 2 ? k ^ (4 * ((k >> 3) & 1)) : k; }
  // The hardware keeps the order of a wavefront's LDS accesses, the fences on both sides the compiler's: these writes come
  // after the reads of the block before and ahead of the reads that other lanes make of them.
  TCCL_D void stage(const Block& v) const {
    asm volatile("" ::: "memory");
    char* at = lds + wave * kWaveBytes;
#pragma unroll
    for (int h = 0; h < 2 * kMB; ++h) {
      const int r = 8 * h + (lane >> 3);
      *(u32x4*)(at + r * 128 + (((lane & 7) ^ ((r >> 1) & 7)) << 4)) = v.a[h];
    }
    at += kMB * 2048;
#pragma unroll
    for (int h = 0; h < 2 * kNB; ++h) {
      if constexpr (kBKMajor) {
        const int r = 8 * h + (lane >> 3);
        *(u32x4*)(at + r * 128 + (((lane & 7) ^ ((r >> 1) & 7)) << 4)) = v.b[h];
      } else {
        const int k = h * kRowsPerLoad + lane / kRowLanes, c = lane % kRowLanes;
        *(u32x4*)(at + row_at(k) * kRowBytes + ((c ^ (kEsz * swizzle(k))) << 4)) = v.b[h];
      }
    }
    asm volatile("" ::: "memory");
  }
  // 16-byte chunk 4 h + l / 16 of row l % 16 of 16-row block `block` (A, k-major B): the 16-bit operand of 32-k half h (k
  // 8 (l / 16) .. + 7 of it); the e4m3 operand of a whole block is both (k 16 (l / 16) .. + 15 and 64 + that).
  TCCL_D u32x4 chunk(int block, int h) const {
    return *(const u32x4*)(lds + wave * kWaveBytes + block * 2048 + i16 * 128 + (((4 * h + kg) ^ ((i16 >> 1) & 7)) << 4));
  }
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  typedef __attribute__((address_space(3))) s16x4 LdsQuad;
  typedef int i32x2 __attribute__((ext_vector_type(2)));
  typedef __attribute__((address_space(3))) i32x2 LdsPair;
  // Column block j of row-major B, transposed on the way out: 16-bit, 32-k half h, two reads (k rows 8 kg + 0 .. 3 and
  // + 4 .. 7); e4m3, the whole block, four reads (k rows 16 kg + 0, 8, 64, 72 and the seven after each).
  TCCL_D Vec turned(int j, int h) const {
    const char* at = lds + wave * kWaveBytes + kMB * 2048;
    if constexpr (kEsz == 2) {
      const int t = i16 >> 2, cq = i16 & 3;
      s16x4 half[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int k = 32 * h + 8 * kg + 4 * q + t;
        const char* p = at + row_at(k) * kRowBytes + (((2 * j + (cq >> 1)) ^ (2 * swizzle(k))) << 4) + (cq & 1) * 8;
        half[q] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsQuad*)p);
      }
      const s16x8 both = __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7);
      return __builtin_bit_cast(Vec, both);
    } else {
      i32x8 v;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = 16 * kg + 8 * (q & 1) + 64 * (q >> 1) + (i16 >> 1);
        const char* p = at + k * kRowBytes + ((j ^ swizzle(k)) << 4) + (i16 & 1) * 8;
        const i32x2 x = __builtin_amdgcn_ds_read_tr8_b64_v2i32((LdsPair*)p);
        v[2 * q] = x[0];
        v[2 * q + 1] = x[1];
      }
      return __builtin_bit_cast(Vec, v);
    }
  }
  TCCL_D Vec staged(int block, int h) const {
    if constexpr (kEsz == 2) {
      return __builtin_bit_cast(Vec, chunk(block, h));
    } else {
      typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));
      const u32x8 both = __builtin_shufflevector(chunk(block, 0), chunk(block, 1), 0, 1, 2, 3, 4, 5, 6, 7);
      return __builtin_bit_cast(Vec, both);
    }
  }

  TCCL_D void multiply(f32x4 (&acc)[kMB][kNB]) const {
#pragma unroll
    for (int h = 0; h < kEsz; ++h) {  // one MFMA deep for e4m3, two for the 16-bit types
      Vec fa[kMB], fb[kNB];
#pragma unroll
      for (int j = 0; j < kNB; ++j) {
        if constexpr (kBKMajor)
          fb[j] = staged(kMB + j, h);
        else
          fb[j] = turned(j, h);
      }
#pragma unroll
      for (int i = 0; i < kMB; ++i) fa[i] = staged(i, h);
#pragma unroll
      for (int i = 0; i < kMB; ++i)
#pragma unroll
        for (int j = 0; j < kNB; ++j) acc[i][j] = Mfma<InT>::run16(fb[j], fa[i], acc[i][j]);
    }
  }

  TCCL_D void refill(Block& v, int kb, int whole, int blocks) const {
    if (kb < whole)
      load<false>(v, kb);
    else if (kb < blocks)
      load<true>(v, kb);
  }

  // `meanwhile` runs once the first blocks have been requested.
  template <typename Meanwhile>
  TCCL_D void k_loop(f32x4 (&acc)[kMB][kNB], Meanwhile meanwhile) const {
    const int blocks = (a.K + kKB - 1) / kKB, whole = a.K / kKB;
    Block v[kDepth];
    // This wavefront's blocks are wave, wave + kWaves, ...; the last one of all may be a partial one.
    int next = wave;
#pragma unroll
    for (int d = 0; d < kDepth; ++d, next += kWaves) refill(v[d], next, whole, blocks);
    meanwhile();
    for (int kb = wave; kb < blocks;) {
#pragma unroll
      for (int d = 0; d < kDepth; ++d) {
        if (kb < blocks) {
          stage(v[d]);
          refill(v[d], next, whole, blocks);  // the block is in LDS: its registers are free
          multiply(acc);
          kb += kWaves;
          next += kWaves;
        }
      }
    }
  }

  // Workgroups behind the tiles (launches that pull).
  TCCL_D void pull(int slot) const {
    if (pull_ready(slot)) pull_share(slot);
  }

  // The units of a block that workgroup `slot` pulls.
  TCCL_D void share(int slot, uint32_t& lo, uint32_t& hi) const {
    const uint32_t units = (uint32_t)a.pull.rows * a.pull.upr, wgs = gridDim.x - a.pull.first, per = (units + wgs - 1) / wgs;
    lo = (uint32_t)(slot - a.pull.first) * per;
    lo = lo < units ? lo : units;
    hi = units - lo < per ? units : lo + per;
  }
  // What the share depends on, for every peer: the TileGroups, or plan tiles, that cover its rows.  Spins until they are
  // complete; false: a deadline passed.
  TCCL_D bool pull_ready(int slot) const {
    uint32_t lo, hi;
    share(slot, lo, hi);
    if (lo >= hi) return true;
    const int r0 = (int)(lo / a.pull.upr), r1 = (int)((hi - 1) / a.pull.upr);
    const int t0 = r0 / a.block_m, tiles = (r1 / a.block_m - t0 + 1) * a.plan_cols;
    const int per_peer = a.s.mode == kSignalTile ? tiles : a.pull.n_groups;
    bool ok = true;
    const int64_t deadline = now_ticks() + a.pull.spin_ticks;
    for (int i = (int)threadIdx.x; i < per_peer * (a.world - 1); i += kWaves * 64) {
      const int q = i / per_peer, k = i - q * per_peer, p = q < a.rank ? q : q + 1;
      const int32_t* words = a.pull.word_stride ? (const int32_t*)((const char*)a.pull.words + (int64_t)(p - a.rank) * a.pull.word_stride)
                                                : translate_ptr(a.pull.words, a.rank, p, a.heap_bases);
      int index = k;
      int32_t need = a.s.epoch;
      if (a.s.mode == kSignalTile) {
        index = tile_id_of(t0 + k / a.plan_cols, k % a.plan_cols, a.plan_rows, a.plan_cols, a.group_m);
      } else {
        if (a.pull.row_starts[k] > r1 || a.pull.row_ends[k] <= r0) continue;
        need = (int32_t)((uint32_t)a.s.epoch * (uint32_t)a.pull.tile_counts[k]);
      }
      ok = ok && tile_wait_ge<true>(words, index, need, deadline);
    }
    if (!ok && a.pull.fault) *a.pull.fault = 1;
    return __syncthreads_and(ok);
  }
  TCCL_D void pull_share(int slot) const {
    uint32_t lo, hi;
    share(slot, lo, hi);
    const int64_t mine = a.heap_bases[a.rank];
    // Several peers' units are requested before any is stored: a wait for a load is also one for every store before it.
    constexpr int kPeers = 4, kBatch = 4;
    for (int q0 = 0; q0 < a.world - 1; q0 += kPeers) {
      for (uint32_t u0 = lo + threadIdx.x; u0 < hi; u0 += kBatch * kWaves * 64) {
        u32x4 v[kPeers][kBatch];
        uint32_t off[kBatch];
#pragma unroll
        for (int b = 0; b < kBatch; ++b) {
          const uint32_t u = u0 + (uint32_t)(b * kWaves * 64), row = u / a.pull.upr;
          off[b] = row * a.pull.pitch + (u - row * a.pull.upr) * 16u;
        }
#pragma unroll
        for (int i = 0; i < kPeers; ++i) {
          const int q = q0 + i, p = q < a.rank ? q : q + 1;
          if (q >= a.world - 1) break;
          const __amdgpu_buffer_rsrc_t from = window((int64_t)(uintptr_t)a.pull.out + p * a.pull.block_bytes + (a.heap_bases[p] - mine));
#pragma unroll
          for (int b = 0; b < kBatch; ++b)
            if (u0 + (uint32_t)(b * kWaves * 64) < hi) v[i][b] = ld16<kCoherent>(from, off[b]);
        }
#pragma unroll
        for (int i = 0; i < kPeers; ++i) {
          const int q = q0 + i, p = q < a.rank ? q : q + 1;
          if (q >= a.world - 1) break;
          const __amdgpu_buffer_rsrc_t to = window((int64_t)(uintptr_t)a.pull.out + p * a.pull.block_bytes);
#pragma unroll
          for (int b = 0; b < kBatch; ++b)
            if (u0 + (uint32_t)(b * kWaves * 64) < hi) st16<kStreaming>(to, off[b], v[i][b]);
        }
      }
    }
  }

  TCCL_D void tile(int slot) {
    // Every segment is spread over all XCDs (an XCD's link to memory would otherwise carry one owner's reductions alone).
    // Within an XCD's part row tiles run fastest: those that share a column slab of B.
    const int per_seg = a.tiles_m * a.tiles_n, slots_per_seg = a.per_xcd << a.xcd_shift;
    int seg = a.segs > 1 ? slot / slots_per_seg : 0;
    const int at = slot - seg * slots_per_seg;
    const int in = (at & ((1 << a.xcd_shift) - 1)) * a.per_xcd + (at >> a.xcd_shift);
    if (in >= per_seg || at >= slots_per_seg) return;
    const int tn = a.tiles_m > 1 ? (int)__umulhi((uint32_t)in, a.tiles_m_magic) : in, tm = in - tn * a.tiles_m;
    seg += a.first_seg;
    if (seg >= a.segs) seg -= a.segs;
    const int row_in = tm * kBM, col0 = tn * kBN;  // relative to the segment
    const int row0 = seg * a.seg_rows + row_in;    // row of C

    i16 = lane & 15;
    kg = lane >> 4;
    const int a_row = a.wrapped ? row_in : row0, a_rows = a.wrapped ? a.seg_rows : a.M;
    const int64_t b_col = (a.wrapped ? (int64_t)seg * a.N : 0) + col0;
    pitch_a = (uint32_t)(a.lda * kEsz);
    pitch_b = (uint32_t)(a.ldb * kEsz);
    const InT* A = (const InT*)a.A + (int64_t)a_row * a.lda;
    ra = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, clamp_u32(((int64_t)(a_rows - 1 - a_row) * a.lda + a.K) * kEsz), 0x00020000);
    off_a = (uint32_t)(lane >> 3) * pitch_a + (uint32_t)(lane & 7) * 16u;
    const int cols_left = a.N - col0;  // columns of this segment from col0 on
    if constexpr (kBKMajor) {
      const InT* B = (const InT*)a.B + b_col * a.ldb;
      rb = __builtin_amdgcn_make_buffer_rsrc((void*)B, 0, clamp_u32(((int64_t)(cols_left - 1) * a.ldb + a.K) * kEsz), 0x00020000);
      off_b = (uint32_t)(lane >> 3) * pitch_b + (uint32_t)(lane & 7) * 16u;
    } else {
      const InT* B = (const InT*)a.B + b_col;
      rb = __builtin_amdgcn_make_buffer_rsrc((void*)B, 0, clamp_u32(((int64_t)(a.K - 1 - a.b_short) * a.ldb + cols_left) * kEsz), 0x00020000);
      const int c = lane % kRowLanes;
      off_b = kVec * c < cols_left ? (uint32_t)(lane / kRowLanes) * pitch_b + (uint32_t)c * 16u : kOutside;
    }

    f32x4 acc[kMB][kNB];
#pragma unroll
    for (int i = 0; i < kMB; ++i)
#pragma unroll
      for (int j = 0; j < kNB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    Signal signal;
    k_loop(acc, [&] { signal = look_up(row0, col0); });

    // The wavefronts' accumulators are added up through LDS ([slot][lane] of each, conflict-free) and the sums
    // staged as rows, from which every thread takes chunks of 8 columns.
#pragma unroll
    for (int i = 0; i < kMB; ++i)
#pragma unroll
      for (int j = 0; j < kNB; ++j) *(f32x4*)(lds + wave * kWaveBytes + ((i * kNB + j) * 64 + lane) * 16) = acc[i][j];
    __syncthreads();
    constexpr int kMine = (kSlots + kWaves - 1) / kWaves;
    f32x4 sum[kMine];
#pragma unroll
    for (int m = 0; m < kMine; ++m) {
      const int slot_no = wave + m * kWaves;
      if (slot_no < kSlots) {
        sum[m] = *(const f32x4*)(lds + (slot_no * 64 + lane) * 16);
#pragma unroll
        for (int w = 1; w < kWaves; ++w) {
          const f32x4 x = *(const f32x4*)(lds + w * kWaveBytes + (slot_no * 64 + lane) * 16);
#pragma unroll
          for (int e = 0; e < 4; ++e) sum[m][e] += x[e];
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < kMine; ++m) {
      const int slot_no = wave + m * kWaves;
      if (slot_no < kSlots) {
        const int i = slot_no / kNB, j = slot_no % kNB;
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[m][e] *= a.alpha;
        *(f32x4*)(lds + (16 * i + i16) * kPitch + (16 * j + 4 * kg) * 4) = sum[m];
      }
    }
    __syncthreads();
    const bool coherent = a.s.mode != kSignalNone;
    const int owner = seg;
    bool ok = true;
    if (a.reduce.active && (owner == a.rank || a.reduce.emulate_peer) && !a.reduce.peers_resident) ok = wait_for_peers(row0, col0);
    constexpr int kChunksPerRow = kBN / 8, kChunks = kBM * kChunksPerRow;
    for (int c = (int)threadIdx.x; c < kChunks; c += kWaves * 64) {
      const int row = c / kChunksPerRow, col = c % kChunksPerRow * 8;
      if (row_in + row >= a.seg_rows || col0 + col >= a.N) continue;
      float f[8];
      const f32x4 lo = *(const f32x4*)(lds + row * kPitch + col * 4), hi = *(const f32x4*)(lds + row * kPitch + col * 4 + 16);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f[e] = lo[e];
        f[4 + e] = hi[e];
      }
      finish(f, signal, owner, row_in, row0, col0, row, col, coherent, ok);
    }
    publish(signal);
  }

  TCCL_D static void put(__amdgpu_buffer_rsrc_t w, uint32_t off, const float (&f)[8], int dtype, bool coherent) {
    if (coherent) {
      if (dtype == kF16)
        store8<_Float16, kCoherent>(w, off, f);
      else if (dtype == kBF16)
        store8<__bf16, kCoherent>(w, off, f);
      else
        store8<float, kCoherent>(w, off, f);
    } else {
      if (dtype == kF16)
        store8<_Float16, 0>(w, off, f);
      else if (dtype == kBF16)
        store8<__bf16, 0>(w, off, f);
      else
        store8<float, 0>(w, off, f);
    }
  }
  TCCL_D static void get(__amdgpu_buffer_rsrc_t w, uint32_t off, float (&f)[8], int dtype) {
    if (dtype == kF16)
      Load8<_Float16, kCoherent>::run(w, off, f);
    else if (dtype == kBF16)
      Load8<__bf16, kCoherent>::run(w, off, f);
    else
      Load8<float, kCoherent>::run(w, off, f);
  }

  // One chunk of 8 columns: to C, to the peers, or into the reduction.
  TCCL_D void finish(float (&f)[8], const Signal& signal, int owner, int row_in, int row0, int col0, int row, int col, bool coherent, bool ok) const {
    const int esz = a.out_dtype == kF32 ? 4 : 2;
    const int64_t c_at = (int64_t)(uintptr_t)a.C + ((int64_t)row0 * a.ldc + col0) * esz;
    const uint32_t off = (uint32_t)((row * a.ldc + col) * esz);
    const bool reduces = a.reduce.active && (owner == a.rank || a.reduce.emulate_peer) && ok;
    const bool store = !(a.reduce.active && owner == a.rank && a.reduce.own_in_registers && ok);
    if (store) put(window(c_at), off, f, a.out_dtype, coherent);
    for (int t = 0; t < a.push.world; ++t) {
      const int c = col0 + col;
      if (t == a.push.rank || c < a.push.col_lo || c >= a.push.col_hi) continue;
      const int64_t to = (int64_t)(uintptr_t)a.C + (base_of(signal, t) - base_of(signal, a.push.rank)) +
                         ((int64_t)row0 * a.push.ld + col0 + a.push.col_shift) * esz;
      put(window(to), (uint32_t)((row * a.push.ld + col) * esz), f, a.out_dtype, true);
    }
    if (!reduces) return;
    // The owner's partial first, then the other ranks ascending; this rank's is the value as stored.
    float mine[8], sum[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) mine[e] = a.out_dtype == kF32 ? f[e] : (a.out_dtype == kF16 ? (float)(_Float16)f[e] : (float)(__bf16)f[e]);
    const int64_t my_base = a.heap_bases[a.rank];
    constexpr int kPeers = 4;  // ranks whose addends are requested together
    for (int i0 = 0; i0 < a.world; i0 += kPeers) {
      float v[kPeers][8];
#pragma unroll
      for (int i = 0; i < kPeers; ++i) {
        const int n = i0 + i, p = n == 0 ? owner : (n <= owner ? n - 1 : n);
        if (n >= a.world) break;
        if (p == a.rank) {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[i][e] = mine[e];
        } else {
          get(window(c_at + (a.heap_bases[p] - my_base)), off, v[i], a.out_dtype);
        }
      }
#pragma unroll
      for (int i = 0; i < kPeers; ++i) {
        if (i0 + i >= a.world) break;
#pragma unroll
        for (int e = 0; e < 8; ++e) sum[e] = i0 + i == 0 ? v[i][e] : sum[e] + v[i][e];
      }
    }
    const int64_t out = (int64_t)(uintptr_t)a.reduce.out + (a.heap_bases[owner] - my_base) + (int64_t)row_in * a.reduce.ld_out_bytes + (int64_t)col0 * 2;
    put(window(out), (uint32_t)(row * a.reduce.ld_out_bytes + col * 2), sum, a.reduce.out_dtype, false);
  }

  TCCL_D int plan_tile(int row0, int col0) const {
    return tile_id_of(row0 / a.block_m, col0 / a.block_n, a.plan_rows, a.plan_cols, a.group_m);
  }

  // The peers' partials of the plan tile under (row0, col0) are published (bounded wait).
  TCCL_D bool wait_for_peers(int row0, int col0) const {
    __shared__ int verdict;
    if (threadIdx.x == 0) {
      const int tile = plan_tile(row0, col0);
      const int64_t deadline = now_ticks() + a.reduce.spin_ticks;
      bool ok = true;
      for (int p = 0; p < a.world && ok; ++p) {
        if (p == a.rank) continue;
        if (a.s.mode == kSignalTile) {
          ok = tile_wait_ge<true>(translate_ptr(a.reduce.locks, a.rank, p, a.heap_bases), tile, a.s.epoch, deadline);
        } else {
          const int g = a.s.group_table[tile];
          const int32_t need = (int32_t)((uint32_t)a.s.epoch * (uint32_t)a.reduce.tile_counts[g]);
          ok = tile_wait_ge<true>(translate_ptr(a.reduce.counter, a.rank, p, a.heap_bases), g, need, deadline);
        }
      }
      if (!ok && a.reduce.fault) *a.reduce.fault = 1;
      verdict = ok ? 1 : 0;
    }
    __syncthreads();
    return verdict != 0;
  }

  TCCL_D Signal look_up(int row0, int col0) const {
    Signal s;
    s.tile = s.word = 0;
    s.tiles = 1;
    s.group = 0;
    s.base = u32x2{0, 0};
    if (a.push.world > 0) s.base = __builtin_amdgcn_raw_buffer_load_b64(window((int64_t)(uintptr_t)a.heap_bases), 8u * (uint32_t)(lane < a.push.world ? lane : 0), 0, 0);
    if (a.s.mode == kSignalNone) return s;
    s.tile = plan_tile(row0, col0);
    s.word = arrival_word(s.tile, a.s.epoch, a.s.mode == kSignalTile);
    if (a.s.mode == kSignalGroup) s.group = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(window((int64_t)(uintptr_t)a.s.group_table), 4u * (uint32_t)s.tile, 0, 0);
    // Tiles of this plan tile: those of its rows and columns that lie inside the segment and N.
    const int pr = row0 / a.block_m * a.block_m, pc = col0 / a.block_n * a.block_n;
    const int seg0 = a.segs > 1 ? row0 / a.seg_rows * a.seg_rows : 0;
    const int rows = (pr + a.block_m < seg0 + a.seg_rows ? pr + a.block_m : seg0 + a.seg_rows) - pr;
    const int cols = (pc + a.block_n < a.N ? pc + a.block_n : a.N) - pc;
    s.tiles = (uint32_t)(((rows + kBM - 1) / kBM) * ((cols + kBN - 1) / kBN));
    return s;
  }
  static TCCL_D int64_t base_of(const Signal& s, int p) {
    const uint32_t lo = __builtin_amdgcn_readlane(s.base[0], p), hi = __builtin_amdgcn_readlane(s.base[1], p);
    return (int64_t)(((uint64_t)hi << 32) | lo);
  }

  TCCL_D void publish(const Signal& signal) const {
    if (a.s.mode == kSignalNone) return;
    wait_vmem();  // this wavefront's write-through stores have landed
    __syncthreads();
    if (threadIdx.x != 0) return;
    const uint32_t n = signal.tiles;
    // Counts to n - 1 and starts over by itself, so the word is zero again when the launch has ended.
    const uint32_t before = n > 1 ? atomicInc(&a.arrivals[signal.word], n - 1) : 0u;
    if (before != n - 1) return;
    if (a.s.mode == kSignalTile)
      tile_publish(a.s.locks, signal.tile, a.s.epoch);
    else
      tile_signal_add<true>(a.s.counter, signal.group, 1);
  }
};
#endif  // __HIP_DEVICE_COMPILE__

// Tile shapes that exist (16 mb x 16 nb, wavefronts), smallest first.
struct StreamShape {
  int mb, nb, waves;
};
constexpr StreamShape kStreamShapes[] = {{1, 1, 16}, {1, 2, 16}, {2, 2, 16}, {2, 4, 8}, {4, 4, 4}};
constexpr int kStreamShapeCount = (int)(sizeof(kStreamShapes) / sizeof(kStreamShapes[0]));

// The workgroups of a launch: `first` for tiles, the rest pull.  Two rules keep every wait finite:
// - In an all-gather only pulling workgroups wait for another rank, and they are numbered, hence started, behind every tile:
//   what a peer waits for never needs a place that one of them holds, however many tiles there are (e4m3: more than are
//   resident).  (In a reduce-scatter the tiles of the own rows wait, the last ones: run_variant().)
// - They are few enough that ranks which share a device find CUs for their tiles, the others' waiting workgroups
//   notwithstanding (a workgroup takes 64 to 128 KiB of LDS, i.e. a CU): a 1/world of the CUs, or a quarter from four
//   ranks on, since no more of one process's launches run at a time (HIP's four hardware queues).
// Where an eighth of the CUs has no tile, they run beside the tiles and are no more than those CUs.
// Measured against shares that every tile's workgroup pulled, and waited for, behind its own tile (peers complete): fp16, two ranks,
// 176 x 1440 x 336 6.9 us both ways, 1000 x 1000 x 512 11.9 -> 9.8, 1024 x 1024 x 1024 13.3 -> 11.3 (eight ranks 19.8 -> 17.8),
// e4m3 1536 x 2048 x 1024 24.6 -> 19.5; slower where 256 tiles of 32 x 32 leave the pulls for a second wave of workgroups:
// 512 x 512 x 256 8.2 -> 8.4, four ranks 8.9 -> 9.5, eight 10.6 -> 11.9.
constexpr int kLiveRanks = 4;
struct StreamGrid {
  int first, wgs;
};
inline StreamGrid stream_grid(int tiles, bool pulls, int cus, int world) {
  if (!pulls) return {tiles, tiles};
  const int ranks = world < kLiveRanks ? world : kLiveRanks;
  int pullers = cus / ranks > 0 ? cus / ranks : 1;
  if (cus - tiles >= cus / 8 && cus - tiles < pullers) pullers = cus - tiles;
  return {tiles, tiles + pullers};
}

// Defined in tccl_stream.hip.  Fills in the tile counts and launches.  0 or a hipError_t.
int launch_stream(int in_dtype, bool b_kmajor, int shape, StreamArgs& a, hipStream_t stream);

}  // namespace tccl
