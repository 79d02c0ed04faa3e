// Stand-alone transfers and reductions between the slices of the symmetric heap: the second kernel of S0,
// the copies and reductions of the stand-alone collectives, and the collectives whose every role is carried
// by one launch.  The inputs of all but the last part (sums behind a wait) are complete when the launch starts (stream order).
//
// What bounds them.  Large ones: HBM (a copy reads and writes each byte once; 128 MiB of traffic at 4096 x 4096
// fp16 in both directions takes 20 us).  Small ones: the launch and one trip to memory, so the work is cut
// finely enough to give every CU a share (launch_bulk_copy, launch_bulk_reduce) and every rank's value of a unit
// is requested before the first is added.  The reduction of eight ranks' 2 MiB fp32 chunks took 45 us as 32
// tasks of 16384 elements, 6.0 us now; eight such reductions and eight 2 MiB gathers, one call after the other: 462 us
// before, 108 us now, 7.2 us of device time a gather.  S0 of the reduce-scatter with bf16 partials
// (16384 x 4096): 184 us before, 171 us now.
#pragma once

#include "tccl_comm.h"

namespace tccl {

// ---- copies: up to kMaxTransfers rectangles of one shape, one per blockIdx.y ------------------------
constexpr int kMaxTransfers = 9;  // an exchange on eight ranks: seven pulls and the push; a gather: eight

struct BulkTransfer {
  int64_t src_shift, dst_shift;  // bytes added to the common source / destination address
  int src_rank;                  // slice read
  uint32_t dst_ranks;            // slices written
};
struct BulkCopyArgs {
  const int64_t* heap_bases;
  int64_t src, dst;  // addresses in slice `rank`
  uint32_t src_pitch, dst_pitch;
  int rank, world;
  int upr;         // 16-byte units per row
  int units;       // rows * upr
  int task_units;  // units a workgroup takes at a time (a multiple of its threads)
  BulkTransfer t[kMaxTransfers];
};

template <int kThreads>
TCCL_D void bulk_copy(const BulkCopyArgs& a, int which, int wg, int num_wgs) {
  const BulkTransfer t = a.t[which];
  const int64_t mine = a.heap_bases[a.rank];
  const CopyBatch<kBulkCopyPolicy, kThreads> b{a.heap_bases, a.world, t.dst_ranks, a.dst + t.dst_shift - mine,
                                               window(a.src + t.src_shift - mine + a.heap_bases[t.src_rank]),
                                               a.src_pitch == (uint32_t)a.upr * 16u && a.dst_pitch == a.src_pitch,
                                               (uint32_t)a.upr, a.src_pitch, a.dst_pitch, (int)threadIdx.x, a.units};
  const int tasks = (a.units + a.task_units - 1) / a.task_units;
  for (int task = wg; task < tasks; task += num_wgs) {
    const int lo = task * a.task_units;
    run_copy(b, lo, lo + a.task_units < a.units ? lo + a.task_units : a.units);
  }
}

// ---- reductions: one owner's rectangle per blockIdx.y ------------------------------------------------
// dst = cast(sum over ranks of src), fp32 accumulation, one rounding; the rank `first` is added first (the
// owner: tile_reduce_scatter, collectives.py:766-781), then the others ascending.
struct BulkReduceArgs {
  const int64_t* heap_bases;
  int64_t src, dst;                // addresses in slice `rank`
  int64_t src_shift, dst_shift;    // bytes per owner: owner o reduces src + o * src_shift into dst + o * dst_shift
  uint32_t src_pitch, dst_pitch;
  int rank, world;
  int upr, units;                  // 8-element units per row and in all
  int first_owner;                 // owner of blockIdx.y == 0
  int ascending;                   // 1: the ranks' values in ascending order, whoever owns the rectangle
  int to_all;                      // 1: every slice receives the sum; 0: the owner's
};

// kRanks: the most ranks this instantiation holds in registers at once (2, 4 or 8; world <= kRanks).
template <typename PT, typename OT, int kRanks, int kThreads, int kLoadPolicy = kBulkReducePolicy>
TCCL_D void bulk_reduce(const BulkReduceArgs& a, int owner, int wg, int num_wgs) {
  constexpr uint32_t kSrcUnit = 8 * sizeof(PT), kDstUnit = 8 * sizeof(OT);
  // Units per thread and round: 256 bytes of requests in flight per thread for fp32, 128 for the 16-bit types.
  // Measured on the bulk reductions of 8192 x 4096 fp32 and 16384 x 4096 bf16 partials of two ranks: 2 units
  // 68 / 126 us, 4 units 66 / 114 us, 8 units 84 / 141 us.
  constexpr int kUnits = 8 / kRanks;
  const int64_t mine = a.heap_bases[a.rank];
  const int64_t src_off = a.src + owner * a.src_shift - mine, dst_off = a.dst + owner * a.dst_shift - mine;
  const int first = a.ascending ? 0 : owner;
  const bool flat = a.src_pitch == (uint32_t)a.upr * kSrcUnit && a.dst_pitch == (uint32_t)a.upr * kDstUnit;
  // Rank order of the addends: `first`, then the others ascending.
  __amdgpu_buffer_rsrc_t from[kRanks];
#pragma unroll
  for (int i = 0; i < kRanks; ++i) {
    const int p = i == 0 ? first : (i <= first ? i - 1 : i);
    from[i] = window(a.heap_bases[p < a.world ? p : first] + src_off);
  }
  for (int u0 = wg * kThreads * kUnits; u0 < a.units; u0 += num_wgs * kThreads * kUnits) {
    uint32_t soff[kUnits], doff[kUnits];
    bool live[kUnits];
    u32x4 raw[kUnits][kRanks][sizeof(PT) / 2];
#pragma unroll
    for (int k = 0; k < kUnits; ++k) {
      const int u = u0 + (int)threadIdx.x + k * kThreads;
      live[k] = u < a.units;
      if (flat) {
        soff[k] = (uint32_t)u * kSrcUnit;
        doff[k] = (uint32_t)u * kDstUnit;
      } else {
        const uint32_t r = (uint32_t)u / (uint32_t)a.upr, c = (uint32_t)u - r * (uint32_t)a.upr;
        soff[k] = r * a.src_pitch + c * kSrcUnit;
        doff[k] = r * a.dst_pitch + c * kDstUnit;
      }
      if (!live[k]) soff[k] = 0;  // idle lane: harmless re-read, nothing stored
    }
#pragma unroll
    for (int i = 0; i < kRanks; ++i)
      if (kRanks == 2 || i < a.world) {
#pragma unroll
        for (int k = 0; k < kUnits; ++k)
#pragma unroll
          for (int h = 0; h < (int)sizeof(PT) / 2; ++h) raw[k][i][h] = ld16<kLoadPolicy>(from[i], soff[k] + 16u * h);
      }
    float acc[kUnits][8];
#pragma unroll
    for (int i = 0; i < kRanks; ++i)
      if (kRanks == 2 || i < a.world) {
#pragma unroll
        for (int k = 0; k < kUnits; ++k) {
          PT e[8];
          __builtin_memcpy(e, raw[k][i], sizeof e);
#pragma unroll
          for (int j = 0; j < 8; ++j) acc[k][j] = i == 0 ? (float)e[j] : acc[k][j] + (float)e[j];
        }
      }
    for (int q = a.to_all ? 0 : owner; q < (a.to_all ? a.world : owner + 1); ++q) {
      const __amdgpu_buffer_rsrc_t to = window(a.heap_bases[q] + dst_off);
#pragma unroll
      for (int k = 0; k < kUnits; ++k)
        if (live[k]) store8<OT, kBulkReducePolicy>(to, doff[k], acc[k]);
    }
  }
}

// ---- reductions behind a wait ---------------------------------------------------------------------
// The sums of a reduce-scatter whose tiles do not sum themselves (run_variant() in tccl_api.hip): this rank's partials are in
// memory, the peers' are once their words say so.  One workgroup looks at all words of an owner's rows, a word per
// lane, until `deadline`; false if some word has not come by then (the fault word is raised).
template <int kThreads>
TCCL_D bool rows_published(const CommArgs& c, int owner, int64_t deadline) {
  const int shard = c.M / c.world, lo = owner * shard, hi = lo + shard, peers = c.world - 1;
  const bool by_tile = c.granularity == kPerTile;
  const int first = lo / c.block_m;
  const int n = by_tile ? ((hi - 1) / c.block_m - first + 1) * c.tile_cols : c.n_groups;  // words per peer
  bool ok = true;
  for (int i = (int)threadIdx.x; i < n * peers && ok; i += kThreads) {
    const int p = i / n, word = i - p * n, peer = p < c.rank ? p : p + 1;
    if (by_tile)
      ok = tile_wait_ge<true>(peer_words(c, c.locks, peer), tile_id_of(first + word / c.tile_cols, word % c.tile_cols, c.tile_rows, c.tile_cols, c.group_m),
                              c.epoch, deadline);
    else if (group_hi(c, word) > lo && group_lo(c, word) < hi)
      ok = tile_wait_ge<true>(peer_words(c, c.counter, peer), word, (int32_t)((uint32_t)c.epoch * (uint32_t)c.tile_counts[word]), deadline);
  }
  const bool all = __syncthreads_and(ok ? 1 : 0) != 0;
  if (!all && threadIdx.x == 0 && c.fault) *c.fault = 1;
  return all;
}

}  // namespace tccl
