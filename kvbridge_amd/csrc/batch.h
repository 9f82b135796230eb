// Per-sequence view of a batched decode call (SplitArgs::seq_starts set).
// Sequence b owns tokens [seq_starts[b], seq_starts[b+1]) of k_positions and
// page-table entries page_offsets[b] .. of page_table; its logical token t
// lives in physical page page_table[page_offsets[b] + t / page_tokens].
// Device metadata is not validated on the host (it may change between
// graph replays), so every index is clamped here to the array sizes the host
// declared: a malformed batch gives wrong numbers for that sequence but
// never reads outside k_positions, page_table or the KV pool.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.h"

namespace kvb {

struct SeqExtent {
  uint32_t start;      // first k_positions entry
  uint32_t tokens;     // clamped token count (<= max_tokens)
  uint32_t table_off;  // first page_table entry
};

__device__ __forceinline__ SeqExtent seq_extent(const SplitArgs& a, uint32_t b) {
  uint32_t s0 = a.seq_starts[b], s1 = a.seq_starts[b + 1];
  s0 = s0 < a.total_tokens ? s0 : a.total_tokens;
  s1 = s1 < s0 ? s0 : (s1 < a.total_tokens ? s1 : a.total_tokens);
  uint32_t t = s1 - s0 < a.max_tokens ? s1 - s0 : a.max_tokens;
  uint32_t off = a.page_offsets[b];
  off = off < a.table_entries ? off : a.table_entries;
  const uint64_t cap = uint64_t(a.table_entries - off) * a.page_tokens;  // tokens the table slice can map
  if (t > cap) t = uint32_t(cap);
  return SeqExtent{s0, t, off};
}

// Which (sequence, split) a work-group of a batched call takes.
struct BatchItem {
  uint32_t seq, split;
  SeqExtent e;
};

// Inclusive sum over the wave's lanes.
__device__ __forceinline__ uint32_t wave_scan(uint32_t x) {
  int v = int(x);
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);  // row_shr 1, 2, 4, 8: sums in 16-lane rows
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast 15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // row_bcast 31 into rows 2 and 3
  return uint32_t(v);
}

// Batched grids are (kv heads [x head-row blocks], splits of max_tokens,
// sequences); the work-groups take the sequences' own splits first, in order,
// and the places past a sequence's end (nothing to read) last.  With the
// place (split, sequence) taken from the block index itself the empty ones
// lie between the others, and as the dispatcher deals work-groups to XCDs and
// CUs by index, some CUs got several times the work of others: 32 sequences
// of 100 .. 4,000 tokens in 8 splits of 512 took 1.4 times as long as 32 of
// 2,048.  Measured (us per call, 32 q / 8 kv heads, dim 128, 64-token pages,
// block index -> packed): 16 sequences of 1K .. 32K tokens in splits of 1,024
// / 2,048 / 5,120 120.7 -> 92.8 / 114.8 -> 94.1 / 91.9 -> 88.5; 32 of 100 ..
// 4,000 in 512 39.8 -> 36.8; 200 of 300 .. 2,000 in 512 123.9 -> 102.3.
// Every wave derives the same item: lane = sequence, a sum over the lanes, 64
// sequences per round (a.packed: at most 256 sequences; above that the rounds
// would cost more than the imbalance).  A grid of at most one work-group per
// CU has nothing to balance and takes the block index as it is (two
// sequences, 144 work-groups: 16.5 against 16.9 us).  Above that sequences of
// one length pay 0.4 to 1.0 us for nothing (11 of 3,326 tokens, dim 64: 20.7 ->
// 21.4), but the host sees neither lengths nor whether the declared totals are
// capacities.  Consecutive work-groups
// are the kv heads of one item, so each XCD gets the same share of every
// sequence when there are 8 of them.
__device__ __forceinline__ BatchItem batch_item(const SplitArgs& a) {
  if (a.packed == 0u) return BatchItem{blockIdx.z, blockIdx.y, seq_extent(a, blockIdx.z)};
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t w = blockIdx.y + a.splits * blockIdx.z;
  BatchItem it{0u, 0u, SeqExtent{0u, 0u, 0u}};
  // Pass 0: the sequences' own splits; pass 1: the places past them.
  uint32_t base = 0;
  for (uint32_t pass = 0; pass < 2u; ++pass) {
    for (uint32_t b0 = 0; b0 < a.batch; b0 += 64u) {
      const bool in = b0 + lane < a.batch;
      const uint32_t b = in ? b0 + lane : a.batch - 1u;
      const SeqExtent e = seq_extent(a, b);
      const uint32_t own = e.tokens > 0u ? (e.tokens - 1u) / a.split_tokens + 1u : 1u;
      const uint32_t count = !in ? 0u : (pass == 0u ? own : a.splits - own);
      const uint32_t upto = base + wave_scan(count);
      const uint64_t hit = __ballot(upto > w);
      if (hit != 0u) {
        const int l = __builtin_ctzll(hit);
        it.seq = b0 + uint32_t(l);
        const uint32_t at = w - uint32_t(__builtin_amdgcn_readlane(int(upto - count), l));
        it.split = at + (pass == 0u ? 0u : uint32_t(__builtin_amdgcn_readlane(int(own), l)));
        it.e.start = uint32_t(__builtin_amdgcn_readlane(int(e.start), l));
        it.e.tokens = uint32_t(__builtin_amdgcn_readlane(int(e.tokens), l));
        it.e.table_off = uint32_t(__builtin_amdgcn_readlane(int(e.table_off), l));
        return it;
      }
      base = uint32_t(__builtin_amdgcn_readlane(int(upto), 63));
    }
  }
  return it;  // not reached: the counts of both passes add up to the grid
}

// Rebase a batched call's arguments on sequence b: its block of row-heads in
// q, q_positions, scratch, counters and the outputs, its k_positions and
// page-table slice, and the token interval [0, T_b).  Splits past the
// sequence's own count see an empty interval and write empty partials
// (m = -inf, l = 0, n = 0), which every merge skips; the single-launch
// kernel instead ends those work-groups at once and merges only the
// sequence's own splits.
__device__ __forceinline__ void rebase_sequence(SplitArgs& a, uint32_t b, const SeqExtent& e) {
  const size_t rh0 = size_t(b) * a.rows * a.q_heads;
  a.q += rh0 * a.dim;
  a.q_positions += size_t(b) * a.rows;
  a.k_positions += e.start;
  a.page_table += e.table_off;
  a.begin = 0;
  a.end = e.tokens;
  a.scratch += rh0 * a.splits * (size_t(a.dim) + 2);
  if (a.counters) a.counters += size_t(b) * a.kv_heads;
  if (a.m) a.m += rh0;
  if (a.l) a.l += rh0;
  if (a.n) a.n += rh0 * a.dim;
  if (a.out) {
    if (a.out_type == 2) a.out = static_cast<_Float16*>(a.out) + rh0 * a.dim;
    else a.out = static_cast<float*>(a.out) + rh0 * a.dim;
  }
}

}  // namespace kvb
