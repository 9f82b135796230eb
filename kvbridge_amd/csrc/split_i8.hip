// Host side of the integer-MFMA split kernel (split_i8.h): shape support,
// the (waves, ring slots) choice, and dispatch to the per-dim translation
// units split_i8_d64/_d128/_d256.hip (built in parallel).
#include <cstdio>
#include <cstdlib>

#include "kernels.h"

namespace kvb {

hipError_t launch_i8_d64(const SplitArgs& a, int cfg, hipStream_t stream);
hipError_t launch_i8_d128(const SplitArgs& a, int cfg, hipStream_t stream);
hipError_t launch_i8_d256(const SplitArgs& a, int cfg, hipStream_t stream);
hipError_t preload_i8_d64();
hipError_t preload_i8_d128();
hipError_t preload_i8_d256();

namespace {

constexpr uint32_t kTiles = 64;  // tokens per tile

// (waves, ring slots) per work-group as 10 * NW + NB; NB = 1: one-tile chunks.
// `single`: the call is to be a single launch (its merge runs in the kernel).
//
// A grid of at most two work-groups per CU of a 256-CU device is bound by
// the latency of its work-groups when its splits are short: a wave that holds
// one tile runs a chunk of one (NB = 1) instead of four items of K and of V,
// three of them empty, and both of its items are in flight from the start.
// Eight waves (two per SIMD, <= 256 registers each) fill a CU and hold a tile
// each up to 8 tiles; a second round of one-tile chunks (9 tiles and more)
// costs as much as the first, where four waves take a chunk of up to four
// tiles each.  Eight-wave work-groups do not share a CU, four-wave ones do, so
// with more than one work-group per CU four waves are faster at any length.
// Dim 256 and 5 to 8 head-rows take a SIMD per wave: four waves.
// Measured (us per call, graph replay, two launches; 8 kv heads, 16 above 256
// work-groups; eight waves in chunks of one / four in chunks of one / of four):
//   dim 128, 4 head-rows, 256 work-groups   4 tiles 11.0 /  9.9 / 13.0
//     8 tiles 12.4 / 12.2 / 13.0   9: 13.4 / 14.1 / 13.1   15: 16.7 / - / 14.5
//   the same, 512 work-groups               5 tiles 19.3 / 14.3 / 16.6
//     8 tiles 22.3 / 17.1 / 18.3   9: 23.8 / 19.2 / 18.7   15: 31.2 / - / 24.4
//   dim 64, 1 head-row, 32 work-groups     11 tiles  9.6 / 10.7 /  9.9
//    12 tiles  9.6 / 10.6 / 9.9   13: 10.4 / 12.2 / 9.8
//   dim 256, 4 head-rows, 128 work-groups   4 tiles - / 14.7 / 18.8
//     8 tiles - / 19.1 / 19.8      9: - / 21.5 / 20.5
//   the same, 512 work-groups               2 tiles - / 22.9 / 28.6; two waves 20.6
// In the single launch, whose merge wants a thread per output, eight waves
// stay ahead to 12 tiles (dim 128, 32 work-groups, 1 / 4 head-rows 11.8 / 12.7
// against 12.0 / two launches 12.6).  From 16 tiles on chunks of four stay
// (65,536 tokens in 2,048 26.5 against 27.8).
//
// Larger grids (batches) run several rounds of work-groups per CU, and
// smaller work-groups that share a CU hide each other's prologue and
// combine: four waves (two per SIMD) for <= 4 head-rows, two waves for 8
// head-rows (whose state takes one SIMD per wave).  Measured on MI355X (16
// ragged sequences of 1K .. 32K tokens / 4 sequences of 128K tokens, 8
// head-rows): 118 / 216 us with these against 140 / 242 us with the
// single-sequence choice.  Large grids of short splits (<= 32 tiles) run one
// wave per work-group: the wave streams its split alone, so there is no wave
// combine, no work-group barrier and no idle wave per split, and eight such
// work-groups share a CU.  Measured: 65,536 tokens through launch_attention
// (its 256-token splits, 2,048 work-groups) 47.7 -> 25.3 us for the split
// launch, 4 x 128K tokens (64 chunks of 2,048 tokens, 8 head-rows) 203.5 ->
// 190.6 us; the ragged batch at 5,120-token splits (80 tiles) stays on four
// waves (91 against 111 us).
// KVB_I8_CFG="NW,NB" overrides (tuning sweeps; unknown pairs fall back).
int i8_config(const SplitArgs& a, bool single) {
  static const int forced = [] {
    const char* e = std::getenv("KVB_I8_CFG");
    int nw = 0, nb = 0;
    char tail = 0;
    if (!e || std::sscanf(e, "%d,%d%c", &nw, &nb, &tail) != 2 || nw < 1 || nw > 9 || nb < 1 || nb > 9) return 0;
    return nw * 10 + nb;
  }();
  const uint32_t tiles = (a.split_tokens - 1u) / kTiles + 1u;
  const uint32_t hr = a.rows * a.group;
  const bool eight = hr <= 4 && a.dim <= 128;
  if (forced == 42 || (forced == 41 && hr <= 4) || forced == 22 || forced == 12 || ((forced == 82 || forced == 81) && eight))
    return forced;
  const uint64_t groups = uint64_t(a.splits) * a.kv_heads * (a.seq_starts ? a.batch : 1u);
  if (groups > 512u) {
    if (tiles <= 32u) return 12;
    return hr <= 4 ? 42 : 22;
  }
  const bool crowded = groups > 256u;  // more than one work-group per CU
  if (tiles >= 16u) return eight ? 82 : 42;
  if (!eight) return hr > 4 || tiles > 8u ? 42 : (crowded && tiles < 4u ? 22 : 41);
  if (tiles <= 4u || (crowded && tiles <= 8u)) return 41;
  return !crowded && (tiles <= 8u || (tiles <= 12u && (a.dim == 64u || single))) ? 81 : 42;
}

}  // namespace

// head_rows <= 8 (<= 4 at dim 256); page_tokens a power of two >= 16 (>= 64
// for batched calls); the small-page path addresses K/V with 32-bit offsets.
bool i8_supported(const SplitArgs& a) {
  const uint32_t hr = a.rows * a.group, P = a.page_tokens;
  if (hr > 8 || (a.dim == 256 && hr > 4)) return false;
  if (a.dim != 64 && a.dim != 128 && a.dim != 256) return false;
  if (P < 16 || (P & (P - 1u)) != 0) return false;
  if (a.seq_starts && P < kTiles) return false;  // batched calls: whole-tile pages only
  if (P < kTiles && uint64_t(a.pages) * a.kv_heads * P * a.dim >= (uint64_t(1) << 32)) return false;
  return true;
}

// Whether the single launch runs its in-kernel merge or the call is two
// launches.  The merge is one work-group per kv head with a thread per output
// and a wave per head-row, at most 32 splits (otherwise the stand-alone merge,
// whose work-groups spread over every CU, is faster: 8 head-rows, 32 splits
// 14.3 against 21.5 us per call, 64 splits 8.5 against 11.0).  A split that is
// alone needs no merge and is one launch whatever its shape (dim 256, 4
// head-rows, 32 sequences of 8 / 20 tiles 18.9 / 37.6 against 23.4 / 42.3).
// Short splits leave the tickets and the merge nothing to hide behind, so below
// 16 tiles only small grids keep it (us per call, single launch against two):
//   64 work-groups, 4 x 64 outputs, 4 tiles  7.6 / 8.2;  256, 1 x 128  11.0 / 10.0
//   128 work-groups of 16 splits, 4 x 128 outputs, 11 tiles  13.2 / 12.8;  of 4
//   splits 13.3 / 13.4
//   256 work-groups, 1 x 128, 16 tiles 17.5 / 18.4
// One head-row of one sequence at dim 128 has the shortest merge and stays one
// launch from 13 tiles on in any grid: 32 / 128 / 256 / 512 work-groups, 14
// tiles 12.1 / 12.9 / 14.9 / 22.9 against 12.3 / 12.7 / 13.7 / 21.7.
// Grids of more than two work-groups per CU (batches) also run two launches:
// every work-group's ticket and the merges then sit between rounds of split
// work (16 ragged sequences: 116 us for two launches against 121-123 us).
bool i8_fusable(const SplitArgs& a) {
  if (!i8_supported(a)) return false;
  const uint64_t groups = uint64_t(a.splits) * a.kv_heads * (a.seq_starts ? a.batch : 1u);
  if (groups > 512u || a.splits > 32u) return false;
  const uint32_t nw = uint32_t(i8_config(a, true)) / 10u, hr = a.rows * a.group, outputs = hr * a.dim;
  if (nw < 4u || hr > 4u) return false;
  if (a.splits == 1u) return true;
  if (outputs > 64u * nw) return false;
  const uint32_t tiles = (a.split_tokens - 1u) / kTiles + 1u;
  const bool one_row = hr == 1u && a.dim == 128u && a.seq_starts == nullptr && tiles > 12u;
  return one_row || tiles >= 16u || (groups <= 128u && (outputs <= 256u || (tiles >= 8u && a.splits <= 8u)));
}

hipError_t launch_i8_fenced_d128(const SplitArgs& a, hipStream_t stream);

// Diagnostic single launch with formal release / acquire fences: only the
// eight-wave dim-128 page-tile configuration (cfg2's) has an instance.  Calls
// of that configuration whose merge is a launch of its own (33 to 128 splits)
// need no fence: the second launch sees what the first one wrote.
bool i8_fenced_supported(const SplitArgs& a) {
  return a.dim == 128 && a.seq_starts == nullptr && a.page_tokens >= kTiles && i8_supported(a) &&
         i8_config(a, true) == 82 && (i8_fusable(a) || (a.splits <= 128u && uint64_t(a.splits) * a.kv_heads <= 512u));
}

hipError_t launch_split_i8_fenced(const SplitArgs& a, hipStream_t stream) {
  return i8_fenced_supported(a) && i8_fusable(a) ? launch_i8_fenced_d128(a, stream) : hipErrorInvalidValue;
}

hipError_t launch_split_i8(const SplitArgs& a, hipStream_t stream) {
  const int cfg = i8_config(a, a.counters != nullptr);
  switch (a.dim) {
    case 64: return launch_i8_d64(a, cfg, stream);
    case 128: return launch_i8_d128(a, cfg, stream);
    case 256: return launch_i8_d256(a, cfg, stream);
    default: return hipErrorInvalidValue;
  }
}

const char* i8_kernel_name(const SplitArgs& a) {
  static thread_local char buf[112];
  const int cfg = i8_config(a, a.counters != nullptr);
  std::snprintf(buf, sizeof(buf), "split_i8_kernel<%u,%d,%d,%s,%d,%s,%s,false>", a.dim, cfg / 10, cfg % 10,
                a.page_tokens >= kTiles ? "true" : "false", a.rows * a.group <= 4 ? 4 : 8,
                a.counters != nullptr ? "true" : "false", a.seq_starts != nullptr ? "true" : "false");
  return buf;
}

hipError_t preload_i8() {
  hipError_t e = preload_i8_d64();
  if (e == hipSuccess) e = preload_i8_d128();
  if (e == hipSuccess) e = preload_i8_d256();
  return e;
}

}  // namespace kvb
