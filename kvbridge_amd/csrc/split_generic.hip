// Split partials of every valid shape that the tiled kernels do not take:
// fp32 KV, other dims, misaligned buffers, ragged batches over small pages or
// with many head-rows, and the tiled shapes of one_block_rows and
// off_grid_rows.  The MFMA kernels (split_generic_mfma.h) serve
// the shapes they can load in whole 16-byte pieces, the scalar kernel here
// (split_generic.h) the rest: dims that are not a multiple of 4, pages that
// are not a multiple of 16 tokens.
//
// Scalar kernel: grid x = row * q_heads + head, y = split, z = sequence of a
// batched call; block of 256 threads (4 waves).
#include <cstdio>

#include "kernels.h"
#include "batch.h"
#include "split_generic.h"

namespace kvb {

hipError_t launch_generic_i8(const SplitArgs& a, int nw, hipStream_t stream);
hipError_t launch_generic_f32(const SplitArgs& a, int nw, hipStream_t stream);
hipError_t preload_generic_i8();
hipError_t preload_generic_f32();

namespace {

constexpr int kThreads = 256;

template <bool kInt8, bool VARLEN>
__global__ __launch_bounds__(kThreads) void split_generic_kernel(SplitArgs a) {
  if constexpr (VARLEN) rebase_sequence(a, blockIdx.z, seq_extent(a, blockIdx.z));
  __shared__ GenericLds<kThreads> lds;
  split_generic_row<kInt8, kThreads>(a, blockIdx.x, blockIdx.y, lds);
}

// Waves per work-group.  int8 (64-token tiles): four -- more leave a wave one
// tile and a longer combine, fewer leave the CUs short of requests (us per
// call, 8 / 4 / 2 waves: dim 96, 8,000 tokens 16.2 / 16.2 / 19.7; 8 ragged
// sequences of up to 4,000 tokens, 8 head-rows 27.4 / 21.8 / 25.8; the same
// 32 sequences 69.4 / 47.9 / 48.2); two where several work-groups per CU
// have only four tiles each (16 sequences, 256-token splits 57.5 / 35.3 /
// 32.7).  fp32 (16-token tiles): eight where the registers allow it and a
// work-group has a CU to itself (dim 64, 8,192 tokens 14.4 / 16.6 / 24.4).
int mfma_waves(const SplitArgs& a, bool int8) {
  const uint32_t tile = int8 ? 64u : 16u, tiles = (a.split_tokens - 1u) / tile + 1u;
  const uint64_t blocks = (uint64_t(a.rows) * a.group + 15u) / 16u;
  const uint64_t groups = blocks * a.kv_heads * a.splits * (a.seq_starts ? a.batch : 1u);
  uint32_t nw = 4;
  if (int8 && groups > 1024u && tiles <= 4u) nw = 2;
  if (!int8 && a.dim <= 128 && groups <= 512u) nw = 8;
  while (nw > tiles) nw /= 2u;
  return int(nw);
}

}  // namespace

// Shapes of the MFMA kernels: K rows and V columns in dword-aligned 16-byte
// loads (dim a multiple of 4, whole 16-token groups in a page), fp32 V slabs
// within 32-bit byte offsets, and a grid of head-row blocks that fits grid.x.
bool generic_mfma_supported(const SplitArgs& a, bool int8) {
  if (a.dim % 4 != 0 || a.page_tokens % 16 != 0) return false;
  if (reinterpret_cast<uintptr_t>(a.k) % 4 != 0 || reinterpret_cast<uintptr_t>(a.v) % 4 != 0) return false;
  if (!int8 && uint64_t(a.dim) * a.page_tokens >= (uint64_t(1) << 30)) return false;
  const uint64_t blocks = (uint64_t(a.rows) * a.group + 15u) / 16u;
  return a.kv_heads * blocks < (uint64_t(1) << 22);
}

// 5 to 16 head-rows at dim 64 and 128 fill the generic kernel's one block of
// columns, which costs it the same for any number of them, and its state fits
// two waves per SIMD.
//  * 5 to 8 (wide GQA): the int8 kernel's state for 8 head-rows takes a SIMD
//    per wave.  us per call, int8 -> generic, 64 q / 8 kv heads, dim 128:
//    splits of 256, 8,192 tokens 14.4 -> 11.3, 65,536 tokens 45.3 -> 40.9; of
//    512, 16,384 tokens 18.3 -> 14.1; dim 64, 16 q / 2 kv heads 12.6 -> 9.9;
//    32 sequences of 100 .. 4,000 in 512 53.3 -> 45.1, 4 of up to 9,000 21.1 ->
//    15.4.  From 16 tiles a split the two are within 4% (20.5 / 19.9, 30.8 /
//    29.5) and the int8 kernel stays.  Above 512 work-groups that one runs four
//    one-wave work-groups per CU and this one two of four waves, so at dim 128
//    grids that all but fill the int8 kernel's first round stay there: 640 / 768
//    / 896 / 1,024 / 1,152 work-groups, 8 head-rows, 4 tiles 19.7 / 20.2 / 22.0 /
//    23.3 / 35.6 -> 19.6 / 20.2 / 23.6 / 24.4 / 27.2, 12 tiles 34.2 / 36.2 / 41.1
//    / 43.8 / 66.4 -> 33.9 / 35.7 / 43.8 / 45.1 / 55.4; later rounds are within
//    4% of each other.  Of a batch this holds where its sequences are as long as
//    the longest (40 of 768 in 256 22.4 -> 26.2, but 40 of 90 .. 1,480 in 960 37.7
//    -> 29.0).  Dim 64 gains on either side (12 tiles, 640 / 1,024 work-groups
//    25.4 / 26.9 -> 19.5 / 24.7).
//  * 9 to 16 (a few query rows of one sequence), up to two work-groups per
//    CU: the rows kernels stage the split through LDS for up to four blocks.
//    4 rows x 32 q / 8 kv heads, dim 128, 16,001 tokens in splits of 512 /
//    1,024 18.2 -> 14.9 / 25.6 -> 19.2, 4,000 tokens in 256 14.8 -> 12.6; dim
//    64, 16,001 tokens in 512 13.3 -> 10.0.
// 17 to 32 head-rows are two blocks that each read the KV (19.6 against 22.8
// at dim 128, 512-token splits) and stay on the rows kernels.
bool one_block_rows(const SplitArgs& a) {
  const uint64_t hr = uint64_t(a.rows) * a.group;
  if (hr <= 4u || hr > 16u || (a.dim != 64 && a.dim != 128) || !generic_mfma_supported(a, true)) return false;
  if (hr > 8u) return a.seq_starts == nullptr && uint64_t(a.splits) * a.kv_heads <= 512u;
  if (a.split_tokens > 15u * 64u) return false;
  const bool batch = a.seq_starts != nullptr;
  if (a.dim == 64 || (batch && uint64_t(a.total_tokens) * 10u < uint64_t(a.batch) * a.max_tokens * 9u)) return true;
  const uint64_t groups = uint64_t(a.splits) * a.kv_heads * (batch ? a.batch : 1u);
  return groups < 768u || groups > 1024u;
}

// More than 8 head-rows over a range that begins off the 64-token tile grid,
// which the rows kernels do not take.  Like split_lds_kernel this one reads the
// KV once per block of 16 head-rows, and it keeps 24 bits of a weight where
// that one keeps 22 of f16 range: n is off by 3.1e-7 of 64 bits against 4e-6,
// and a v-scale of 2^30 times the others' costs them nothing (3e-3 there).
// us per call, split_lds_kernel -> this one, dense geometry (8 rows, group 6,
// dim 256, 256-token splits) 1,500 / 8,000 / 57,338 tokens 28.7 -> 21.5 / 55.4
// -> 41.2 / 286 -> 144; one 8,192-token split 276 -> 155; 8 rows x 32 q / 8 kv
// heads, dim 128, 16,000 / 65,536 tokens 28.2 -> 23.7 / 74.3 -> 51.0; dim 64,
// 65,536 tokens 72.7 -> 31.1; 512 head-rows 45.9 -> 39.9.  Counting the tokens
// from the begin would let the rows kernels take page-aligned begins (57,338
// tokens 55), but their weights are fixed point below the largest v-scale of
// an epoch, where a v-scale of 2^20 times the others' leaves them an error of
// 0.3 and a NaN becomes a number: not for calls that had neither.
bool off_grid_rows(const SplitArgs& a) {
  return uint64_t(a.rows) * a.group > 8u && a.begin % 64u != 0 && generic_mfma_supported(a, true);
}

hipError_t launch_split_generic(const SplitArgs& a, bool int8, hipStream_t stream) {
  if (generic_mfma_supported(a, int8)) {
    const int nw = mfma_waves(a, int8);
    return int8 ? launch_generic_i8(a, nw, stream) : launch_generic_f32(a, nw, stream);
  }
  const bool varlen = a.seq_starts != nullptr;
  const dim3 grid(a.rows * a.q_heads, a.splits, varlen ? a.batch : 1u);
  if (int8 && varlen)
    hipLaunchKernelGGL((split_generic_kernel<true, true>), grid, dim3(kThreads), 0, stream, a);
  else if (int8)
    hipLaunchKernelGGL((split_generic_kernel<true, false>), grid, dim3(kThreads), 0, stream, a);
  else if (varlen)
    hipLaunchKernelGGL((split_generic_kernel<false, true>), grid, dim3(kThreads), 0, stream, a);
  else
    hipLaunchKernelGGL((split_generic_kernel<false, false>), grid, dim3(kThreads), 0, stream, a);
  return hipGetLastError();
}

// The family, and after a colon the MFMA instance that serves the call.
const char* generic_kernel_name(const SplitArgs& a, bool int8) {
  static thread_local char buf[128];
  const char* const t = int8 ? "true" : "false";
  const char* const v = a.seq_starts != nullptr ? "true" : "false";
  const int at = std::snprintf(buf, sizeof(buf), "split_generic_kernel<%s, %s>", t, v);
  if (generic_mfma_supported(a, int8))
    std::snprintf(buf + at, sizeof(buf) - at, ": split_generic_%s_kernel<%d, %d, %s>", int8 ? "i8" : "f32",
                  a.dim <= 64 ? 64 : (a.dim <= 128 ? 128 : 256), mfma_waves(a, int8), v);
  return buf;
}

hipError_t preload_generic() {
  const void* fns[] = {reinterpret_cast<const void*>(&split_generic_kernel<true, false>),
                       reinterpret_cast<const void*>(&split_generic_kernel<false, false>),
                       reinterpret_cast<const void*>(&split_generic_kernel<true, true>),
                       reinterpret_cast<const void*>(&split_generic_kernel<false, true>)};
  hipFuncAttributes attr{};
  for (const void* f : fns) {
    const hipError_t e = hipFuncGetAttributes(&attr, f);
    if (e != hipSuccess) return e;
  }
  const hipError_t e = preload_generic_i8();
  return e != hipSuccess ? e : preload_generic_f32();
}

}  // namespace kvb
