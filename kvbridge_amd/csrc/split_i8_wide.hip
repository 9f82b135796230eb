// The integer-MFMA split kernel with four digits for ragged batches over
// pages of 16 or 32 tokens (dim 128, at most 4 head-rows): the same stream and
// the same MFMA count as three digits -- 4 head-rows x 4 digits fill the 16
// columns -- and as exact as the fp32 arithmetic of the other generic kernels,
// without their conversions of the codes (n off by 2.1e-7 of 64 bits, relative,
// where the scalar kernel is off by 3.9e-7; 5.5e-7 while 2^kp sat in the
// weights' exponent).
#include "split_i8.h"

namespace kvb {
namespace {

template <int D, int NW, int NB, int HS>
__global__ __launch_bounds__(64 * NW) void split_i8_wide_kernel(
    const uint32_t* __restrict__ table_in, const int8_t* __restrict__ kdata, const float* __restrict__ kscale,
    const float* __restrict__ vscale, uint32_t p_begin, uint32_t p_end, uint32_t p_split_tokens,
    uint32_t p_page_tokens, uint32_t p_kv_heads, uint32_t p_pages, SplitArgs a_in,
    const float* __restrict__ q_in, const int64_t* __restrict__ qpos_in, const int64_t* __restrict__ kpos_in,
    const int8_t* __restrict__ vdata, float* __restrict__ scratch_in) {
  constexpr int ND = 4;
  constexpr bool PT = false, FUSED = false, VARLEN = true, FENCE = false;
#include "split_i8_body.h"
}

template <int D, int NW, int NB, int HS>
hipError_t launch_wide(const SplitArgs& a, hipStream_t stream) {
  hipLaunchKernelGGL((split_i8_wide_kernel<D, NW, NB, HS>), dim3(a.kv_heads, a.splits, a.batch), dim3(64 * NW), 0,
                     stream, KVB_I8_ARGS);
  return hipGetLastError();
}

// (waves, ring slots) as in split_i8.hip: one-tile chunks on four waves for
// short splits of a grid that the chip holds at once, one wave for them in
// larger grids, two waves up to 32 tiles, four beyond.  Measured (us per call,
// 32 q / 8 kv heads, 16-token pages; waves x ring 1x2 / 2x2 / 4x1 / 4x2, and
// split_generic_i8_kernel):
//   32 sequences of 100 .. 4,000, splits of 512  38.5 / 37.5 / 42.8 / 47.4  43.9
//   the same, splits of 256                      40.2 / 47.8 / 53.4 / 75.3  44.2
//   12 of up to 3,000 (4 kv heads)               24.0 / 16.0 / 14.5 / 16.3  14.9
//   2 of 32,768, splits of 2,048                 66.1 / 37.7 / 31.8 / 28.6  32.2
// Dim 64 and 8 head-rows stay on split_generic_i8_kernel, which was faster
// there (15.5 against 13.6, 58.8 against 47.9 us).
int wide_config(const SplitArgs& a) {
  const uint32_t tiles = (a.split_tokens - 1u) / kTileTokens + 1u;
  const uint64_t groups = uint64_t(a.splits) * a.kv_heads * a.batch;
  if (groups <= 512u) return tiles < 16u ? 41 : 42;
  return tiles <= 4u ? 12 : (tiles <= 32u ? 22 : 42);
}

}  // namespace

bool i8_wide_supported(const SplitArgs& a) {
  if (a.seq_starts == nullptr || (a.page_tokens != 16 && a.page_tokens != 32)) return false;
  if (a.dim != 128 || a.rows * a.group > 4) return false;
  if (uint64_t(a.pages) * a.kv_heads * a.page_tokens * a.dim >= (uint64_t(1) << 32)) return false;
  const auto al = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  return al(a.k) && al(a.v) && al(a.q);
}

hipError_t launch_split_i8_wide(const SplitArgs& a, hipStream_t stream) {
  switch (wide_config(a)) {
    case 12: return launch_wide<128, 1, 2, 4>(a, stream);
    case 22: return launch_wide<128, 2, 2, 4>(a, stream);
    case 41: return launch_wide<128, 4, 1, 4>(a, stream);
    default: return launch_wide<128, 4, 2, 4>(a, stream);
  }
}

const char* i8_wide_kernel_name(const SplitArgs& a) {
  switch (wide_config(a)) {
    case 12: return "split_i8_wide_kernel<128, 1, 2, 4>";
    case 22: return "split_i8_wide_kernel<128, 2, 2, 4>";
    case 41: return "split_i8_wide_kernel<128, 4, 1, 4>";
    default: return "split_i8_wide_kernel<128, 4, 2, 4>";
  }
}

hipError_t preload_i8_wide() {
  const void* fns[] = {reinterpret_cast<const void*>(&split_i8_wide_kernel<128, 1, 2, 4>),
                       reinterpret_cast<const void*>(&split_i8_wide_kernel<128, 2, 2, 4>),
                       reinterpret_cast<const void*>(&split_i8_wide_kernel<128, 4, 1, 4>),
                       reinterpret_cast<const void*>(&split_i8_wide_kernel<128, 4, 2, 4>)};
  return preload_fns(fns, 4);
}

}  // namespace kvb
