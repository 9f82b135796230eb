// Split partials of every valid shape that the tiled kernels do not take:
// fp32 KV, other dims, misaligned buffers, and ragged batches over small
// pages or with many head-rows.  The MFMA kernels (split_generic_mfma.h) serve
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

// Shapes of the MFMA kernels: K rows and V columns in dword-aligned 16-byte
// loads (dim a multiple of 4, whole 16-token groups in a page), fp32 V slabs
// within 32-bit byte offsets, and a grid of head-row blocks that fits grid.x.
bool mfma_supported(const SplitArgs& a, bool int8) {
  if (a.dim % 4 != 0 || a.page_tokens % 16 != 0) return false;
  if (reinterpret_cast<uintptr_t>(a.k) % 4 != 0 || reinterpret_cast<uintptr_t>(a.v) % 4 != 0) return false;
  if (!int8 && uint64_t(a.dim) * a.page_tokens >= (uint64_t(1) << 30)) return false;
  const uint64_t blocks = (uint64_t(a.rows) * a.group + 15u) / 16u;
  return a.kv_heads * blocks < (uint64_t(1) << 22);
}

// Waves per work-group.  Up to two work-groups per CU: as many as the split
// has tiles for, because a lone work-group is bound by latency (8,000 tokens,
// dim 96, 128 work-groups of 8 tiles: split kernel 11.5 us with 8 waves,
// 15.0 with 2).  Larger grids: two waves, so that four work-groups share a CU
// and hide each other's prologue and combine (32 sequences of 100 .. 4,000
// tokens, dim 128, 2,048 work-groups: 49 us per call with 2 waves, 51 with 4,
// 73 with 8).  The state of dims above 128 takes a SIMD per wave.
int mfma_waves(const SplitArgs& a, bool int8) {
  const uint32_t tile = int8 ? 64u : 16u, tiles = (a.split_tokens - 1u) / tile + 1u;
  const uint64_t blocks = (uint64_t(a.rows) * a.group + 15u) / 16u;
  const uint64_t groups = blocks * a.kv_heads * a.splits * (a.seq_starts ? a.batch : 1u);
  int nw = groups > 512u ? 2 : (a.dim <= 128 ? 8 : 4);
  while (nw > 1 && uint32_t(nw) > tiles) nw /= 2;
  return nw;
}

}  // namespace

hipError_t launch_split_generic(const SplitArgs& a, bool int8, hipStream_t stream) {
  if (mfma_supported(a, int8)) {
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
  if (mfma_supported(a, int8))
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
