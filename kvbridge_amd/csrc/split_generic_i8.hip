// int8 instances of the generic MFMA split kernels (split_generic_mfma.h).
#include "split_generic_mfma.h"

namespace kvb {
namespace {

template <int DP, int NW>
hipError_t launch_nw(const SplitArgs& a, hipStream_t stream) {
  const bool varlen = a.seq_starts != nullptr;
  const dim3 grid(a.kv_heads * ((a.rows * a.group + 15u) / 16u), a.splits, varlen ? a.batch : 1u);
  if (varlen) hipLaunchKernelGGL((split_generic_i8_kernel<DP, NW, true>), grid, dim3(64 * NW), 0, stream, a);
  else hipLaunchKernelGGL((split_generic_i8_kernel<DP, NW, false>), grid, dim3(64 * NW), 0, stream, a);
  return hipGetLastError();
}

template <int DP>
hipError_t launch_dim(const SplitArgs& a, int nw, hipStream_t stream) {
  return nw == 4 ? launch_nw<DP, 4>(a, stream) : (nw == 2 ? launch_nw<DP, 2>(a, stream) : launch_nw<DP, 1>(a, stream));
}

template <int DP, int NW>
hipError_t preload_nw() {
  hipFuncAttributes attr{};
  const hipError_t e = hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(&split_generic_i8_kernel<DP, NW, false>));
  return e != hipSuccess
             ? e
             : hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(&split_generic_i8_kernel<DP, NW, true>));
}

template <int DP>
hipError_t preload_dim() {
  hipError_t e = preload_nw<DP, 1>();
  if (e == hipSuccess) e = preload_nw<DP, 2>();
  if (e == hipSuccess) e = preload_nw<DP, 4>();
  return e;
}

}  // namespace

hipError_t launch_generic_i8(const SplitArgs& a, int nw, hipStream_t stream) {
  if (a.dim <= 64) return launch_dim<64>(a, nw, stream);
  return a.dim <= 128 ? launch_dim<128>(a, nw, stream) : launch_dim<256>(a, nw, stream);
}

hipError_t preload_generic_i8() {
  hipError_t e = preload_dim<64>();
  if (e == hipSuccess) e = preload_dim<128>();
  return e == hipSuccess ? preload_dim<256>() : e;
}

}  // namespace kvb
