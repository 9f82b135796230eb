// Scalar split partial of one row-head: any valid Shape (dim 1..256, any page
// size, any begin, int8 or fp32 KV, any GQA group) and any values, on a
// work-group of NT threads.  The arithmetic follows the per-split semantics
// of the reference src/attention_shared.cu:42-209 / :213-293 (visible =
// k_pos <= q_pos, score = (q . k_code) * k_scale * scale, weights exp(score -
// split max), numerator weighted by v_scale; a zero weight leaves its V row
// out, whatever it holds), evaluated as an online softmax over 256-token
// chunks so that one work-group can cover a split of any length.
#pragma once
#include "kernels.h"
#include "device_common.h"

namespace kvb {

constexpr uint32_t kGenericChunk = 256;  // tokens per online-softmax step

template <int NT>
struct GenericLds {
  float q[256];
  float pw[kGenericChunk];
  uint32_t vbase[kGenericChunk];
  float red[2][NT / 64];
};

template <int NT>
__device__ __forceinline__ float block_max(float x, float* red) {
  x = wave_max(x);
  const int wave = threadIdx.x >> 6;
  __syncthreads();  // red is reused; previous readers must be done
  if ((threadIdx.x & 63) == 0) red[wave] = x;
  __syncthreads();
  float r = red[0];
#pragma unroll
  for (int w = 1; w < NT / 64; ++w) r = fmaxf(r, red[w]);
  return r;
}
template <int NT>
__device__ __forceinline__ float block_sum(float x, float* red) {
  x = wave_sum(x);
  const int wave = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[wave] = x;
  __syncthreads();
  float r = red[0];
#pragma unroll
  for (int w = 1; w < NT / 64; ++w) r += red[w];
  return r;
}

template <bool kInt8>
__device__ __forceinline__ float kv_value(const void* base, uint32_t i) {
  if constexpr (kInt8) return float(static_cast<const int8_t*>(base)[i]);
  else return static_cast<const float*>(base)[i];
}

// The whole work-group calls this with the same rh and split.
template <bool kInt8, int NT>
__device__ __forceinline__ void split_generic_row(const SplitArgs& a, uint32_t rh, uint32_t split,
                                                  GenericLds<NT>& lds) {
  // Tokens and dims per thread (a work-group of 512 leaves its upper half idle).
  constexpr uint32_t kPer = NT < int(kGenericChunk) ? kGenericChunk / NT : 1u;
  static_assert(kPer * NT % kGenericChunk == 0, "threads cover a chunk in whole rounds");
  const uint32_t tid = threadIdx.x;
  const uint32_t row = rh / a.q_heads, head = rh % a.q_heads;
  const uint32_t kv = head / a.group;
  const uint32_t D = a.dim, P = a.page_tokens;

  const uint64_t s0_64 = uint64_t(a.begin) + uint64_t(split) * a.split_tokens;
  const uint32_t s0 = s0_64 < a.end ? uint32_t(s0_64) : a.end;
  const uint32_t s1 = uint64_t(s0) + a.split_tokens < a.end ? s0 + a.split_tokens : a.end;
  const int64_t qpos = a.q_positions[row];

  __syncthreads();  // the LDS area may still be read
  for (uint32_t d = tid; d < D; d += NT) lds.q[d] = a.q[size_t(rh) * D + d];
  __syncthreads();

  float m_run = neg_inf(), l_run = 0.f, acc[kPer];
#pragma unroll
  for (uint32_t i = 0; i < kPer; ++i) acc[i] = 0.f;
  for (uint32_t c0 = s0; c0 < s1; c0 += kGenericChunk) {
    float score[kPer], vsc[kPer], smax = neg_inf();
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) {
      const uint32_t j = tid + i * NT, t = c0 + j;
      score[i] = neg_inf();
      vsc[i] = 0.f;
      uint32_t vb = 0;
      if (j < kGenericChunk && t < s1 && a.k_positions[t] <= qpos) {
        uint32_t page = a.page_table[t / P];
        page = page < a.pages ? page : a.pages - 1;
        const uint32_t slot = t % P;
        const uint32_t si = (page * a.kv_heads + kv) * P + slot;
        float dot = 0.f;
        for (uint32_t d = 0; d < D; ++d) dot = fmaf(lds.q[d], kv_value<kInt8>(a.k, si * D + d), dot);
        const float ks = kInt8 ? a.k_scales[si] : 1.f;
        vsc[i] = kInt8 ? a.v_scales[si] : 1.f;
        score[i] = dot * ks * a.scale;
        vb = (page * a.kv_heads + kv) * D * P + slot;
      }
      if (j < kGenericChunk) lds.vbase[j] = vb;
      smax = fmaxf(smax, score[i]);
    }
    const float cmax = block_max<NT>(smax, lds.red[0]);
    const float m_new = fmaxf(m_run, cmax);
    const float m_use = m_new == neg_inf() ? 0.f : m_new;
    const float alpha = exp_e(m_run - m_use);  // m_run = -inf -> 0
    float wsum = 0.f;
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) {
      const float w = exp_e(score[i] - m_use);  // score = -inf -> 0
      wsum += w;
      if (tid + i * NT < kGenericChunk) lds.pw[tid + i * NT] = w * vsc[i];
    }
    const float csum = block_sum<NT>(wsum, lds.red[1]);
    l_run = l_run * alpha + csum;
    m_run = m_new;
    __syncthreads();
    const uint32_t cnt = s1 - c0 < kGenericChunk ? s1 - c0 : kGenericChunk;
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) {
      const uint32_t d = tid + i * NT;
      if (d >= D) continue;
      float part = 0.f;
      for (uint32_t j = 0; j < cnt; ++j) {
        const float p = lds.pw[j];
        if (p != 0.f) part = fmaf(p, kv_value<kInt8>(a.v, lds.vbase[j] + d * P), part);
      }
      acc[i] = fmaf(acc[i], alpha, part);
    }
    __syncthreads();
  }
  const size_t out = (size_t(rh) * a.splits + split) * (size_t(D) + 2);
  if (tid == 0) {
    a.scratch[out] = m_run;
    a.scratch[out + 1] = l_run;
  }
#pragma unroll
  for (uint32_t i = 0; i < kPer; ++i) {
    const uint32_t d = tid + i * NT;
    if (d < D) a.scratch[out + 2 + d] = acc[i];
  }
}

}  // namespace kvb
