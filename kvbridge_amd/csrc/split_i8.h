// Integer-MFMA split-partial kernel for paged INT8 KV with few grouped
// head-rows per KV head (head_rows = rows * q_heads/kv_heads <= 8).
//
// The INT8 codes are never converted: both contractions run on
// v_mfma_i32_16x16x64_i8 with the raw K and V bytes as the A operand.
//  * QK: Q of each head-row is scaled by a power of two to a 23-bit integer
//    and split into three int8 digits (q = hi*2^16 + mid*2^8 + lo, exact).
//    The digits of all head-rows sit side by side in the 16 MFMA columns
//    (column = digit * HS + head), so one MFMA per 64 dims gives all three
//    digit dot products for 16 tokens.
//  * PV: the weights w * v_scale are scaled by 2^kp to integers below 2^21
//    and split into three 7-bit digits (p = d0*2^14 + d1*2^7 + d2); the
//    per-digit integer numerators accumulate exactly in int32.
// Digit recombination and the softmax run in a transposed view where each
// lane owns one token of the tile for every head-row (data moves through a
// small per-wave LDS exchange area), so no VALU work is spent on padding
// columns.
//
// Two passes per chunk of up to 4 tiles (NB = 1: one tile, for waves that
// hold one or two): the K images of the chunk are
// streamed first (scores kept in registers, exact chunk maximum), then the V
// images; the int32 numerators therefore never need an online rescale and
// are folded into fp32 once per chunk.
//
// Staging: K and V bytes go from HBM straight into VGPRs, already in the
// MFMA operand layout, with non-temporal 16-byte buffer loads (per-lane
// constant voffset; the descriptor is rebased per tile on its page, so
// every access is bounded by the page).  Each wave keeps a ring of NB item
// slots in registers and issues item j+NB-1 before computing item j; items
// run in fixed chunks (K images of 4 tiles, then their V images) so every
// ring slot is a compile-time register set and the issue is unconditional
// (an item past the wave's last tile gets a zero-sized descriptor and moves
// no data), which lets the compiler's wait-count pass keep exact
// per-register waits.  Eight waves per work-group (two per SIMD) where the
// state fits in 256 registers.
//
// Partial layout and semantics are those of every split kernel here:
// scratch[((row*q_heads + head)*splits + split)*(dim+2) + col], col 0 = split
// max score (natural log units), 1 = sum of exp(score - max), 2.. =
// sum of exp(score - max) * v_scale * v_code -- except in the single launch,
// which packs the same values differently in the same scratch
// (PackedPartials below).
#pragma once
#include <cstdint>

#include "kernels.h"
#include "batch.h"
#include "device_common.h"
#include "lds_stream.h"

namespace kvb {
namespace {

using lds::static_for;
using lds::u32x4_t;
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kTileTokens = 64;
constexpr float kLn2 = 0.6931471805599453f;
constexpr int32_t kRsrcWord3 = 0x00020000;   // raw 32-bit buffer, gfx9 dword3

// ---- loads.  Compiler builtins, so that its wait-count pass tracks every
// loaded register (in-order vmcnt; exact for this static schedule).
constexpr int kAuxNT = 2;  // non-temporal
__device__ __forceinline__ u32x4_t bload16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, int(voff), int(soff), kAuxNT);
}
__device__ __forceinline__ uint32_t bload4(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_amdgcn_raw_buffer_load_b32(r, int(voff), int(soff), kAuxNT);
}
__device__ __forceinline__ u32x4_t gload16(const int8_t* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
}
__device__ __forceinline__ uint32_t gload4(const float* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(p));
}

// One item in registers: the K image (d[mb * D/64 + j] = 16 bytes of K row
// 16*(m/4) + 4*mb + m%4, dims 64*j + 16*g ..; with PAIR the half-row layout
// below) plus k- and v-scale of token lane, or the V image (d[mb] = V row
// 16*mb + m, slots 16g .. 16g+15), which reuses its tile's scales.
template <int D>
struct Slot {
  u32x4_t d[D / 16];
  uint32_t ks, vs;
};

struct IssueCtx {
  __amdgpu_buffer_rsrc_t rk, rv, rks, rvs;  // whole-array descriptors (small-page path)
  uint32_t voff_k, voff_v, voff_s;          // per-lane constant offsets (page-tile path)
  const int8_t* k;
  const int8_t* v;
  const float* ks;
  const float* vs;
  const uint32_t* table;
  uint32_t kv, kv_heads, P, lg_p, pages, lp_lo, lp_hi, lane, ptab;
  uint32_t kv_bytes, sc_bytes;  // small-page path: whole-array sizes (< 4 GiB)
};

typedef const __attribute__((address_space(4))) uint32_t* const_u32_ptr;

// Physical page of logical page lp (uniform), clamped to the split's pages
// and to the pool; the first 64 come from the wave's page-table window.
__device__ __forceinline__ uint32_t page_of(const IssueCtx& c, uint32_t lp) {
  lp = clampu(lp, c.lp_lo, c.lp_hi);
  const uint32_t rel = lp - c.lp_lo;
  uint32_t x = rel < 64u ? uint32_t(__builtin_amdgcn_readlane(int(c.ptab), int(rel)))
                         : ((const_u32_ptr)(c.table))[lp];  // scalar load
  x = uint32_t(__builtin_amdgcn_readfirstlane(int(x)));
  return x < c.pages ? x : c.pages - 1u;
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, int(bytes), kRsrcWord3);
}

// Issue one item (D/16 + 2 loads for K, D/16 for V, unconditionally: an
// item past the wave's last tile gets zero-sized descriptors, so its loads
// return 0 and move no data).  PT: page_tokens is a power of two >= 64, the tile lies in one page
// and the descriptors are rebased on it (any pool size).  Otherwise
// page_tokens is 16 or 32: every 16-token group lies in one page and lanes
// address their group's page through whole-array descriptors.
// PAIR (K image of the paired-row QK layout): MFMA row m of M-block mb is
// half m%2 of token 8*mb + m/2, so the 16 lanes of a k-block read 8 rows x
// 2 segments of one 128-byte line each instead of 16 rows.
template <int D, bool PT, bool IS_V, bool PAIR>
__device__ __forceinline__ void issue_item(const IssueCtx& c, uint32_t tile, bool real, Slot<D>& s) {
  const uint32_t t0 = tile * kTileTokens;
  if constexpr (PT) {
    const uint64_t slab = page_of(c, t0 >> c.lg_p) * uint64_t(c.kv_heads) + c.kv;
    const uint32_t slot0 = t0 & (c.P - 1u);
    const uint64_t tok = slab * c.P + slot0;
    if constexpr (!IS_V && PAIR) {
      const __amdgpu_buffer_rsrc_t r = rsrc(c.k + tok * D, real ? 64u * D : 0u);
#pragma unroll
      for (uint32_t mb = 0; mb < 8; ++mb) s.d[mb] = bload16(r, c.voff_k + 1024u * mb, 0u);
    } else if constexpr (!IS_V) {
      const __amdgpu_buffer_rsrc_t r = rsrc(c.k + tok * D, real ? 64u * D : 0u);
      static_for<0, 4>([&](auto mbc) __attribute__((always_inline)) {
        constexpr uint32_t mb = decltype(mbc)::value;
        static_for<0, D / 64>([&](auto jc) __attribute__((always_inline)) {
          constexpr uint32_t j = decltype(jc)::value;
          s.d[mb * (D / 64) + j] = bload16(r, c.voff_k + (4 * mb * D + 64 * j), 0u);
        });
      });
    } else {
      const __amdgpu_buffer_rsrc_t r = rsrc(c.v + slab * D * c.P + slot0, real ? D * c.P - slot0 : 0u);
#pragma unroll
      for (uint32_t mb = 0; mb < D / 16; ++mb) s.d[mb] = bload16(r, c.voff_v, 16u * mb * c.P);
    }
    if constexpr (!IS_V) {  // the tile's V item reuses these
      s.ks = bload4(rsrc(c.ks + tok, real ? 256u : 0u), c.voff_s, 0u);
      s.vs = bload4(rsrc(c.vs + tok, real ? 256u : 0u), c.voff_s, 0u);
    }
  } else {
    const uint32_t lane = c.lane, m = lane & 15u, g = lane >> 4;
    uint32_t slab[4];  // slab of token group q (tokens t0+16q ..), uniform
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) slab[q] = page_of(c, (t0 + 16u * q) >> c.lg_p) * c.kv_heads + c.kv;
    auto pick = [&](uint32_t q) __attribute__((always_inline)) {
      return q == 0 ? slab[0] : (q == 1 ? slab[1] : (q == 2 ? slab[2] : slab[3]));
    };
    const __amdgpu_buffer_rsrc_t none = rsrc(c.k, 0u);
    if constexpr (!IS_V && PAIR) {
      const __amdgpu_buffer_rsrc_t r = real ? c.rk : none;
      static_for<0, 8>([&](auto mbc) __attribute__((always_inline)) {
        constexpr uint32_t mb = decltype(mbc)::value;
        constexpr uint32_t q = mb >> 1;  // 16-token group of tokens 8*mb ..
        const uint32_t row = pick(q) * c.P + ((t0 + 16u * q) & (c.P - 1u)) + 8u * (mb & 1u) + (m >> 1);
        s.d[mb] = bload16(r, row * uint32_t(D) + 64u * (m & 1u) + 16u * g, 0u);
      });
    } else if constexpr (!IS_V) {
      const uint32_t grp = m >> 2;
      const uint32_t row = pick(grp) * c.P + ((t0 + 16u * grp) & (c.P - 1u)) + (m & 3u);
      const uint32_t voff = row * uint32_t(D) + 16u * g;
      const __amdgpu_buffer_rsrc_t r = real ? c.rk : none;
      static_for<0, 4>([&](auto mbc) __attribute__((always_inline)) {
        constexpr uint32_t mb = decltype(mbc)::value;
        static_for<0, D / 64>([&](auto jc) __attribute__((always_inline)) {
          constexpr uint32_t j = decltype(jc)::value;
          s.d[mb * (D / 64) + j] = bload16(r, voff + (4 * mb * D + 64 * j), 0u);
        });
      });
    } else {
      const uint32_t voff = (pick(g) * uint32_t(D) + m) * c.P + ((t0 + 16u * g) & (c.P - 1u));
      const __amdgpu_buffer_rsrc_t r = real ? c.rv : none;
#pragma unroll
      for (uint32_t mb = 0; mb < D / 16; ++mb) s.d[mb] = bload16(r, voff, 16u * mb * c.P);
    }
    if constexpr (!IS_V) {  // the tile's V item reuses these
      const uint32_t si = (pick(g) * c.P + ((t0 + 16u * g) & (c.P - 1u)) + m) * 4u;
      s.ks = bload4(real ? c.rks : none, si, 0u);
      s.vs = bload4(real ? c.rvs : none, si, 0u);
    }
  }
}

template <int D, int NW, int HS>
struct I8Layout {
  static constexpr int NC = (3 * HS + 15) / 16;       // MFMA column tiles
  static constexpr uint32_t kExchCol = 272;           // int32 column of 64 tokens + pad
  static constexpr uint32_t kDigCol = 80;             // int8 column of 64 tokens + pad
  static constexpr uint32_t kExch = NC * 16 * kExchCol;
  static constexpr uint32_t kDig = NC * 16 * kDigCol;
  static constexpr uint32_t kWave = kExch + kDig;
  // Wave combine area after the exchange areas: [NW][HS] maxima, [NW][HS]
  // denominators, [NW][HS][D] numerators.
  static constexpr uint32_t kComb = NW * kWave;
  // Q digit area after it: [64 lanes][kQdBytes] (written before the main
  // loop, read by every wave; waves with no tiles reach the combine early,
  // so it must not overlap the combine area).
  static constexpr bool kPair = D == 128 && HS <= 4;  // paired-row QK layout
  static constexpr uint32_t kQdBytes = (kPair ? 2 : NC) * (kPair ? 1 : D / 64) * 16;
  static constexpr uint32_t kQd = kComb + NW * HS * (D + 2) * 4;
  static constexpr uint32_t kBytes = kQd + 64 * kQdBytes;
};

// Agent-scope (all XCDs) coherent load of a partial written by another
// work-group with an agent-scope atomic store.
__device__ __forceinline__ float ld_agent(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The single launch's merge (at most 32 splits, one output column per
// thread) reads a packed partial layout of its own instead of the
// [row-head][split][m, l, n] rows above (same size, internal to the call):
//   m: scratch[rh*splits + j]             (RS = rows * q_heads * splits)
//   l: scratch[RS + rh*splits + j]
//   n: scratch[2*RS + (rh*splits + j)*D + d]
// so the merger's (m_j, l_j) of one row-head are one 128-byte line each
// instead of a line per split, and every 256-byte numerator request of a
// wave covers two whole 128-byte lines (numerator rows start 512-byte apart,
// at a 128-byte boundary when the scratch base has one) instead of three.
// The merge is bound by those line requests: agent-scope loads miss the
// L2, and one work-group issues all of them.
template <int D>
struct PackedPartials {
  const size_t rs;
  float* base;
  __device__ __forceinline__ PackedPartials(float* scratch, const SplitArgs& a)
      : rs(size_t(a.rows) * a.q_heads * a.splits), base(scratch) {}
  __device__ __forceinline__ float* m(size_t rh, uint32_t splits, uint32_t j) const { return base + rh * splits + j; }
  __device__ __forceinline__ float* l(size_t rh, uint32_t splits, uint32_t j) const { return base + rs + rh * splits + j; }
  __device__ __forceinline__ float* n(size_t rh, uint32_t splits, uint32_t j) const {
    return base + 2 * rs + (rh * splits + j) * D;
  }
};

// Merge of all splits of one kv head's head-rows, by the last work-group,
// with the reference merge semantics (src/attention_shared.cu:295-335):
// M = max_j m_j; L = sum_{l_j > 0} e^{m_j - M} l_j; N[d] likewise (N in four
// interleaved sums, L by a wave tree); an all-empty head-row gives M = -inf,
// L = 0, N = 0.  Optional normalized output out = L > 0 ? N / L : 0 (fp32 or
// fp16).  Splits 0 .. ns-1 are merged; a.splits is the partial stride.
// i8_fusable admits at most 32 splits, one output per thread and one head-row
// per wave: straight-line code that requests every operand at once -- the
// wave's (m_j, l_j) and the thread's 32 numerators, split indices clamped
// instead of branched on -- so the merge costs one memory round trip.  The 64
// outputs of a wave lie in one head-row (64 divides D), so every wave turns
// its own head-row's (m_j, l_j) into the factors e^{m_j - M} (lane j holds
// split j), without a work-group barrier.  f_s: LDS [NW][32] split factors.
template <int D, int NW>
__device__ __forceinline__ void fused_merge(const SplitArgs& a, uint32_t kv, uint32_t head_rows, uint32_t ns,
                                            const float* __restrict__ scratch, float* f_s) {
  constexpr uint32_t kCh = 32;  // splits
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t outs = head_rows * D;
  auto row_head = [&](uint32_t hh) __attribute__((always_inline)) {
    return size_t(hh / a.group) * a.q_heads + kv * a.group + hh % a.group;
  };
  static_assert(D % 64 == 0, "a wave's outputs lie in one head-row");
  static_assert(kCh == 32, "the short merge covers 32 splits");
  if (64u * wave >= outs) return;
  const uint32_t jmax = ns - 1u;
  const uint32_t hh = (64u * wave) / D;
  const PackedPartials<D> pp(const_cast<float*>(scratch), a);
  const size_t rhh = row_head(hh);
  const uint32_t jl = lane < ns ? lane : jmax;
  const float mj = ld_agent(pp.m(rhh, a.splits, jl));
  const float lj = ld_agent(pp.l(rhh, a.splits, jl));
  const uint32_t d = tid % D;
  // Numerator j of column d through one descriptor over the head-row's
  // numerator rows, with the row offset in the instruction's scalar offset
  // (no per-load vector address arithmetic); agent-coherent cache policy.
  // Rows past ns - 1 re-read row ns - 1 and are masked below.
  const float* nb = pp.n(rhh, a.splits, 0) + d;
  float pre[kCh];
#pragma unroll
  for (uint32_t j = 0; j < kCh; ++j) pre[j] = ld_agent(nb + size_t(j < jmax ? j : jmax) * D);
  const bool in = lane < ns;
  const float mx = wave_max(in ? mj : neg_inf());
  const float f = in && lj > 0.f ? exp_e(mj - mx) : 0.f;
  const float lsum = wave_sum(f * lj);
  // The factors reach every lane as LDS broadcasts (this wave's own 32
  // floats of f_s), and the 32 products go into four interleaved sums
  // added as (s0 + s1) + (s2 + s3): a fixed order, four times shorter
  // dependency chains.
  float* const fw = f_s + wave * kCh;
  if (lane < kCh) fw[lane] = f;
  float fv[kCh];
#pragma unroll
  for (uint32_t q4 = 0; q4 < kCh / 4u; ++q4) {
    const float4 x = reinterpret_cast<const float4*>(fw)[q4];
    fv[4 * q4] = x.x;
    fv[4 * q4 + 1] = x.y;
    fv[4 * q4 + 2] = x.z;
    fv[4 * q4 + 3] = x.w;
  }
  float s4[4] = {0.f, 0.f, 0.f, 0.f};
  if (ns == kCh) {
#pragma unroll
    for (uint32_t j = 0; j < kCh; ++j) s4[j & 3u] = fmaf(fv[j], pre[j], s4[j & 3u]);
  } else {
#pragma unroll
    for (uint32_t j = 0; j < kCh; ++j) s4[j & 3u] = fmaf(fv[j], j <= jmax ? pre[j] : 0.f, s4[j & 3u]);
  }
  const float nacc = (s4[0] + s4[1]) + (s4[2] + s4[3]);
  const size_t rh = row_head(hh);
  if (d == 0) {
    a.m[rh] = mx;
    a.l[rh] = lsum;
  }
  a.n[rh * D + d] = nacc;
  if (a.out_type != 0) {
    const float ov = lsum > 0.f ? nacc / lsum : 0.f;
    if (a.out_type == 1) static_cast<float*>(a.out)[rh * D + d] = ov;
    else static_cast<_Float16*>(a.out)[rh * D + d] = (_Float16)ov;
  }
}

// VARLEN: batched call, grid (kv heads, splits, sequences) in the order of
// batch_item (arguments rebased per work-group).
// The leading scalar arguments are everything the first KV request depends
// on; the translation units that instantiate this kernel are built with
// kernel-argument preloading for them (the dispatcher places them in SGPRs),
// so the page-table load is issued without waiting for a kernel-argument
// load.  They duplicate fields of a_in, which the kernel overrides with them.
//
// FENCE (one diagnostic instance, kvb_decode_attention_fused_fenced): the
// single launch with the formal agent-scope release fence before every
// ticket and an acquire fence after the merger's -- the ordering the other
// instances get from agent-scope atomic partials, without the L2 write-back
// and invalidate these fences add.
template <int D, int NW, int NB, bool PT, int HS, bool FUSED, bool VARLEN, bool FENCE>
__global__ __launch_bounds__(64 * NW) void split_i8_kernel(
    const uint32_t* __restrict__ table_in, const int8_t* __restrict__ kdata, const float* __restrict__ kscale,
    const float* __restrict__ vscale, uint32_t p_begin, uint32_t p_end, uint32_t p_split_tokens,
    uint32_t p_page_tokens, uint32_t p_kv_heads, uint32_t p_pages, SplitArgs a_in,
    const float* __restrict__ q_in, const int64_t* __restrict__ qpos_in, const int64_t* __restrict__ kpos_in,
    const int8_t* __restrict__ vdata, float* __restrict__ scratch_in) {
#include "split_i8_body.h"
}

#define KVB_I8_ARGS                                                                                        \
  a.page_table, static_cast<const int8_t*>(a.k), a.k_scales, a.v_scales, a.begin, a.end, a.split_tokens,     \
      a.page_tokens, a.kv_heads, a.pages, a, a.q, a.q_positions, a.k_positions, static_cast<const int8_t*>(a.v), \
      a.scratch

// Single-launch instances exist where i8_fusable can choose them.
template <int NW, int HS>
constexpr bool kFusedInstance = NW >= 4 && HS <= 4;

template <int D, int NW, int NB, int HS>
hipError_t launch_cfg(const SplitArgs& a, hipStream_t stream) {
  const bool pt = a.page_tokens >= kTileTokens, fused = a.counters != nullptr, varlen = a.seq_starts != nullptr;
  const dim3 grid = varlen ? dim3(a.kv_heads, a.splits, a.batch) : dim3(a.splits, a.kv_heads, 1u);  // batch_item
  const dim3 block(64 * NW);
  if (varlen && !pt) return hipErrorInvalidValue;  // batched calls need whole-tile pages (i8_supported)
  if (fused) {
    if constexpr (kFusedInstance<NW, HS>) {
      if (varlen)
        hipLaunchKernelGGL((split_i8_kernel<D, NW, NB, true, HS, true, true, false>), grid, block, 0, stream, KVB_I8_ARGS);
      else if (pt)
        hipLaunchKernelGGL((split_i8_kernel<D, NW, NB, true, HS, true, false, false>), grid, block, 0, stream, KVB_I8_ARGS);
      else
        hipLaunchKernelGGL((split_i8_kernel<D, NW, NB, false, HS, true, false, false>), grid, block, 0, stream, KVB_I8_ARGS);
      return hipGetLastError();
    } else {
      return hipErrorInvalidValue;
    }
  }
  if (varlen)
    hipLaunchKernelGGL((split_i8_kernel<D, NW, NB, true, HS, false, true, false>), grid, block, 0, stream, KVB_I8_ARGS);
  else if (pt)
    hipLaunchKernelGGL((split_i8_kernel<D, NW, NB, true, HS, false, false, false>), grid, block, 0, stream, KVB_I8_ARGS);
  else
    hipLaunchKernelGGL((split_i8_kernel<D, NW, NB, false, HS, false, false, false>), grid, block, 0, stream, KVB_I8_ARGS);
  return hipGetLastError();
}

inline hipError_t preload_fns(const void* const* fns, int count) {
  hipFuncAttributes attr{};
  for (int i = 0; i < count; ++i) {
    const hipError_t e = hipFuncGetAttributes(&attr, fns[i]);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

template <int D, int NW, int NB, int HS>
hipError_t preload_cfg() {
  const void* fns[] = {reinterpret_cast<const void*>(&split_i8_kernel<D, NW, NB, true, HS, false, false, false>),
                       reinterpret_cast<const void*>(&split_i8_kernel<D, NW, NB, false, HS, false, false, false>),
                       reinterpret_cast<const void*>(&split_i8_kernel<D, NW, NB, true, HS, false, true, false>)};
  hipError_t e = preload_fns(fns, 3);
  if constexpr (kFusedInstance<NW, HS>) {
    const void* one[] = {reinterpret_cast<const void*>(&split_i8_kernel<D, NW, NB, true, HS, true, false, false>),
                         reinterpret_cast<const void*>(&split_i8_kernel<D, NW, NB, false, HS, true, false, false>),
                         reinterpret_cast<const void*>(&split_i8_kernel<D, NW, NB, true, HS, true, true, false>)};
    if (e == hipSuccess) e = preload_fns(one, 3);
  }
  return e;
}

// Launch / preload of every (waves, ring) configuration of one dim; cfg =
// 10 * waves + ring slots (82 and 81 only for head_rows <= 4 and dim <= 128).
template <int D>
hipError_t launch_dim(const SplitArgs& a, int cfg, hipStream_t stream) {
  if (a.rows * a.group <= 4) {
    if constexpr (D <= 128) {
      if (cfg == 82) return launch_cfg<D, 8, 2, 4>(a, stream);
      if (cfg == 81) return launch_cfg<D, 8, 1, 4>(a, stream);
    }
    if (cfg == 41) return launch_cfg<D, 4, 1, 4>(a, stream);
    if (cfg == 12) return launch_cfg<D, 1, 2, 4>(a, stream);
    return cfg == 42 ? launch_cfg<D, 4, 2, 4>(a, stream) : launch_cfg<D, 2, 2, 4>(a, stream);
  }
  if constexpr (D <= 128) {
    if (cfg == 12) return launch_cfg<D, 1, 2, 8>(a, stream);
    return cfg == 42 ? launch_cfg<D, 4, 2, 8>(a, stream) : launch_cfg<D, 2, 2, 8>(a, stream);
  }
  return hipErrorInvalidValue;
}

template <int D>
hipError_t preload_dim() {
  hipError_t e = hipSuccess;
  if constexpr (D <= 128) {
    e = preload_cfg<D, 8, 2, 4>();
    if (e == hipSuccess) e = preload_cfg<D, 8, 1, 4>();
    if (e == hipSuccess) e = preload_cfg<D, 4, 2, 8>();
    if (e == hipSuccess) e = preload_cfg<D, 2, 2, 8>();
    if (e == hipSuccess) e = preload_cfg<D, 1, 2, 8>();
  }
  if (e == hipSuccess) e = preload_cfg<D, 4, 1, 4>();
  if (e == hipSuccess) e = preload_cfg<D, 4, 2, 4>();
  if (e == hipSuccess) e = preload_cfg<D, 2, 2, 4>();
  if (e == hipSuccess) e = preload_cfg<D, 1, 2, 4>();
  return e;
}

}  // namespace
}  // namespace kvb
