// MFMA split-partial kernels of the generic family: int8 or fp32 KV, any dim
// that is a multiple of 4, any page size that is a multiple of 16 tokens, any
// number of head-rows, one sequence or a ragged batch.
//
// One work-group of NW waves per (split, kv head, block of 16 head-rows[,
// sequence]): every wave streams its tiles (round-robin over the waves)
// straight into registers in MFMA operand layout and runs the whole online
// softmax for all 16 head-rows of the block, so the KV is read once for a
// block instead of once per head-row.  The score tile leaves the QK MFMA with
// lane (n, g) = head-row n and the tokens 4g .. of its 16-row block, which is
// the lane that feeds those tokens' weights to PV: nothing moves between
// lanes except the row maximum.  The waves' states meet in LDS at the end.
//
// fp32 accuracy throughout, as the scalar kernel:
//  * int8 KV (64-token tiles): the codes are converted to bf16 (exact, 8
//    bits), Q and the weights are cut into three bf16 pieces (8 bits each:
//    the 24 bits of an fp32 exactly), and v_mfma_f32_16x16x32_bf16 sums the
//    exact products in fp32.  The maximum carries every rounding of its score
//    into m and l, so a score takes as few as it can: Q comes times the score
//    scale, the sums of the high pieces are kept from the low ones' bits, and
//    one fma applies the k-scale.  Error of m against 64 bits, relative, dim
//    256 / 128 / 64: 9.5e-8 / 6.5e-8 / 5.8e-8 with one sum and log2 units,
//    5.2e-8 / 4.4e-8 / 3.9e-8 so; l 3.9e-7 / 2.5e-7 / 2.1e-7 -> 2.2e-7 /
//    1.8e-7 / 1.4e-7.
//  * fp32 KV (16-token tiles): v_mfma_f32_16x16x4_f32.
//
// What bounds it: below two work-groups per CU, latency -- the page table, Q
// and positions in one round trip, the first tile in a second, and ~2,500
// VALU cycles of conversion and softmax per 64-token int8 tile; a second tile
// in registers (ring of two) gained nothing (head size 96, 8,000 tokens: 16.9
// us per call with it, 15.9 without).  Measured per call against one scalar
// work-group per head-row (32 q / 8 kv heads): dim 96, 8,000 tokens 132 ->
// 13.2 us; fp32 KV, dim 128, 8,192 tokens 150 -> 25.6 us (16-token tiles on
// 128 work-groups, 26 GB/s per CU); 32 sequences of 100 .. 4,000 tokens over
// 16-token pages, dim 128, 915 -> 42.0 us.  Error of n against 64 bits, relative:
// 2.3e-7 / 4.4e-7 / 2.0e-7, scalar 4.0e-7 / 8.3e-7 / 3.9e-7.
//
// Non-finite values: a masked token's K, V and scales never reach the
// arithmetic; a split whose result is not finite (infinities or NaN in the
// cache, Q or the scales, or an overflow) is computed again by
// split_generic_row, whose rule (a zero weight leaves its V row out) a matrix
// product cannot follow.
#pragma once
#include <cstdio>
#include <cstdint>

#include "kernels.h"
#include "batch.h"
#include "device_common.h"
#include "split_generic.h"

namespace kvb {
namespace {

typedef uint32_t u32x4_g __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kGenericNT = 2;  // non-temporal
__device__ __forceinline__ __amdgpu_buffer_rsrc_t g_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, int(bytes), 0x00020000);
}
// The whole offset sits in the vector offset, so that the descriptor's bound
// is checked against it.
__device__ __forceinline__ u32x4_g g_load16(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, int(off), 0, kGenericNT);
}
// Smallest dim that a padded size serves: blocks below it need no check.
template <int DP>
constexpr uint32_t kDimFloor = DP == 64 ? 4u : DP / 2u + 4u;

// Four signed codes of one dword as floats, exact.
__device__ __forceinline__ f32x4 codes_f32(uint32_t w) {
  return f32x4{float(int8_t(w)), float(int8_t(w >> 8)), float(int8_t(w >> 16)), float(int32_t(w) >> 24)};
}
// The upper halves (bf16, truncated) of two floats in one dword.
__device__ __forceinline__ uint32_t hi_pair(float lo, float hi) {
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}
// Eight signed codes (two dwords) -> eight exactly equal bf16 values.
__device__ __forceinline__ bf16x8 codes_bf16(uint32_t w0, uint32_t w1) {
  const f32x4 a = codes_f32(w0), b = codes_f32(w1);
  const u32x4_g r = {hi_pair(a[0], a[1]), hi_pair(a[2], a[3]), hi_pair(b[0], b[1]), hi_pair(b[2], b[3])};
  return __builtin_bit_cast(bf16x8, r);
}
// Eight floats as three bf16 vectors whose sum is exactly the floats (8 + 8 +
// 8 significant bits, each piece the truncated rest; exact while the rest is
// a normal number).
__device__ __forceinline__ void cut3(const float (&x)[8], bf16x8 (&piece)[3]) {
  float r[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = x[i];
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    const u32x4_g w = {hi_pair(r[0], r[1]), hi_pair(r[2], r[3]), hi_pair(r[4], r[5]), hi_pair(r[6], r[7])};
    piece[p] = __builtin_bit_cast(bf16x8, w);
    if (p < 2) {
#pragma unroll
      for (int i = 0; i < 8; ++i) r[i] -= __uint_as_float(__float_as_uint(r[i]) & 0xffff0000u);
    }
  }
}

// Rows of the wave's coming tiles.  Lane l holds 16-token group l % GT of the
// wave's tile i0 + l / GT (GT groups per tile): the index of its first row in
// [page][kv head][slot] order, its slot in the page, and the element index of
// its first V column.  Groups outside the split's tokens are clamped to one
// inside, so every address is one the split may read.  The page id is
// requested a window ahead (PageWindow) and only turned into rows when the
// window starts, so nothing waits for it in between.
struct PageWindow {
  uint32_t page, slot;
};
struct RowWindow {
  uint32_t row, vcol, slot;
};

struct SplitRange {
  uint32_t s0, s1;       // the split's tokens
  uint32_t first, step;  // the wave's tile i starts at token (first + i * step) * tile
};

template <uint32_t TILE>
__device__ __forceinline__ PageWindow load_window(const SplitArgs& a, const SplitRange& s, uint32_t i0,
                                                  uint32_t lane) {
  constexpr uint32_t GT = TILE / 16u;
  // 64-bit: a group past the end may lie past 2^32 tokens.
  const uint64_t t64 = uint64_t(s.first + uint64_t(i0 + lane / GT) * s.step) * TILE + 16u * (lane % GT);
  const uint32_t lo = s.s0 & ~15u, hi = (s.s1 - 1u) & ~15u;
  const uint32_t t = t64 < lo ? lo : (t64 > hi ? hi : uint32_t(t64));
  const uint32_t lp = t / a.page_tokens, slot = t - lp * a.page_tokens;
  return PageWindow{a.page_table[lp], slot};
}

__device__ __forceinline__ RowWindow window_rows(const SplitArgs& a, const PageWindow& w, uint32_t kv) {
  const uint32_t page = w.page < a.pages ? w.page : a.pages - 1u;
  const uint32_t slab = page * a.kv_heads + kv;
  return RowWindow{slab * a.page_tokens + w.slot, slab * a.dim * a.page_tokens + w.slot, w.slot};
}

__device__ __forceinline__ uint32_t lane_pick(uint32_t x, uint32_t from) {
  return uint32_t(__builtin_amdgcn_ds_bpermute(int(4u * from), int(x)));
}

// Row of the lane's head-row (lanes past the last one repeat it).
__device__ __forceinline__ uint32_t block_row(const SplitArgs& a, uint32_t hb, uint32_t lane) {
  const uint32_t hr = a.rows * a.group, mine = 16u * hb + (lane & 15u);
  return (mine < hr ? mine : hr - 1u) / a.group;
}

// The block's head-rows as the lane (n, g) sees them: head-row hb * 16 + n.
struct HeadLane {
  uint32_t hr;            // head-rows of the kv head
  uint32_t end;           // this lane's visible tokens end here
  uint32_t e_min, e_max;  // over the block's head-rows
};

// The last key position and the lane's query position (requested together by
// the caller, before anything waits) decide the common case; a row that does
// not see the whole split searches its end.
__device__ __forceinline__ HeadLane head_lane(const SplitArgs& a, const SplitRange& s, uint32_t hb, uint32_t lane,
                                              int64_t klast, int64_t qp) {
  HeadLane h;
  h.hr = a.rows * a.group;
  h.end = s.s1;
  h.e_min = s.s1;
  h.e_max = s.s1;
  if (__all(klast <= qp)) return h;
  const uint32_t last = 16u * hb + 15u < h.hr - 1u ? 16u * hb + 15u : h.hr - 1u;
  const uint32_t row = block_row(a, hb, lane);
  h.e_min = 0xffffffffu;
  h.e_max = s.s0;
  for (uint32_t r = 16u * hb / a.group; r <= last / a.group; ++r) {
    const int64_t qr = a.q_positions[r];
    const uint32_t e =
        __builtin_amdgcn_readfirstlane(klast <= qr ? s.s1 : visible_end(a.k_positions, s.s0, s.s1, qr, lane));
    h.end = row == r ? e : h.end;
    h.e_min = e < h.e_min ? e : h.e_min;
    h.e_max = e > h.e_max ? e : h.e_max;
  }
  return h;
}

// Combine area of the waves, and the scalar path's area after it is done.
template <int DP, int NW>
union GenericSmem {
  u32x4_g q[DP / 64][2][3][64];  // int8: Q pieces of every lane
  struct {
    float m[NW][16], l[NW][16], f[NW][16];
    float acc[NW][16][DP + 4];  // padded rows: 16 head-rows of one column spread over the banks
  } c;
  GenericLds<64 * NW> scalar;
};

// Combines the waves (the visible part of a short split: dim 128, 16
// head-rows, 3.2 of the split kernel's 12.7 us while every thread computed the
// factors and took one column per step; a quad per thread took 2 us off; l
// summed over the lanes of a head-row already) and writes the block's partials; a block with a non-finite result
// goes through the scalar rows instead.
template <int DP, int NW, bool kInt8>
__device__ __forceinline__ void write_partials(const SplitArgs& a, const HeadLane& h, uint32_t kv, uint32_t hb,
                                               uint32_t split, float m, float l, const f32x4 (&acc)[DP / 16],
                                               GenericSmem<DP, NW>& sm) {
  const uint32_t tid = threadIdx.x, lane = tid & 63u, n = lane & 15u, g = lane >> 4;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t rows_here = h.hr - 16u * hb < 16u ? h.hr - 16u * hb : 16u;
  __syncthreads();  // the main loop's area is free
  float z = l * 0.f;  // 0 while everything is finite, else NaN
  if (n < rows_here) {
    if (g == 0) {
      sm.c.m[wave][n] = m;
      sm.c.l[wave][n] = l;
    }
#pragma unroll
    for (int mb = 0; mb < DP / 16; ++mb) {
      *reinterpret_cast<f32x4*>(&sm.c.acc[wave][n][16 * mb + 4 * g]) = acc[mb];
      if (16u * mb + 4u * g < a.dim) {  // dim is a multiple of 4; rows past it hold anything
#pragma unroll
        for (int e = 0; e < 4; ++e) z = fmaf(acc[mb][e], 0.f, z);
      }
    }
  }
  if (__syncthreads_or(n < rows_here && z != 0.f)) {
    for (uint32_t r = 0; r < rows_here; ++r) {
      const uint32_t hh = 16u * hb + r;
      split_generic_row<kInt8, 64 * NW>(a, (hh / a.group) * a.q_heads + kv * a.group + hh % a.group, split, sm.scalar);
    }
    return;
  }
  // Factors of the waves, one (wave, head-row) per lane of wave 0, then a
  // quad of columns per thread: independent 16-byte LDS loads and one store.
  if (tid < 16u * NW) {
    const uint32_t r = tid & 15u, w = tid >> 4;
    if (r < rows_here) {
      float mm = sm.c.m[0][r];
#pragma unroll
      for (int i = 1; i < NW; ++i) mm = fmaxf(mm, sm.c.m[i][r]);
      const float mw = sm.c.m[w][r];
      sm.c.f[w][r] = mw == neg_inf() ? 0.f : exp_e(mw - mm);
    }
  }
  __syncthreads();
  constexpr uint32_t QT = DP / 4;  // threads per head-row
  const uint32_t q = tid % QT;
  for (uint32_t r = tid / QT; r < rows_here; r += 64u * NW / QT) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    float ls = 0.f, mm = neg_inf();
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = sm.c.f[w][r];
      const f32x4 x = *reinterpret_cast<const f32x4*>(&sm.c.acc[w][r][4u * q]);
      ls = fmaf(f, sm.c.l[w][r], ls);
      mm = fmaxf(mm, sm.c.m[w][r]);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = fmaf(f, x[e], v[e]);
    }
    const uint32_t hh = 16u * hb + r;
    const size_t rh = size_t(hh / a.group) * a.q_heads + kv * a.group + hh % a.group;
    float* const dst = a.scratch + (rh * a.splits + split) * (size_t(a.dim) + 2);
    if (4u * q < a.dim) {  // dim is a multiple of 4; partial rows are only 4-byte aligned
      typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));
      *reinterpret_cast<f32x4_u*>(dst + 2u + 4u * q) = v;
    }
    if (q == 0u) {
      dst[0] = mm;
      dst[1] = ls;
    }
  }
}

// The partials of a split without tokens (past the end of a batched call's
// shorter sequences): m = -inf, l = 0, n = 0.
template <int NW>
__device__ __forceinline__ void write_empty(const SplitArgs& a, uint32_t kv, uint32_t hb, uint32_t split) {
  const uint32_t hr = a.rows * a.group, w = a.dim + 2u;
  for (uint32_t hh = 16u * hb; hh < hr && hh < 16u * hb + 16u; ++hh) {
    const size_t rh = size_t(hh / a.group) * a.q_heads + kv * a.group + hh % a.group;
    float* const dst = a.scratch + (rh * a.splits + split) * size_t(w);
    for (uint32_t c = threadIdx.x; c < w; c += 64u * NW) dst[c] = c == 0u ? neg_inf() : 0.f;
  }
}

// Online-softmax state of lane (n, g): head-row n, its own tokens' share of l.
template <int DP>
struct OnlineState {
  float m = neg_inf(), l = 0.f;
  f32x4 acc[DP / 16];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int mb = 0; mb < DP / 16; ++mb) acc[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // y: the lane's scores -> its weights.  Scores and maxima are in natural
  // units: in log2 units the rounding of the constant would reach every weight.
  template <int N>
  __device__ __forceinline__ void weights(float (&y)[N]) {
    float t = y[0];
#pragma unroll
    for (int i = 1; i < N; ++i) t = fmaxf(t, y[i]);
    const float m_new = fmaxf(m, rows_max(t));
    const float mu = m_new == neg_inf() ? 0.f : m_new;
    if (__any(m_new > m)) {  // else every factor is 1
      const float f = m == neg_inf() ? 0.f : __builtin_amdgcn_exp2f((m - mu) * kLog2e);
      l *= f;
#pragma unroll
      for (int mb = 0; mb < DP / 16; ++mb) acc[mb] *= f;
      m = m_new;
    }
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      y[i] = __builtin_amdgcn_exp2f((y[i] - mu) * kLog2e);
      s += y[i];
    }
    l += s;
  }
};

template <int NW>
__device__ __forceinline__ SplitRange split_range(const SplitArgs& a, uint32_t split, uint32_t tile) {
  SplitRange s;
  const uint64_t s0_64 = uint64_t(a.begin) + uint64_t(split) * a.split_tokens;
  s.s0 = s0_64 < a.end ? uint32_t(s0_64) : a.end;
  s.s1 = uint64_t(s.s0) + a.split_tokens < a.end ? s.s0 + a.split_tokens : a.end;
  s.first = s.s0 / tile + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  s.step = NW;
  return s;
}

// The wave's tiles that hold a visible token.
template <uint32_t TILE>
__device__ __forceinline__ uint32_t wave_tiles(const SplitRange& s, uint32_t e_max) {
  if (e_max <= s.s0) return 0u;
  const uint32_t last = (e_max - 1u) / TILE;
  return last < s.first ? 0u : (last - s.first) / s.step + 1u;
}

// Grid: x = kv head + kv_heads * head-row block, y = split, z = sequence (see
// batch_item).
//
// int8 KV.  MFMA row m of QK M-block mb is token 16 (m / 4) + 4 mb + m % 4 of
// the 64-token tile, so lane (n, g) ends up with the scores of tokens 16g ..
// 16g + 15 (register 4 mb + e = token 16g + 4 mb + e), which are the bytes
// of the V rows that lane (m, g) loads: 16 slots of one page from one
// 16-byte load.  K bytes past dim (a padded 64-dim step) meet zeros of Q; V
// rows past dim give accumulators that are never stored.
template <int DP, int NW, bool VARLEN>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(DP <= 128 ? 2 : 1)))
void split_generic_i8_kernel(SplitArgs a) {
  uint32_t split = blockIdx.y;
  if constexpr (VARLEN) {
    const BatchItem item = batch_item(a);
    split = item.split;
    rebase_sequence(a, item.seq, item.e);
  }
  __shared__ __attribute__((aligned(16))) GenericSmem<DP, NW> sm;
  constexpr uint32_t TILE = 64;
  constexpr int KS = DP / 64;   // 64-dim steps
  constexpr int MB = DP / 16;   // V row blocks
  const uint32_t lane = threadIdx.x & 63u, n = lane & 15u, g = lane >> 4;
  const uint32_t kv = blockIdx.x % a.kv_heads, hb = blockIdx.x / a.kv_heads;
  const SplitRange s = split_range<NW>(a, split, TILE);
  if (s.s1 <= s.s0) return write_empty<NW>(a, kv, hb, split);
  OnlineState<DP> st;
  st.clear();

  RowWindow win{0u, 0u, 0u};
  PageWindow next_win = load_window<TILE>(a, s, 0u, lane);
  const int64_t klast = a.k_positions[s.s1 - 1u], qpos = a.q_positions[block_row(a, hb, lane)];
  // Q of this lane's head-row times the score scale (rounded once per element,
  // which averages out, instead of once per score): dims 64 s + 16 g .. + 15 of
  // step s, as bf16 pieces.
  const uint32_t hr = a.rows * a.group, mine = 16u * hb + n;
  const bool real_head = mine < hr;
  float qv[KS][16];
  {
    const uint32_t hh = real_head ? mine : 0u;
    const float* const src = a.q + (size_t(hh / a.group) * a.q_heads + kv * a.group + hh % a.group) * a.dim;
#pragma unroll
    for (int k = 0; k < KS; ++k)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t d = 64u * k + 16u * g + 4u * j;
        const bool in = real_head && d < a.dim;  // dim is a multiple of 4
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float x = src[(in ? d : 0u) + i];
          qv[k][4 * j + i] = in ? x * a.scale : 0.f;
        }
      }
  }
  const HeadLane h = head_lane(a, s, hb, lane, klast, qpos);
  const uint32_t nt = wave_tiles<TILE>(s, h.e_max);

  const uint32_t rows_all = a.pages * a.kv_heads * a.page_tokens;
  const __amdgpu_buffer_rsrc_t rk = g_rsrc(a.k, rows_all * a.dim), rv = g_rsrc(a.v, rows_all * a.dim);
  const __amdgpu_buffer_rsrc_t rks = g_rsrc(a.k_scales, rows_all * 4u), rvs = g_rsrc(a.v_scales, rows_all * 4u);
  const __amdgpu_buffer_rsrc_t none = g_rsrc(a.k, 0u);
  // A step or row block past dim loads nothing.
  auto step = [&](__amdgpu_buffer_rsrc_t r, uint32_t d) __attribute__((always_inline)) {
    return d < kDimFloor<DP> || d < a.dim ? r : none;
  };
  struct Slot {
    u32x4_g k[KS * 4], v[MB];
    uint32_t ks, vs;
  };
  Slot it;
  auto window = [&](uint32_t i) __attribute__((always_inline)) {
    if ((i & 15u) == 0u) {  // the coming 16 tiles; the ones after them are requested here
      win = window_rows(a, next_win, kv);
      if (i + 16u < nt) next_win = load_window<TILE>(a, s, i + 16u, lane);
    }
  };
  auto issue_k = [&](uint32_t i, Slot& t) __attribute__((always_inline)) {
    const bool real = i < nt;
    const uint32_t at = 4u * (i & 15u);
    const uint32_t voff = (lane_pick(win.row, at + (n >> 2)) + (n & 3u)) * a.dim + 16u * g;
    const __amdgpu_buffer_rsrc_t r = real ? rk : none;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int k = 0; k < KS; ++k) t.k[mb * KS + k] = g_load16(step(r, 64u * k), voff + 4u * mb * a.dim + 64u * k);
    const uint32_t soff = (lane_pick(win.row, at + g) + n) * 4u;  // lane = token
    t.ks = __builtin_amdgcn_raw_buffer_load_b32(real ? rks : none, int(soff), 0, kGenericNT);
    t.vs = __builtin_amdgcn_raw_buffer_load_b32(real ? rvs : none, int(soff), 0, kGenericNT);
  };
  auto issue_v = [&](uint32_t i, Slot& t) __attribute__((always_inline)) {
    const uint32_t voff = lane_pick(win.vcol, 4u * (i & 15u) + g) + n * a.page_tokens;
    const __amdgpu_buffer_rsrc_t r = i < nt ? rv : none;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) t.v[mb] = g_load16(step(r, 16u * mb), voff + 16u * mb * a.page_tokens);
  };
  window(0u);
  issue_k(0u, it);
  issue_v(0u, it);
  // Every wave needs the same pieces: wave w cuts steps w, w + NW, ...
#pragma unroll
  for (int k = 0; k < KS; ++k)
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      if ((2 * k + hf) % NW != int(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6))) continue;
      float x[8];
      bf16x8 piece[3];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = qv[k][8 * hf + i];
      cut3(x, piece);
#pragma unroll
      for (int p = 0; p < 3; ++p) sm.q[k][hf][p][lane] = __builtin_bit_cast(u32x4_g, piece[p]);
    }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the tiles stay in flight

  for (uint32_t i = 0; i < nt; ++i) {
    const uint32_t t0 = (s.first + i * s.step) * TILE;
    // The two low pieces of Q and the high one in accumulators of their own
    // (cl, c): the high products are short, so their sum hardly rounds.  Up to
    // dim 128 the low pieces of all steps go first, while the codes of the next
    // step are converted; above, the converted codes would not fit.
    f32x4 c[4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    f32x4 cl[4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    constexpr bool kLowFirst = DP <= 128, kOneSum = DP == 64;
    bf16x8 kb[kLowFirst ? 2 * KS : 1][4];
#pragma unroll
    for (int k = 0; k < 2 * KS; ++k) {
      auto& kbs = kb[kLowFirst ? k : 0];
#pragma unroll
      for (int mb = 0; mb < 4; ++mb)
        kbs[mb] = codes_bf16(it.k[mb * KS + k / 2][2 * (k % 2)], it.k[mb * KS + k / 2][2 * (k % 2) + 1]);
#pragma unroll
      for (int p = 2; p >= (kLowFirst ? 1 : 0); --p) {
        const bf16x8 qb = __builtin_bit_cast(bf16x8, sm.q[k / 2][k % 2][p][lane]);
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) {
          f32x4& x = p == 0 ? c[mb] : cl[mb];
          x = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kbs[mb], qb, x, 0, 0, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);  // one step's operands at a time
    }
    if constexpr (kLowFirst) {
#pragma unroll
      for (int k = 0; k < 2 * KS; ++k) {
        const bf16x8 qb = __builtin_bit_cast(bf16x8, sm.q[k / 2][k % 2][0][lane]);
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) {
          f32x4& x = kOneSum ? cl[mb] : c[mb];  // two steps round little either way
          x = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb[k][mb], qb, x, 0, 0, 0);
        }
      }
    }
    // Lane = token: its scales, 0 for a token no row sees.
    const uint32_t tok = t0 + lane;
    const bool seen = tok >= s.s0 && tok < h.e_max;
    float ksl = seen ? __uint_as_float(it.ks) : 0.f;
    float vsl = seen ? __uint_as_float(it.vs) : 0.f;
    asm volatile("" : "+v"(ksl), "+v"(vsl));  // the scales' registers are free for the next tile
    if (i + 1u < nt) window(i + 1u);
    issue_k(i + 1u, it);
    float y[16];
#define KVB_SCORE(j)                                        \
  y[j] = cl[(j) / 4][(j) % 4] * row_bcast<j>(ksl);          \
  if constexpr (!kOneSum) y[j] = fmaf(c[(j) / 4][(j) % 4], row_bcast<j>(ksl), y[j]);
    KVB_SCORE(0) KVB_SCORE(1) KVB_SCORE(2) KVB_SCORE(3) KVB_SCORE(4) KVB_SCORE(5) KVB_SCORE(6) KVB_SCORE(7)
    KVB_SCORE(8) KVB_SCORE(9) KVB_SCORE(10) KVB_SCORE(11) KVB_SCORE(12) KVB_SCORE(13) KVB_SCORE(14) KVB_SCORE(15)
#undef KVB_SCORE
    if (t0 < s.s0 || t0 + TILE > h.e_min) {
#pragma unroll
      for (uint32_t j = 0; j < 16; ++j) {
        const uint32_t t = t0 + 16u * g + j;
        if (t < s.s0 || t >= h.end) y[j] = neg_inf();
      }
    }
    st.weights(y);
#define KVB_WEIGHT(j) y[j] *= row_bcast<j>(vsl);
    KVB_WEIGHT(0) KVB_WEIGHT(1) KVB_WEIGHT(2) KVB_WEIGHT(3) KVB_WEIGHT(4) KVB_WEIGHT(5) KVB_WEIGHT(6) KVB_WEIGHT(7)
    KVB_WEIGHT(8) KVB_WEIGHT(9) KVB_WEIGHT(10) KVB_WEIGHT(11) KVB_WEIGHT(12) KVB_WEIGHT(13) KVB_WEIGHT(14)
    KVB_WEIGHT(15)
#undef KVB_WEIGHT
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      float x[8];
      bf16x8 pb[3];
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = y[8 * hf + j];
      cut3(x, pb);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const bf16x8 vb = codes_bf16(it.v[mb][2 * hf], it.v[mb][2 * hf + 1]);
#pragma unroll
        for (int p = 2; p >= 0; --p)
          st.acc[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vb, pb[p], st.acc[mb], 0, 0, 0);
        if (mb % 2 == 1) __builtin_amdgcn_sched_barrier(0);
      }
    }
    issue_v(i + 1u, it);
  }
  write_partials<DP, NW, true>(a, h, kv, hb, split, st.m, rows_sum(st.l), st.acc, sm);
}

// fp32 KV, 16-token tiles: a tile lies in one page, so its rows are addressed
// through descriptors of the tile's own K rows and V slab (any pool size).
// MFMA step (S, j) takes dims 16 S + 4 g + j of K and Q, step e of PV the
// token 4 g + e: whole 16-byte loads on both sides.
template <int DP, int NW, bool VARLEN>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(DP <= 128 ? 2 : 1)))
void split_generic_f32_kernel(SplitArgs a) {
  uint32_t split = blockIdx.y;
  if constexpr (VARLEN) {
    const BatchItem item = batch_item(a);
    split = item.split;
    rebase_sequence(a, item.seq, item.e);
  }
  __shared__ __attribute__((aligned(16))) GenericSmem<DP, NW> sm;
  constexpr uint32_t TILE = 16;
  constexpr int MB = DP / 16;  // 16-dim steps of QK, V row blocks
  const uint32_t lane = threadIdx.x & 63u, n = lane & 15u, g = lane >> 4;
  const uint32_t kv = blockIdx.x % a.kv_heads, hb = blockIdx.x / a.kv_heads;
  const SplitRange s = split_range<NW>(a, split, TILE);
  if (s.s1 <= s.s0) return write_empty<NW>(a, kv, hb, split);
  OnlineState<DP> st;
  st.clear();

  RowWindow win{0u, 0u, 0u};
  PageWindow next_win = load_window<TILE>(a, s, 0u, lane);
  const int64_t klast = a.k_positions[s.s1 - 1u], qpos = a.q_positions[block_row(a, hb, lane)];
  const uint32_t hr = a.rows * a.group, mine = 16u * hb + n;
  const bool real_head = mine < hr;
  f32x4 qv[MB];
  {
    const uint32_t hh = real_head ? mine : 0u;
    const float* const src = a.q + (size_t(hh / a.group) * a.q_heads + kv * a.group + hh % a.group) * a.dim;
#pragma unroll
    for (int k = 0; k < MB; ++k) {
      const uint32_t d = 16u * k + 4u * g;
      const bool in = real_head && d < a.dim;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x = src[(in ? d : 0u) + i];
        qv[k][i] = in ? x : 0.f;
      }
    }
  }
  const HeadLane h = head_lane(a, s, hb, lane, klast, qpos);
  const uint32_t nt = wave_tiles<TILE>(s, h.e_max);
  const float* const kbase = static_cast<const float*>(a.k);
  const float* const vbase = static_cast<const float*>(a.v);
  const __amdgpu_buffer_rsrc_t none = g_rsrc(a.k, 0u);
  auto step = [&](__amdgpu_buffer_rsrc_t r, uint32_t d) __attribute__((always_inline)) {
    return d < kDimFloor<DP> || d < a.dim ? r : none;
  };
  struct Slot {
    f32x4 k[MB], v[MB];
  };
  Slot it;
  auto window = [&](uint32_t i) __attribute__((always_inline)) {
    if ((i & 63u) == 0u) {
      win = window_rows(a, next_win, kv);
      if (i + 64u < nt) next_win = load_window<TILE>(a, s, i + 64u, lane);
    }
  };
  auto issue_k = [&](uint32_t i, Slot& t) __attribute__((always_inline)) {
    const uint32_t row = uint32_t(__builtin_amdgcn_readlane(int(win.row), int(i & 63u)));
    const __amdgpu_buffer_rsrc_t r = g_rsrc(kbase + size_t(row) * a.dim, i < nt ? 64u * a.dim : 0u);
    const uint32_t voff = n * 4u * a.dim + 16u * g;
#pragma unroll
    for (int k = 0; k < MB; ++k) t.k[k] = __builtin_bit_cast(f32x4, g_load16(step(r, 16u * k), voff + 64u * k));
  };
  auto issue_v = [&](uint32_t i, Slot& t) __attribute__((always_inline)) {
    const uint32_t col = uint32_t(__builtin_amdgcn_readlane(int(win.vcol), int(i & 63u)));
    const uint32_t slot = uint32_t(__builtin_amdgcn_readlane(int(win.slot), int(i & 63u)));
    const __amdgpu_buffer_rsrc_t r = g_rsrc(vbase + col, i < nt ? (a.dim * a.page_tokens - slot) * 4u : 0u);
    const uint32_t voff = n * 4u * a.page_tokens + 16u * g;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
      t.v[mb] = __builtin_bit_cast(f32x4, g_load16(step(r, 16u * mb), voff + 64u * mb * a.page_tokens));
  };
  window(0u);
  issue_k(0u, it);
  issue_v(0u, it);
  const float cs = a.scale;
  const bool ragged_dim = a.dim < uint32_t(DP);
  for (uint32_t i = 0; i < nt; ++i) {
    const uint32_t t0 = (s.first + i * s.step) * TILE;
    if (ragged_dim) {  // past dim lie the next row's values, whatever they are
#pragma unroll
      for (int k = 0; k < MB; ++k)
        if (16u * k + 4u * g >= a.dim) it.k[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    f32x4 c[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int k = 0; k < MB; ++k)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        c[j & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(it.k[k][j], qv[k][j], c[j & 1], 0, 0, 0);
    if (i + 1u < nt) window(i + 1u);
    issue_k(i + 1u, it);
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = (c[0][e] + c[1][e]) * cs;
    if (t0 < s.s0 || t0 + TILE > h.e_min) {
#pragma unroll
      for (uint32_t e = 0; e < 4; ++e) {
        const uint32_t t = t0 + 4u * g + e;
        if (t < s.s0 || t >= h.end) y[e] = neg_inf();
        if (t < s.s0 || t >= h.e_max) {  // no row sees the token: its V may hold anything
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) it.v[mb][e] = 0.f;
        }
      }
    }
    st.weights(y);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        st.acc[mb] = __builtin_amdgcn_mfma_f32_16x16x4f32(it.v[mb][e], y[e], st.acc[mb], 0, 0, 0);
    issue_v(i + 1u, it);
  }
  write_partials<DP, NW, false>(a, h, kv, hb, split, st.m, rows_sum(st.l), st.acc, sm);
}

}  // namespace
}  // namespace kvb
