// Body of the integer-MFMA split kernel (split_i8.h), included in the kernel
// function.
  SplitArgs a = a_in;
  a.begin = p_begin;
  a.end = p_end;
  a.split_tokens = p_split_tokens;
  a.page_tokens = p_page_tokens;
  a.kv_heads = p_kv_heads;
  a.pages = p_pages;
  uint32_t split = blockIdx.x, kv = blockIdx.y;
  if constexpr (VARLEN) {
    const BatchItem item = batch_item(a);
    split = item.split;
    kv = blockIdx.x;
    rebase_sequence(a, item.seq, item.e);
  }
  const float* __restrict__ q = VARLEN ? a.q : q_in;
  const int64_t* __restrict__ qpos = VARLEN ? a.q_positions : qpos_in;
  const int64_t* __restrict__ kpos = VARLEN ? a.k_positions : kpos_in;
  const uint32_t* __restrict__ table = VARLEN ? a.page_table : table_in;
  float* __restrict__ scratch = VARLEN ? a.scratch : scratch_in;
  constexpr int CH = NB == 1 ? 1 : 4;  // tiles per two-pass chunk
  using L = I8Layout<D, NW, HS>;
  constexpr int ND = 3;  // int8 digits of Q and of the weights
  constexpr int NC = L::NC;  // MFMA column tiles of the digit columns (PV; QK unless PAIR)
  // Paired-row QK (dim 128, <= 4 head-rows): MFMA row m of M-block mb is
  // half m%2 (dims 64*(m%2) ..) of token 8*mb + m/2; column tile h of the Q
  // digits holds half h, so rows and tiles of equal half give the two half
  // dot products of a token, which add exactly in int32.  The K loads of a
  // k-block then read whole 64-byte half rows, two per 128-byte line.
  constexpr bool PAIR = L::kPair;
  constexpr int NCQ = PAIR ? 2 : NC;        // MFMA column tiles of the QK B operand
  constexpr int KS = PAIR ? 1 : D / 64;     // 64-dim steps per QK M-block
  __shared__ __attribute__((aligned(16))) uint8_t smem[L::kBytes];

  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t n = lane & 15u, g = lane >> 4;
  const uint32_t head_rows = a.rows * a.group;  // <= HS
  // Splits that take part in the fused merge.  A batched single-launch call
  // merges only the sequence's own splits (at least one, so that an empty
  // sequence still gets its empty result); work-groups past them write no
  // partial and take no ticket.  In a two-launch batched call they write the
  // empty partial (m = -inf, l = 0, n = 0) straight away, without loading
  // anything.
  uint32_t nsplit = a.splits;
  if constexpr (VARLEN) {
    nsplit = a.end > 0u ? (a.end - 1u) / a.split_tokens + 1u : 1u;
    if (split >= nsplit) {
      if constexpr (!FUSED) {
        constexpr uint32_t W = D + 2;
        for (uint32_t o = threadIdx.x; o < head_rows * W; o += 64u * NW) {
          const uint32_t hh = o / W, col = o % W;
          const uint32_t row2 = hh / a.group, head2 = kv * a.group + hh % a.group;
          scratch[((size_t(row2) * a.q_heads + head2) * a.splits + split) * W + col] = col == 0 ? neg_inf() : 0.f;
        }
      }
      return;
    }
  }

  const uint64_t s0_64 = uint64_t(a.begin) + uint64_t(split) * a.split_tokens;
  const uint32_t s0 = s0_64 < a.end ? uint32_t(s0_64) : a.end;
  const uint32_t s1 = uint64_t(s0) + a.split_tokens < a.end ? s0 + a.split_tokens : a.end;
  const uint32_t k_first = s0 / kTileTokens;

  IssueCtx c;
  c.k = kdata;
  c.v = vdata;
  c.ks = kscale;
  c.vs = vscale;
  c.table = table;
  c.kv = kv;
  c.kv_heads = a.kv_heads;
  c.P = a.page_tokens;
  c.pages = a.pages;
  c.lp_lo = s0 / a.page_tokens;
  c.lp_hi = s1 > s0 ? (s1 - 1u) / a.page_tokens : c.lp_lo;
  c.lane = lane;
  c.lg_p = 31u - __builtin_clz(a.page_tokens);  // page_tokens is a power of two
  {
    // Page-table window of the split (no load for an empty split, whose
    // lp_lo may be one past the last page).
    const uint32_t lp = c.lp_lo + lane;
    c.ptab = s1 > s0 && lp <= c.lp_hi ? table[lp] : 0u;
  }
  if constexpr (PT) {
    c.voff_k = PAIR ? 128u * (n >> 1) + 64u * (n & 1u) + 16u * g
                    : (16u * (n >> 2) + (n & 3u)) * uint32_t(D) + 16u * g;
    c.voff_v = n * a.page_tokens + 16u * g;
    c.voff_s = 4u * lane;
  } else {
    const uint32_t kv_bytes = a.pages * a.kv_heads * a.page_tokens * uint32_t(D);  // < 4 GiB (host check)
    const uint32_t sc_bytes = a.pages * a.kv_heads * a.page_tokens * 4u;
    c.rk = rsrc(kdata, kv_bytes);
    c.rv = rsrc(vdata, kv_bytes);
    c.rks = rsrc(kscale, sc_bytes);
    c.rvs = rsrc(vscale, sc_bytes);
  }

  // Per-wave LDS exchange areas (plain LDS accesses: the compiler inserts
  // the MFMA-result hazards and lgkmcnt waits).
  uint8_t* const wbase = smem + wave * L::kWave;

  // ---- everything the KV stream and the Q digits depend on is loaded in
  // one memory round trip: the page-table window (above), the split's last
  // key position, the query positions, and the Q elements this lane turns
  // into MFMA digit columns (straight into registers; no LDS staging and no
  // work-group barrier before the stream starts).
  const int64_t klast = s1 > s0 ? kpos[s1 - 1u] : 0;
  int64_t qp[HS];
#pragma unroll
  for (int r = 0; r < HS; ++r) qp[r] = qpos[uint32_t(r) < a.rows ? uint32_t(r) : 0u];
  // Lane (n, g) of MFMA column tile nc feeds a digit column: column
  // 16*nc + n (digit dg = col / HS of head-row col % HS), or with PAIR column
  // n of tile nc = half nc.  MFMA s of a 64-dim step takes dims 64*s + 16*g
  // .. +15 of Q and K alike (PAIR: dims 64*nc + 16*g ..), so the K loads
  // read whole 64-byte row segments.
  float qv[NCQ][16 * KS];
#pragma unroll
  for (int nc = 0; nc < NCQ; ++nc) {
    const uint32_t col = PAIR ? n : 16u * nc + n;
    const uint32_t h = col % HS;
    const bool valid = col < uint32_t(ND * HS) && h < head_rows;
    const uint32_t hq = valid ? h : 0u;
    const float* src = q + (size_t(hq / a.group) * a.q_heads + kv * a.group + hq % a.group) * D + 16u * g +
                       (PAIR ? 64u * nc : 0u);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float4 w = reinterpret_cast<const float4*>(src + 64 * s)[j];
        qv[nc][16 * s + 4 * j] = valid ? w.x : 0.f;
        qv[nc][16 * s + 4 * j + 1] = valid ? w.y : 0.f;
        qv[nc][16 * s + 4 * j + 2] = valid ? w.z : 0.f;
        qv[nc][16 * s + 4 * j + 3] = valid ? w.w : 0.f;
      }
    }
  }

  // ---- visibility per head-row: tokens [s0, eh[h]) (k_positions nondecreasing)
  uint32_t eh[HS];
  {
    uint32_t erow[HS];
#pragma unroll
    for (int r = 0; r < HS; ++r) {
      erow[r] = s0;
      if (s1 > s0 && uint32_t(r) < a.rows)
        erow[r] = klast <= qp[r] ? s1 : visible_end(kpos, s0, s1, qp[r], lane);
    }
#pragma unroll
    for (int h = 0; h < HS; ++h) {
      const uint32_t r = uint32_t(h) / a.group;
      uint32_t e = s0;
#pragma unroll
      for (int rr = 0; rr < HS; ++rr)
        if (uint32_t(rr) == r) e = erow[rr];
      eh[h] = uint32_t(h) < head_rows ? __builtin_amdgcn_readfirstlane(e) : s0;
    }
  }
  uint32_t e_min = 0xffffffffu, e_max = s0;
#pragma unroll
  for (int h = 0; h < HS; ++h) {
    if (uint32_t(h) < head_rows) e_min = eh[h] < e_min ? eh[h] : e_min;
    e_max = eh[h] > e_max ? eh[h] : e_max;
  }

  // ---- the wave's tiles (round-robin over the work-group).  Items run in
  // chunks of 2*CH: K images of tiles 4c..4c+3, then their V images.
  // Items of tiles past the wave's last tile load nothing (zero-sized
  // descriptors); their stale slot contents are masked by tok_ok and zero
  // weights.
  const uint32_t k_vis = e_max > s0 ? (e_max - 1u) / kTileTokens : 0u;
  const uint32_t k_count = e_max > s0 ? k_vis + 1u - k_first : 0u;
  const uint32_t nt = k_count > wave ? (k_count - wave + NW - 1u) / NW : 0u;
  const uint32_t n_chunks = (nt + CH - 1u) / CH;
  auto tile_k = [&](uint32_t i) __attribute__((always_inline)) { return k_first + wave + i * NW; };
  // Item at chunk position POS (0 .. 2*CH-1) of chunk ch.
  auto issue = [&](auto posc, uint32_t ch, Slot<D>& slot) __attribute__((always_inline)) {
    constexpr uint32_t pos = decltype(posc)::value;
    const uint32_t i = ch * CH + pos % CH;
    issue_item<D, PT, (pos >= uint32_t(CH)), PAIR>(c, tile_k(i), i < nt, slot);
  };
  constexpr int kRing = NB == 1 ? 2 : NB;
  constexpr int kAhead = NB == 1 ? 2 : NB - 1;
  Slot<D> ring[kRing];
  // Start streaming before the Q digits are built.
  static_for<0, kAhead>([&](auto uc) __attribute__((always_inline)) { issue(uc, 0u, ring[decltype(uc)::value]); });

  // ---- Q digits (B operand of QK) and per-head score factors.  A column's
  // scale 2^kq comes from its head-row's whole Q row (with PAIR both tiles
  // of a lane hold the same column).  Every wave needs the same digits (its
  // lanes are the same MFMA columns), so the digit dwords are built once per
  // work-group: wave w builds dwords d = w, w + NW, ... of every lane and
  // stores them in the Q digit area of LDS; after one barrier (LDS only: the
  // first KV item stays in flight) each wave reads its lanes' digits back.
  i32x4 qd[NCQ][KS];
  float cql[HS];
  static_assert(L::kQdBytes == NCQ * KS * 16, "digit bytes per lane");
  uint8_t* const qd_s = smem + L::kQd + lane * L::kQdBytes;
  {
    int kq_lane = 0;
    auto col_kq = [&](float amax) __attribute__((always_inline)) {
      amax = rows_max(amax);
      int kq = 0;
      if (amax > 0.f) {
        kq = 22 - __builtin_amdgcn_frexp_expf(amax);  // |2^kq q| < 2^22: top digit in [-64, 64]
        kq = kq < -100 ? -100 : (kq > 100 ? 100 : kq);
      }
      return kq;
    };
    int kq_pair = 0;
    if constexpr (PAIR) {
      float amax = 0.f;
#pragma unroll
      for (int nc = 0; nc < NCQ; ++nc)
#pragma unroll
        for (int i = 0; i < 16 * KS; ++i) amax = fmaxf(amax, fabsf(qv[nc][i]));
      kq_pair = col_kq(amax);
    }
#pragma unroll
    for (int nc = 0; nc < NCQ; ++nc) {
      const uint32_t col = PAIR ? n : 16u * nc + n;
      const uint32_t dg = col / HS;
      const bool valid = col < uint32_t(ND * HS) && col % HS < head_rows;
      int kq = kq_pair;
      if constexpr (!PAIR) {
        float amax = 0.f;
#pragma unroll
        for (int i = 0; i < 16 * KS; ++i) amax = fmaxf(amax, fabsf(qv[nc][i]));
        kq = col_kq(amax);
      }
      if (nc == 0) kq_lane = kq;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t dw = (uint32_t(nc) * KS + s) * 4u + j;  // digit dword of the lane
          if (dw % NW != wave) continue;                       // uniform: built by wave dw % NW
          uint32_t packed = 0;
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            const int qi = int(__builtin_rintf(__builtin_amdgcn_ldexpf(qv[nc][16 * s + 4 * j + b], kq)));
            // Balanced digits from the last (dg = ND - 1) up.
            int r = qi, d = 0;
#pragma unroll
            for (int x = ND - 1; x >= 0; --x) {
              const int lo = x > 0 ? int(int8_t(r & 0xff)) : r;
              d = dg == uint32_t(x) ? lo : d;
              r = (r - lo) >> 8;
            }
            packed |= (uint32_t(d) & 0xffu) << (8 * b);
          }
          *reinterpret_cast<uint32_t*>(qd_s + 4u * dw) = valid ? packed : 0u;
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int nc = 0; nc < NCQ; ++nc)
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const u32x4_t w = *reinterpret_cast<const u32x4_t*>(qd_s + 16u * (uint32_t(nc) * KS + s));
        qd[nc][s] = i32x4{int(w[0]), int(w[1]), int(w[2]), int(w[3])};
      }
#pragma unroll
    for (int h = 0; h < HS; ++h) {
      const int kq = __builtin_amdgcn_readlane(kq_lane, h);
      cql[h] = __builtin_amdgcn_ldexpf(a.scale, -kq) * kLog2e;
    }
  }

  uint8_t* const exch_w = wbase + n * L::kExchCol + 64u * g;              // C write base (MFMA view)
  uint8_t* const exch_w2 = wbase + n * L::kExchCol + 8u * g;              // PAIR: summed C write base
  const uint8_t* const exch_r = wbase + 4u * lane;                        // lane-as-token read base
  uint8_t* const dig_w = wbase + L::kExch + lane;                         // digit write (lane-as-token)
  const uint8_t* const dig_r = wbase + L::kExch + n * L::kDigCol + 16u * g;  // B operand read

  // State.  Lane-as-token view: sc, mx, lw, lrun per head-row.  MFMA view:
  // int32 digit numerators acc_i, fp32 numerators acc_f (head = lane & 15).
  float sc[CH][HS];
  float vsc[CH];  // v-scale of token lane, per tile of the chunk
  float mx[HS], lw[HS], lrun[HS];
  float m_run[HS], m_new[HS], mu[HS];
  float vmx = 0.f;
  int kp = 0;
  i32x4 acc_i[NC][D / 16];
  f32x4 acc_f[D / 16];
#pragma unroll
  for (int h = 0; h < HS; ++h) {
    mx[h] = neg_inf();
    lw[h] = 0.f;
    lrun[h] = 0.f;
    m_run[h] = neg_inf();
    m_new[h] = neg_inf();
    mu[h] = 0.f;
#pragma unroll
    for (int r = 0; r < CH; ++r) sc[r][h] = neg_inf();
  }
#pragma unroll
  for (int mb = 0; mb < D / 16; ++mb) {
    acc_f[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int nc = 0; nc < NC; ++nc) acc_i[nc][mb] = i32x4{0, 0, 0, 0};
  }

  // ---- pass 1 item: scores of chunk tile r (tile index i).
  auto process_k = [&](auto rc, uint32_t i, const Slot<D>& it) __attribute__((always_inline)) {
    constexpr uint32_t r = decltype(rc)::value;
    const uint32_t t0 = tile_k(i) * kTileTokens;
    const uint32_t tok = t0 + lane;
    const bool real = i < nt;
    const bool full = real && t0 >= s0 && t0 + kTileTokens <= e_min;
    const bool tok_ok = full || (real && tok >= s0 && tok < e_max);
    if constexpr (PAIR) {
      // Rows 4g+e of M-block mb: e even = half 0, e odd = half 1 of tokens
      // 8mb+2g (e < 2) and 8mb+2g+1; tile 0 gives the half-0 and tile 1 the
      // half-1 dot products, summed exactly here.
      static_for<0, 8>([&](auto mbc) __attribute__((always_inline)) {
        constexpr uint32_t mb = decltype(mbc)::value;
        const u32x4_t w = it.d[mb];
        const i32x4 av = {int(w[0]), int(w[1]), int(w[2]), int(w[3])};
        const i32x4 zero = {0, 0, 0, 0};
        const i32x4 c0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, qd[0][0], zero, 0, 0, 0);
        const i32x4 c1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, qd[1][0], zero, 0, 0, 0);
        typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
        const u32x2_t cw = {uint32_t(c0[0] + c1[1]), uint32_t(c0[2] + c1[3])};
        *reinterpret_cast<u32x2_t*>(exch_w2 + 32 * mb) = cw;
      });
    } else {
      static_for<0, NC>([&](auto ncc) __attribute__((always_inline)) {
        constexpr uint32_t nc = decltype(ncc)::value;
        static_for<0, 4>([&](auto mbc) __attribute__((always_inline)) {
          constexpr uint32_t mb = decltype(mbc)::value;
          i32x4 cc = {0, 0, 0, 0};
#pragma unroll
          for (int s = 0; s < D / 64; ++s) {
            const u32x4_t w = it.d[mb * (D / 64) + s];
            const i32x4 av = {int(w[0]), int(w[1]), int(w[2]), int(w[3])};
            cc = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, qd[nc][s], cc, 0, 0, 0);
          }
          const u32x4_t cw = {uint32_t(cc[0]), uint32_t(cc[1]), uint32_t(cc[2]), uint32_t(cc[3])};
          *reinterpret_cast<u32x4_t*>(exch_w + (nc * 16 * L::kExchCol + 16 * mb)) = cw;
        });
      });
    }
    int dv[HS][ND];
    static_for<0, HS>([&](auto hc) __attribute__((always_inline)) {
      constexpr uint32_t h = decltype(hc)::value;
      static_for<0, ND>([&](auto dc) __attribute__((always_inline)) {
        constexpr uint32_t dg = decltype(dc)::value;
        constexpr uint32_t col = dg * HS + h;
        dv[h][dg] = *reinterpret_cast<const int*>(exch_r + col * L::kExchCol);
      });
    });
    const float ks_l = __uint_as_float(it.ks);
    const float vs_l = __uint_as_float(it.vs);
    vsc[r] = vs_l;  // for the tile's V item (which loads no scales)
    vmx = fmaxf(vmx, tok_ok ? fabsf(vs_l) : 0.f);
#pragma unroll
    for (int h = 0; h < HS; ++h) {
      const float si = fmaf(fmaf(float(dv[h][0]), 256.f, float(dv[h][1])), 256.f, float(dv[h][2]));
      float s2 = si * (ks_l * cql[h]);
      if (!full && !(real && tok >= s0 && tok < eh[h])) s2 = neg_inf();
      if (uint32_t(h) >= head_rows) s2 = neg_inf();
      sc[r][h] = s2;
      mx[h] = fmaxf(mx[h], s2);
    }
  };

  // ---- pass 2 item: weights of chunk tile r, PV.
  auto process_v = [&](auto rc, uint32_t i, const Slot<D>& it) __attribute__((always_inline)) {
    constexpr uint32_t r = decltype(rc)::value;
    const uint32_t t0 = tile_k(i) * kTileTokens;
    const uint32_t tok = t0 + lane;
    const bool real = i < nt;
    const bool tok_ok = real && ((t0 >= s0 && t0 + kTileTokens <= e_min) || (tok >= s0 && tok < e_max));
    const float vs_l = tok_ok ? vsc[r] : 0.f;
    static_for<0, HS>([&](auto hc) __attribute__((always_inline)) {
      constexpr uint32_t h = decltype(hc)::value;
      const float w = __builtin_amdgcn_exp2f(sc[r][h] - mu[h]);  // w * 2^kp
      lw[h] += w;
      // p = w * v_scale rounded to an integer (0 <= p < 2^21) in one fma:
      // 1.5 * 2^23 + p lies in [2^23, 2^24), where the float's ulp is 1, so
      // its low 22 bits are p mod 2^22 (two's complement), and bits 0-6,
      // 7-13 and 14-21 are the three digits of p.
      const uint32_t pb = __float_as_uint(fmaf(w, vs_l, 12582912.f));
      const uint32_t d0 = (pb >> 14) & 0xffu;
      const uint32_t d1 = (pb >> 7) & 0x7fu;
      const uint32_t d2 = pb & 0x7fu;
      dig_w[h * L::kDigCol] = uint8_t(d0);
      dig_w[(HS + h) * L::kDigCol] = uint8_t(d1);
      dig_w[(2 * HS + h) * L::kDigCol] = uint8_t(d2);
    });
    u32x4_t bd[NC];
    static_for<0, NC>([&](auto ncc) __attribute__((always_inline)) {
      constexpr uint32_t nc = decltype(ncc)::value;
      bd[nc] = *reinterpret_cast<const u32x4_t*>(dig_r + nc * 16 * L::kDigCol);
    });
#pragma unroll
    for (int nc = 0; nc < NC; ++nc) {
      const i32x4 bv = {int(bd[nc][0]), int(bd[nc][1]), int(bd[nc][2]), int(bd[nc][3])};
#pragma unroll
      for (int mb = 0; mb < D / 16; ++mb) {
        const u32x4_t w = it.d[mb];
        const i32x4 av = {int(w[0]), int(w[1]), int(w[2]), int(w[3])};
        acc_i[nc][mb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, bv, acc_i[nc][mb], 0, 0, 0);
      }
    }
  };

  // ---- chunk maximum and weight exponent kp (after the chunk's K items).
  auto chunk_max = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < HS; ++h) {
      const float mc = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(wave_max(mx[h]))));
      m_new[h] = fmaxf(m_run[h], mc);
      mx[h] = neg_inf();
    }
    const float vmax = wave_max(vmx);
    vmx = 0.f;
    kp = 0;
    if (vmax > 0.f) {
      kp = 21 - __builtin_amdgcn_frexp_expf(vmax * kVmaxMargin);
      kp = kp < -100 ? -100 : (kp > 100 ? 100 : kp);
    }
#pragma unroll
    for (int h = 0; h < HS; ++h) mu[h] = (m_new[h] == neg_inf() ? 0.f : m_new[h]) - float(kp);
  };

  // ---- fold the chunk's int32 digit numerators into the fp32 state.
  auto fold = [&]() __attribute__((always_inline)) {
    float fh[HS];
#pragma unroll
    for (int h = 0; h < HS; ++h) {
      fh[h] = m_run[h] == neg_inf() ? 0.f : __builtin_amdgcn_exp2f(m_run[h] - m_new[h]);
      lrun[h] = fmaf(lrun[h], fh[h], __builtin_amdgcn_ldexpf(lw[h], -kp));
      lw[h] = 0.f;
      m_run[h] = m_new[h];
    }
    float f_lane = 0.f;  // head (lane & 15) of the MFMA view
#pragma unroll
    for (int h = 0; h < HS; ++h)
      if (n == uint32_t(h)) f_lane = fh[h];
    const float inv = __builtin_amdgcn_ldexpf(1.f, -kp);
#pragma unroll
    for (int mb = 0; mb < D / 16; ++mb) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        // digit dg of head h is column dg*HS + h: tile (dg*HS+h)/16, lane shift (dg*HS)%16.
        const float x0 = float(acc_i[0][mb][e]);
        float x1, x2;
        if constexpr (HS <= 4) {
          x1 = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x0), 0x100 + HS, 0xF, 0xF, true));
          x2 = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x0), 0x100 + 2 * HS, 0xF, 0xF, true));
        } else {
          x1 = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x0), 0x100 + (HS % 16), 0xF, 0xF, true));
          x2 = float(acc_i[NC - 1][mb][e]);  // column 2*HS + h = 16 + h for HS == 8
        }
        const float comb = fmaf(fmaf(x0, 128.f, x1), 128.f, x2);
        acc_f[mb][e] = fmaf(acc_f[mb][e], f_lane, comb * inv);
      }
#pragma unroll
      for (int nc = 0; nc < NC; ++nc) acc_i[nc][mb] = i32x4{0, 0, 0, 0};
    }
  };

  if constexpr (NB == 1) {
    // ---- main loop of one-tile chunks: each slot is refilled as soon as its
    // item is consumed.
    for (uint32_t ch = 0; ch < n_chunks; ++ch) {
      process_k(std::integral_constant<uint32_t, 0>(), ch, ring[0]);
      chunk_max();
      issue(std::integral_constant<uint32_t, 0>(), ch + 1u, ring[0]);
      process_v(std::integral_constant<uint32_t, 0>(), ch, ring[1]);
      issue(std::integral_constant<uint32_t, 1>(), ch + 1u, ring[1]);
      fold();
    }
  } else {
    // ---- main loop: one chunk per iteration, items unrolled so that ring
    // slots (item % NB, NB divides 2*CH) are compile-time.
    static_assert((2 * CH) % kRing == 0, "ring size must divide the chunk");
    for (uint32_t ch = 0; ch < n_chunks; ++ch) {
      static_for<0, 2 * CH>([&](auto uc) __attribute__((always_inline)) {
        constexpr uint32_t u = decltype(uc)::value;
        issue(std::integral_constant<uint32_t, (u + NB - 1) % (2 * CH)>(), ch + (u + NB - 1) / (2 * CH),
              ring[(u + NB - 1) % NB]);
        if constexpr (u < uint32_t(CH)) {
          process_k(std::integral_constant<uint32_t, u>(), ch * CH + u, ring[u % NB]);
          if constexpr (u == uint32_t(CH) - 1) chunk_max();
        } else {
          process_v(std::integral_constant<uint32_t, u - CH>(), ch * CH + (u - CH), ring[u % NB]);
          if constexpr (u == 2u * CH - 1) fold();
        }
      });
    }
  }

  // ---- combine the waves through LDS and write the split partial.  Each
  // wave publishes its maxima, denominators and numerators in its own rows
  // of the combine area (disjoint from every exchange area, so no barrier is
  // needed before), then one barrier.  Each output then requests the NW
  // wave values of its column together (independent LDS loads, one latency)
  // and adds them in wave order; a wave with no visible token (m = -inf)
  // contributes factor 0 to its zero values, which leaves the sum unchanged.
  float* const wm_s = reinterpret_cast<float*>(smem + L::kComb);  // [NW][HS]
  float* const wl_s = wm_s + NW * HS;                              // [NW][HS]
  float* const wacc_s = wl_s + NW * HS;                            // [NW][HS][D]
#pragma unroll
  for (int h = 0; h < HS; ++h) {
    const float lsum = wave_sum(lrun[h]);
    if (lane == 0) {
      wm_s[wave * HS + h] = m_run[h] * kLn2;
      wl_s[wave * HS + h] = lsum;
    }
  }
  if (n < uint32_t(HS)) {
#pragma unroll
    for (int mb = 0; mb < D / 16; ++mb) {
      float4 y;
      y.x = acc_f[mb][0];
      y.y = acc_f[mb][1];
      y.z = acc_f[mb][2];
      y.w = acc_f[mb][3];
      *reinterpret_cast<float4*>(&wacc_s[(wave * HS + n) * D + 16 * mb + 4 * g]) = y;
    }
  }
  __syncthreads();
  // One numerator column per thread and iteration (no branches: the LDS
  // loads of all waves are requested together); the thread of column 0 also
  // writes the head-row's maximum and denominator.
  constexpr uint32_t W = D + 2;
  for (uint32_t o = threadIdx.x; o < head_rows * uint32_t(D); o += 64u * NW) {
    // A wave's 64 columns lie in one head-row (64 divides D), so the NW
    // wave maxima, denominators and factors of its iteration are scalars:
    // lane w < NW reads wave w's pair and computes its factor once.
    const uint32_t hh = __builtin_amdgcn_readfirstlane(o / D), d = o % D;
    const uint32_t wl = lane < uint32_t(NW) ? lane : 0u;
    const float m_l = wm_s[wl * HS + hh], l_l = wl_s[wl * HS + hh];
    float mw[NW], lv[NW], xw[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      mw[w] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(m_l), w));
      lv[w] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(l_l), w));
      xw[w] = wacc_s[(w * HS + hh) * D + d];
    }
    float mm = mw[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) mm = fmaxf(mm, mw[w]);
    const float f_l = m_l == neg_inf() ? 0.f : exp_e(m_l - mm);
    float val = 0.f, lsum = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f_l), w));
      val = fmaf(f, xw[w], val);
      lsum = fmaf(f, lv[w], lsum);
    }
    const uint32_t row2 = hh / a.group, head2 = kv * a.group + hh % a.group;
    const size_t rh = size_t(row2) * a.q_heads + head2;
    float* const dst = scratch + (rh * a.splits + split) * W;
    if constexpr (FUSED) {  // agent-coherent, in the merge's packed layout
      const PackedPartials<D> pp(scratch, a);
      __hip_atomic_store(pp.n(rh, a.splits, split) + d, val, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (d == 0) {
        __hip_atomic_store(pp.m(rh, a.splits, split), mm, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(pp.l(rh, a.splits, split), lsum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    } else {
      dst[2 + d] = val;
      if (d == 0) {
        dst[0] = mm;
        dst[1] = lsum;
      }
    }
  }

  // ---- fused merge: the last work-group to finish for this kv head merges
  // its splits (agent-scope release of every partial, then a ticket).
  if constexpr (FUSED) {
    __shared__ uint32_t last_s;
    // The partials were stored with agent-scope atomic stores (coherent
    // across XCDs, no L2 write-back needed) and are read back with
    // agent-scope atomic loads.  Every wave waits until its stores have
    // completed, the work-group synchronizes, and only then takes a ticket,
    // so the work-group that draws the last ticket sees every partial.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if constexpr (FENCE) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __syncthreads();
    if (threadIdx.x == 0) {
      const uint32_t t = __hip_atomic_fetch_add(a.counters + kv, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last_s = t + 1u == nsplit ? 1u : 0u;
    }
    __syncthreads();
    if (last_s != 0u) {
      if constexpr (FENCE) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      static_assert(NW * 32 * 4 <= L::kBytes, "the merge's factors fit the kernel's LDS");
      fused_merge<D, NW>(a, kv, head_rows, nsplit, scratch, reinterpret_cast<float*>(smem));
      if (threadIdx.x == 0) __hip_atomic_store(a.counters + kv, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
