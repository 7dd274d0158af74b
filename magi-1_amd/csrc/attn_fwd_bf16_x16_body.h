// The body of the kernels of attn_fwd_bf16_x16.hip, included in each: QMODE, QB; a: the call's arguments; X16_BLOCK: the workgroup's number in it.
// (Not a function of them: behind a reference to the arguments the compiler treats the single calls' tile loop differently, which costs them up
// to half a per cent.)
  constexpr bool CHECK = QMODE == Q_CHECK;
  constexpr int NW = 4, WROWS = 16 * QB, BM = WROWS * NW;
  static_assert(QB == 4 || (QB == 2 && !CHECK), "two query blocks: no verdicts, no shared keys");
  constexpr int LOADS = BN / (4 * NW);  // direct loads per wave per matrix per tile (4 rows each)
  constexpr int RING = 4;               // operand fragments in flight between LDS and the MFMAs
  // K and V double buffered in four separate LDS objects that are only named statically (an operand read then
  // never waits for the direct loads in flight to the other pair of slots)
  __shared__ __attribute__((aligned(1024))) unsigned char sK0[K_TILE_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char sV0[V_TILE_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char sK1[K_TILE_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char sV1[V_TILE_BYTES];
  __shared__ int s_sel[LOCATE_WORDS];
  __shared__ int s_over;  // CHECK: the first tile overflowed

  if (gate_closed(a)) return;
  const int tid = threadIdx.x;
  if (CHECK && tid == 0) s_over = 0;
  unsigned block = X16_BLOCK;
  SplitPiece sp = {nullptr, 0u};
  if constexpr (QB == 4) sp = split_piece<SPLIT_FLOATS>(a, block);
  const WorkItem wi = locate_work(a, BM, tid, s_sel, block);
  if (!wi.valid) return;
  const int qe = wi.qe;
  int ks = wi.ks, ke = wi.ke;

  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63, n = l & 15, g = l >> 4;
  const int row0 = wi.q0 + WROWS * w;  // first row of this wave
  if (ke <= ks) {
#pragma unroll
    for (int b = 0; b < QB / 2; ++b)
      if (row0 + 32 * b + (l & 31) < qe) store_empty_row(a, wi, row0 + 32 * b + (l & 31), l >> 5);
    if (CHECK && l == 0) a.verdict[4 * (long)wi.item + w] = 0;
    return;
  }
  if (sp.out) {
    const unsigned tiles = (unsigned)(ke - ks + BN - 1) / BN;
    const int b = (int)split_cut(a, tiles, sp.piece), e = (int)split_cut(a, tiles, sp.piece + 1);
    if (b == e) {  // (a range with fewer tiles than pieces)
      store_partial_zero(sp.out, w, l);
      return;
    }
    ke = min(ke, ks + e * BN);
    ks += b * BN;
  }

  // ---- K/V tile loader: wave w fills rows 4 * (w + 4 j) .. +3; lane l sits at row +(l >> 4), slot l & 15 ----
  const long ks_t = a.ks_t, vs_t = a.vs_t;
  const int k_split = a.k_split;
  const long k2_delta = a.k2 ? (a.k2 - a.k) - (long)k_split * ks_t : 0;
  const long v2_delta = a.v2 ? (a.v2 - a.v) - (long)k_split * vs_t : 0;
  const char* const kcolp = a.k + (long)wi.kvh * a.ks_h;
  const char* const vcolp = a.v + (long)wi.kvh * a.vs_h;

  auto issue_mat = [&](int k0, unsigned char* tile_base, bool is_v) __attribute__((always_inline)) {
    const int group = is_v ? V_GROUP : K_GROUP;
    unsigned char* dst = tile_base + w * group;
    const long st = is_v ? vs_t : ks_t;
    const char* colp = is_v ? vcolp : kcolp;
    const long d2 = is_v ? v2_delta : k2_delta;
    // the lane geometry is re-derived from an opaque copy of the lane index at every call, so that nothing of it
    // occupies registers across the main loop
    int lane = l;
    asm volatile("" : "+v"(lane));
    const int lr = lane >> 4, sl = lane & 15;
    // logical 16-byte chunk that belongs at this lane's fixed LDS slot.  Row r of a tile (row r & 3 = lr of its
    // group) keeps chunk c at
    //   K: c ^ (r & 3)         (ds_read_b128 down 16 rows: four groups 64 bytes apart x four chunks)
    //   V: c ^ ((r & 3) << 1)  (transposing reads of 32 bytes from each of 8 rows: two groups 128 bytes apart x
    //                           four 32-byte slots)
    const int chunk = is_v ? (sl ^ (lr << 1)) : (sl ^ lr);
    const bool interior = (k0 + BN <= ke) && (k0 + BN <= k_split || k0 >= k_split);
    if (interior) {
      // buffer-addressed direct loads: tile base in the resource descriptor, one 32-bit lane offset, the row
      // group of load j in the scalar offset
      const char* b = colp + (long)k0 * st + (k0 >= k_split ? d2 : 0);
      const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)b, 0, 0x7fffffff, 0x00020000);
      const unsigned voff = (unsigned)(4 * w + lr) * (unsigned)st + (unsigned)(chunk * 16);
#pragma unroll
      for (int j = 0; j < LOADS; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, LDS_PTR(void, dst + j * NW * group), 16, voff,
                                                 (int)((unsigned)(4 * NW * j) * (unsigned)st), 0, 0);
    } else {
      // Ragged end of the range, or a tile that straddles the two key segments: per-lane rows, clamped to the last
      // valid key, each lane reading through the descriptor of the segment its row lives in.  Still buffer loads
      // (a global_load ... lds anywhere in the kernel counts as a possible FLAT access to LDS, after which the
      // compiler waits for ALL outstanding LDS reads in front of every MFMA instead of counting them).
      const char* b1 = colp + (long)k0 * st;  // row k0 of the first segment, of the second: (rows >= k_split only)
      const char* b2 = b1 + d2;
      const __amdgpu_buffer_rsrc_t rs1 = __builtin_amdgcn_make_buffer_rsrc((void*)b1, 0, 0x7fffffff, 0x00020000);
      const __amdgpu_buffer_rsrc_t rs2 = __builtin_amdgcn_make_buffer_rsrc((void*)b2, 0, 0x7fffffff, 0x00020000);
#pragma unroll
      for (int j = 0; j < LOADS; ++j) {
        const int row = min(k0 + 4 * w + lr + 4 * NW * j, ke - 1);
        const unsigned voff = (unsigned)(row - k0) * (unsigned)st + (unsigned)(chunk * 16);
        if (row < k_split)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs1, LDS_PTR(void, dst + j * NW * group), 16, voff, 0, 0, 0);
        else
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs2, LDS_PTR(void, dst + j * NW * group), 16, voff, 0, 0, 0);
      }
    }
  };

  // The first tile (the LAST one of the key range, see below) is requested before q is loaded and normalised, so that
  // the two latencies overlap: it matters where a workgroup sees few tiles (the text cross attention).
  const int n_tiles = (ke - ks + BN - 1) / BN;
  const int last = n_tiles - 1;
  issue_mat(ks + last * BN, sK0, false);
  issue_mat(ks + last * BN, sV0, true);

  // ---- Q fragments (B operand of S^T = K Q^T): lane (n, g) holds Q[row 16 qb + n][32 kk + 8 g .. +8] ----
  bf16x8 qf[QB][4];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int qr = min(row0 + 16 * qb + n, qe - 1);
    const char* qp = a.q + row_offset(a, qr, a.qs_t, a.qs_b) + (long)wi.h * a.qs_h + g * 16;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) qf[qb][kk] = *(const bf16x8*)(qp + kk * 64);
  }
  if constexpr (QMODE == Q_SCALE) {
    const float cs = a.scale_log2;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int e = 0; e < 8; ++e) qf[qb][kk][e] = (__bf16)((float)qf[qb][kk][e] * cs);
  }
  if (QMODE == Q_NORM || (QMODE == Q_EITHER && a.q_norm_gamma)) {
    // q holds the raw projection: per-(token, head) norm over the 128 features in fp32, times the softmax scale,
    // one rounding to bf16.  A row's features are spread over the four lanes (n, 0..3): 32 each, feature
    // 32 kk + 8 g + e in fragment kk, element e.
    const float inv_d = 1.f / 128.f;
    float mean[QB], rstd[QB];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      float sum = 0.f;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int e = 0; e < 8; ++e) sum += (float)qf[qb][kk][e];
      sum += __shfl_xor(sum, 16);
      sum += __shfl_xor(sum, 32);
      mean[qb] = a.q_norm_kind == 0 ? sum * inv_d : 0.f;  // (RMS form: no centring)
      float sq = 0.f;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float d = (float)qf[qb][kk][e] - mean[qb];
          sq += d * d;
        }
      sq += __shfl_xor(sq, 16);
      sq += __shfl_xor(sq, 32);
      rstd[qb] = __builtin_amdgcn_rsqf(sq * inv_d + a.q_norm_eps) * a.scale_log2;
    }
    // (one fragment index at a time, so that the parameters of one fragment are all that is in registers)
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      __builtin_amdgcn_sched_barrier(0);
      const f32x4* gp = (const f32x4*)(a.q_norm_gamma + 32 * kk + 8 * g);
      const f32x4 g0 = gp[0], g1 = gp[1];
      f32x4 b0 = {0.f, 0.f, 0.f, 0.f}, b1 = b0;
      if (a.q_norm_beta) {
        const f32x4* bp = (const f32x4*)(a.q_norm_beta + 32 * kk + 8 * g);
        b0 = bp[0];
        b1 = bp[1];
      }
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float gm = (e < 4 ? g0[e & 3] : g1[e & 3]) + 1.f;
          const float bt = (e < 4 ? b0[e & 3] : b1[e & 3]) * a.scale_log2;
          qf[qb][kk][e] = (__bf16)(((float)qf[qb][kk][e] - mean[qb]) * rstd[qb] * gm + bt);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
  }

  // ---- per-lane LDS read bases ----
  // K as A operand: row 16 kb + n, 16-byte chunk 4 kk + g, kept at (4 kk + g) ^ (n & 3) = 4 kk + (g ^ (n & 3)) of row
  // n & 3 of group 4 kb + n / 4: everything but the lane's own part is a constant offset of the read.  The 16 lanes
  // of one g touch four groups (64 bytes apart in bank terms) x four chunks: all 64 banks once.
  const int base_k = (n >> 2) * K_GROUP + (n & 3) * ROW_BYTES + ((g ^ (n & 3)) << 4);
  // V^T through the transposing read: the 16-lane group g serves key rows 4 g + r4 (r4 = (l % 16) / 4) of a 16-key
  // block, i.e. row r4 of group g (+ 4 per key block); lane 4 r4 + c4 of the group points at the four features
  // 16 db + 4 c4 .. +3 of its row, and receives the four rows' values of feature 16 db + l % 16.  Those 32 bytes of
  // the row are 32-byte slot db, kept at db ^ r4 = 4 (db / 4) + ((db % 4) ^ r4): one v_xor per value of db % 4,
  // the rest constant offsets.  Half a wave touches two groups (128 bytes apart in bank terms) x four slots x 32 bytes.
  const int r4 = n >> 2, c4 = n & 3;
  const int base_v = g * V_GROUP + r4 * ROW_BYTES + (r4 << 5) + (c4 << 3);

  f32x4v o_acc[8][QB];  // [d block][query block]; zeroed below, right ahead of the first tile
  float l_run[QB] = {};  // this lane's share of the row sums, per query block
  const bool wave_on = row0 < qe;
  const f32x4v zero4 = {0.f, 0.f, 0.f, 0.f};

  // One 64-key tile for this wave.  The 32 operand fragments of a tile are consumed in this order:
  //   half t = 0, 1:  K(t, kb = 0..1, kk = 0..3)  [scores of 32 keys x 64 queries]   then   V^T(t, db = 0, 4, 1, 5,
  //   2, 6, 3, 7: the two of a pair share their address)
  // each fragment feeding four MFMAs (the query blocks); fragment o is requested RD fragments ahead of its use.
  auto compute_tile = [&](const unsigned char* Kt, const unsigned char* Vt, int k0, auto ragged) __attribute__((always_inline)) {
    auto read_op = [&](auto oc) __attribute__((always_inline)) -> bf16x8 {
      constexpr int o = decltype(oc)::value;
      constexpr int t = o >> 4, j = o & 15;
      if constexpr (j < 8)
        return read_k<2 * t + (j >> 2), (j & 3)>(Kt, base_k);
      else
        return read_v<t, v_block(j - 8)>(Vt, base_v, k0);
    };
    constexpr int RD = RING;
    bf16x8 ring[RD];
    static_for<0, RD>([&](auto oc) __attribute__((always_inline)) { ring[decltype(oc)::value] = read_op(oc); });
    __builtin_amdgcn_sched_barrier(0);

    f32x4v sc[2][QB];  // scores of the current half: [key block][query block]
    u32x4 pf[QB];     // their probabilities as the B operand of the PV MFMAs, per query block
    auto consume = [&](auto oc) __attribute__((always_inline)) {
      constexpr int o = decltype(oc)::value;
      constexpr int t = o >> 4, j = o & 15;
      // ---- softmax of half t (32 keys x 64 queries: 32 values per lane, one query per lane and query block), one
      // (key block, query block) piece at a time: four exponentials, their sum, two packed pairs of the P operand.
      // (Keys past the end of the range need nothing here: their scores start from a large negative value, see below.)
      auto soft = [&](auto kc, auto qc) __attribute__((always_inline)) {
        constexpr int kb = decltype(kc)::value, qb = decltype(qc)::value;
        // Row sums in fp32 by plain additions on the unrounded values (rounding to bf16 is unbiased, so this is as
        // good a denominator; dot instructions would hold the matrix pipe up)
        const float c = CHECK ? a.scale_log2 : 1.f;
        const float p0 = __builtin_amdgcn_exp2f(sc[kb][qb][0] * c), p1 = __builtin_amdgcn_exp2f(sc[kb][qb][1] * c);
        const float p2 = __builtin_amdgcn_exp2f(sc[kb][qb][2] * c), p3 = __builtin_amdgcn_exp2f(sc[kb][qb][3] * c);
        l_run[qb] += (p0 + p1) + (p2 + p3);
        pf[qb][2 * kb] = pack_bf16x2(p0, p1);
        pf[qb][2 * kb + 1] = pack_bf16x2(p2, p3);
      };
      if constexpr (j == 8) {
        static_for<0, QB>([&](auto qc) __attribute__((always_inline)) {
          soft(std::integral_constant<int, 0>{}, qc);
          soft(std::integral_constant<int, 1>{}, qc);
        });
        __builtin_amdgcn_sched_barrier(0);
        static_for<0, RD>([&](auto pc) __attribute__((always_inline)) {
          constexpr int nf = 16 * t + 8 + decltype(pc)::value;
          ring[nf % RD] = read_op(std::integral_constant<int, nf>{});
        });
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (j < 8) {
        // scores: S^T[key][q] += K[key][32 kk ..] Q[q][32 kk ..]
        constexpr int kb = j >> 2, kk = j & 3;
        // The accumulators of a key block start from 0.  In the ragged copy of the body, keys past the end of the
        // range (whose LDS rows hold copies of the last valid key: the loader clamps) start from -1e4 instead: their
        // scores stay far below any real one (|score| <= 64), 2^score is exactly 0, and neither the row sums nor
        // the P operand see them.  (CHECK multiplies the scores by the caller's scale afterwards: -inf there.)  Register r of the lanes of group g is key 16 kb + 4 g + r of the half.
        f32x4v c0 = zero4;
        if constexpr (decltype(ragged)::value && kk == 0) {
          const int left = ke - (k0 + 32 * t) - 16 * kb - 4 * (l >> 4);  // valid keys from this lane's first one on
#pragma unroll
          for (int r = 0; r < 4; ++r) c0[r] = r < left ? 0.f : (CHECK ? -__builtin_inff() : -1.0e4f);
        }
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
          sc[kb][qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ring[o % RD], qf[qb][kk], kk == 0 ? c0 : sc[kb][qb], 0, 0, 0);
      } else {
        // O^T[d][q] += V^T[d][key] P^T[key][q]
        constexpr int db = v_block(j - 8);
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
          o_acc[db][qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ring[o % RD], __builtin_bit_cast(bf16x8, pf[qb]), o_acc[db][qb], 0, 0, 0);
      }
      // refill the slot just consumed with the fragment RD ahead; the first RD V^T fragments of a half are requested
      // right after the softmax instead (they would occupy registers across it)
      if constexpr (o + RD < 32) {
        constexpr int nj = (o + RD) & 15;
        if constexpr (!(nj >= 8 && nj < 8 + RD)) ring[o % RD] = read_op(std::integral_constant<int, o + RD>{});
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    static_for<0, 16>(consume);
    // (the ragged tile: a second half without a valid key has nothing to add.  Short key ranges, the text cross
    // attention with its dozen tiles per workgroup, are where this is noticeable.)
    if (!decltype(ragged)::value || ke - k0 > 32) static_for<16, 32>(consume);
  };

  // Tile order: the LAST tile of the key range first (it may hold the ragged end, so it runs the copy of the tile
  // body that masks the tail; the order of keys is immaterial to a softmax), then tiles 0 .. n_tiles-2 with the
  // mask-free body, two per loop iteration so that every LDS slot is named statically.  Tile `last` uses slot
  // pair 0, tile j slot pair (j + 1) & 1.
  const std::integral_constant<int, 0> slot0;
  const std::integral_constant<int, 1> slot1;
  // The accumulators start from zeros the compiler cannot see through: left to fold them into the first tile's
  // MFMAs it allocates that tile's registers differently from the steady-state body and spills two accumulators
  // there, a round trip to scratch memory for every workgroup.  (Here, behind the q fragments, so that the 128
  // registers are not held while q is loaded and normalised: the statement below pins the finished q fragments
  // ahead of them, or the compiler sinks the norm arithmetic to its first use, behind the zeros.)
  if constexpr (QB == 2)
    asm volatile("" ::"v"(qf[0][0]), "v"(qf[0][1]), "v"(qf[0][2]), "v"(qf[0][3]), "v"(qf[1][0]), "v"(qf[1][1]), "v"(qf[1][2]), "v"(qf[1][3]));
  if constexpr (QB == 4)
    asm volatile("" ::"v"(qf[0][0]), "v"(qf[0][1]), "v"(qf[0][2]), "v"(qf[0][3]), "v"(qf[1][0]), "v"(qf[1][1]), "v"(qf[1][2]),
               "v"(qf[1][3]), "v"(qf[2][0]), "v"(qf[2][1]), "v"(qf[2][2]), "v"(qf[2][3]), "v"(qf[3][0]), "v"(qf[3][1]),
               "v"(qf[3][2]), "v"(qf[3][3]));
#pragma unroll
  for (int db = 0; db < 8; ++db)
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      o_acc[db][qb] = f32x4v{0.f, 0.f, 0.f, 0.f};
      asm volatile("" : "+v"(o_acc[db][qb]));
    }
  // one tile: wait for it, request the next one (tile `nxt` of the range, if any) into the other slot pair, compute
  auto step = [&](int cur, int nxt, auto sc_, auto ragged) __attribute__((always_inline)) {
    constexpr int B = decltype(sc_)::value;
    wait_vmcnt<0>();
    __syncthreads();  // the tile landed in everybody's view; the other slot pair is free
    if (nxt < last) {
      issue_mat(ks + nxt * BN, B ? sK0 : sK1, false);
      issue_mat(ks + nxt * BN, B ? sV0 : sV1, true);
    }
    if (!wave_on) return;
    compute_tile(B ? sK1 : sK0, B ? sV1 : sV0, ks + cur * BN, ragged);
  };
  step(last, 0, slot0, std::true_type{});
  int end = last;
  if constexpr (CHECK) {
    // Inputs with large scores throughout show it in the first tile: no need to go on (a sum that is too small so far
    // may still grow; an overflow is final).
    bool over = false;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) over |= !(l_run[qb] <= SUM_MAX);
    if (wave_on && over) s_over = 1;
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(s_over) != 0) {
      end = 0;
      wait_vmcnt<0>();  // (the next tile is on its way into LDS)
    }
  }
  int j = 0;
  for (; j + 1 < end; j += 2) {
    step(j, j + 1, slot1, std::false_type{});
    step(j + 1, j + 2, slot0, std::false_type{});
  }
  if (j < end) step(j, j + 1, slot1, std::false_type{});

  // ---- a piece of an item: accumulators and row sums as they are, one contiguous 1 KB per instruction ----
  if (sp.out) {
    if (!wave_on) return;
    f32x4v* const dst = (f32x4v*)sp.out + w * 2048 + l;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      float s = l_run[qb];
      s += __shfl_xor(s, 16);
      s += __shfl_xor(s, 32);
      if (CHECK && end != last) s = __builtin_nanf("");
      if (g == 0) sp.out[256 * 128 + 64 * w + 16 * qb + n] = s;
#pragma unroll
      for (int db = 0; db < 8; ++db) dst[(4 * db + qb) * 64] = o_acc[db][qb];
    }
    return;
  }

  // ---- epilogue: normalise, transpose through LDS, store whole rows ----
  __syncthreads();  // every wave is done with the tile slots: wave w takes slot w as its staging area of 256 bytes a row
  if (!wave_on) {
    if (CHECK && l == 0) a.verdict[4 * (long)wi.item + w] = 0;
    return;
  }
  unsigned char* const stage = w == 0 ? sK0 : w == 1 ? sV0 : w == 2 ? sK1 : sV1;
  int lane_e = l;
  asm volatile("" : "+v"(lane_e));
  const int ne = lane_e & 15, ge = lane_e >> 4;
  bool bad = false;
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    float s = l_run[qb];
    s += __shfl_xor(s, 16);
    s += __shfl_xor(s, 32);
    if constexpr (CHECK) {
      float fine = 0.f;  // (NaN once an accumulator is not finite)
#pragma unroll
      for (int db = 0; db < 8; ++db)
#pragma unroll
        for (int r = 0; r < 4; ++r) fine = __builtin_fmaf(o_acc[db][qb][r], 0.f, fine);
      bad |= end != last || !(s >= SUM_MIN && s <= SUM_MAX) || fine != fine;
    }
    const float inv = 1.f / s;
    // lane (ne, ge) holds O[row 16 qb + ne][d = 16 db + 4 ge + r]: 8 bytes of bf16 at byte 32 db + 8 ge of the row,
    // i.e. half (ge & 1) of 16-byte chunk 2 db + ge / 2, kept at chunk ^ (row & 15) = chunk ^ ne
    unsigned char* const rowp = stage + (16 * qb + ne) * ROW_BYTES + ((ge & 1) << 3);
#pragma unroll
    for (int db = 0; db < 8; ++db) {
      const u32x2 v = {pack_bf16x2(o_acc[db][qb][0] * inv, o_acc[db][qb][1] * inv),
                       pack_bf16x2(o_acc[db][qb][2] * inv, o_acc[db][qb][3] * inv)};
      *LDS_PTR(u32x2, rowp + (((2 * db + (ge >> 1)) ^ ne) << 4)) = v;
    }
    const int q_row = row0 + 16 * qb + ne;
    if (a.lse && ge == 0 && q_row < qe)
      a.lse[(long)wi.h * a.total_q + q_row] = __builtin_amdgcn_logf(s) * 0.6931471805599453f;
  }
  if constexpr (CHECK) {
    const bool any = __builtin_amdgcn_ballot_w64(bad) != 0;
    if (lane_e == 0) a.verdict[4 * (long)wi.item + w] = any ? 1 : 0;
  }
  // (the staging area is this wave's own: its LDS operations complete in order, no workgroup barrier is needed)
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // 16 lanes x 16 bytes = one row; the wave stores four rows per instruction
#pragma unroll
  for (int it = 0; it < 4 * QB; ++it) {
    const int r = 4 * it + ge;
    const u32x4 v = *LDS_PTR(const u32x4, stage + r * ROW_BYTES + ((ne ^ (r & 15)) << 4));
    const int q_row = row0 + r;
    if (q_row < qe) *(u32x4*)(a.out + row_offset(a, q_row, a.os_t, a.os_b) + wi.o_head + 16 * ne) = v;
  }
