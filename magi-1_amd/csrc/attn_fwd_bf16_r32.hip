// Range attention forward, bf16, 32 query rows per wavefront on v_mfma_f32_16x16x32_bf16, three workgroups of 128 rows per CU, for gfx950
// (MI355X): the online softmax on unscaled q, and the softmax of bounded scores without a running maximum.
//
// 64-key tiles, two K slots and one V slot (three of them fit a CU's LDS) filled by direct global->LDS loads.  The MFMA shape, its operand
// layouts and the layout of the tiles in LDS are those of attn_fwd_bf16_x16.hip (there: why that shape, and the reads' banks), with two
// query blocks of 16 per wavefront; without a running maximum a row's bits are the same.  160 to 164 registers.
// What bounds it: per tile and wavefront the matrix pipe has 1024 cycles of work, the LDS 32 KB of operand reads, the vector pipe 32
// exponentials and 60 to 100 other instructions, about as long each; long launches run at the power limit.
//   Online softmax, in launches of more than a round: the 16x16x32 shape takes less energy per FLOP, 9360 rows x 2 chunks x 24 heads over
// 28080 and 37440 keys 6604 us on 32x32x16 (attn_fwd_bf16.hip) and 6407 so (1.18 PFLOP/s); whole rows go out through LDS, 16 lanes a row:
// 74880 x 24 rows over 20 keys, which is mostly the way of q and out, 223 -> 202 us, and 174 with the first tile requested ahead of q.
//   Bounded scores: 64 rows per wavefront read half as much from LDS and win in full launches (attn_fwd_bf16_x16.hip); this form where its
// 128-row workgroups are one round, three per CU, and 256-row ones a partly empty round (r32_plan in api.cpp): 2700 rows x 24 heads over
// 2700 keys 125 -> 107 us, four ranges of 792 rows over 1584 to 3960 138 -> 114.
//
// Shared keys (SHARE).  A launch of few items leaves most of the chip idle: 24 items over 127 tiles take 127 tiles in a row, 181 us.
// Their keys are cut in pieces of a.share_tiles tiles, a workgroup each; a piece leaves unnormalised accumulators, row sums
// and row maxima in fp32 (65 KB), a second launch brings them to a common maximum and adds them up in the order of the keys: 41 us.
// The grid has the pieces of the longest range for every item: the surplus ones of shorter ranges return at once.  An item of one piece
// is written right away.  Relative error against float64, pieces over whole: 0.95 to 0.99, 0.97 on average (online, 24 drawn sizes).
#include "attn_bf16_tiles.h"

namespace magi {
namespace {

// The maxima of two values over the four lanes n, n + 16, n + 32, n + 48 of a query, in every one of them.  The first exchange
// serves both values (the lower half of the wave then works on a, the upper on b), the last one hands both to everybody.
__device__ __forceinline__ void quad_max2(float& a, float& b) {
  asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1\n\tv_max_f32 %0, %0, %1\n\tv_mov_b32 %1, %0\n\ts_nop 1\n\t"
      "v_permlane16_swap_b32 %0, %1\n\ts_nop 1\n\tv_max_f32 %0, %0, %1\n\tv_mov_b32 %1, %0\n\ts_nop 1\n\t"
      "v_permlane32_swap_b32 %0, %1\n\ts_nop 1"
      : "+v"(a), "+v"(b));
}

// What q holds, and what is known about the scores.  ONLINE: unscaled bf16 q, nothing: running maximum, scores scaled in fp32.  The others
// as in attn_fwd_bf16_x16.hip, scores bounded, no maximum: AS_IS, q carries the scale; NORM, the raw projection; SCALE, unscaled.
constexpr int AS_IS = 0, NORM = 1, SCALE = 2, ONLINE = 3;
// SHARE: the keys of an item are shared by several workgroups, a.share_tiles tiles each (share_plan and r32_plan in api.cpp).
template <int QMODE, bool SHARE>
__global__ __launch_bounds__(256, 3) void attn_fwd_bf16_r32_kernel(const AttnKernArgs a) {
  constexpr bool MAX = QMODE == ONLINE;
  constexpr int QB = 2, NW = 4, WROWS = 16 * QB, BM = WROWS * NW;
  constexpr int LOADS = BN / (4 * NW);  // direct loads per wave per matrix per tile (4 rows each)
  constexpr int RD = 4;                 // operand fragments in flight between LDS and the MFMAs
  __shared__ __attribute__((aligned(1024))) unsigned char sK0[K_TILE_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char sK1[K_TILE_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char sV[V_TILE_BYTES];
  __shared__ int s_sel[LOCATE_WORDS];

  if (gate_closed(a)) return;
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63, n = l & 15, g = l >> 4;

  // ---- which piece of work is this workgroup? ----
  unsigned block = blockIdx.x, piece = 0;
  if constexpr (SHARE) {  // (the first pieces of all items, then the second ones, ...)
    const unsigned pos = block >> 3, xcd = block & 7u;
    piece = pos / a.per_xcd;
    block = (pos - piece * a.per_xcd) << 3 | xcd;
  }
  const WorkItem wi = locate_work(a, BM, tid, s_sel, block);
  if (!wi.valid) return;
  const int qe = wi.qe, row0 = wi.q0 + WROWS * w;  // first row of this wave
  int ks = wi.ks, ke = wi.ke;
  if (ke <= ks) {
    if (piece == 0 && row0 + (l & 31) < qe) store_empty_row(a, wi, row0 + (l & 31), l >> 5);
    return;
  }
  float* part = nullptr;
  if constexpr (SHARE) {
    // (the last piece takes what is left: ranges may be longer than the max_seqlen_k that the pieces were planned with; counted from
    // the range's first key, unsigned: a stated max_seqlen_k of up to 2^31 - 1 puts pieces behind the last key that an int could name)
    const unsigned keys = (unsigned)(ke - ks), per = a.share_tiles * BN, first = piece * per;
    if (first >= keys) return;
    const unsigned end = piece + 1 < a.share_pieces ? min(first + per, keys) : keys;
    if (piece != 0 || end < keys) part = a.partial + ((long)block * a.share_pieces + piece) * ONLINE_PARTIAL_FLOATS;
    ke = ks + (int)end;
    ks += (int)first;
  }

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
    int lane = l;
    asm volatile("" : "+v"(lane));
    const int lr = lane >> 4, sl = lane & 15;
    const int chunk = is_v ? (sl ^ (lr << 1)) : (sl ^ lr);
    const bool interior = (k0 + BN <= ke) && (k0 + BN <= k_split || k0 >= k_split);
    if (interior) {
      const char* b = colp + (long)k0 * st + (k0 >= k_split ? d2 : 0);
      const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)b, 0, 0x7fffffff, 0x00020000);
      const unsigned voff = (unsigned)(4 * w + lr) * (unsigned)st + (unsigned)(chunk * 16);
#pragma unroll
      for (int j = 0; j < LOADS; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, LDS_PTR(void, dst + j * NW * group), 16, voff,
                                                 (int)((unsigned)(4 * NW * j) * (unsigned)st), 0, 0);
    } else {
      const char* b1 = colp + (long)k0 * st;
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

  // The LAST tile of the range goes first: it may be ragged, so it has a copy of the tile's code of its own, which also knows that there
  // is no maximum yet, and the others' code has neither.  It is on its way into LDS, V too, while q is loaded.  (The text cross attention,
  // a few tiles: 93600 x 24 rows 511 -> 509 us, 42196 x 24 over 115 keys 137 -> 133, 74880 x 24 over 64 keys 194 -> 187, over 20 191 -> 174.)
  const int last = (ke - ks - 1) / BN;
  issue_mat(ks + last * BN, sK0, false);
  issue_mat(ks + last * BN, sV, true);

  // ---- Q fragments (B operand of S^T = K Q^T): lane (n, g) holds Q[row 16 qb + n][32 kk + 8 g .. +8] ----
  bf16x8 qf[QB][4];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int qr = min(row0 + 16 * qb + n, qe - 1);
    const char* qp = a.q + row_offset(a, qr, a.qs_t, a.qs_b) + (long)wi.h * a.qs_h + g * 16;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) qf[qb][kk] = *(const bf16x8*)(qp + kk * 64);
  }
  if constexpr (QMODE == SCALE) {
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int e = 0; e < 8; ++e) qf[qb][kk][e] = (__bf16)((float)qf[qb][kk][e] * a.scale_log2);
  }
  if constexpr (QMODE == NORM) norm_q<QB>(a, qf, g);

  const int base_k = (n >> 2) * K_GROUP + (n & 3) * ROW_BYTES + ((g ^ (n & 3)) << 4);
  const int r4 = n >> 2, c4 = n & 3;
  const int base_v = g * V_GROUP + r4 * ROW_BYTES + (r4 << 5) + (c4 << 3);

  f32x4v o_acc[8][QB];
#pragma unroll
  for (int db = 0; db < 8; ++db)
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) o_acc[db][qb] = f32x4v{0.f, 0.f, 0.f, 0.f};
  float l_run[QB] = {};                                        // this lane's share of the row sums, per query block
  float m_run[QB] = {-__builtin_inff(), -__builtin_inff()};  // running maxima of the raw scores
  const float c = a.scale_log2;
  const f32x4v zero4 = {0.f, 0.f, 0.f, 0.f};
  const f32x4v none4 = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff(), -__builtin_inff()};

  auto compute_tile = [&](const unsigned char* Kt, const unsigned char* Vt, int k0, auto first, auto before_pv) __attribute__((always_inline)) {
    constexpr bool FIRST = decltype(first)::value;
    // scores, S^T[key][q]: fragment o = (half t, kk, kb of the half), so that four accumulators are in turn
    auto read_kf = [&](auto oc) __attribute__((always_inline)) -> bf16x8 {
      constexpr int o = decltype(oc)::value;
      return read_k<2 * (o >> 3) + (o & 1), ((o >> 1) & 3)>(Kt, base_k);
    };
    auto read_vf = [&](auto oc) __attribute__((always_inline)) -> bf16x8 {
      constexpr int o = decltype(oc)::value;
      return read_v<(o >> 3), v_block(o & 7)>(Vt, base_v, k0);
    };
    bf16x8 ring[RD];
    f32x4v sc[4][QB];
    const bool half = FIRST && ke - k0 <= BN / 2;  // no key in the second half
    static_for<0, RD>([&](auto oc) __attribute__((always_inline)) { ring[decltype(oc)::value] = read_kf(oc); });
    __builtin_amdgcn_sched_barrier(0);
    auto scores = [&](auto oc) __attribute__((always_inline)) {
      constexpr int o = decltype(oc)::value;
      constexpr int kb = 2 * (o >> 3) + (o & 1), kk = (o >> 1) & 3;
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
        sc[kb][qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ring[o % RD], qf[qb][kk], kk == 0 ? zero4 : sc[kb][qb], 0, 0, 0);
      if constexpr (o + RD < 16) ring[o % RD] = read_kf(std::integral_constant<int, o + RD>{});
      __builtin_amdgcn_sched_barrier(0);
    };
    static_for<0, 8>(scores);
    if (!half) {
      static_for<8, 16>(scores);
    } else {
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) sc[2][qb] = sc[3][qb] = none4;
    }
    if (FIRST && k0 + BN > ke) {  // ragged: keys >= ke do not exist
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (k0 + 16 * kb + 4 * g + r >= ke) {
#pragma unroll
            for (int qb = 0; qb < QB; ++qb) sc[kb][qb][r] = -__builtin_inff();
          }
    }
    // softmax: lane (n, g) holds keys 16 kb + 4 g + r of query n of each block
    if constexpr (MAX) {
      float mx[QB];
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        float m = max3(sc[0][qb][0], sc[0][qb][1], sc[0][qb][2]);
        m = max3(m, sc[0][qb][3], sc[1][qb][0]);
        m = max3(m, sc[1][qb][1], sc[1][qb][2]);
        m = max3(m, sc[1][qb][3], sc[2][qb][0]);
        m = max3(m, sc[2][qb][1], sc[2][qb][2]);
        m = max3(m, sc[2][qb][3], sc[3][qb][0]);
        m = max3(m, sc[3][qb][1], sc[3][qb][2]);
        mx[qb] = fmaxf(m, sc[3][qb][3]);
      }
      quad_max2(mx[0], mx[1]);
      const float m0 = fmaxf(m_run[0], mx[0]), m1 = fmaxf(m_run[1], mx[1]);
      if constexpr (FIRST) {
        m_run[0] = m0;
        m_run[1] = m1;
      } else if (__builtin_amdgcn_ballot_w64(m0 != m_run[0] || m1 != m_run[1]) != 0) {  // some row of this wave saw a new maximum
        const float a0 = __builtin_amdgcn_exp2f((m_run[0] - m0) * c), a1 = __builtin_amdgcn_exp2f((m_run[1] - m1) * c);
        m_run[0] = m0;
        m_run[1] = m1;
        l_run[0] *= a0;
        l_run[1] *= a1;
#pragma unroll
        for (int db = 0; db < 8; ++db) {
          o_acc[db][0] *= a0;
          o_acc[db][1] *= a1;
        }
      }
    }
    u32x4 pf[2][QB];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      const float mc = fmaxf(m_run[qb], -3.0e38f) * c;  // (a piece whose scores are all -inf so far adds zeros)
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        const float p0 = __builtin_amdgcn_exp2f(MAX ? sc[kb][qb][0] * c - mc : sc[kb][qb][0]), p1 = __builtin_amdgcn_exp2f(MAX ? sc[kb][qb][1] * c - mc : sc[kb][qb][1]);
        const float p2 = __builtin_amdgcn_exp2f(MAX ? sc[kb][qb][2] * c - mc : sc[kb][qb][2]), p3 = __builtin_amdgcn_exp2f(MAX ? sc[kb][qb][3] * c - mc : sc[kb][qb][3]);
        l_run[qb] += (p0 + p1) + (p2 + p3);
        pf[kb >> 1][qb][2 * (kb & 1)] = pack_bf16x2(p0, p1);
        pf[kb >> 1][qb][2 * (kb & 1) + 1] = pack_bf16x2(p2, p3);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    before_pv();
    // O^T[d][q] += V^T[d][key] P^T[key][q]
    static_for<0, RD>([&](auto oc) __attribute__((always_inline)) { ring[decltype(oc)::value] = read_vf(oc); });
    __builtin_amdgcn_sched_barrier(0);
    auto products = [&](auto oc) __attribute__((always_inline)) {
      constexpr int o = decltype(oc)::value;
      constexpr int db = v_block(o & 7);
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
        o_acc[db][qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ring[o % RD], __builtin_bit_cast(bf16x8, pf[o >> 3][qb]), o_acc[db][qb], 0, 0, 0);
      if constexpr (o + RD < 16) ring[o % RD] = read_vf(std::integral_constant<int, o + RD>{});
      __builtin_amdgcn_sched_barrier(0);
    };
    static_for<0, 8>(products);
    if (!half) static_for<8, 16>(products);
  };

  // one tile (`nxt`: the one behind it, if below `last`): the last one in K slot 0, then tile j in slot (j + 1) & 1
  auto step = [&](int cur, int nxt, auto bc, auto first) __attribute__((always_inline)) {
    constexpr int B = decltype(bc)::value;
    wait_vmcnt<0>();
    barrier_loads_in_flight();  // the K tile landed in everybody's view; the other K slot and the V slot are free
    if constexpr (!decltype(first)::value) issue_mat(ks + cur * BN, sV, true);
    if (nxt < last) issue_mat(ks + nxt * BN, B ? sK0 : sK1, false);
    compute_tile(B ? sK1 : sK0, sV, ks + cur * BN, first, [&]() __attribute__((always_inline)) {
      if (nxt < last)
        wait_vmcnt<LOADS>();  // the V tile landed, the next K tile stays in flight
      else
        wait_vmcnt<0>();
      barrier_loads_in_flight();
    });
  };
  const std::integral_constant<int, 0> slot0;
  const std::integral_constant<int, 1> slot1;
  step(last, 0, slot0, std::true_type{});
  for (int j = 0; j < last; j += 2) {
    step(j, j + 1, slot1, std::false_type{});
    if (j + 1 >= last) break;
    step(j + 1, j + 2, slot0, std::false_type{});
  }

  if (row0 >= qe) return;
  int lane_e = l;
  asm volatile("" : "+v"(lane_e));
  const int ne = lane_e & 15, ge = lane_e >> 4;
  float sum[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    sum[qb] = l_run[qb] + __shfl_xor(l_run[qb], 16);
    sum[qb] += __shfl_xor(sum[qb], 32);
  }
  // ---- a piece of an item: accumulators, row sums and maxima as they are, one contiguous 1 KB per instruction ----
  if (SHARE && part) {
    f32x4v* const dst = (f32x4v*)part + w * 1024 + lane_e;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      if (ge == 0) {
        part[128 * 128 + WROWS * w + 16 * qb + ne] = sum[qb];
        part[128 * 128 + 128 + WROWS * w + 16 * qb + ne] = MAX ? m_run[qb] * c : 0.f;
      }
#pragma unroll
      for (int db = 0; db < 8; ++db) dst[(2 * db + qb) * 64] = o_acc[db][qb];
    }
    return;
  }
  // ---- epilogue: normalise, transpose through LDS (behind the last tile's second barrier the K slots are free), whole rows ----
  unsigned char* const stage = (w < 2 ? sK0 : sK1) + (w & 1) * (WROWS * ROW_BYTES);
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const float inv = 1.f / sum[qb];
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
      a.lse[(long)wi.h * a.total_q + q_row] = ((MAX ? m_run[qb] * c : 0.f) + __builtin_amdgcn_logf(sum[qb])) * 0.6931471805599453f;
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
}

constexpr unsigned MERGE_SHARES = 4;
// The items of a SHARE launch that are in pieces: brings the pieces to a common maximum, adds them up in the order of the keys,
// normalises, writes the rows.  Four workgroups per item (query block, half of the features), on the item's XCD.
__global__ __launch_bounds__(256) void attn_fwd_bf16_r32_merge_kernel(const AttnKernArgs a) {
  constexpr unsigned SHARES = MERGE_SHARES;
  __shared__ int s_sel[LOCATE_WORDS];
  if (gate_closed(a)) return;
  const int tid = threadIdx.x, l = tid & 63, n = l & 15, g = l >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned share = (blockIdx.x >> 3) % SHARES, block = ((blockIdx.x >> 3) / SHARES << 3) | (blockIdx.x & 7u);
  const int qb = (int)(share >> 1), half = (int)(share & 1);
  const WorkItem wi = locate_work(a, 128, tid, s_sel, block);
  if (!wi.valid || wi.ke <= wi.ks) return;
  const int tiles = (wi.ke - wi.ks + BN - 1) / BN, pieces = (int)min(((unsigned)tiles + a.share_tiles - 1) / a.share_tiles, a.share_pieces);
  if (pieces < 2) return;
  const int q_row = wi.q0 + 32 * w + 16 * qb + n;
  if (wi.q0 + 32 * w >= wi.qe) return;  // (wavefronts without rows leave nothing)
  const float* const base = a.partial + (long)block * a.share_pieces * ONLINE_PARTIAL_FLOATS;
  const float* const stat = base + 128 * 128 + 32 * w + 16 * qb + n;
  float M = -__builtin_inff();
  for (int i = 0; i < pieces; ++i) M = fmaxf(M, stat[(long)i * ONLINE_PARTIAL_FLOATS + 128]);
  float s = 0.f;
  f32x4v o[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) o[d] = f32x4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
  for (int i = 0; i < pieces; ++i) {
    const float* const p = base + (long)i * ONLINE_PARTIAL_FLOATS;
    const float f = __builtin_amdgcn_exp2f(stat[(long)i * ONLINE_PARTIAL_FLOATS + 128] - M);
    const f32x4v* const src = (const f32x4v*)p + w * 1024 + l;
#pragma unroll
    for (int d = 0; d < 4; ++d) o[d] += src[(2 * (4 * half + d) + qb) * 64] * f;
    s += stat[(long)i * ONLINE_PARTIAL_FLOATS] * f;
  }
  if (q_row >= wi.qe) return;
  const float inv = 1.f / s;
  char* const op = a.out + row_offset(a, q_row, a.os_t, a.os_b) + wi.o_head + 128 * half + 8 * g;
#pragma unroll
  for (int d = 0; d < 4; ++d)
    *(u32x2*)(op + 32 * d) = u32x2{pack_bf16x2(o[d][0] * inv, o[d][1] * inv), pack_bf16x2(o[d][2] * inv, o[d][3] * inv)};
  if (a.lse && half == 0 && g == 0) a.lse[(long)wi.h * a.total_q + q_row] = (M + __builtin_amdgcn_logf(s)) * 0.6931471805599453f;
}

}  // namespace

namespace {
template <int QMODE>
void launch(const AttnKernArgs& a, hipStream_t stream) {
  if (a.share_pieces > 1) {
    hipLaunchKernelGGL((attn_fwd_bf16_r32_kernel<QMODE, true>), dim3(8u * a.per_xcd * a.share_pieces), dim3(256), 0, stream, a);
    AttnKernArgs m = a;
    m.flags &= ~ATTN_ZERO_GAPS;  // (the rows no range covers are clear by now)
    hipLaunchKernelGGL(attn_fwd_bf16_r32_merge_kernel, dim3(8u * a.per_xcd * MERGE_SHARES), dim3(256), 0, stream, m);
  } else {
    hipLaunchKernelGGL((attn_fwd_bf16_r32_kernel<QMODE, false>), dim3(8u * a.per_xcd), dim3(256), 0, stream, a);
  }
}
}  // namespace

hipError_t launch_attn_fwd_bf16_r32(const AttnKernArgs& a, hipStream_t stream) {
  if (!(a.flags & ATTN_BOUNDED))
    launch<ONLINE>(a, stream);
  else if (a.q_norm_gamma)
    launch<NORM>(a, stream);
  else if (a.flags & ATTN_SCALE_Q)
    launch<SCALE>(a, stream);
  else
    launch<AS_IS>(a, stream);
  return hipGetLastError();
}

}  // namespace magi
