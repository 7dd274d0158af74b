// The text cross attention beside something else in a launch (attn_fwd_fp8_text.hip, attn_text_merge.hip): little LDS, so that the
// workgroups around it keep their places.  128 rows a workgroup, 32 to a wavefront, on v_mfma_f32_16x16x32_bf16, scores bounded, q the raw
// projection; layouts and order of the keys are attn_fwd_bf16_r32.hip's, so the same bits, but the keys come in tiles of 32, K and V double
// buffered: 36 KB.
#pragma once
#include "attn_bf16_tiles.h"

namespace magi {
namespace {

constexpr int HN = 32;  // keys of a text tile
constexpr int HK_BYTES = (HN / 4) * K_GROUP, HV_BYTES = (HN / 4) * V_GROUP;

// sK0, sK1: HK_BYTES; sV0, sV1: HV_BYTES
__device__ __forceinline__ void text_rows(const AttnKernArgs& a, unsigned block, unsigned char* sK0, unsigned char* sV0, unsigned char* sK1,
                                          unsigned char* sV1, int* s_sel) {
  constexpr int QB = 2, NW = 4, WROWS = 16 * QB, BM = WROWS * NW;
  constexpr int LOADS = HN / (4 * NW);  // direct loads per wave per matrix per tile (4 rows each)
  constexpr int RD = 4;                 // operand fragments in flight between LDS and the MFMAs
  static_assert(HK_BYTES >= WROWS * ROW_BYTES, "a wavefront's rows of out in a slot");
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63, n = l & 15, g = l >> 4;
  const WorkItem wi = locate_work(a, BM, tid, s_sel, block);
  if (!wi.valid) return;
  const int qe = wi.qe, row0 = wi.q0 + WROWS * w, ks = wi.ks, ke = wi.ke;
  if (ke <= ks) {
    if (row0 + (l & 31) < qe) store_empty_row(a, wi, row0 + (l & 31), l >> 5);
    return;
  }
  const long ks_t = a.ks_t, vs_t = a.vs_t;
  const int k_split = a.k_split;
  const long k2_delta = a.k2 ? (a.k2 - a.k) - (long)k_split * ks_t : 0;
  const long v2_delta = a.v2 ? (a.v2 - a.v) - (long)k_split * vs_t : 0;
  const char* const kcolp = a.k + (long)wi.kvh * a.ks_h;
  const char* const vcolp = a.v + (long)wi.kvh * a.vs_h;

  auto issue_mat = [&](int k0, unsigned char* tile_base, bool is_v) __attribute__((always_inline)) {
    const int group = is_v ? V_GROUP : K_GROUP;
    unsigned char* const dst = tile_base + w * group;
    const long st = is_v ? vs_t : ks_t;
    const char* const b1 = (is_v ? vcolp : kcolp) + (long)k0 * st;  // row k0 of the first segment, of the second: (rows >= k_split only)
    const char* const b2 = b1 + (is_v ? v2_delta : k2_delta);
    int lane = l;
    asm volatile("" : "+v"(lane));
    const int lr = lane >> 4, sl = lane & 15;
    const int chunk = is_v ? (sl ^ (lr << 1)) : (sl ^ lr);
    const __amdgpu_buffer_rsrc_t rs1 = __builtin_amdgcn_make_buffer_rsrc((void*)b1, 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t rs2 = __builtin_amdgcn_make_buffer_rsrc((void*)b2, 0, 0x7fffffff, 0x00020000);
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {  // (rows past the last valid key: copies of it)
      const int row = min(k0 + 4 * w + lr + 4 * NW * j, ke - 1);
      const unsigned voff = (unsigned)(row - k0) * (unsigned)st + (unsigned)(chunk * 16);
      if (row < k_split)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs1, LDS_PTR(void, dst + j * NW * group), 16, voff, 0, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs2, LDS_PTR(void, dst + j * NW * group), 16, voff, 0, 0, 0);
    }
  };

  // The order of the keys of attn_fwd_bf16_r32.hip: the last 64 of a walk in steps of 64 (or what there is of them), then the others.
  const int last = (ke - ks - 1) / BN, at_end = ke - ks - last * BN > HN ? 2 : 1, tiles = 2 * last + at_end;
  auto key_of = [&](int t) { return ks + HN * (t < at_end ? 2 * last + t : t - at_end); };
  issue_mat(key_of(0), sK0, false);
  issue_mat(key_of(0), sV0, true);

  // ---- Q fragments (B operand of S^T = K Q^T): lane (n, g) holds Q[row 16 qb + n][32 kk + 8 g .. +8] ----
  bf16x8 qf[QB][4];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int qr = min(row0 + 16 * qb + n, qe - 1);
    const char* qp = a.q + row_offset(a, qr, a.qs_t, a.qs_b) + (long)wi.h * a.qs_h + g * 16;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) qf[qb][kk] = *(const bf16x8*)(qp + kk * 64);
  }
  norm_q<QB>(a, qf, g);

  const int base_k = (n >> 2) * K_GROUP + (n & 3) * ROW_BYTES + ((g ^ (n & 3)) << 4);
  const int r4 = n >> 2, c4 = n & 3;
  const int base_v = g * V_GROUP + r4 * ROW_BYTES + (r4 << 5) + (c4 << 3);
  f32x4v o_acc[8][QB];
#pragma unroll
  for (int db = 0; db < 8; ++db)
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) o_acc[db][qb] = f32x4v{0.f, 0.f, 0.f, 0.f};
  float l_run[QB] = {};  // this lane's share of the row sums, per query block
  const f32x4v zero4 = {0.f, 0.f, 0.f, 0.f};

  auto compute = [&](const unsigned char* Kt, const unsigned char* Vt, int k0) __attribute__((always_inline)) {
    auto read_kf = [&](auto oc) __attribute__((always_inline)) -> bf16x8 {
      constexpr int o = decltype(oc)::value;
      return read_k<(o & 1), (o >> 1)>(Kt, base_k);
    };
    auto read_vf = [&](auto oc) __attribute__((always_inline)) -> bf16x8 {
      return read_v<0, v_block(decltype(oc)::value)>(Vt, base_v, k0);
    };
    bf16x8 ring[RD];
    f32x4v sc[2][QB];
    static_for<0, RD>([&](auto oc) __attribute__((always_inline)) { ring[decltype(oc)::value] = read_kf(oc); });
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, 8>([&](auto oc) __attribute__((always_inline)) {
      constexpr int o = decltype(oc)::value;
      constexpr int kb = o & 1, kk = o >> 1;
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
        sc[kb][qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ring[o % RD], qf[qb][kk], kk == 0 ? zero4 : sc[kb][qb], 0, 0, 0);
      if constexpr (o + RD < 8) ring[o % RD] = read_kf(std::integral_constant<int, o + RD>{});
      __builtin_amdgcn_sched_barrier(0);
    });
    if (k0 + HN > ke) {  // ragged: keys >= ke do not exist
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (k0 + 16 * kb + 4 * g + r >= ke) {
#pragma unroll
            for (int qb = 0; qb < QB; ++qb) sc[kb][qb][r] = -__builtin_inff();
          }
    }
    u32x4 pf[QB];  // lane (n, g) holds keys 16 kb + 4 g + r of query n of each block
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const float p0 = __builtin_amdgcn_exp2f(sc[kb][qb][0]), p1 = __builtin_amdgcn_exp2f(sc[kb][qb][1]);
        const float p2 = __builtin_amdgcn_exp2f(sc[kb][qb][2]), p3 = __builtin_amdgcn_exp2f(sc[kb][qb][3]);
        l_run[qb] += (p0 + p1) + (p2 + p3);
        pf[qb][2 * kb] = pack_bf16x2(p0, p1);
        pf[qb][2 * kb + 1] = pack_bf16x2(p2, p3);
      }
    __builtin_amdgcn_sched_barrier(0);
    // O^T[d][q] += V^T[d][key] P^T[key][q]
    static_for<0, RD>([&](auto oc) __attribute__((always_inline)) { ring[decltype(oc)::value] = read_vf(oc); });
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, 8>([&](auto oc) __attribute__((always_inline)) {
      constexpr int o = decltype(oc)::value;
      constexpr int db = v_block(o);
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
        o_acc[db][qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ring[o % RD], __builtin_bit_cast(bf16x8, pf[qb]), o_acc[db][qb], 0, 0, 0);
      if constexpr (o + RD < 8) ring[o % RD] = read_vf(std::integral_constant<int, o + RD>{});
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  // tile t in the slots of its parity; the tile behind it is on its way while it is worked on
  auto step = [&](int t, const unsigned char* Kt, const unsigned char* Vt, unsigned char* Kn, unsigned char* Vn) __attribute__((always_inline)) {
    wait_vmcnt<0>();
    barrier_loads_in_flight();  // the tile landed in everybody's view, the other slots are free
    if (t + 1 < tiles) {
      issue_mat(key_of(t + 1), Kn, false);
      issue_mat(key_of(t + 1), Vn, true);
    }
    compute(Kt, Vt, key_of(t));
  };
  for (int t = 0; t < tiles; t += 2) {
    step(t, sK0, sV0, sK1, sV1);
    if (t + 1 >= tiles) break;
    step(t + 1, sK1, sV1, sK0, sV0);
  }
  barrier_loads_in_flight();  // (every slot is free)

  if (row0 >= qe) return;
  // ---- epilogue: normalise, transpose through LDS, whole rows (as in attn_fwd_bf16_r32.hip) ----
  int lane_e = l;
  asm volatile("" : "+v"(lane_e));
  const int ne = lane_e & 15, ge = lane_e >> 4;
  unsigned char* const stage = w == 0 ? sK0 : w == 1 ? sV0 : w == 2 ? sK1 : sV1;
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    float sum = l_run[qb] + __shfl_xor(l_run[qb], 16);
    sum += __shfl_xor(sum, 32);
    const float inv = 1.f / sum;
    unsigned char* const rowp = stage + (16 * qb + ne) * ROW_BYTES + ((ge & 1) << 3);
#pragma unroll
    for (int db = 0; db < 8; ++db) {
      const u32x2 v = {pack_bf16x2(o_acc[db][qb][0] * inv, o_acc[db][qb][1] * inv), pack_bf16x2(o_acc[db][qb][2] * inv, o_acc[db][qb][3] * inv)};
      *LDS_PTR(u32x2, rowp + (((2 * db + (ge >> 1)) ^ ne) << 4)) = v;
    }
    const int q_row = row0 + 16 * qb + ne;
    if (a.lse && ge == 0 && q_row < qe) a.lse[(long)wi.h * a.total_q + q_row] = __builtin_amdgcn_logf(sum) * 0.6931471805599453f;
  }
  // (the staging area is this wave's own: its LDS operations complete in order, no workgroup barrier is needed)
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int it = 0; it < 4 * QB; ++it) {
    const int r = 4 * it + ge;
    const u32x4 v = *LDS_PTR(const u32x4, stage + r * ROW_BYTES + ((ne ^ (r & 15)) << 4));
    const int q_row = row0 + r;
    if (q_row < qe) *(u32x4*)(a.out + row_offset(a, q_row, a.os_t, a.os_b) + wi.o_head + 16 * ne) = v;
  }
}

}  // namespace
}  // namespace magi
