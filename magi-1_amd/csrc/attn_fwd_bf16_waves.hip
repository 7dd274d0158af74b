// Range attention forward, bf16, bounded scores, launches of a few rows: the wavefronts of a workgroup share the keys of 32 query rows, for
// gfx950 (MI355X).  One or two calls in a launch (a layer's core and text attention, which do not depend on each other).
//
// What bounds such launches is latency: 12 items of 128 rows over 480 keys are eight tiles in a row on twelve CUs, 14.3 us, while the rest
// of the chip waits, and the text attention behind it lives for 7.8 us of launch and trips to memory.  So: workgroups of 32 rows x four
// wavefronts (up to 1024 keys, and more than a workgroup per CU) or eight, each wavefront every fourth or eighth slab of 32 keys, with LDS slots
// of its own (no barriers in the loop); without a running maximum the wavefronts' accumulators and row sums simply add up, through LDS.
// The two calls in one launch 10.1 us.  MFMA shape, operand layouts and the layout of keys in LDS are those
// of attn_fwd_bf16_r32.hip.  A slab is fetched for 32 rows only, four times the bytes per row of a 128-row workgroup: 130 GB/s and CU, what
// direct loads hold, are 1 us per 256 keys, so this is for launches of about one workgroup per CU (waves_plan in api.cpp).
#include "attn_bf16_tiles.h"

namespace magi {
namespace {

constexpr int ROWS = 32, SLAB = 32, GROUPS = SLAB / 4;
constexpr int K_SLAB = GROUPS * K_GROUP, V_SLAB = GROUPS * V_GROUP;
constexpr int PART = ROWS * 128 * 4;  // a wavefront's accumulators in LDS, ahead of their sum
static_assert(PART <= 2 * K_SLAB && PART <= 2 * V_SLAB, "the accumulators of half of the wavefronts in each of the two arrays");

// WAVES: wavefronts of a workgroup.  a.waves of them, all or the first four of eight, work on an item: a row's bits depend on that number
// and not on what else is in the launch.
template <int WAVES>
__global__ __launch_bounds__(64 * WAVES, 2) void attn_fwd_bf16_waves_kernel(const AttnPairArgs) {
  __shared__ __attribute__((aligned(1024))) unsigned char sK[WAVES * K_SLAB];
  __shared__ __attribute__((aligned(1024))) unsigned char sV[WAVES * V_SLAB];
  __shared__ float s_sum[WAVES][ROWS];
  __shared__ int s_sel[LOCATE_WORDS];
  // (the arguments where they are: copied by value, both jobs' would be loaded and chosen between field by field)
  const AttnPairArgs& pair = *(const AttnPairArgs*)__builtin_amdgcn_kernarg_segment_ptr();

  // ---- which job, which 32 rows ----
  const unsigned pos = blockIdx.x >> 3, xcd = blockIdx.x & 7u, ahead = pair.job[0].per_xcd;
  const bool second = pos >= ahead;
  const AttnKernArgs& a = pair.job[second ? 1 : 0];
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63, n = l & 15, g = l >> 4;
  const WorkItem wi = locate_work(a, ROWS, tid, s_sel, (second ? pos - ahead : pos) << 3 | xcd);
  if (!wi.valid) return;
  const int qe = wi.qe, row0 = wi.q0, ks = wi.ks, ke = wi.ke;
  if (ke <= ks) {
    if (w == 0 && row0 + (l & 31) < qe) store_empty_row(a, wi, row0 + (l & 31), l >> 5);
    return;
  }
  const int waves = WAVES == 4 ? 4 : a.waves;
  const int slabs = (int)((unsigned)(ke - ks + SLAB - 1) / SLAB);

  const long ks_t = a.ks_t, vs_t = a.vs_t;
  const int k_split = a.k_split;
  const long k2_delta = a.k2 ? (a.k2 - a.k) - (long)k_split * ks_t : 0;
  const long v2_delta = a.v2 ? (a.v2 - a.v) - (long)k_split * vs_t : 0;
  const char* const kcolp = a.k + (long)wi.kvh * a.ks_h;
  const char* const vcolp = a.v + (long)wi.kvh * a.vs_h;
  unsigned char* const Kt = sK + w * K_SLAB;
  unsigned char* const Vt = sV + w * V_SLAB;

  // slab j into this wavefront's slot: a load fills four rows, lane l sits at row l / 16, slot l % 16 (see issue_mat of attn_fwd_bf16_r32.hip)
  auto issue = [&](int j, unsigned char* dst, bool is_v) __attribute__((always_inline)) {
    const int k0 = ks + j * SLAB, group = is_v ? V_GROUP : K_GROUP;
    const long st = is_v ? vs_t : ks_t;
    const char* const b1 = (is_v ? vcolp : kcolp) + (long)k0 * st;  // row k0 of the first segment, of the second: (rows >= k_split only)
    const char* const b2 = b1 + (is_v ? v2_delta : k2_delta);
    const int lr = l >> 4, sl = l & 15, chunk = is_v ? (sl ^ (lr << 1)) : (sl ^ lr);
    if (k0 + SLAB <= ke && (k0 + SLAB <= k_split || k0 >= k_split)) {
      const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(k0 >= k_split ? b2 : b1), 0, 0x7fffffff, 0x00020000);
      const unsigned voff = (unsigned)lr * (unsigned)st + (unsigned)(chunk * 16);
#pragma unroll
      for (int i = 0; i < GROUPS; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, LDS_PTR(void, dst + i * group), 16, voff, (int)((unsigned)(4 * i) * (unsigned)st), 0, 0);
    } else {  // the ragged end, or a slab in both key segments: rows clamped to the last key, each through the segment it lives in
      const __amdgpu_buffer_rsrc_t rs1 = __builtin_amdgcn_make_buffer_rsrc((void*)b1, 0, 0x7fffffff, 0x00020000);
      const __amdgpu_buffer_rsrc_t rs2 = __builtin_amdgcn_make_buffer_rsrc((void*)b2, 0, 0x7fffffff, 0x00020000);
#pragma unroll
      for (int i = 0; i < GROUPS; ++i) {
        const int row = min(k0 + lr + 4 * i, ke - 1);
        const unsigned voff = (unsigned)(row - k0) * (unsigned)st + (unsigned)(chunk * 16);
        if (row < k_split)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs1, LDS_PTR(void, dst + i * group), 16, voff, 0, 0, 0);
        else
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs2, LDS_PTR(void, dst + i * group), 16, voff, 0, 0, 0);
      }
    }
  };

  f32x4v o_acc[8][2];
#pragma unroll
  for (int db = 0; db < 8; ++db)
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) o_acc[db][qb] = f32x4v{0.f, 0.f, 0.f, 0.f};
  float l_run[2] = {0.f, 0.f};  // this lane's share of the row sums

  if (w < min(slabs, waves)) {
    issue(w, Kt, false);
    issue(w, Vt, true);
    // ---- Q fragments, as every wavefront of the workgroup has them: lane (n, g) holds Q[row 16 qb + n][32 kk + 8 g .. +8] ----
    bf16x8 qf[2][4];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      const int qr = min(row0 + 16 * qb + n, qe - 1);
      const char* qp = a.q + row_offset(a, qr, a.qs_t, a.qs_b) + (long)wi.h * a.qs_h + g * 16;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) qf[qb][kk] = *(const bf16x8*)(qp + kk * 64);
    }
    if (a.q_norm_gamma) {
      norm_q<2>(a, qf, g);
    } else if (a.flags & ATTN_SCALE_Q) {
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
          for (int e = 0; e < 8; ++e) qf[qb][kk][e] = (__bf16)((float)qf[qb][kk][e] * a.scale_log2);
    }

    const int base_k = (n >> 2) * K_GROUP + (n & 3) * ROW_BYTES + ((g ^ (n & 3)) << 4);
    const int r4 = n >> 2, c4 = n & 3;
    const int base_v = g * V_GROUP + r4 * ROW_BYTES + (r4 << 5) + (c4 << 3);
    for (int j = w; j < slabs; j += waves) {
      const bool more = j + waves < slabs;
      const int left = ke - (ks + j * SLAB) - 4 * g;  // valid keys from this lane's first one on
      wait_vmcnt<GROUPS>();  // (K of this slab landed, V may be on its way)
      f32x4v sc[2][2];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        // (keys past the end, copies of the last one in LDS, start from a score whose exponential is 0)
        f32x4v c0;
#pragma unroll
        for (int r = 0; r < 4; ++r) c0[r] = r + 16 * kb < left ? 0.f : -1.0e4f;
        sc[kb][0] = sc[kb][1] = c0;
      }
      static_for<0, 4>([&](auto kc) __attribute__((always_inline)) {
        constexpr int kk = decltype(kc)::value;
        const bf16x8 k0f = read_k<0, kk>(Kt, base_k), k1f = read_k<1, kk>(Kt, base_k);
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
          sc[0][qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0f, qf[qb][kk], sc[0][qb], 0, 0, 0);
          sc[1][qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1f, qf[qb][kk], sc[1][qb], 0, 0, 0);
        }
      });
      u32x4 pf[2];
#pragma unroll
      for (int qb = 0; qb < 2; ++qb)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          const float p0 = __builtin_amdgcn_exp2f(sc[kb][qb][0]), p1 = __builtin_amdgcn_exp2f(sc[kb][qb][1]);
          const float p2 = __builtin_amdgcn_exp2f(sc[kb][qb][2]), p3 = __builtin_amdgcn_exp2f(sc[kb][qb][3]);
          l_run[qb] += (p0 + p1) + (p2 + p3);
          pf[qb][2 * kb] = pack_bf16x2(p0, p1);
          pf[qb][2 * kb + 1] = pack_bf16x2(p2, p3);
        }
      __builtin_amdgcn_sched_barrier(0);
      if (more) {
        issue(j + waves, Kt, false);  // (the products above have this slab's operands in hand)
        wait_vmcnt<GROUPS>();         // (V of this slab landed)
      } else {
        wait_vmcnt<0>();
      }
      static_for<0, 8>([&](auto dc) __attribute__((always_inline)) {
        constexpr int db = v_block(decltype(dc)::value);
        const bf16x8 vf = read_v<0, db>(Vt, base_v, j);
#pragma unroll
        for (int qb = 0; qb < 2; ++qb)
          o_acc[db][qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, __builtin_bit_cast(bf16x8, pf[qb]), o_acc[db][qb], 0, 0, 0);
      });
      __builtin_amdgcn_sched_barrier(0);
      if (more) issue(j + waves, Vt, true);
    }
  }

  // ---- the wavefronts' sums: 16-byte piece (db, qb, g, n) of a wavefront at n ^ (2 db + g / 2), so that both the write and the read below
  // spread over the banks ----
  __syncthreads();  // (everybody is done with the slots)
  const int parts = min(slabs, waves);
  auto part = [&](int i) __attribute__((always_inline)) { return (i < WAVES / 2 ? sK : sV) + i % (WAVES / 2) * PART; };
  if (w < parts) {
    unsigned char* const dst = part(w);
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
      float s = l_run[qb];
      s += __shfl_xor(s, 16);
      s += __shfl_xor(s, 32);
      if (g == 0) s_sum[w][16 * qb + n] = s;
#pragma unroll
      for (int db = 0; db < 8; ++db) *LDS_PTR(f32x4v, dst + ((2 * db + qb) * 64 + g * 16 + (n ^ (2 * db + (g >> 1)))) * 16) = o_acc[db][qb];
    }
  }
  __syncthreads();
  // 16 lanes to a row, eight features each
  const int c = tid & 15;
#pragma unroll
  for (int it = 0; it < 8 / WAVES; ++it) {
    const int r = 4 * WAVES * it + (tid >> 4), q_row = row0 + r;
    const int piece = ((c >> 1) * 2 + (r >> 4)) * 64 + (c & 1) * 32 + ((r & 15) ^ c);
    f32x4v lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < WAVES; ++i)
      if (i < parts) {
        lo += *LDS_PTR(const f32x4v, part(i) + piece * 16);
        hi += *LDS_PTR(const f32x4v, part(i) + (piece + 16) * 16);
        s += s_sum[i][r];
      }
    if (q_row >= qe) continue;
    const float inv = 1.f / s;
    *(u32x4*)(a.out + row_offset(a, q_row, a.os_t, a.os_b) + wi.o_head + 16 * c) =
        u32x4{pack_bf16x2(lo[0] * inv, lo[1] * inv), pack_bf16x2(lo[2] * inv, lo[3] * inv), pack_bf16x2(hi[0] * inv, hi[1] * inv),
              pack_bf16x2(hi[2] * inv, hi[3] * inv)};
    if (a.lse && c == 0) a.lse[(long)wi.h * a.total_q + q_row] = __builtin_amdgcn_logf(s) * 0.6931471805599453f;
  }
}

}  // namespace

hipError_t launch_attn_fwd_bf16_waves(const AttnPairArgs& p, hipStream_t stream) {
  const dim3 grid(8u * (p.job[0].per_xcd + p.job[1].per_xcd));
  if (p.job[0].waves == 4 && (p.job[1].per_xcd == 0 || p.job[1].waves == 4))
    hipLaunchKernelGGL(attn_fwd_bf16_waves_kernel<4>, grid, dim3(256), 0, stream, p);
  else
    hipLaunchKernelGGL(attn_fwd_bf16_waves_kernel<8>, grid, dim3(512), 0, stream, p);
  return hipGetLastError();
}

}  // namespace magi
