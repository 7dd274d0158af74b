// What brings the pieces of the bounded-score kernel's shared items together (attn_fwd_bf16_x16.hip): its launch behind that kernel, and the
// one that the text attention shares with it (attn_text_merge.hip).
#pragma once
#include "attn_common.h"

namespace magi {
namespace {

// Row sums that the kernel without a running maximum can be trusted with (CHECK, below).
constexpr float SUM_MIN = 0x1p-16f, SUM_MAX = 0x1p64f;

// workgroups per item of the function below
template <bool CHECK>
constexpr int MERGE_SHARES = CHECK ? 1 : 4;

// The split items of a launch of attn_fwd_bf16_x16_kernel: sums their pieces, normalises, writes the rows (CHECK: and the verdicts).
// A wavefront for each 64 rows, lane layout of the accumulators as there.  Memory bound: SPLIT_FLOATS * 4 bytes read per piece.
// Four workgroups per item, one for each query block (CHECK: one, which leaves the wavefronts' verdicts), on the item's XCD: with
// one for all four a launch of 48 items read 0.5 MB per workgroup and nothing beside it.
template <bool CHECK>
__device__ __forceinline__ void merge_pieces(const AttnKernArgs& a, unsigned block, int* s_sel) {
  constexpr int SHARES = MERGE_SHARES<CHECK>;
  const int tid = threadIdx.x, l = tid & 63, n = l & 15, g = l >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned share = (block >> 3) % SHARES, item = ((block >> 3) / SHARES << 3) | (block & 7u);
  const WorkItem wi = locate_work(a, 256, tid, s_sel, item + 8u * a.split_from);
  const int row0 = wi.q0 + 64 * w;
  if (!wi.valid || wi.ke <= wi.ks) return;  // (nothing there, or without keys: done)
  if (row0 >= wi.qe) {
    if (CHECK && l == 0) a.verdict[4 * (long)wi.item + w] = 0;
    return;
  }
  const float* const base = a.partial + (long)item * a.split_pieces * SPLIT_FLOATS;
  const int pieces = (int)a.split_pieces;
  bool bad = false;
#pragma unroll
  for (int k = 0; k < 4 / SHARES; ++k) {
    const int qb = CHECK ? k : (int)share;
    const float* p = base;
    float s = 0.f;
    f32x4 o[8];
#pragma unroll
    for (int db = 0; db < 8; ++db) o[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int i = 0; i < pieces; ++i, p += SPLIT_FLOATS) {
      const f32x4* const src = (const f32x4*)p + w * 2048 + l;
#pragma unroll
      for (int db = 0; db < 8; ++db) o[db] += src[(4 * db + qb) * 64];
      s += p[256 * 128 + 64 * w + 16 * qb + n];
    }
    if constexpr (CHECK) {
      float fine = 0.f;
#pragma unroll
      for (int db = 0; db < 8; ++db)
#pragma unroll
        for (int r = 0; r < 4; ++r) fine = __builtin_fmaf(o[db][r], 0.f, fine);
      bad |= !(s >= SUM_MIN && s <= SUM_MAX) || fine != fine;
    }
    const int q_row = row0 + 16 * qb + n;
    if (q_row >= wi.qe) continue;
    const float inv = 1.f / s;
    char* const op = a.out + row_offset(a, q_row, a.os_t, a.os_b) + wi.o_head + 8 * g;
#pragma unroll
    for (int db = 0; db < 8; ++db)
      *(u32x2*)(op + 32 * db) = u32x2{pack_bf16x2(o[db][0] * inv, o[db][1] * inv), pack_bf16x2(o[db][2] * inv, o[db][3] * inv)};
    if (a.lse && g == 0) a.lse[(long)wi.h * a.total_q + q_row] = __builtin_amdgcn_logf(s) * 0.6931471805599453f;
  }
  if constexpr (CHECK) {
    // (rows beyond the range repeat its last row, as in the kernel that left the pieces: they raise no flag of their own)
    const bool any = __builtin_amdgcn_ballot_w64(bad) != 0;
    if (l == 0) a.verdict[4 * (long)wi.item + w] = any ? 1 : 0;
  }
}

}  // namespace
}  // namespace magi
