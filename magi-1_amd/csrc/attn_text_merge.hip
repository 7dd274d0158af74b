// The text cross attention and what brings the pieces of the core attention's shared items together, in one launch, for gfx950 (MI355X).
//
// A layer of less than a few rounds of 256-row workgroups has the keys of its core attention in pieces, and behind that launch a merge that
// is bound by memory (10 to 25 us, 64 to 137 MB) and then the text attention, bound by latency and the matrix pipe: neither needs the other.
// Here the text's workgroups come first and the merge's fill the places they leave: 36 KB of LDS, 168 registers, three workgroups per CU
// (attn_text_rows.h, attn_bf16_merge.h).
// Layers around the two, 24 heads, one by one -> together: 2112 rows over 14784 keys 390 -> 381 us, 3024 (four ranges) 386 -> 372, 2964 over 5928
// 403 -> 389, 2640 (two) 373 -> 364.
#include "attn_bf16_merge.h"
#include "attn_text_rows.h"

namespace magi {
namespace {

// job[0]: the arguments of the launch that left the pieces; job[1]: the text's, in 128-row tiles, pair.ahead workgroups of each XCD
__global__ __launch_bounds__(256, 3) void attn_text_merge_kernel(const AttnPairArgs) {
  __shared__ __attribute__((aligned(1024))) unsigned char sK0[HK_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char sV0[HV_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char sK1[HK_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char sV1[HV_BYTES];
  __shared__ int s_sel[LOCATE_WORDS];
  const AttnPairArgs& pair = *(const AttnPairArgs*)__builtin_amdgcn_kernarg_segment_ptr();  // (see attn_fwd_bf16_waves.hip)
  const unsigned ahead = 8u * pair.ahead;
  if (blockIdx.x < ahead)
    text_rows(pair.job[1], blockIdx.x, sK0, sV0, sK1, sV1, s_sel);
  else
    merge_pieces<false>(pair.job[0], blockIdx.x - ahead, s_sel);
}

}  // namespace

hipError_t launch_attn_text_merge(const AttnPairArgs& p, hipStream_t stream) {
  AttnPairArgs pair = p;
  pair.ahead = p.job[1].per_xcd;
  pair.job[0].flags &= ~ATTN_ZERO_GAPS;  // (the rows no range covers are clear by now)
  const dim3 grid(8u * (pair.ahead + split_items(p.job[0]) * MERGE_SHARES<false>));
  hipLaunchKernelGGL(attn_text_merge_kernel, grid, dim3(256), 0, stream, pair);
  return hipGetLastError();
}

}  // namespace magi
