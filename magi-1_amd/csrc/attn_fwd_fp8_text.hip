// Core attention of e4m3 rows and the text cross attention of bf16 rows in one launch, for gfx950 (MI355X).
//
// The two do not depend on each other, and one after the other the e4m3 launch ends with slots empty for the length of a workgroup and the
// text's launch, which waits for all of it, is a round or two of short workgroups of its own.  Here the text's workgroups follow the core's.
// They must not cost the core its three workgroups per CU, 36 KB of LDS and 168 registers each: the forms of the bf16 kernels take 53 and
// 70 KB.  So the text is walked in tiles of 32 keys in the four slots of the e4m3 tiles (attn_text_rows.h).  168 registers, 3 of them spilled
// outside the tile loops (the e4m3 kernel by itself: 2).
// The layers around the two, one by one -> together, 24 heads: 9360 rows over 46800 keys, 400 of text 2997 -> 2955 us; 5400 rows 551 -> 513; 14472
// 2644 -> 2586; 3600 318 -> 306; 86400 rows x 48 heads 79.50 -> 79.45 ms.  28 drawn layers from 122 rows per CU (of all heads) on: 1.006 to
// 1.096 times as fast; below 64 the two do not fill the chip and are launched one by one (module.py).
#include "attn_fp8_tiles.h"
#include "attn_text_rows.h"

namespace magi {
namespace {

constexpr int SK_BYTES = HK_BYTES > e4m3::K_TILE_BYTES ? HK_BYTES : e4m3::K_TILE_BYTES;
constexpr int SV_BYTES = HV_BYTES > e4m3::V_TILE_BYTES ? HV_BYTES : e4m3::V_TILE_BYTES;

// job[0]: the core's arguments, pair.ahead workgroups of each XCD; job[1]: the text's, in 128-row tiles
template <bool FASTP>
__global__ __launch_bounds__(256, 3) void attn_fwd_fp8_text_kernel(const AttnPairArgs) {
  __shared__ __attribute__((aligned(1024))) unsigned char sK0[SK_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char sV0[SV_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char sK1[SK_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char sV1[SV_BYTES];
  __shared__ int s_sel[LOCATE_WORDS];
  const AttnPairArgs& pair = *(const AttnPairArgs*)__builtin_amdgcn_kernarg_segment_ptr();  // (see attn_fwd_bf16_waves.hip)
  const unsigned ahead = 8u * pair.ahead;
  if (blockIdx.x >= ahead) {
    text_rows(pair.job[1], blockIdx.x - ahead, sK0, sV0, sK1, sV1, s_sel);
    return;
  }
  constexpr bool POW2 = true;
  const AttnKernArgs& a = pair.job[0];
  using e4m3::BM;
  using e4m3::BN;
  using e4m3::i32x2;
  using e4m3::i32x4;
  using e4m3::i32x8;
  using e4m3::K_GROUP;
  using e4m3::LOADS;
  using e4m3::NW;
  using e4m3::P_SHIFT;
  using e4m3::ROW_BYTES;
  using e4m3::store_rows;
  using e4m3::V_GROUP;
#define FP8_BLOCK blockIdx.x
#include "attn_fwd_fp8_body.h"
#undef FP8_BLOCK
}

}  // namespace

hipError_t launch_attn_fwd_fp8_text(const AttnPairArgs& p, hipStream_t stream) {
  AttnPairArgs pair = p;
  pair.ahead = split_grid(p.job[0]) / 8u;
  const dim3 grid(split_grid(p.job[0]) + 8u * p.job[1].per_xcd);
  if (p.job[0].flags & 4)
    hipLaunchKernelGGL(attn_fwd_fp8_text_kernel<true>, grid, dim3(256), 0, stream, pair);
  else
    hipLaunchKernelGGL(attn_fwd_fp8_text_kernel<false>, grid, dim3(256), 0, stream, pair);
  launch_fp8_merge(p.job[0], stream);
  return hipGetLastError();
}

}  // namespace magi
