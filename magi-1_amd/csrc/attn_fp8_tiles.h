// What the kernels of e4m3 rows share (attn_fwd_fp8.hip, attn_fwd_fp8_text.hip): the layout of their tiles in LDS and the stores of
// their results.  In a namespace of its own, beside the bf16 tiles' names.
#pragma once
#include "attn_common.h"

namespace magi {
namespace {
namespace e4m3 {

typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

constexpr int BN = 64;
constexpr int ROW_BYTES = 128;  // D = 128 fp8
// A tile in LDS is eight groups of eight rows (what one wave-wide direct load fills: 64 lanes x 16 bytes), in key
// order.  The groups are spaced by a little more than their 1024 bytes and the MFMAs take the keys of a tile in an
// order that spreads every operand read over the groups (see the read bases below): consecutive groups start 16
// (K) or 32 (V) bytes further round the banks, so no swizzle is needed and every read address is the lane's base
// plus a constant.
constexpr int K_GROUP = 1024 + 16, V_GROUP = 1024 + 32;
constexpr int K_TILE_BYTES = (BN / 8) * K_GROUP, V_TILE_BYTES = (BN / 8) * V_GROUP;
constexpr int NW = 4;
constexpr int BM = 32 * NW;
constexpr int LOADS = 8 / NW;  // direct loads per wave per matrix per tile (8 rows each)
constexpr float P_SHIFT = 8.f;

// acc * inv as bf16, features 32 mb .. +31 of this lane's row (op: the row's bytes + 16 g); acc in the lane layout of the PV MFMAs.
// A lane holds four consecutive features per b, its partner in the other half wave the next four: the halves trade the odd-b
// registers of the lower half for the even-b registers of the upper one, after which every lane owns eight consecutive features
// and stores 16 bytes at a time.
__device__ __forceinline__ void store_block(bool row_ok, char* op, int mb, const f32x16& acc, float inv) {
#pragma unroll
  for (int bp = 0; bp < 2; ++bp) {
    unsigned ev[2], od[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      ev[e] = pack_bf16x2(acc[8 * bp + 2 * e] * inv, acc[8 * bp + 2 * e + 1] * inv);
      od[e] = pack_bf16x2(acc[8 * bp + 4 + 2 * e] * inv, acc[8 * bp + 4 + 2 * e + 1] * inv);
      half_swap(ev[e], od[e]);  // lower half: (own even, partner's even); upper half: (partner's odd, own odd)
    }
    if (row_ok) *(u32x4*)(op + (32 * mb + 16 * bp) * 2) = u32x4{ev[0], ev[1], od[0], od[1]};
  }
}
// acc * inv as bf16 rows wi.q0 + row0 .. + 31 of out.  (The row address is derived from
// an opaque copy of the lane index so that it is computed here and not carried through the main loop.)
__device__ __forceinline__ void store_rows(const AttnKernArgs& a, const WorkItem& wi, int row0, int l, const f32x16 (&acc)[4], float inv) {
  int lane_e = l;
  asm volatile("" : "+v"(lane_e));
  const bool row_ok = wi.q0 + row0 + (l & 31) < wi.qe;
  char* const op = a.out + (long)(wi.q0 + row0 + (lane_e & 31)) * a.os_t + wi.o_head + 16 * (lane_e >> 5);
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) store_block(row_ok, op, mb, acc[mb], inv);
}

}  // namespace e4m3
}  // namespace
}  // namespace magi
