// K / V tiles of bf16 rows in LDS as the 16x16x32 MFMAs of 32 query rows per wavefront read them, and the norm of q on its way into
// registers (gfx950): shared by attn_fwd_bf16_r32.hip and attn_fwd_bf16_waves.hip.  (attn_fwd_bf16_x16.hip, which explains the
// layouts, has its own copies: its tile loop is sensitive to what the compiler does around it.)
#pragma once
#include "attn_common.h"

namespace magi {
namespace {

constexpr int ROW_BYTES = 256;  // D = 128 bf16
constexpr int BN = 64;          // keys per LDS tile
// a tile in LDS: 16 groups of four rows, spaced so that the operand reads are free of bank conflicts
constexpr int K_GROUP = 1024 + 64, V_GROUP = 1024 + 128;
constexpr int K_TILE_BYTES = (BN / 4) * K_GROUP, V_TILE_BYTES = (BN / 4) * V_GROUP;

typedef float f32x4v __attribute__((ext_vector_type(4)));

// base ^ M, neither hoisted out of the tile loop nor shared between its uses (see attn_fwd_bf16_x16.hip)
template <int M, int TAG>
__device__ __forceinline__ int swz(int base, int tie) {
  if constexpr (M == 0) return base;
  int r;
  asm("v_xor_b32 %0, %1, %2" : "=v"(r) : "n"(M), "v"(base), "s"(tie), "n"(TAG));
  return r;
}
// K as the A operand of the score MFMAs: rows 16 KB + n of a tile, features 32 KK + 8 g .. +8
template <int KB, int KK>
__device__ __forceinline__ bf16x8 read_k(const unsigned char* Kt, int base) {
  return *LDS_PTR(const bf16x8, Kt + (base + KK * 64 + 4 * KB * K_GROUP));
}
// V^T as the A operand of the PV MFMAs: feature block DB, the two 16-key blocks of half T of a tile
template <int T, int DB>
__device__ __forceinline__ bf16x8 read_v(const unsigned char* Vt, int base, int tie) {
  const int bv = swz<((DB & 3) << 5), 16 * T + (DB & 3)>(base, tie) + (DB >> 2) * 128;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(s16x4, Vt + (bv + (8 * T) * V_GROUP)));
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(s16x4, Vt + (bv + (8 * T + 4) * V_GROUP)));
  const s16x8 va = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(bf16x8, va);
}
// order in which the feature blocks are visited: 0, 4, 1, 5, 2, 6, 3, 7 (the two of a pair share their address)
constexpr int v_block(int i) { return (i >> 1) + 4 * (i & 1); }

// NORM: qf holds the raw projection, lane (n, g) features 32 kk + 8 g .. +8 of row 16 qb + n in fragment kk: per-(token, head) norm over the
// 128 features in fp32, times the softmax scale, one rounding to bf16 (the bits of attn_fwd_bf16_x16.hip's)
template <int QB>
__device__ __forceinline__ void norm_q(const AttnKernArgs& a, bf16x8 (&qf)[QB][4], int g) {
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

}  // namespace
}  // namespace magi
