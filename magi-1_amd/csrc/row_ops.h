// Row helpers shared by the prologue, norm and small-projection kernels (gfx950): bf16 / e4m3 packing of eight elements, the
// per-head norm of a row held by eight lanes.
#pragma once
#include "kernels.h"

namespace magi {
namespace {

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int D = 128;

__device__ __forceinline__ void unpack8(const u32x4 v, float* f) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __builtin_bit_cast(float, v[i] << 16);
    f[2 * i + 1] = __builtin_bit_cast(float, v[i] & 0xffff0000u);
  }
}
__device__ __forceinline__ unsigned pack2(float a, float b) {
  f32x2 x = {a, b};
  bf16x2 r = __builtin_convertvector(x, bf16x2);
  return __builtin_bit_cast(unsigned, r);
}
__device__ __forceinline__ u32x4 pack8(const float* f) {
  u32x4 v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = pack2(f[2 * i], f[2 * i + 1]);
  return v;
}
// 8 floats -> 8 saturating OCP e4m3fn bytes (the conversion itself does not saturate: clamp first)
__device__ __forceinline__ u32x2 pack8_e4m3(const float* f) {
  u32x2 o;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    float c[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) c[i] = fminf(fmaxf(f[4 * j + i], -448.f), 448.f);
    int u = 0;
    u = __builtin_amdgcn_cvt_pk_fp8_f32(c[0], c[1], u, false);
    u = __builtin_amdgcn_cvt_pk_fp8_f32(c[2], c[3], u, true);
    o[j] = (unsigned)u;
  }
  return o;
}
__device__ __forceinline__ float group8_sum(float x) {
  x += __shfl_xor(x, 1);
  x += __shfl_xor(x, 2);
  x += __shfl_xor(x, 4);
  return x;
}

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) x += __shfl_xor(x, m);
  return x;
}

// Normalise the 16 values of this lane (8 lanes = one row of 128) in place; gam(i), bet(i): the parameters of its value i.  The
// roundings are spelled out (no contraction that the compiler is free to choose), so that every kernel that norms heads gives
// the same bits.
template <class G, class B>
__device__ __forceinline__ void norm16_by(float* x, G gam, B bet, int kind, float eps, bool has_beta) {
#pragma clang fp contract(off)
  if (kind == 2) return;
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) s += x[i];
  float mean = 0.f;
  if (kind == 0) mean = group8_sum(s) * (1.f / D);
#pragma unroll
  for (int i = 0; i < 16; ++i) x[i] -= mean;
  float q = __builtin_fmaf(x[0], x[0], x[1] * x[1]);
#pragma unroll
  for (int i = 2; i < 16; ++i) q = __builtin_fmaf(x[i], x[i], q);
  const float rstd = __builtin_amdgcn_rsqf(__builtin_fmaf(group8_sum(q), 1.f / D, eps));
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    float y = x[i] * rstd * (gam(i) + 1.f);
    if (kind == 0 && has_beta) y += bet(i);
    x[i] = y;
  }
}
__device__ __forceinline__ void norm16(float* x, const float* gam, const float* bet, int ea, int eb, int kind, float eps,
                                       bool has_beta) {
  auto at = [&](int i) { return i < 8 ? ea + i : eb + (i - 8); };
  norm16_by(x, [&](int i) { return gam[at(i)]; }, [&](int i) { return bet[at(i)]; }, kind, eps, has_beta);
}
// Rotate the eight pairs (x[i], x[8 + i]), with the roundings spelled out as above
template <class S, class C>
__device__ __forceinline__ void rotate8(float* x, S sn, C cs) {
#pragma clang fp contract(off)
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float x1 = x[i], x2 = x[8 + i];
    x[i] = __builtin_fmaf(x1, cs(i), -(x2 * sn(i)));
    x[8 + i] = __builtin_fmaf(x1, sn(i), x2 * cs(i));
  }
}

// elements 8 vi .. 8 vi + 7 of a norm parameter
template <bool PF32>
__device__ __forceinline__ void param8(const char* p, int vi, float* out) {
  if (PF32) {
    const f32x4 lo = *(const f32x4*)(p + (long)vi * 32), hi = *(const f32x4*)(p + (long)vi * 32 + 16);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      out[k] = lo[k];
      out[4 + k] = hi[k];
    }
  } else {
    unpack8(*(const u32x4*)(p + (long)vi * 16), out);
  }
}

}  // namespace
}  // namespace magi
