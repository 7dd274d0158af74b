// The projections of a small layer with everything around them, in one launch, for gfx950: LayerNorm of the layer input,
// q | k | v | qx projections, per-head norm, rotary, cast, KV-cache append; and for the text tokens the K | V projection with
// the K norm.  Every rounding that the separate launches make is made here too, in fp32 and to bf16 (the normalised input, the raw
// projections, the results): norms and rotary in their arithmetic and order of sums, the products as one fp32 sum over K from its
// first element to its last, 32 at a time, whatever the row's place.  That is the library's order as well wherever it does not cut
// K in pieces: the same bits for 32 rows and more at K up to 1024, for more than 2^17 results above (700 drawn shapes; with fewer
// rows one result of some thousand is the neighbouring bf16).
//
// What bounds it: latency.  Below about a thousand rows the library's GEMM, the norm ahead of it and the prologue behind it
// each live for little more than a launch and a few trips to memory, and a library call costs the host 18 us to issue.
// So: many small workgroups.  A workgroup of four wavefronts forms 32 or 64 rows x one head (128 columns); the weight rows stream
// through LDS in steps of 64 elements of K, three to six stages filled by direct global->LDS loads, 128 bytes of a row per eight
// lanes.  (Operands loaded straight into registers, 16 bytes per lane from 16 rows at a time, move 16 bytes per clock and CU: 33 us
// for 400 text tokens at K = 3072, 16 so.)  The loads stay in flight over the barriers; __syncthreads() would wait for them (layers of 768
// rows 121 against 116 us, of 840 rows 158 against 148).
// The product is formed transposed, W X^T on v_mfma_f32_16x16x32_bf16 with the weight rows as the A operand: register r of lane
// (n, g) of a result block is column 4 g + r of the block, row n; it goes through LDS to eight lanes per row, which do with it
// what the prologue does.
// With e4m3 attention q and k leave quantised with their constant scales, v as it is for the quantiser that follows: the layer's norm,
// product, prologue and text product in this launch (240 rows x 20 heads and 45 x 4, hidden 768: 153 -> 66 us for the layer, most of it the host's time).
// RES: the workgroup's rows are in LDS whole (K up to 1024), normalised ahead of the product.  Otherwise the rows, not to be
// normalised, stream beside the weights.  All workgroups then walk K in step, at the same bytes of weight rows that are a multiple
// of the caches' interleave apart, i.e. on one or two channels; so the workgroups of a head first touch a piece of K each of its weights
// (they are on one XCD: its L2 then has or awaits the lines, from all channels): 300 rows x 16 heads at K = 3072, weights out of memory,
// 21.7 -> 17.7 us, 100 rows 20.5 -> 19.4, out of L2 the same 15.5.  (Walking K from different places gains as much, 17.8, but the order of
// a row's sums then depends on its place among the rows.)
#include "attn_common.h"
#include "row_ops.h"

namespace magi {
namespace {

constexpr int NW = 4;    // wavefronts
constexpr int BK = 64;   // elements of K per stage: 128 bytes of a row
constexpr int STAGE_W = D * BK * 2;
constexpr int LDS_MAX = 160 * 1024;
// bytes per resident row: 16 more than its elements, so that the 16 rows of an operand read fall on different banks
__device__ __forceinline__ int resident_row(int K) { return 2 * K + 16; }
// Resident rows (RES): how long they may be, beside the stages of weights.  (64 rows of 832 elements would fit too; they would be a
// thirteenth piece per lane for a width that no layer here has.)
template <int ROWS>
constexpr int res_max_k() { return ROWS == 32 ? 1024 : 768; }

// What a thread needs from memory to finish its row (eight lanes per row, as in the prologue: a rotary pair (i, i + R2) in one
// lane): requested ahead of the product, not behind it.
template <int HALVES>
struct RowParams {
  f32x4 gam[4], bet[4], sin_cos[HALVES][4];  // elements ea .. +7, eb .. +7; the lane's eight sines and cosines
  bool normed, rot;
  int ea, eb;
};
template <int HALVES>
__device__ __forceinline__ void load_row_params(const SmallProjKernArgs& a, RowParams<HALVES>& p, bool text, int head, int row0, int rows, int tid) {
  const int j = tid & 7, nr = a.R2 >> 3;
  const bool rot_lane = j < nr;
  p.ea = rot_lane ? 8 * j : 2 * a.R2 + 16 * (j - nr);
  p.eb = rot_lane ? a.R2 + 8 * j : p.ea + 8;
  const float *gam = nullptr, *bet = nullptr;
  const bool q = !text && head < a.Hq, k = !text && !q && head < a.Hq + a.Hkv;
  if (q || k) {
    gam = k ? a.gk : a.gq;
    bet = k ? a.bk : a.bq;
  } else if (text && (head & 1) == 0) {
    gam = a.gkx;
    bet = a.bkx;
  }
  p.normed = gam != nullptr;
  p.rot = (q || k) && a.rope && rot_lane;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = (i < 2 ? p.ea : p.eb) + 4 * (i & 1);
    p.gam[i] = gam ? *(const f32x4*)(gam + e) : f32x4{0.f, 0.f, 0.f, 0.f};
    p.bet[i] = gam && bet ? *(const f32x4*)(bet + e) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  if (p.rot) {
#pragma unroll
    for (int h = 0; h < HALVES; ++h) {
      const float* rp = a.rope + (long)(min(row0 + 32 * h + (tid >> 3), rows - 1) / a.batch) * (2 * a.R2) + 8 * j;
#pragma unroll
      for (int i = 0; i < 4; ++i) p.sin_cos[h][i] = *(const f32x4*)(rp + (i < 2 ? 0 : a.R2) + 4 * (i & 1));
    }
  }
}

// The 32 rows row0 .. of one head as the product left them in LDS
template <int HALVES>
__device__ __forceinline__ void store_rows32(const SmallProjKernArgs& a, const RowParams<HALVES>& p, int half, const float* out, bool text, int head,
                                             int row0, int rows, int tid) {
  const int r = tid >> 3, s = row0 + r;
  float v[16];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const f32x4 y = *LDS_PTR(const f32x4, out + r * D + (((((q < 2 ? p.ea : p.eb) >> 2) + (q & 1)) ^ (r & 15)) << 2));
#pragma unroll
    for (int e = 0; e < 4; ++e) v[4 * q + e] = (float)(__bf16)y[e];  // what the projection by itself returns
  }
  if (s >= rows) return;
  char* dst;
  float mul = 1.f, inv = 0.f;  // inv: 1 / the scale of what leaves as e4m3
  if (text) {
    dst = a.text_out + ((long)s * a.Hkv * 2 + head) * (D * 2);
  } else if (head < a.Hq) {
    mul = a.q_premul;
    inv = a.out_fp8 ? a.q_inv_scale : 0.f;
    dst = a.q_out + ((long)s * a.Hq + head) * (a.out_fp8 ? D : D * 2);
  } else if (head < a.Hq + 2 * a.Hkv) {
    const bool is_v = head >= a.Hq + a.Hkv;
    char* const row = s < a.n_cache_rows ? a.kv_out + (long)s * a.kv_stride_t : a.kv_tail + (long)(s - a.n_cache_rows) * a.kv_tail_stride_t;
    if (!a.out_fp8) {
      dst = row + (long)(head - a.Hq - (is_v ? a.Hkv : 0)) * (2 * D * 2) + (is_v ? D * 2 : 0);
    } else if (is_v) {
      dst = a.v_out + ((long)s * a.Hkv + (head - a.Hq - a.Hkv)) * (D * 2);
    } else {
      inv = a.k_inv_scale;
      dst = row + (long)(head - a.Hq) * D;
    }
  } else {
    dst = a.qx_out + ((long)s * a.Hqx + (head - a.Hq - 2 * a.Hkv)) * (D * 2);
  }
  // (the arithmetic of the prologue and, for the text, of the head norm: the bits of the separate launches)
  if (p.normed) norm16_by(v, [&](int i) { return p.gam[i >> 2][i & 3]; }, [&](int i) { return p.bet[i >> 2][i & 3]; }, 0, a.eps, !text || a.bkx);
  if (p.rot)
    rotate8(v, [&](int i) { return p.sin_cos[half][i >> 2][i & 3]; }, [&](int i) { return p.sin_cos[half][2 + (i >> 2)][i & 3]; });
  if (mul != 1.f) {
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] *= mul;
  }
  if (inv != 0.f) {
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] *= inv;
    *(u32x2*)(dst + p.ea) = pack8_e4m3(v);
    *(u32x2*)(dst + p.eb) = pack8_e4m3(v + 8);
    return;
  }
  *(u32x4*)(dst + p.ea * 2) = pack8(v);
  *(u32x4*)(dst + p.eb * 2) = pack8(v + 8);
}

// x of the lane whose number differs in bit M (1, 2 or 4)
template <int M>
__device__ __forceinline__ float lane_xor(float x) {
  int v = __builtin_bit_cast(int, x);
  if constexpr (M == 4) v = __builtin_amdgcn_mov_dpp(v, 0x141, 0xf, 0xf, true);  // row_half_mirror: lane ^ 7
  constexpr int QUAD = M == 1 ? 0xb1 : M == 2 ? 0x4e : 0x1b;                     // quad_perm: lane ^ 1, ^ 2, ^ 3
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(v, QUAD, 0xf, 0xf, true));
}
// The sum over a wavefront's 64 lanes of wave_sum, for eight lanes that stand for them: x[p] of lane j is lane 8 p + j's.  Same pairs in
// the same order, so the same bits: the lanes' bits 1, 2, 4 first (each step a lane hands on the half of the sums that it does not
// keep, and lane j is left with that of p = j), then the bits of p.
__device__ __forceinline__ float wave_sum8(const float (&x)[8], int j) {
  float y[4], z[2];
#pragma unroll
  for (int i = 0; i < 4; ++i) y[i] = (j & 1 ? x[2 * i + 1] : x[2 * i]) + lane_xor<1>(j & 1 ? x[2 * i] : x[2 * i + 1]);
#pragma unroll
  for (int i = 0; i < 2; ++i) z[i] = (j & 2 ? y[2 * i + 1] : y[2 * i]) + lane_xor<2>(j & 2 ? y[2 * i] : y[2 * i + 1]);
  float s = (j & 4 ? z[1] : z[0]) + lane_xor<4>(j & 4 ? z[0] : z[1]);
  s += lane_xor<1>(s);
  s += lane_xor<2>(s);
  return s + lane_xor<4>(s);
}
// Mean and reciprocal standard deviation of a row that eight lanes hold packed, pieces j, j + 8, ... of eight elements in lane j's raw
// (nv of them), as row_stats of the layer norm's kernel forms them: its wavefront has piece 64 i + l in lane l, so lane j here
// stands for lanes j, j + 8, ... j + 56 with up to two pieces each.
template <int NV>
__device__ __forceinline__ void row_stats8(const u32x4 (&raw)[NV], int j, int nv, float inv_n, float eps, float& mean, float& rstd) {
#pragma clang fp contract(off)
  static_assert(NV <= 16, "two pieces per lane of a wavefront");
  float part[8];
#pragma unroll
  for (int p = 0; p < 8; ++p) part[p] = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {  // (zeros past the end)
    float f[8];
    unpack8(raw[i], f);
#pragma unroll
    for (int e = 0; e < 8; ++e) part[i & 7] += f[e];
  }
  mean = wave_sum8(part, j) * inv_n;
#pragma unroll
  for (int p = 0; p < 8; ++p) part[p] = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (i >= nv) continue;
    float f[8];
    unpack8(raw[i], f);
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] -= mean;
    float q = i < 8 ? __builtin_fmaf(f[0], f[0], f[1] * f[1]) : __builtin_fmaf(f[1], f[1], __builtin_fmaf(f[0], f[0], part[i & 7]));
#pragma unroll
    for (int e = 2; e < 8; ++e) q = __builtin_fmaf(f[e], f[e], q);
    part[i & 7] = q;
  }
  rstd = __builtin_amdgcn_rsqf(__builtin_fmaf(inv_n, wave_sum8(part, j), eps));
}

// RES: the rows whole in LDS ahead of the product, normalised on the way there; else they stream beside the weights, as they are
template <bool RES, int ROWS>
__global__ __launch_bounds__(64 * NW, 1) void small_proj_kernel(const SmallProjKernArgs a) {
  constexpr int NST = RES ? (ROWS == 64 ? 3 : 4) : 6;  // stages
  constexpr int TB = ROWS / 16;                        // blocks of 16 rows
  constexpr int STAGE_X = RES ? 16 : ROWS * BK * 2;
  // the stages, named statically (an operand read then does not wait for the loads in flight to another stage)
  __shared__ __attribute__((aligned(1024))) unsigned char sW0[STAGE_W], sW1[STAGE_W], sW2[STAGE_W], sW3[NST > 3 ? STAGE_W : 16],
      sW4[NST > 4 ? STAGE_W : 16], sW5[NST > 5 ? STAGE_W : 16];
  __shared__ __attribute__((aligned(1024))) unsigned char sX0[STAGE_X], sX1[STAGE_X], sX2[STAGE_X], sX3[STAGE_X], sX4[STAGE_X], sX5[STAGE_X];
  __shared__ __attribute__((aligned(1024))) unsigned char sR[RES ? ROWS * (2 * res_max_k<ROWS>() + 16) : 16];
  __shared__ __attribute__((aligned(1024))) unsigned char sT[RES ? 16 : NW * 256];
  static_assert(NST * (STAGE_X + STAGE_W) + (int)sizeof(sR) + (int)sizeof(sT) <= LDS_MAX - 512, "LDS");
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63, n = l & 15, g = l >> 4;

  // ---- which rows, which head: the hidden rows' workgroups, then the text rows' ----
  const bool text = blockIdx.x >= (unsigned)a.hidden_blocks;
  const unsigned b = text ? blockIdx.x - (unsigned)a.hidden_blocks : blockIdx.x;
  const unsigned heads = text ? 2u * (unsigned)a.Hkv : (unsigned)(a.Hq + 2 * a.Hkv + a.Hqx);
  const unsigned tile = b / heads;
  const int head = (int)(b - tile * heads);
  const int row0 = (int)tile * ROWS, rows = text ? a.T : a.S, K = text ? a.Kt : a.K;
  const char* const x = text ? a.text : a.x;
  const long xs = text ? a.text_stride : a.x_stride;
  const char* const wt = (text ? a.w_text : a.w) + (long)head * D * K * 2;
  const int steps = K / BK;
  const bool ln = RES && !text && a.ln_w != nullptr;

  // ---- loader: a wave-wide load of 64 x 16 bytes fills eight rows of 128 bytes; lane l sits at row l / 8, slot l % 8, and fetches
  // the chunk that belongs there: row r keeps chunk c at c ^ ((r / 2) % 8), so that the 16 rows of an operand read fall on
  // different banks.  Wavefront w fills rows 8 (w + 4 j) .. +7 of the weights, j = 0 .. 3, and rows 8 w .. +7 of x (where they stream).
  const int lr = l >> 3, chunk = (l & 7) ^ ((4 * w + (lr >> 1)) & 7);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)wt, 0, 0x7fffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void*)(x + (long)row0 * xs), 0, 0x7fffffff, 0x00020000);
  const unsigned vw = (unsigned)(8 * w + lr) * (unsigned)(K * 2) + 16u * (unsigned)chunk;
  const unsigned vx = (unsigned)min(8 * w + lr, rows - 1 - row0) * (unsigned)xs + 16u * (unsigned)chunk;
  const unsigned vx2 = (unsigned)min(8 * w + lr + 32, rows - 1 - row0) * (unsigned)xs + 16u * (unsigned)chunk;
  constexpr int LOADS = RES ? 4 : 4 + ROWS / 32;  // per wavefront and stage
  auto load = [&](int step, unsigned char* W, unsigned char* X) __attribute__((always_inline)) {
    if (step >= steps) return;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, LDS_PTR(void, W + (w + 4 * j) * 1024), 16, vw,
                                               (int)((unsigned)step * (BK * 2) + (unsigned)(32 * j) * (unsigned)(K * 2)), 0, 0);
    if constexpr (!RES) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, LDS_PTR(void, X + w * 1024), 16, vx, (int)((unsigned)step * (BK * 2)), 0, 0);
      if constexpr (ROWS == 64)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, LDS_PTR(void, X + (w + 4) * 1024), 16, vx2, (int)((unsigned)step * (BK * 2)), 0, 0);
    }
  };
  if constexpr (!RES) {  // the touches: four bytes of each row and stage, a line per lane, into LDS that nothing reads
    const int tiles = (rows + ROWS - 1) / ROWS, end = (int)((long)steps * (tile + 1) / tiles);
    for (int st = (int)((long)steps * tile / tiles) + w; st < end; st += NW)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, LDS_PTR(void, sT + w * 256), 4, (unsigned)(64 * j + l) * (unsigned)(K * 2), st * (BK * 2), 0, 0);
  }
  RowParams<ROWS / 32> params;
  load_row_params(a, params, text, head, row0, rows, tid);
  load(0, sW0, sX0);
  load(1, sW1, sX1);
  if constexpr (NST > 3) load(2, sW2, sX2);
  if constexpr (!RES) load(3, sW3, sX3);

  // ---- RES: the workgroup's rows, their statistics and norm, eight lanes a row ----
  const int x_row = resident_row(K);
  if constexpr (RES) {
#pragma unroll
    for (int half = 0; half < ROWS / 32; ++half) {
      const int r = 32 * half + (tid >> 3), j = tid & 7;
      const char* const rp = x + (long)min(row0 + r, rows - 1) * xs;
      constexpr int NV = res_max_k<ROWS>() / 64;  // pieces of eight elements per lane: j, j + 8, ...
      const int nv = K >> 6;
      u32x4 raw[NV];
#pragma unroll
      for (int i = 0; i < NV; ++i) raw[i] = i < nv ? *(const u32x4*)(rp + (8 * i + j) * 16) : u32x4{0u, 0u, 0u, 0u};
      u32x4 lnw[NV], lnb[NV];  // bf16 parameters, requested with the rows
      if (ln && !a.ln_fp32) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          lnw[i] = i < nv ? *(const u32x4*)(a.ln_w + (8 * i + j) * 16) : u32x4{0u, 0u, 0u, 0u};
          lnb[i] = i < nv ? *(const u32x4*)(a.ln_b + (8 * i + j) * 16) : u32x4{0u, 0u, 0u, 0u};
        }
      }
      float mean = 0.f, rstd = 1.f;
      if (ln) row_stats8<NV>(raw, j, nv, 1.f / (float)K, a.ln_eps, mean, rstd);
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        if (i >= nv) continue;
        float f[8], wf[8], bf[8];
        unpack8(raw[i], f);
        if (!ln) {
          *LDS_PTR(u32x4, sR + r * x_row + (8 * i + j) * 16) = raw[i];
          continue;
        }
        if (a.ln_fp32) {
          param8<true>(a.ln_w, 8 * i + j, wf);
          param8<true>(a.ln_b, 8 * i + j, bf);
        } else {
          unpack8(lnw[i], wf);
          unpack8(lnb[i], bf);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = __builtin_fmaf((f[e] - mean) * rstd, wf[e], bf[e]);
        *LDS_PTR(u32x4, sR + r * x_row + (8 * i + j) * 16) = pack8(f);
      }
    }
  }

  // ---- operand reads: lane (n, g) holds elements 32 kk + 8 g .. +8 of weight row 32 w + 16 fb + n and of row 16 tb + n ----
  const int sw = (g ^ ((n >> 1) & 3)) << 4, sh = ((n >> 3) & 1) << 6;  // chunk (4 kk + g) ^ (n / 2): the low bits, the high bit
  const int base_w = (32 * w + n) * (BK * 2) + sw, base_x = RES ? n * x_row + 16 * g : n * (BK * 2) + sw;
  f32x4 acc[2][TB];
#pragma unroll
  for (int fb = 0; fb < 2; ++fb)
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) acc[fb][tb] = f32x4{0.f, 0.f, 0.f, 0.f};
  struct Operands {
    bf16x8 w[2][2], x[2][TB];
  };
  auto read = [&](Operands& o, int s, const unsigned char* W, const unsigned char* X) __attribute__((always_inline)) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
      for (int fb = 0; fb < 2; ++fb) o.w[kk][fb] = *LDS_PTR(const bf16x8, W + ((base_w + ((64 * kk) ^ sh)) + fb * 16 * (BK * 2)));
#pragma unroll
      for (int tb = 0; tb < TB; ++tb)
        o.x[kk][tb] = RES ? *LDS_PTR(const bf16x8, sR + (base_x + tb * 16 * x_row + s * (BK * 2) + 64 * kk))
                          : *LDS_PTR(const bf16x8, X + ((base_x + ((64 * kk) ^ sh)) + tb * 16 * (BK * 2)));
    }
  };
  auto multiply = [&](const Operands& o) __attribute__((always_inline)) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int fb = 0; fb < 2; ++fb)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
          acc[fb][tb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(o.w[kk][fb], o.x[kk][tb], acc[fb][tb], 0, 0, 0);
  };
  if constexpr (RES) {
    auto step = [&](int s, const unsigned char* W, unsigned char* Wn) __attribute__((always_inline)) {
      if (s >= steps) return;
      // (the loads of the stages behind this one may be outstanding; the barrier also publishes the rows)
      const int behind = steps - 1 - s;
      if (behind >= NST - 2)
        wait_vmcnt<LOADS * (NST - 2)>();
      else if (NST > 3 && behind == 1)
        wait_vmcnt<LOADS>();
      else
        wait_vmcnt<0>();
      barrier_loads_in_flight();
      load(s + NST - 1, Wn, nullptr);
      Operands o;
      read(o, s, W, nullptr);
      __builtin_amdgcn_sched_barrier(0);  // (all reads of a stage ahead of its products: their latency once; 1.5 % of a layer of 768 rows)
      multiply(o);
    };
    for (int s = 0; s < steps; s += NST) {
      if constexpr (NST == 4) {
        step(s, sW0, sW3);
        step(s + 1, sW1, sW0);
        step(s + 2, sW2, sW1);
        step(s + 3, sW3, sW2);
      } else {
        step(s, sW0, sW2);
        step(s + 1, sW1, sW0);
        step(s + 2, sW2, sW1);
      }
    }
  } else {
    // Two stages per barrier, the four behind them on the way (their bytes arrive at 130 GB/s per CU, what the direct path holds).  A
    // last stage without a partner is multiplied by itself.
    auto pair = [&](int s, const unsigned char* Wa, const unsigned char* Xa, const unsigned char* Wb, const unsigned char* Xb, unsigned char* Wan,
                    unsigned char* Xan, unsigned char* Wbn, unsigned char* Xbn) __attribute__((always_inline)) {
      if (s >= steps) return;
      const int behind = steps - 2 - s;
      if (behind >= 2)
        wait_vmcnt<LOADS * 2>();
      else if (behind == 1)
        wait_vmcnt<LOADS>();
      else
        wait_vmcnt<0>();
      barrier_loads_in_flight();
      load(s + 4, Wan, Xan);
      load(s + 5, Wbn, Xbn);
      Operands o;
      read(o, s, Wa, Xa);
      multiply(o);
      if (s + 1 < steps) {
        read(o, s + 1, Wb, Xb);
        multiply(o);
      }
    };
    for (int s = 0; s < steps; s += 6) {
      pair(s, sW0, sX0, sW1, sX1, sW4, sX4, sW5, sX5);
      pair(s + 2, sW2, sX2, sW3, sX3, sW0, sX0, sW1, sX1);
      pair(s + 4, sW4, sX4, sW5, sX5, sW2, sX2, sW3, sX3);
    }
  }
  // 32 rows at a time through LDS: 512 bytes a row, its 16-byte chunk c at c ^ (row % 16)
  float* const out = (float*)sW0;
#pragma unroll
  for (int half = 0; half < ROWS / 32; ++half) {
    __syncthreads();
#pragma unroll
    for (int fb = 0; fb < 2; ++fb)
#pragma unroll
      for (int tb = 0; tb < 2; ++tb)
        *LDS_PTR(f32x4, out + (16 * tb + n) * D + (((8 * w + 4 * fb + g) ^ n) << 2)) = acc[fb][2 * half + tb];
    __syncthreads();
    store_rows32(a, params, half, out, text, head, row0 + 32 * half, rows, tid);
  }
}

}  // namespace

hipError_t launch_small_proj(const SmallProjKernArgs& a_in, int compute_units, hipStream_t stream) {
  SmallProjKernArgs a = a_in;
  const int heads = a.Hq + 2 * a.Hkv + a.Hqx;
  auto blocks = [&](int rows) { return ((a.S + rows - 1) / rows) * heads + ((a.T + rows - 1) / rows) * 2 * a.Hkv; };
  if (blocks(32) == 0) return hipSuccess;
  const int K = (a.S > 0 && a.K > a.Kt) || a.T == 0 ? a.K : a.Kt;  // the longer rows
  const bool res = K <= res_max_k<32>(), tall = (!res || K <= res_max_k<64>()) && blocks(32) > compute_units;
  a.hidden_blocks = (tall ? (a.S + 63) / 64 : (a.S + 31) / 32) * heads;
  const dim3 grid((unsigned)blocks(tall ? 64 : 32)), threads(64 * NW);
  if (!res && tall)
    hipLaunchKernelGGL((small_proj_kernel<false, 64>), grid, threads, 0, stream, a);
  else if (!res)
    hipLaunchKernelGGL((small_proj_kernel<false, 32>), grid, threads, 0, stream, a);
  else if (tall)
    hipLaunchKernelGGL((small_proj_kernel<true, 64>), grid, threads, 0, stream, a);
  else
    hipLaunchKernelGGL((small_proj_kernel<true, 32>), grid, threads, 0, stream, a);
  return hipGetLastError();
}

}  // namespace magi
