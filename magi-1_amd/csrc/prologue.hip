// HBM-bound prologue kernels for gfx950: per-head QK norm + partial non-interleaved rotary +
// bf16 cast + KV-cache write in one pass, plus the norm-only and rotary-only variants.  With e4m3 outputs the
// same pass quantises q and k with constant scales (rows of a QK norm have a known bound, so no absmax pass is
// needed) and leaves v to the chunk quantiser.
//
// Layout: 8 lanes serve one (token, head) row of D = 128 elements, 16 elements (two 16-byte
// vectors) per lane, chosen so that a rotary pair (i, i + R2) lives in ONE lane: lanes
// j < R2/8 hold x[8j..8j+7] and x[R2+8j..R2+8j+7], the remaining lanes hold the pass-through
// tail in two consecutive vectors.  The rotation therefore needs no cross-lane traffic and the
// norm statistics need three butterfly steps.  A wavefront covers 8 rows, a workgroup 32; all
// global accesses are 16 bytes per lane and contiguous per row.
#include "row_ops.h"

namespace magi {
namespace {

constexpr int THREADS = 256;
constexpr int GROUPS = THREADS / 8;  // rows in flight per workgroup

// TPB: tokens that share a workgroup (1, 2, 4 or 8).  OUT8: q and k leave as e4m3 bytes (q_out [S, Hq, D],
// K rows [*, Hkv, D] at kv_out / kv_tail), each multiplied by its constant inverse scale; v is not touched, but for the largest
// magnitude of each of its rows where a.v_row_max asks for them: its quantiser then finds a group's scale in two bytes per row
// ([9360, 24 + 8 heads], out of memory: 32 -> 37 us here, 46 -> 11 there).
template <int TPB, bool OUT8>
__global__ __launch_bounds__(THREADS) void prologue_kernel(const PrologueKernArgs a) {
  __shared__ float s_par[4][D];  // gq, bq, gk, bk
  const int tid = threadIdx.x;
  // Everything a workgroup needs from memory is requested in one go: the norm parameters (two per thread, on their way
  // to LDS), the token's rotary row and each row group's first row; the barrier that publishes the parameters is where
  // they are waited for.  (Parameters, barrier, then the rows: two memory latencies in a workgroup that lives for
  // little more than that.)
  float par[4 * D / THREADS];
#pragma unroll
  for (int k = 0; k < 4 * D / THREADS; ++k) {
    const int i = tid + k * THREADS, which = i / D, e = i % D;
    const float* src = which == 0 ? a.gq : which == 1 ? a.bq : which == 2 ? a.gk : a.bk;
    par[k] = src ? src[e] : 0.f;
  }

  // The 32 row groups of the workgroup form tok_per_block teams of equal size, one token each, so that layers
  // with few heads (e.g. one rank's share of a head-parallel split: 8 rows per token) still fill the workgroup.
  const int j = tid & 7;
  constexpr int gpt = GROUPS / TPB;  // row groups per token
  const int team = TPB == 1 ? 0 : (tid >> 3) / gpt;  // (a constant keeps the token index in a scalar register)
  const int grp = (tid >> 3) % gpt;
  const int nr = a.R2 >> 3;  // lanes that hold rotary pairs
  const bool rot_lane = j < nr;
  const int ea = rot_lane ? 8 * j : 2 * a.R2 + 16 * (j - nr);  // first element of vector A
  const int eb = rot_lane ? a.R2 + 8 * j : ea + 8;             // first element of vector B
  const int U = a.Hq + (OUT8 && !a.v_row_max ? 1 : 2) * a.Hkv;
  constexpr int ES = OUT8 ? 1 : 2;  // bytes per output element

  const int s = blockIdx.x * TPB + team;
  const bool live = s < a.S;
  float sn[8], cs[8];
  if (live && rot_lane && a.rope) {
    const float* rp = a.rope + (long)(s / a.batch) * (2 * a.R2);
    const f32x4 s0 = *(const f32x4*)(rp + 8 * j), s1 = *(const f32x4*)(rp + 8 * j + 4);
    const f32x4 c0 = *(const f32x4*)(rp + a.R2 + 8 * j), c1 = *(const f32x4*)(rp + a.R2 + 8 * j + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sn[i] = s0[i];
      sn[4 + i] = s1[i];
      cs[i] = c0[i];
      cs[4 + i] = c1[i];
    }
  }
  const int sc = live ? s : 0;  // (a valid row for the address arithmetic of a team past the end)
  char* kvrow = (sc < a.n_cache_rows) ? a.kv_out + (long)sc * a.kv_stride_t
                                      : a.kv_tail + (long)(sc - a.n_cache_rows) * a.kv_tail_stride_t;
  // row u of the token: 0 = q, 1 = k, 2 = v; where it comes from and where it goes
  auto locate = [&](int u, const char*& src, char*& dst, int& kind) __attribute__((always_inline)) {
    if (u < a.Hq) {
      kind = 0;
      src = a.q_raw + (long)sc * a.q_raw_stride_t + (long)u * (D * 2);
      dst = a.q_out + ((long)sc * a.Hq + u) * (D * ES);
    } else if (u < a.Hq + a.Hkv) {
      kind = 1;
      const int hh = u - a.Hq;
      src = a.k_raw + (long)sc * a.k_raw_stride_t + (long)hh * (D * 2);
      dst = kvrow + (long)hh * (OUT8 ? D : 2 * D * 2);
    } else {
      kind = 2;
      const int hh = u - a.Hq - a.Hkv;
      src = a.v_raw + (long)sc * a.v_raw_stride_t + (long)hh * (D * 2);
      dst = kvrow + (long)hh * (2 * D * 2) + D * 2;
    }
  };
  int u = grp;
  const char* src = nullptr;
  char* dst = nullptr;
  int kind = 0;
  u32x4 va = {0u, 0u, 0u, 0u}, vb = va;
  if (live && u < U) {
    locate(u, src, dst, kind);
    va = *(const u32x4*)(src + ea * 2);
    vb = *(const u32x4*)(src + eb * 2);
  }
#pragma unroll
  for (int k = 0; k < 4 * D / THREADS; ++k) {
    const int i = tid + k * THREADS;
    s_par[i / D][i % D] = par[k];
  }
  __syncthreads();
  if (!live) return;

  while (u < U) {
    // the next row of this group is requested before the current one is worked on
    const int u_next = u + gpt;
    const char* src_n = nullptr;
    char* dst_n = nullptr;
    int kind_n = 0;
    u32x4 va_n = va, vb_n = vb;
    if (u_next < U) {
      locate(u_next, src_n, dst_n, kind_n);
      va_n = *(const u32x4*)(src_n + ea * 2);
      vb_n = *(const u32x4*)(src_n + eb * 2);
    }
    if (OUT8 && kind == 2) {
      // (two magnitudes per word, which order like unsigned 16-bit integers, a NaN above all)
      typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
      u16x2 mp = {0, 0};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        mp = __builtin_elementwise_max(mp, __builtin_bit_cast(u16x2, va[i] & 0x7fff7fffu));
        mp = __builtin_elementwise_max(mp, __builtin_bit_cast(u16x2, vb[i] & 0x7fff7fffu));
      }
      unsigned m = max(mp[0], mp[1]);
      m = max(m, (unsigned)__shfl_xor((int)m, 1));
      m = max(m, (unsigned)__shfl_xor((int)m, 2));
      m = max(m, (unsigned)__shfl_xor((int)m, 4));
      if (j == 0) a.v_row_max[(long)(u - a.Hq - a.Hkv) * a.S + sc] = (unsigned short)m;
    } else if (kind == 2) {
      *(u32x4*)(dst + ea * 2) = va;
      *(u32x4*)(dst + eb * 2) = vb;
    } else {
      float x[16];
      unpack8(va, x);
      unpack8(vb, x + 8);
      norm16(x, s_par[2 * kind], s_par[2 * kind + 1], ea, eb, a.norm_kind, a.eps, true);
      if (rot_lane && a.rope) rotate8(x, [&](int i) { return sn[i]; }, [&](int i) { return cs[i]; });
      if (kind == 0 && a.q_premul != 1.f) {  // e.g. softmax_scale * log2(e), ahead of the one rounding to bf16
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] *= a.q_premul;
      }
      if constexpr (OUT8) {
        const float inv = kind == 0 ? a.q_inv_scale : a.k_inv_scale;
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] *= inv;
        *(u32x2*)(dst + ea) = pack8_e4m3(x);
        *(u32x2*)(dst + eb) = pack8_e4m3(x + 8);
      } else {
        *(u32x4*)(dst + ea * 2) = pack8(x);
        *(u32x4*)(dst + eb * 2) = pack8(x + 8);
      }
    }
    u = u_next;
    src = src_n;
    dst = dst_n;
    kind = kind_n;
    va = va_n;
    vb = vb_n;
  }
}

// x [S, H, 128] bf16 with strides -> y contiguous, norm only.
__global__ __launch_bounds__(THREADS) void head_norm_kernel(const char* x, long xs_t, long xs_h, const float* gamma,
                                                            const float* beta, char* y, int S, int H, int norm_kind,
                                                            float eps) {
  __shared__ float s_par[2][D];
  const int tid = threadIdx.x;
  for (int i = tid; i < 2 * D; i += THREADS) {
    const float* src = i < D ? gamma : beta;
    s_par[i / D][i % D] = src ? src[i % D] : 0.f;
  }
  __syncthreads();
  const int j = tid & 7;
  const long row = (long)blockIdx.x * GROUPS + (tid >> 3);
  if (row >= (long)S * H) return;
  const long s = row / H, h = row % H;
  const char* src = x + s * xs_t + h * xs_h;
  char* dst = y + row * (D * 2);
  const int ea = 16 * j, eb = ea + 8;
  float v[16];
  unpack8(*(const u32x4*)(src + ea * 2), v);
  unpack8(*(const u32x4*)(src + eb * 2), v + 8);
  norm16(v, s_par[0], s_par[1], ea, eb, norm_kind, eps, beta != nullptr);
  *(u32x4*)(dst + ea * 2) = pack8(v);
  *(u32x4*)(dst + eb * 2) = pack8(v + 8);
}

// Mean and reciprocal standard deviation of a row of nvec 16-byte vectors that a wavefront holds packed (vector
// i * 64 + lane in raw[i], zeros past the end), fp32, in two passes over the registers.  The row stays packed between the
// passes (48 registers for 6144 columns instead of 96 more for its fp32 form): the empty asm makes the compiler
// unpack again rather than keep the first pass's values.
template <int NV>
__device__ __forceinline__ void row_stats(u32x4* raw, int lane, int nvec, float inv_n, float eps, float& mean, float& rstd) {
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    float f[8];
    unpack8(raw[i], f);
#pragma unroll
    for (int k = 0; k < 8; ++k) s += f[k];
  }
  mean = wave_sum(s) * inv_n;
#pragma unroll
  for (int i = 0; i < NV; ++i) asm volatile("" : "+v"(raw[i]));
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (i * 64 + lane < nvec) {
      float f[8];
      unpack8(raw[i], f);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float d = f[k] - mean;
        q += d * d;
      }
    }
  }
  rstd = __builtin_amdgcn_rsqf(wave_sum(q) * inv_n + eps);
#pragma unroll
  for (int i = 0; i < NV; ++i) asm volatile("" : "+v"(raw[i]));
}

// Row LayerNorm of the layer input: one wavefront per row, the row held packed in registers as NV 16-byte
// vectors per lane (vector i of lane l covers elements (64 i + l) * 8 ...), fp32 statistics in two passes over
// the registers.  Weight and bias are read straight from global memory in the last pass (they stay in L1 / L2);
// a persistent variant that staged them in LDS once per workgroup measured 7-8 % slower.
template <int NV, bool PF32>
__global__ __launch_bounds__(THREADS) void layer_norm_kernel(const char* x, long xs, const char* w, const char* b,
                                                             char* y, long ys, long rows, int cols, float eps) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int nvec = cols >> 3;
  const float inv_n = 1.f / (float)cols;
  const long row = (long)blockIdx.x * (THREADS / 64) + (tid >> 6);
  if (row >= rows) return;
  const char* src = x + row * xs;
  u32x4 raw[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int vi = i * 64 + lane;
    raw[i] = vi < nvec ? *(const u32x4*)(src + (long)vi * 16) : u32x4{0u, 0u, 0u, 0u};
  }
  float mean, rstd;
  row_stats<NV>(raw, lane, nvec, inv_n, eps, mean, rstd);
  char* dst = y + row * ys;
  if (w && b) {  // the usual case, free of branches so that the parameter loads of all vectors go out together
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int vi = i * 64 + lane;
      if (vi < nvec) {
        float f[8], wf[8], bf[8];
        unpack8(raw[i], f);
        param8<PF32>(w, vi, wf);
        param8<PF32>(b, vi, bf);
#pragma unroll
        for (int k = 0; k < 8; ++k) f[k] = (f[k] - mean) * rstd * wf[k] + bf[k];
        *(u32x4*)(dst + (long)vi * 16) = pack8(f);
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int vi = i * 64 + lane;
      if (vi < nvec) {
        float f[8], wf[8], bf[8];
        unpack8(raw[i], f);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          wf[k] = 1.f;
          bf[k] = 0.f;
        }
        if (w) param8<PF32>(w, vi, wf);
        if (b) param8<PF32>(b, vi, bf);
#pragma unroll
        for (int k = 0; k < 8; ++k) f[k] = (f[k] - mean) * rstd * wf[k] + bf[k];
        *(u32x4*)(dst + (long)vi * 16) = pack8(f);
      }
    }
  }
}

// 8 quotients -> e4m3(bf16(clamp(q, +-448))); the clamp keeps a NaN (IEEE 754-2019 minimum / maximum)
__device__ __forceinline__ u32x2 clamp8_e4m3(const float* q) {
  u32x2 o;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    float c[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      c[i] = (float)(__bf16)__builtin_elementwise_minimum(__builtin_elementwise_maximum(q[4 * j + i], -448.f), 448.f);
    int u = 0;
    u = __builtin_amdgcn_cvt_pk_fp8_f32(c[0], c[1], u, false);
    u = __builtin_amdgcn_cvt_pk_fp8_f32(c[2], c[3], u, true);
    o[j] = (unsigned)u;
  }
  return o;
}

// Row LayerNorm whose result leaves only as the e4m3 inputs of up to four fp8 linear layers, each with its own input
// scales: y_k = e4m3(bf16(clamp(bf16(norm(x)) / scale_k))).  The normalised rows never reach memory: 2 + n bytes per
// element instead of 4 for the norm and 3 n for the quantisers behind it.
// One workgroup per CU walks a contiguous piece of the rows, one wavefront per row, with the scales in LDS (two planes of
// four floats, so that consecutive lanes read consecutive 16 bytes): fetched per row they would be 16 bytes per element
// through L1.  Outputs whose scales are equal bit for bit (one calibration of the shared input) are converted once and
// stored n times.
// No division per element: y = v_rcp(s) (within one ulp), q0 = f y, q = q0 + (f - q0 s) y.  The bf16 rounding of q (the
// intermediate that is part of the quantiser) equals that of the IEEE quotient for every pair of an 8-bit and a 24-bit
// mantissa and every reciprocal within one ulp: checked exhaustively, 3.2e9 cases.  q0 is clamped to +-2^10 so that it
// cannot overflow (q comes out above 448 all the same).  A scale outside 2^+-60, whose residual could leave the normal
// range, sends the workgroup's rows through divisions instead.
// Bound: HBM with equal scales, the vector ALU with four different ones.  [86400, 6144], four outputs: 711 us (4.5 TB/s)
// with equal scales, 1011 us with four different ones, against 2070 us for the norm and four quantisers; [9360, 3072]:
// 36 and 63 against 105 us.
template <int NV, bool PF32, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void layer_norm_quant_kernel(const LnQuantKernArgs a) {
  __shared__ __attribute__((aligned(16))) f32x4 s_scale[4][2][NV * 64];
  __shared__ int s_diff[4][4];  // [k][j], j < k: scale vectors k and j differ
  __shared__ int s_wide;        // some scale is not within 2^+-60
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nvec = a.cols >> 3;
  if (tid < 16) s_diff[tid >> 2][tid & 3] = 0;
  if (tid == 16) s_wide = 0;
  __syncthreads();
  for (int c = tid; c < 2 * nvec; c += 64 * WAVES) {  // four columns per thread and pass
    f32x4 sc[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (k < a.n_out) {
        sc[k] = *(const f32x4*)(a.scale[k] + 4 * c);
#pragma unroll
        for (int j = 0; j < k; ++j) {
          bool same = true;
#pragma unroll
          for (int i = 0; i < 4; ++i) same &= __float_as_uint(sc[k][i]) == __float_as_uint(sc[j][i]);
          if (!same) s_diff[k][j] = 1;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float m = fabsf(sc[k][i]);
          if (!(m >= 0x1p-60f && m <= 0x1p60f)) s_wide = 1;
        }
        s_scale[k][c & 1][c >> 1] = sc[k];
      }
  }
  __syncthreads();
  const bool exact = __builtin_amdgcn_readfirstlane(s_wide) != 0;
  int rep[4];  // the first output with the same scales
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    rep[k] = k;
#pragma unroll
    for (int j = k - 1; j >= 0; --j)
      if (__builtin_amdgcn_readfirstlane(s_diff[k][j]) == 0) rep[k] = j;
  }
  const float inv_n = 1.f / (float)a.cols;
  const long per = (a.rows + gridDim.x - 1) / gridDim.x;
  const long r0 = (long)blockIdx.x * per, r1 = r0 + per < a.rows ? r0 + per : a.rows;
  for (long row = r0 + w; row < r1; row += WAVES) {
    const char* src = a.x + row * a.xs;
    int lane = tid & 63;  // (opaque: or every address below is computed ahead of the loop and does not fit the registers)
    asm volatile("" : "+v"(lane));
    u32x4 raw[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int vi = i * 64 + lane;
      raw[i] = vi < nvec ? *(const u32x4*)(src + (long)vi * 16) : u32x4{0u, 0u, 0u, 0u};
    }
    float mean, rstd;
    row_stats<NV>(raw, lane, nvec, inv_n, a.eps, mean, rstd);
    // the normalised elements of vector vi, as the bf16 rows the linear layers would be handed
    auto norm8 = [&](const u32x4 v, int vi, float* f) __attribute__((always_inline)) {
      float wf[8], bf[8];
      unpack8(v, f);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        wf[k] = 1.f;
        bf[k] = 0.f;
      }
      if (a.w) param8<PF32>(a.w, vi, wf);
      if (a.b) param8<PF32>(a.b, vi, bf);
#pragma unroll
      for (int k = 0; k < 8; ++k) f[k] = (f[k] - mean) * rstd * wf[k] + bf[k];
      unpack8(pack8(f), f);
    };
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int vi = i * 64 + lane;
      if (vi < nvec) {
        float f[8];
        norm8(raw[i], vi, f);
        u32x2 o[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (k < a.n_out) {
            if (rep[k] == k) {
              const f32x4 s0 = s_scale[k][0][vi], s1 = s_scale[k][1][vi];
              float q[8];
#pragma unroll
              for (int e = 0; e < 8; ++e) {
                const float sc = e < 4 ? s0[e & 3] : s1[e & 3];
                const float y = __builtin_amdgcn_rcpf(sc);
                const float q0 = __builtin_amdgcn_fmed3f(f[e] * y, -1024.f, 1024.f);
                q[e] = __builtin_fmaf(__builtin_fmaf(-q0, sc, f[e]), y, q0);
              }
              o[k] = clamp8_e4m3(q);
            } else {
              o[k] = rep[k] == 0 ? o[0] : rep[k] == 1 ? o[1] : o[2];
            }
            *(u32x2*)(a.y[k] + row * a.cols + 8 * vi) = o[k];
          }
      }
      __builtin_amdgcn_sched_barrier(0);  // (one vector at a time: interleaved, they do not fit the registers)
    }
    if (exact) {
      for (int vi = lane; vi < nvec; vi += 64)
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (k < a.n_out) {
            float f[8];
            norm8(*(const u32x4*)(src + (long)vi * 16), vi, f);
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = f[e] / s_scale[k][e >> 2][vi][e & 3];
            *(u32x2*)(a.y[k] + row * a.cols + 8 * vi) = clamp8_e4m3(f);
          }
    }
  }
}

// Rotary only, x and y contiguous [B, S, H, D] (may be the same memory): HBM bound, every element read and written
// once.  A lane owns the 16-byte vector at pair offset p and the one at p + R2, so a rotated pair never leaves it (and in
// place works), or two vectors of the pass-through tail; a row is 2^lpr_log2 lanes and a workgroup owns one contiguous
// piece of ROT_ROWS rows per row slot, all of whose loads are in flight together.  cos / sin rows come from the
// caches: the heads of a token read the same one.  fp32 [37440, 24, 128]: 160 us, 5.8 TB/s (what a plain copy
// reaches), against 300-313 us, 3.0 TB/s, with one pair of elements per lane (the form below); bf16 86 against 263 us.
constexpr int ROT_ROWS = 2;  // rows per lane
template <bool BF16>
__global__ __launch_bounds__(THREADS) void rotary_vec_kernel(const char* xin, const float* cosp, const float* sinp, char* yout,
                                                             unsigned rows, int S, int H, int R2, int lpr_log2) {
  constexpr int VE = BF16 ? 8 : 4;  // elements per vector
  const int row_bytes = 32 << lpr_log2;
  const int slots = THREADS >> lpr_log2;  // rows in flight per pass of the workgroup
  const int j = threadIdx.x & ((1 << lpr_log2) - 1), slot = threadIdx.x >> lpr_log2;
  const unsigned first = blockIdx.x * (unsigned)(slots * ROT_ROWS);
  const bool rot = j < R2 / VE;
  const int ea = rot ? VE * j : 2 * R2 + 2 * VE * (j - R2 / VE);
  const int eb = rot ? ea + R2 : ea + VE;
  constexpr int ES = BF16 ? 2 : 4;
  u32x4 va[ROT_ROWS], vb[ROT_ROWS];
  f32x4 cs[ROT_ROWS][VE / 4], sn[ROT_ROWS][VE / 4];
#pragma unroll
  for (int k = 0; k < ROT_ROWS; ++k) {
    const unsigned row = first + (unsigned)(slot + k * slots);
    if (row < rows) {
      const char* src = xin + (long)row * row_bytes;
      va[k] = *(const u32x4*)(src + ea * ES);
      vb[k] = *(const u32x4*)(src + eb * ES);
      if (rot) {
        const long at = (long)(row / (unsigned)H % (unsigned)S) * R2 + VE * j;
#pragma unroll
        for (int i = 0; i < VE / 4; ++i) {
          cs[k][i] = *(const f32x4*)(cosp + at + 4 * i);
          sn[k][i] = *(const f32x4*)(sinp + at + 4 * i);
        }
      }
    }
  }
#pragma unroll
  for (int k = 0; k < ROT_ROWS; ++k) {
    const unsigned row = first + (unsigned)(slot + k * slots);
    if (row >= rows) break;
    if (rot) {
      float a[VE], b[VE];
      if constexpr (BF16) {
        unpack8(va[k], a);
        unpack8(vb[k], b);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // (whole vectors: a bit cast of one element of a vector reads element 0)
          a[i] = __builtin_bit_cast(f32x4, va[k])[i];
          b[i] = __builtin_bit_cast(f32x4, vb[k])[i];
        }
      }
#pragma unroll
      for (int i = 0; i < VE; ++i) {
        const float x1 = a[i], x2 = b[i], c = cs[k][i >> 2][i & 3], sv = sn[k][i >> 2][i & 3];
        a[i] = x1 * c - x2 * sv;
        b[i] = x1 * sv + x2 * c;
      }
      if constexpr (BF16) {
        va[k] = pack8(a);
        vb[k] = pack8(b);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          va[k][i] = __builtin_bit_cast(unsigned, a[i]);
          vb[k][i] = __builtin_bit_cast(unsigned, b[i]);
        }
      }
    }
    char* dst = yout + (long)row * row_bytes;
    *(u32x4*)(dst + ea * ES) = va[k];
    *(u32x4*)(dst + eb * ES) = vb[k];
  }
}

// The same for row lengths, rotary widths or addresses that do not split into 16-byte vectors; one thread per
// (row, pair).
template <bool BF16>
__global__ __launch_bounds__(THREADS) void rotary_kernel(const void* xin, const float* cosp, const float* sinp,
                                                         void* yout, long rows, int S, int H, int Dd, int R2) {
  const long gid = (long)blockIdx.x * THREADS + threadIdx.x;
  const int half = Dd / 2;  // threads per row: each handles elements p and p + half ... see below
  const long row = gid / half;
  const int p = (int)(gid % half);
  if (row >= rows) return;
  const long s = (row / H) % S;
  // thread p < R2 rotates the pair (p, p + R2); threads R2 <= p < half copy the tail two at a time
  auto ld = [&](long idx) -> float {
    if (BF16) return __builtin_bit_cast(float, (unsigned)((const unsigned short*)xin)[idx] << 16);
    return ((const float*)xin)[idx];
  };
  auto st = [&](long idx, float v) {
    if (BF16) {
      f32x2 t = {v, 0.f};
      bf16x2 r = __builtin_convertvector(t, bf16x2);
      ((unsigned short*)yout)[idx] = (unsigned short)(__builtin_bit_cast(unsigned, r) & 0xffffu);
    } else {
      ((float*)yout)[idx] = v;
    }
  };
  const long base = row * Dd;
  if (p < R2) {
    const float c = cosp[s * R2 + p], sn = sinp[s * R2 + p];
    const float x1 = ld(base + p), x2 = ld(base + R2 + p);
    st(base + p, x1 * c - x2 * sn);
    st(base + R2 + p, x1 * sn + x2 * c);
  } else {
    const int e = 2 * R2 + 2 * (p - R2);
    st(base + e, ld(base + e));
    st(base + e + 1, ld(base + e + 1));
  }
}

// div_clamp_to: y = e4m3(bf16(clamp(float(x) / scale, -448, 448))), the fp8 linears' input quantiser with its bf16
// intermediate (a double rounding that is part of the definition).  One thread per 8 consecutive elements of a row;
// scale: one value, or one per column.  IEEE division (the reference divides in fp32).
__global__ __launch_bounds__(THREADS) void div_clamp_kernel(const char* x, long xs, const float* scale, int per_column,
                                                            char* y, long ys, long rows, int cols8) {
  const long t = (long)blockIdx.x * THREADS + threadIdx.x;
  if (t >= rows * cols8) return;
  const long r = t / cols8;
  const int c = (int)(t - r * cols8);
  float f[8];
  unpack8(*(const u32x4*)(x + r * xs + (long)c * 16), f);
  float sc[8];
  if (per_column) {
    const f32x4 s0 = *(const f32x4*)(scale + 8 * c), s1 = *(const f32x4*)(scale + 8 * c + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sc[i] = s0[i];
      sc[4 + i] = s1[i];
    }
  } else {
    const float s = scale[0];
#pragma unroll
    for (int i = 0; i < 8; ++i) sc[i] = s;
  }
  float q[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float d = f[i] / sc[i];
    const float cl = d != d ? d : fminf(fmaxf(d, -448.f), 448.f);  // (a NaN stays a NaN, as torch.clamp leaves it)
    q[i] = (float)(__bf16)cl;                                     // the bf16 intermediate
  }
  u32x2 o;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    int u = 0;
    u = __builtin_amdgcn_cvt_pk_fp8_f32(q[4 * j], q[4 * j + 1], u, false);
    u = __builtin_amdgcn_cvt_pk_fp8_f32(q[4 * j + 2], q[4 * j + 3], u, true);
    o[j] = (unsigned)u;
  }
  *(u32x2*)(y + r * ys + (long)c * 8) = o;
}

}  // namespace

hipError_t launch_div_clamp(const char* x, long x_stride, const float* scale, int per_column, char* y, long y_stride,
                            long rows, int cols, hipStream_t stream) {
  const long n = rows * (cols / 8);
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(div_clamp_kernel, dim3((unsigned)((n + THREADS - 1) / THREADS)), dim3(THREADS), 0, stream, x, x_stride,
                     scale, per_column, y, y_stride, rows, cols / 8);
  return hipGetLastError();
}

hipError_t launch_prologue(const PrologueKernArgs& a_in, hipStream_t stream) {
  if (a_in.S <= 0) return hipSuccess;
  const PrologueKernArgs& a = a_in;
  const int rows = a.Hq + (a.out_fp8 && !a.v_row_max ? 1 : 2) * a.Hkv;
  int tpb = 1;
  while (tpb < 8 && 2 * tpb * rows <= GROUPS) tpb *= 2;
  const dim3 grid((unsigned)((a.S + tpb - 1) / tpb)), block(THREADS);
#define MAGI_PROLOGUE(TPB)                                                                  \
  do {                                                                                      \
    if (a.out_fp8)                                                                          \
      hipLaunchKernelGGL((prologue_kernel<TPB, true>), grid, block, 0, stream, a);          \
    else                                                                                    \
      hipLaunchKernelGGL((prologue_kernel<TPB, false>), grid, block, 0, stream, a);         \
  } while (0)
  switch (tpb) {
    case 1: MAGI_PROLOGUE(1); break;
    case 2: MAGI_PROLOGUE(2); break;
    case 4: MAGI_PROLOGUE(4); break;
    default: MAGI_PROLOGUE(8); break;
  }
#undef MAGI_PROLOGUE
  return hipGetLastError();
}

hipError_t launch_head_norm(const char* x, long x_stride_t, long x_stride_h, const float* gamma, const float* beta,
                            char* y, int S, int H, int norm_kind, float eps, hipStream_t stream) {
  const long rows = (long)S * H;
  if (rows <= 0) return hipSuccess;
  const unsigned grid = (unsigned)((rows + GROUPS - 1) / GROUPS);
  hipLaunchKernelGGL(head_norm_kernel, dim3(grid), dim3(THREADS), 0, stream, x, x_stride_t, x_stride_h, gamma, beta, y,
                     S, H, norm_kind, eps);
  return hipGetLastError();
}

hipError_t launch_layer_norm(const char* x, long x_stride, const void* w, const void* b, int params_fp32, char* y,
                             long y_stride, long rows, int cols, float eps, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  const int need = (cols / 8 + 63) / 64;  // 16-byte vectors per lane
  const dim3 grid((unsigned)((rows + THREADS / 64 - 1) / (THREADS / 64))), block(THREADS);
  const char* wp = static_cast<const char*>(w);
  const char* bp = static_cast<const char*>(b);
#define MAGI_LN(NV)                                                                                               \
  do {                                                                                                            \
    if (params_fp32)                                                                                              \
      hipLaunchKernelGGL((layer_norm_kernel<NV, true>), grid, block, 0, stream, x, x_stride, wp, bp, y, y_stride, \
                         rows, cols, eps);                                                                        \
    else                                                                                                          \
      hipLaunchKernelGGL((layer_norm_kernel<NV, false>), grid, block, 0, stream, x, x_stride, wp, bp, y,          \
                         y_stride, rows, cols, eps);                                                              \
  } while (0)
  if (need <= 2) MAGI_LN(2);
  else if (need <= 4) MAGI_LN(4);
  else if (need <= 6) MAGI_LN(6);
  else if (need <= 8) MAGI_LN(8);
  else if (need <= 12) MAGI_LN(12);
  else MAGI_LN(16);
#undef MAGI_LN
  return hipGetLastError();
}

hipError_t launch_layer_norm_quant(const LnQuantKernArgs& a, int params_fp32, int compute_units, hipStream_t stream) {
  if (a.rows <= 0) return hipSuccess;
  const int need = (a.cols / 8 + 63) / 64;  // 16-byte vectors per lane
#define MAGI_LNQ(NV, WAVES, PER_CU)                                                                                      \
  do {                                                                                                                   \
    const long wgs = (a.rows + WAVES - 1) / WAVES, most = (long)compute_units * PER_CU;                                  \
    const dim3 grid((unsigned)(wgs < most ? wgs : most)), block(64 * WAVES);                                             \
    if (params_fp32)                                                                                                     \
      hipLaunchKernelGGL((layer_norm_quant_kernel<NV, true, WAVES>), grid, block, 0, stream, a);                         \
    else                                                                                                                 \
      hipLaunchKernelGGL((layer_norm_quant_kernel<NV, false, WAVES>), grid, block, 0, stream, a);                        \
  } while (0)
  // (workgroups per CU: what the scales in LDS and the registers allow)
  if (need <= 2) MAGI_LNQ(2, 8, 3);
  else if (need <= 6) MAGI_LNQ(6, 8, 3);
  else if (need <= 12) MAGI_LNQ(12, 16, 1);
  else MAGI_LNQ(16, 16, 1);
#undef MAGI_LNQ
  return hipGetLastError();
}

hipError_t launch_rotary(const void* x, const float* cos, const float* sin, void* y, int B, int S, int H, int Dd, int R2,
                         int is_bf16, hipStream_t stream) {
  const long rows = (long)B * S * H;
  const long threads = rows * (Dd / 2);
  if (threads <= 0) return hipSuccess;
  const int ve = is_bf16 ? 8 : 4;
  const int lpr = Dd / (2 * ve);  // lanes per row of the vector form
  const uintptr_t addr = (uintptr_t)x | (uintptr_t)y | (R2 > 0 ? (uintptr_t)cos | (uintptr_t)sin : 0);
  if (Dd % (2 * ve) == 0 && (lpr & (lpr - 1)) == 0 && lpr <= THREADS && R2 % ve == 0 && (addr & 15u) == 0 &&
      rows < 0x7fffff00L) {
    const long per_wg = (long)(THREADS / lpr) * ROT_ROWS;
    const dim3 grid((unsigned)((rows + per_wg - 1) / per_wg));
    const char* xp = static_cast<const char*>(x);
    char* yp = static_cast<char*>(y);
    if (is_bf16)
      hipLaunchKernelGGL(rotary_vec_kernel<true>, grid, dim3(THREADS), 0, stream, xp, cos, sin, yp, (unsigned)rows, S, H, R2,
                         __builtin_ctz(lpr));
    else
      hipLaunchKernelGGL(rotary_vec_kernel<false>, grid, dim3(THREADS), 0, stream, xp, cos, sin, yp, (unsigned)rows, S, H, R2,
                         __builtin_ctz(lpr));
    return hipGetLastError();
  }
  const unsigned grid = (unsigned)((threads + THREADS - 1) / THREADS);
  if (is_bf16)
    hipLaunchKernelGGL(rotary_kernel<true>, dim3(grid), dim3(THREADS), 0, stream, x, cos, sin, y, rows, S, H, Dd, R2);
  else
    hipLaunchKernelGGL(rotary_kernel<false>, dim3(grid), dim3(THREADS), 0, stream, x, cos, sin, y, rows, S, H, Dd, R2);
  return hipGetLastError();
}

}  // namespace magi
