// fp8 (OCP e4m3fn) range attention forward and the per-(chunk, head) quantiser, for gfx950.
//
// Same organisation as the bf16 kernel (S^T = K Q^T, one query per lane column, online softmax in
// fp32, O^T = V^T P^T), built on v_mfma_f32_32x32x64_f8f6f4, which runs at twice the bf16 rate:
//   * K / V tiles are 64 rows x 128 bytes; the transposing LDS read is ds_read_b64_tr_b8;
//   * P is quantised to e4m3 after scaling by 2^8 (P <= 1 so P * 256 <= 256 < 448), the factor is
//     folded into the exponent of exp2 and divided out with the row sum;
//   * Q, K, V carry one fp32 scale per (chunk of `scale_chunk_tokens` tokens, head).  The key axis
//     is walked in pieces that never cross a scale chunk (nor the boundary between the two key
//     segments), so inside a tile the K and V scales are wave-uniform scalars: the K scale joins
//     the softmax scale, the V scale (relative to the largest V scale of the range) joins the exp2
//     exponent, and the Q scale is a per-lane constant because a lane owns one query.
#include "attn_fp8_tiles.h"

namespace magi {
namespace {

using namespace e4m3;

// FASTP (with POW2): the probabilities come from a piecewise-linear exp2 built on the matrix pipe's scaling
// instead of the quarter-rate v_exp_f32: the score registers hold e4m3 codes (see the softmax below).
template <bool POW2, bool FASTP = false>
__global__ __launch_bounds__(64 * NW, 3) void attn_fwd_fp8_kernel(const AttnKernArgs a) {
  // Two (K tile, V tile) buffers as four separate objects that are only ever indexed statically: the compiler
  // then knows that a read of one buffer cannot alias the direct-to-LDS loads in flight to the other and does
  // not make it wait for them (with one array and a run-time buffer index every LDS read waited for vmcnt(0),
  // i.e. for the tile that had just been requested).
  __shared__ __attribute__((aligned(1024))) unsigned char sK0[K_TILE_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char sV0[V_TILE_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char sK1[K_TILE_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char sV1[V_TILE_BYTES];
  __shared__ int s_sel[LOCATE_WORDS];

#define FP8_BLOCK blockIdx.x
#include "attn_fwd_fp8_body.h"
#undef FP8_BLOCK
}

// The split items of a launch of the kernel above (a.split_*): brings the pieces' sums to a common maximum, adds them in the order
// of the keys, normalises, writes the rows.  Lanes and wavefronts as there, four workgroups per item, one for each 32 features, on the
// item's XCD.  Memory bound.
__global__ __launch_bounds__(64 * NW) void attn_fwd_fp8_merge_kernel(const AttnKernArgs a) {
  __shared__ int s_sel[LOCATE_WORDS];
  const int tid = threadIdx.x, l = tid & 63, i = l & 31, g = l >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int mb = (int)(blockIdx.x >> 3) & 3;
  const unsigned item = (blockIdx.x >> 5 << 3) | (blockIdx.x & 7u);
  const WorkItem wi = locate_work(a, BM, tid, s_sel, item + 8u * a.split_from);
  if (!wi.valid || wi.ke <= wi.ks || wi.q0 + 32 * w >= wi.qe) return;
  const int pieces = (int)a.split_pieces, row = 32 * w + i;
  const float* const base = a.partial + (long)item * pieces * SPLIT_FLOATS_FP8;
  float m = -__builtin_inff();
  for (int p = 0; p < pieces; ++p) m = fmaxf(m, base[(long)p * SPLIT_FLOATS_FP8 + 128 * 128 + 128 + row]);
  float sum = 0.f;
  f32x16 o;
#pragma unroll
  for (int v = 0; v < 16; ++v) o[v] = 0.f;
  for (int p = 0; p < pieces; ++p) {
    const float* const src = base + (long)p * SPLIT_FLOATS_FP8;
    const float f = __builtin_amdgcn_exp2f(src[128 * 128 + 128 + row] - m);
    sum += src[128 * 128 + row] * f;
    const f32x4* const acc = (const f32x4*)src + w * 1024 + l;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const f32x4 x = acc[(4 * mb + b) * 64];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[4 * b + e] += x[e] * f;
    }
  }
  store_block(wi.q0 + row < wi.qe, a.out + (long)(wi.q0 + row) * a.os_t + wi.o_head + 16 * g, mb, o, 1.f / sum);
  if (a.lse && mb == 0 && g == 0 && wi.q0 + row < wi.qe) a.lse[(long)wi.h * a.total_q + wi.q0 + row] = (m + __builtin_amdgcn_logf(sum)) * 0.6931471805599453f;
}

// ------------------------------------------------------------------------------------------------
// Quantiser: absmax per (chunk, head) -> scale = max(absmax, tiny) / 448; y = e4m3(clamp(x / scale)).
// ------------------------------------------------------------------------------------------------
constexpr int QT = 256;

__global__ __launch_bounds__(QT) void fill_zero_kernel(unsigned* p, int n) {
  const int i = blockIdx.x * QT + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// grid (slices, H, n_chunks); 16 lanes x 16 bytes per (token, head) row; result: max |x| bits in amax[c*H + h]
__global__ __launch_bounds__(QT) void absmax_kernel(const char* x, long xs_t, long xs_h, unsigned* amax, int T, int H,
                                                    int chunk_tokens) {
  __shared__ unsigned s_red[QT / 64];
  const int c = blockIdx.z, h = blockIdx.y;
  const int t_begin = c * chunk_tokens, t_end = min(T, t_begin + chunk_tokens);
  const int lane16 = threadIdx.x & 15, sub = threadIdx.x >> 4;
  unsigned m = 0u;
  for (int t = t_begin + blockIdx.x * (QT / 16) + sub; t < t_end; t += gridDim.x * (QT / 16)) {
    const u32x4 v = *(const u32x4*)(x + (long)t * xs_t + (long)h * xs_h + lane16 * 16);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      m = max(m, (v[j] << 16) & 0x7fffffffu);
      m = max(m, v[j] & 0x7fff0000u);
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o));
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int j = 1; j < QT / 64; ++j) m = max(m, s_red[j]);
    atomicMax(&amax[c * H + h], m);  // non-negative floats order like their bit patterns
  }
}

// absmax of a (chunk, head) group -> its scale
__device__ __forceinline__ float scale_of_absmax(float amax, float premul, int pow2) {
  float f = fmaxf(amax * fabsf(premul) / 448.f, 1e-12f);
  if (pow2) {  // round up to a power of two
    unsigned b = __builtin_bit_cast(unsigned, f);
    b = ((b >> 23) + ((b & 0x7fffffu) ? 1u : 0u)) << 23;
    f = __builtin_bit_cast(float, b);
  }
  return f;
}

__global__ __launch_bounds__(QT) void finalize_scales_kernel(float* scales, int n, float premul, int pow2) {
  const int i = blockIdx.x * QT + threadIdx.x;
  if (i >= n) return;
  scales[i] = scale_of_absmax(scales[i], premul, pow2);
}

// 16 bytes of bf16 (8 elements) -> 8 bytes of e4m3: y = sat(x * premul / sc)
__device__ __forceinline__ u32x2 quantize8(const u32x4 v, float premul, float sc) {
  float fv[8];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    fv[2 * j] = __builtin_bit_cast(float, v[j] << 16);
    fv[2 * j + 1] = __builtin_bit_cast(float, v[j] & 0xffff0000u);
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) fv[j] = fminf(fmaxf(fv[j] * premul / sc, -448.f), 448.f);
  u32x2 o;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    int u = 0;
    u = __builtin_amdgcn_cvt_pk_fp8_f32(fv[4 * j], fv[4 * j + 1], u, false);
    u = __builtin_amdgcn_cvt_pk_fp8_f32(fv[4 * j + 2], fv[4 * j + 3], u, true);
    o[j] = (unsigned)u;
  }
  return o;
}

// one thread per 8 elements
__global__ __launch_bounds__(QT) void quantize_kernel(const char* x, long xs_t, long xs_h, char* y, const float* scales,
                                                      int T, int H, int chunk_tokens, float premul) {
  const long gid = (long)blockIdx.x * QT + threadIdx.x;
  const long row = gid >> 4;
  const int part = (int)(gid & 15);
  if (row >= (long)T * H) return;
  const int t = (int)(row / H), h = (int)(row % H);
  const float sc = scales[(long)(t / chunk_tokens) * H + h];
  const u32x4 v = *(const u32x4*)(x + (long)t * xs_t + (long)h * xs_h + part * 16);
  *(u32x2*)(y + row * 128 + part * 8) = quantize8(v, premul, sc);
}

// The whole job in one launch with no memory beyond the inputs and outputs: a workgroup takes the absmax of its
// (chunk, head) group (a video chunk of one head is 5.5 MB at the 720p shape), reduces it through LDS, and
// quantises with the resulting scale.  To fill the chip when there are few groups, gridDim.z workgroups share a
// group: each of them takes the absmax of the WHOLE group (a maximum does not depend on the order, so all arrive
// at the same scale; the repeated reads are served by the caches, HBM sees the group once) and quantises its own
// slice of the rows; slice 0 writes the scale.  Groups that start at or after token n_first go to the second
// destination.
// Bound by what a CU pulls through its vector ALU and L1 in the first pass: hence two instructions per word there, not five.
// `apart`: each workgroup starts at its own slice and wraps round, so that they wait for different rows from memory and find
// the others' in L2, instead of all for the same ones.  Together, [9360, 8] rows in one group per head: 50.5 -> 41.4 us out of
// memory, 34.2 -> 29.4 out of the caches; [3120, 8] 22.0 -> 19.0; [86400, 8] in four (not apart) 165.8 -> 163.4.
constexpr int QT1 = 1024;
constexpr int QROWS = QT1 / 16;  // rows per pass of a workgroup
__global__ __launch_bounds__(QT1) void quantize_groups_kernel(const char* x, long xs_t, long xs_h, char* y, float* scales,
                                                              int T, int H, int chunk_tokens, float premul, int pow2,
                                                              int n_first, char* y2, float* scales2, int apart) {
  __shared__ unsigned s_red[QT1 / 64];
  const int h = blockIdx.x, c = blockIdx.y;
  const int t_begin = c * chunk_tokens, t_end = min(T, t_begin + chunk_tokens);
  const int lane16 = threadIdx.x & 15, sub = threadIdx.x >> 4;
  const char* const xcol = x + (long)h * xs_h + lane16 * 16;
  // (two magnitudes per word, which order like unsigned 16-bit integers: two instructions per word)
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  u16x2 mp = {0, 0};
  auto fold = [&](const u32x4 v) {
#pragma unroll
    for (int j = 0; j < 4; ++j) mp = __builtin_elementwise_max(mp, __builtin_bit_cast(u16x2, v[j] & 0x7fff7fffu));
  };
  constexpr int UN = 8;  // loads in flight per lane
  const int per = (t_end - t_begin + (int)gridDim.z - 1) / (int)gridDim.z;  // rows of a workgroup's slice
  auto absmax = [&](int from, int to) __attribute__((always_inline)) {
    int t = from + sub;
    for (; t + (UN - 1) * QROWS < to; t += UN * QROWS) {
      u32x4 v[UN];
#pragma unroll
      for (int u = 0; u < UN; ++u) v[u] = *(const u32x4*)(xcol + (long)(t + u * QROWS) * xs_t);
#pragma unroll
      for (int u = 0; u < UN; ++u) fold(v[u]);
    }
    for (; t < to; t += QROWS) fold(*(const u32x4*)(xcol + (long)t * xs_t));
  };
  const int start = apart ? min(t_end, t_begin + (int)blockIdx.z * per) : t_begin;
#pragma nounroll
  for (int part = 0; part < (apart ? 2 : 1); ++part) absmax(part ? t_begin : start, part ? start : t_end);
  unsigned m = (unsigned)max(mp[0], mp[1]) << 16;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o));
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = m;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < QT1 / 64; ++j) m = max(m, s_red[j]);  // non-negative floats order like their bit patterns
  const float sc = scale_of_absmax(__builtin_bit_cast(float, m), premul, pow2);
  const bool second = t_begin >= n_first;
  const int t_off = second ? n_first : 0;
  if (threadIdx.x == 0 && blockIdx.z == 0) (second ? scales2 : scales)[(long)(c - t_off / chunk_tokens) * H + h] = sc;
  // this workgroup's slice of the rows
  const int s_begin = t_begin + (int)blockIdx.z * per, s_end = min(t_end, s_begin + per);
  char* const ycol = (second ? y2 : y) + (long)h * 128 + lane16 * 8 - (long)t_off * H * 128;
  int t = s_begin + sub;
  for (; t + (UN - 1) * QROWS < s_end; t += UN * QROWS) {
    u32x4 v[UN];
#pragma unroll
    for (int u = 0; u < UN; ++u) v[u] = *(const u32x4*)(xcol + (long)(t + u * QROWS) * xs_t);
#pragma unroll
    for (int u = 0; u < UN; ++u) *(u32x2*)(ycol + (long)(t + u * QROWS) * H * 128) = quantize8(v[u], premul, sc);
  }
  for (; t < s_end; t += QROWS)
    *(u32x2*)(ycol + (long)t * H * 128) = quantize8(*(const u32x4*)(xcol + (long)t * xs_t), premul, sc);
}

// The quantiser with the largest magnitude of each row in hand (row_max [H, T], bf16 bits): a workgroup takes its group's scale from two
// bytes per row and quantises its slice, whose first rows are requested ahead of that.  Bound by HBM, below some thousand
// rows by two trips to memory.  Out of memory, a pass over the rows first / this: [9360, 8] in one group per head 46 / 11 us, [3000, 8] 13.5 / 7.3,
// [37440, 8] in four 61 / 31, [86400, 8] in four 142 / 59 (4.5 TB/s); the prologue pays 5, 1, 16 and 13 us for the maxima.
constexpr int UNK = 4;  // rows in flight per lane
__global__ __launch_bounds__(QT1) void quantize_row_max_kernel(const char* x, long xs_t, long xs_h, char* y, float* scales, int T, int H,
                                                               int chunk_tokens, float premul, int pow2, int n_first, char* y2,
                                                               float* scales2, const unsigned short* row_max) {
  __shared__ unsigned s_red[QT1 / 64];
  const int h = blockIdx.x, c = blockIdx.y;
  const int t_begin = c * chunk_tokens, t_end = (int)min((long)T, (long)t_begin + chunk_tokens);
  const int per = (t_end - t_begin + (int)gridDim.z - 1) / (int)gridDim.z;  // rows of a workgroup's slice
  const int s_begin = t_begin + (int)blockIdx.z * per, s_end = min(t_end, s_begin + per);
  if (s_begin >= s_end) return;  // (never slice 0, which writes the scale)
  const int lane16 = threadIdx.x & 15, sub = threadIdx.x >> 4;
  const char* const xcol = x + (long)h * xs_h + lane16 * 16;
  u32x4 v[UNK];
  auto request = [&](int t) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < UNK; ++u) v[u] = *(const u32x4*)(xcol + (long)min(t + u * QROWS, s_end - 1) * xs_t);
  };
  request(s_begin + sub);
  const unsigned short* const rm = row_max + (long)h * T;
  unsigned m = 0u;
#pragma unroll 8
  for (int t = t_begin + (int)threadIdx.x; t < t_end; t += QT1) m = max(m, (unsigned)rm[t]);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o));
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = m;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < QT1 / 64; ++j) m = max(m, s_red[j]);
  const float sc = scale_of_absmax(__builtin_bit_cast(float, m << 16), premul, pow2);
  const bool second = t_begin >= n_first;
  const int t_off = second ? n_first : 0;
  if (threadIdx.x == 0 && blockIdx.z == 0) (second ? scales2 : scales)[(long)(c - t_off / chunk_tokens) * H + h] = sc;
  char* const ycol = (second ? y2 : y) + (long)h * 128 + lane16 * 8 - (long)t_off * H * 128;
  for (int t = s_begin + sub;; t += UNK * QROWS) {
#pragma unroll
    for (int u = 0; u < UNK; ++u)
      if (t + u * QROWS < s_end) *(u32x2*)(ycol + (long)(t + u * QROWS) * H * 128) = quantize8(v[u], premul, sc);
    if (t + UNK * QROWS >= s_end) break;
    request(t + UNK * QROWS);
  }
}

}  // namespace

void launch_fp8_merge(const AttnKernArgs& a, hipStream_t stream) {
  if (const unsigned items = split_items(a)) {
    AttnKernArgs m = a;
    m.flags &= ~ATTN_ZERO_GAPS;  // (the rows no range covers are clear by now)
    hipLaunchKernelGGL(attn_fwd_fp8_merge_kernel, dim3(32u * items), dim3(64 * NW), 0, stream, m);
  }
}

hipError_t launch_attn_fwd_fp8(const AttnKernArgs& a, hipStream_t stream) {
  const unsigned grid = split_grid(a);
  if ((a.flags & 1) && (a.flags & 4))
    hipLaunchKernelGGL((attn_fwd_fp8_kernel<true, true>), dim3(grid), dim3(64 * NW), 0, stream, a);
  else if (a.flags & 1)
    hipLaunchKernelGGL(attn_fwd_fp8_kernel<true>, dim3(grid), dim3(64 * NW), 0, stream, a);
  else
    hipLaunchKernelGGL(attn_fwd_fp8_kernel<false>, dim3(grid), dim3(64 * NW), 0, stream, a);
  launch_fp8_merge(a, stream);
  return hipGetLastError();
}

hipError_t launch_quantize_fp8(const char* x, long x_stride_t, long x_stride_h, char* y, float* scales, int T, int H,
                               int chunk_tokens, float premul, int pow2_scales, int n_first, char* y2, float* scales2,
                               bool one_launch, int compute_units, hipStream_t stream, int* n_launches) {
  const int n_chunks = (T + chunk_tokens - 1) / chunk_tokens;
  const int n = n_chunks * H;
  *n_launches = 0;
  if (n <= 0) return hipSuccess;
  // Unless asked for, one launch only when a group is small enough for one workgroup's two passes and there are
  // enough groups to spread over the chip (a second destination is served by that kernel alone); both paths give
  // the same bytes.
  if (n_first < T || (min(chunk_tokens, T) <= 8192 && (n >= 64 || (long)T * H <= 65536))) one_launch = true;
  if (one_launch) {
    if (n_chunks > 65535) return hipErrorInvalidValue;
    // workgroups per group: towards one per CU over the launch (every workgroup reads its whole group for the absmax, so
    // a second one per CU doubles what a CU pulls through its caches: 162 instead of 105 us at the 720p shape), each
    // slice at least four passes long
    int share = (compute_units + n - 1) / n;
    share = max(1, min(share, min(16, min(chunk_tokens, T) / (4 * QROWS))));
    // the groups of an XCD (workgroup ids deal them out by head) have to stay in its 4 MB of L2 for that: beyond, starting
    // together is what reads them once
    const int apart = share > 1 && (double)min(chunk_tokens, T) * 256 * ((n + 7) / 8) <= 3.0e6;
    hipLaunchKernelGGL(quantize_groups_kernel, dim3(H, n_chunks, share), dim3(QT1), 0, stream, x, x_stride_t, x_stride_h, y,
                       scales, T, H, chunk_tokens, premul, pow2_scales, n_first, y2, scales2, apart);
    *n_launches = 1;
    return hipGetLastError();
  }
  hipLaunchKernelGGL(fill_zero_kernel, dim3((n + QT - 1) / QT), dim3(QT), 0, stream, (unsigned*)scales, n);
  const int rows_per_pass = QT / 16;
  int slices = (min(chunk_tokens, T) + rows_per_pass * 8 - 1) / (rows_per_pass * 8);
  slices = max(1, min(slices, 256));
  hipLaunchKernelGGL(absmax_kernel, dim3(slices, H, n_chunks), dim3(QT), 0, stream, x, x_stride_t, x_stride_h,
                     (unsigned*)scales, T, H, chunk_tokens);
  hipLaunchKernelGGL(finalize_scales_kernel, dim3((n + QT - 1) / QT), dim3(QT), 0, stream, scales, n, premul, pow2_scales);
  const long threads = (long)T * H * 16;
  hipLaunchKernelGGL(quantize_kernel, dim3((unsigned)((threads + QT - 1) / QT)), dim3(QT), 0, stream, x, x_stride_t,
                     x_stride_h, y, scales, T, H, chunk_tokens, premul);
  *n_launches = 4;
  return hipGetLastError();
}

hipError_t launch_quantize_fp8_row_max(const char* x, long x_stride_t, long x_stride_h, char* y, float* scales, int T, int H,
                                       int chunk_tokens, float premul, int pow2_scales, int n_first, char* y2, float* scales2,
                                       const unsigned short* row_max, int compute_units, hipStream_t stream) {
  if (T <= 0 || H <= 0) return hipSuccess;
  const int n_chunks = (int)(((long)T + chunk_tokens - 1) / chunk_tokens);
  if (n_chunks > 65535) return hipErrorInvalidValue;
  // two workgroups per CU over the launch, each slice at least one pass long
  const long n = (long)n_chunks * H;
  const int share = (int)max(1L, min((2L * compute_units + n - 1) / n, (long)min(chunk_tokens, T) / QROWS));
  hipLaunchKernelGGL(quantize_row_max_kernel, dim3(H, n_chunks, share), dim3(QT1), 0, stream, x, x_stride_t, x_stride_h, y, scales, T,
                     H, chunk_tokens, premul, pow2_scales, n_first, y2, scales2, row_max);
  return hipGetLastError();
}

}  // namespace magi
