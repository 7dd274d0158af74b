// Internal launch interface between the C-ABI layer (api.cpp) and the HIP kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace magi {

// Arguments of the range-attention forward kernels.  All strides are in BYTES.
struct AttnKernArgs {
  const char* q;
  const char* k;
  const char* v;
  const char* k2;
  const char* v2;
  char* out;
  float* lse;
  const int* q_ranges;
  const int* k_ranges;
  const float* q_scale;
  const float* k_scale;
  const float* v_scale;
  const float* q_norm_gamma;  // non-null: q is raw, normalise each (token, head) row while loading it
  const float* q_norm_beta;
  long qs_t, qs_h, ks_t, ks_h, vs_t, vs_h, os_t, os_h;
  // fp8, side segment with scale tables of its own: element offsets that lead from row c of k_scale / v_scale to
  // row c - scale_split_chunk of those tables (0 without them)
  long k2_scale_delta, v2_scale_delta;
  long os_g;     // byte stride between output head groups (out_group > 0)
  int out_group; // heads per output group, 0 = heads addressed by os_h alone
  long qs_b, os_b;  // strides between blocks of batch_rows q rows (batch_rows > 0)
  int batch_rows;   // 0: row r at r * qs_t / r * os_t
  int total_q, total_k, k_split;
  int n_ranges, ranges_mode, tiles_per_range;
  int block_m;  // q rows per workgroup (the launchers map it to an instantiation)
  int Hq, Hkv, G;
  int scale_chunk_tokens;
  int scale_split_chunk;  // first chunk served by the side segment's scale tables (INT_MAX without them)
  int flags;  // MAGI_ATTN_* bits of the public header, plus ATTN_BOUNDED / ATTN_SCALE_Q
  unsigned per_xcd;  // workgroups per XCD (the grid is 8 of these)
  float scale_log2;  // softmax_scale * log2(e)
  float q_norm_eps;
  int q_norm_kind;  // MAGI_NORM_LAYERNORM_1P / MAGI_NORM_RMSNORM_1P
  // Measured score bound (MAGI_ATTN_AUTO_BOUND): gate[0] / gate[1] = the largest squared length of a q row / a k row
  // as launch_row_norm_max left them.  A kernel that is handed a gate first tests whether
  // sqrt(gate[0] gate[1]) * scale_log2 * 1.01 <= MAGI_SCORE_BOUND_MAX and runs only if the answer equals
  // gate_want (the bounded-score kernel: 1, the online-softmax kernel launched behind it: 0).  NULL: no test.
  const float* gate;
  int gate_want;
  // Checked launches (MAGI_ATTN_CHECKED): four words per item, one per wavefront of the 256-row kernel
  int* verdict;
  // Items whose keys are shared by several workgroups (split_plan in api.cpp; the 256-row bf16 kernel and the fp8 kernel): the items from
  // position split_from of each XCD's list on, in split_pieces pieces each.  Piece p starts at tile n_tiles * (split_num +
  // p - 1) / split_den of the item's key range, piece 0 at tile 0.  `partial`: SPLIT_FLOATS floats per piece.
  float* partial;
  unsigned split_from, split_pieces, split_num, split_den;  // split_from: UINT_MAX = nothing is split
  // Online softmax, 128-row workgroups: the keys of every item in up to share_pieces pieces of share_tiles tiles each (0 or 1:
  // whole; `partial`: ONLINE_PARTIAL_FLOATS floats per item and piece).
  unsigned share_pieces, share_tiles;
  int waves;  // attn_fwd_bf16_waves.hip: wavefronts that share the keys of a workgroup's rows, 4 or 8
};
// online softmax: 128 rows x 128 accumulators, 128 row sums, 128 row maxima
constexpr int ONLINE_PARTIAL_FLOATS = 128 * 128 + 256;
// 256 rows x 128 accumulators, and the 256 row sums behind them
constexpr int SPLIT_FLOATS = 256 * 128 + 256;
// fp8: 128 rows x 128 accumulators, 128 row sums, 128 row maxima
constexpr int SPLIT_FLOATS_FP8 = 128 * 128 + 256;
// the items of one XCD's list that are split, and the workgroups of the launch
inline unsigned split_items(const AttnKernArgs& a) { return a.split_from < a.per_xcd ? a.per_xcd - a.split_from : 0u; }
inline unsigned split_grid(const AttnKernArgs& a) {
  const unsigned items = split_items(a);
  return 8u * (a.per_xcd - items + items * a.split_pieces);
}


// internal flag: the caller promised bounded scores (magi_attn_args.score_bound within MAGI_SCORE_BOUND_MAX)
constexpr int ATTN_BOUNDED = 1 << 8;
// internal flag (with ATTN_BOUNDED): q is unscaled, the kernel multiplies it by scale_log2 while loading it
constexpr int ATTN_SCALE_Q = 1 << 9;
// MAGI_ATTN_ZERO_UNCOVERED of the public header
constexpr int ATTN_ZERO_GAPS = 32;

hipError_t launch_attn_fwd_bf16(const AttnKernArgs& a, hipStream_t stream);
hipError_t launch_attn_fwd_bf16_r32(const AttnKernArgs& a, hipStream_t stream);
// One or two calls (job[1].per_xcd = 0: one), bounded scores, block_m 32: the wavefronts of a workgroup share the keys of 32 rows
struct AttnPairArgs {
  AttnKernArgs job[2];
  unsigned ahead;  // attn_fwd_bf16_x16.hip, attn_fwd_fp8_text.hip: workgroups of the first per XCD
};
hipError_t launch_attn_fwd_bf16_waves(const AttnPairArgs& p, hipStream_t stream);
hipError_t launch_attn_fwd_bf16_w64(const AttnKernArgs& a, hipStream_t stream);
// (with items to split: and behind it the launch that adds their pieces up)
hipError_t launch_attn_fwd_bf16_x16(const AttnKernArgs& a, hipStream_t stream, bool merge = true);
hipError_t launch_attn_fwd_bf16_merge(const AttnKernArgs& a, hipStream_t stream);  // that launch by itself
// and it beside a call in 128-row tiles, bounded scores, raw q, nothing to split
hipError_t launch_attn_text_merge(const AttnPairArgs& p, hipStream_t stream);
// two such calls in 256-row workgroups, the second without items to split, q as it is or raw
hipError_t launch_attn_fwd_bf16_x16_pair(const AttnPairArgs& p, hipStream_t stream);
// the bounded-score kernel without a promise, and behind it the launch that repeats what it could not be trusted with
hipError_t launch_attn_fwd_bf16_checked(const AttnKernArgs& a, int compute_units, hipStream_t stream);
hipError_t launch_attn_fwd_fp8(const AttnKernArgs& a, hipStream_t stream);
void launch_fp8_merge(const AttnKernArgs& a, hipStream_t stream);  // the launch behind one with items to split
// a call of e4m3 rows with power-of-two scales and one of bf16 rows in 128-row tiles, bounded scores, raw q, nothing to split
hipError_t launch_attn_fwd_fp8_text(const AttnPairArgs& p, hipStream_t stream);
// ws[0..3] = 0 (a kernel, not a memset: the call may be under graph capture)
hipError_t launch_gate_init(unsigned* ws, hipStream_t stream);
// *out_bits = max(*out_bits, bit pattern of the largest sum of squares over a [T, H, 128] bf16 tensor's rows);
// strides in BYTES.  Bit patterns of non-negative floats order like the floats, and a NaN row ends up on top.
hipError_t launch_row_norm_max(const char* x, long stride_t, long stride_h, int T, int H, unsigned* out_bits,
                               hipStream_t stream);

struct PrologueKernArgs {
  const char* q_raw;
  const char* k_raw;
  const char* v_raw;
  const float* rope;
  const float* gq;
  const float* bq;
  const float* gk;
  const float* bk;
  char* q_out;
  char* kv_out;
  char* kv_tail;
  long q_raw_stride_t, k_raw_stride_t, v_raw_stride_t;  // bytes
  long kv_stride_t, kv_tail_stride_t;                   // bytes
  int S, n_cache_rows;
  int Hq, Hkv, R2;
  int norm_kind;
  float eps;
  int batch;
  float q_premul;  // factor on q before the bf16 rounding (1 = none)
  int out_fp8;     // q and k leave as e4m3 (kv_out / kv_tail then hold K rows only, strides in bytes); v untouched
  float q_inv_scale, k_inv_scale;  // out_fp8: 1 / the constant scale of q (after q_premul) and of k
  unsigned short* v_row_max;       // out_fp8, or nullptr: [Hkv, S] receives the largest magnitude of each row of v, as bf16 bits
};
hipError_t launch_prologue(const PrologueKernArgs& a, hipStream_t stream);

// The four projections as one GEMM with the prologue as its epilogue.  Strides in BYTES.
struct QkvGemmKernArgs {
  const char* x;  // [S, K] bf16
  const char* w;  // [(Hq + 2 Hkv + Hqx) * 128, K] bf16, rows ordered q | k | v | qx heads
  const float* rope;
  const float* gq;
  const float* bq;
  const float* gk;
  const float* bk;
  char* q_out;
  char* kv_out;
  char* kv_tail;
  char* qx_out;
  long x_stride, w_stride;
  long kv_stride_t, kv_tail_stride_t;
  int S, K, n_cache_rows;
  int Hq, Hkv, Hqx;
  int norm_kind;
  float eps;
  int batch;
  float q_premul;
  int n_row_tiles, n_col_tiles;  // filled by the launcher
};
hipError_t launch_qkv_gemm_prologue(const QkvGemmKernArgs& a, hipStream_t stream);

// The projections of a small layer and what comes around them, in one launch (small_proj.hip).  Strides in BYTES.
struct SmallProjKernArgs {
  // S rows of the layer input (0: none): LayerNorm (ln_w null: as they are), then columns [q | k | v | qx] heads of w [.., K]
  const char* x;
  const char* w;
  const char* ln_w;
  const char* ln_b;
  const float* rope;
  const float* gq;
  const float* bq;
  const float* gk;
  const float* bk;
  char* q_out;
  char* kv_out;
  char* kv_tail;
  char* qx_out;
  // T text rows (0: none): columns [head][K | V] of w_text [2 Hkv 128, Kt], K normed
  const char* text;
  const char* w_text;
  const float* gkx;
  const float* bkx;
  char* text_out;
  long x_stride, text_stride, kv_stride_t, kv_tail_stride_t;
  int S, K, T, Kt, n_cache_rows;
  int Hq, Hkv, Hqx, R2;
  int ln_fp32, batch;
  float ln_eps, eps, q_premul;
  // out_fp8: q and k leave as e4m3 (kv_out / kv_tail then hold K rows only, strides in bytes), v as it is in rows of v_out [S, Hkv, 128] bf16
  int out_fp8;
  float q_inv_scale, k_inv_scale;  // out_fp8: 1 / the constant scale of q (after q_premul) and of k
  char* v_out;
  int hidden_blocks;  // filled by the launcher
};
hipError_t launch_small_proj(const SmallProjKernArgs& a, int compute_units, hipStream_t stream);

hipError_t launch_head_norm(const char* x, long x_stride_t, long x_stride_h, const float* gamma, const float* beta,
                            char* y, int S, int H, int norm_kind, float eps, hipStream_t stream);
hipError_t launch_layer_norm(const char* x, long x_stride, const void* w, const void* b, int params_fp32, char* y,
                             long y_stride, long rows, int cols, float eps, hipStream_t stream);
// LayerNorm of x [rows, cols] bf16 leaving as n_out e4m3 tensors [rows, cols] (contiguous): y[k] = e4m3(bf16(clamp(bf16(norm)
// / scale[k], +-448))), scale[k] [cols] fp32.  xs in BYTES.
struct LnQuantKernArgs {
  const char* x;
  long xs;
  const char* w;
  const char* b;
  const float* scale[4];
  char* y[4];
  long rows;
  int cols, n_out;
  float eps;
};
hipError_t launch_layer_norm_quant(const LnQuantKernArgs& a, int params_fp32, int compute_units, hipStream_t stream);
// y = e4m3(bf16(clamp(x / scale, +-448))): x [rows, cols] bf16, y [rows, cols] e4m3, strides in BYTES
hipError_t launch_div_clamp(const char* x, long x_stride, const float* scale, int per_column, char* y, long y_stride,
                            long rows, int cols, hipStream_t stream);
hipError_t launch_rotary(const void* x, const float* cos, const float* sin, void* y, int B, int S, int H, int D,
                         int R2, int is_bf16, hipStream_t stream);
// Rows below n_first go to y / scales, the rest (row index and chunk index counted from n_first, a multiple of
// chunk_tokens) to y2 / scales2.  one_launch: always the single-launch kernel (else only where it is the faster).
// *n_launches receives the number of kernels launched.
hipError_t launch_quantize_fp8(const char* x, long x_stride_t, long x_stride_h, char* y, float* scales, int T, int H,
                               int chunk_tokens, float premul, int pow2_scales, int n_first, char* y2, float* scales2,
                               bool one_launch, int compute_units, hipStream_t stream, int* n_launches);
// The same with the largest magnitude of each row in hand: row_max [H, T], bf16 bits
hipError_t launch_quantize_fp8_row_max(const char* x, long x_stride_t, long x_stride_h, char* y, float* scales, int T, int H,
                                       int chunk_tokens, float premul, int pow2_scales, int n_first, char* y2, float* scales2,
                                       const unsigned short* row_max, int compute_units, hipStream_t stream);

}  // namespace magi
