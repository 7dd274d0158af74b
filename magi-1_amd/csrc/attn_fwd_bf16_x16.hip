// Range attention forward, bf16, bounded scores, 64 query rows per wavefront on v_mfma_f32_16x16x32_bf16,
// for gfx950 (MI355X).
//
// Same algorithm, tile loop and LDS staging as attn_fwd_bf16_w64.hip (S^T = K Q^T and O^T = V^T P^T, p = 2^score
// without a running maximum, K / V tiles of 64 keys double buffered in LDS by direct global->LDS loads, transposing
// LDS reads for V^T), on the other bf16 MFMA shape.  Why: this part runs at its board power limit, and a
// 16x16x32 MFMA spends less energy per FLOP than a 32x32x16 one (it sums 32 products into each accumulator element
// instead of 16, so half as many fp32 accumulator reads and writes per FLOP): an MFMA-only loop on random operands
// holds ~14 % more FLOP/s at the limit with this shape, measured on the same box.
//
// Shape of a wave's work.  A wave owns 64 query rows as FOUR blocks of 16 (qb).  Lane l = (n = l % 16, g = l / 16):
//   S^T block (16 keys x 16 queries) = K[16 keys x 32 d] Q^T[32 d x 16 queries], accumulated over 4 d steps (kk):
//       A = K fragment : lane holds K[key n][d = 32 kk + 8 g .. +8]          (one ds_read_b128, 1 KB per wave)
//       B = Q fragment : lane holds Q[query n][d = 32 kk + 8 g .. +8]        (registers, 64 in all)
//       D             : lane holds S^T[key 4 g + r][query n], r = 0..3
//     every K fragment feeds the four query blocks: 4 MFMAs per 1 KB read from LDS, the same bytes per FLOP as the
//     32x32x16 kernel's two.
//   O^T block (16 d x 16 queries) += V^T[16 d x 32 keys] P^T[32 keys x 16 queries]:
//       B = P fragment : lane holds the probabilities of query n for 8 keys; the D layout above hands a lane keys
//                        4 g + r of each 16-key block, so the 32 keys of a step are two key blocks (kb = 0, 1) and
//                        operand element e is key 16 (e / 4) + 4 g + e % 4: two S^T accumulators, packed, no
//                        lane exchange
//       A = V^T fragment: lane holds V[those 8 keys][d = 16 db + n]: two transposing reads (ds_read_b64_tr_b16),
//                        one per key block; feeds the four query blocks
//       D             : lane holds O^T[d = 16 db + 4 g + r][query n]
// Registers: Q 64 + O 128 + the scores of one 32-key half tile 32 + a ring of four operand fragments 16.
//
// The epilogue goes through LDS (the tile slots are free by then): every wave writes its 64 x 128 normalised
// outputs as bf16 rows and reads them back 16 bytes per lane, so that 16 consecutive lanes store one whole 256-byte
// row: every global store instruction writes four complete rows.
#include "attn_bf16_merge.h"

namespace magi {
namespace {

constexpr int ROW_BYTES = 256;  // D = 128 bf16
constexpr int BN = 64;          // keys per LDS tile
// A tile in LDS is 16 groups of four rows (what one wave-wide direct load fills: 64 lanes x 16 bytes).  The groups are
// spaced by a little more than their 1024 bytes, so that consecutive groups start in different banks and the operand
// reads need no address arithmetic beyond constant offsets (see the read bases below).
constexpr int K_GROUP = 1024 + 64, V_GROUP = 1024 + 128;
constexpr int K_TILE_BYTES = (BN / 4) * K_GROUP, V_TILE_BYTES = (BN / 4) * V_GROUP;

typedef float f32x4v __attribute__((ext_vector_type(4)));

// base ^ M computed where it is used (one v_xor per operand read instead of a register per address across the tile
// loop): inline assembly that also names a loop-variant scalar (`tie`, unused by the instruction) and a tag unique
// to the call site, so that the result is neither hoisted out of the loop nor shared.  Not `asm volatile`: behind a
// volatile statement the compiler waits for ALL outstanding LDS reads instead of counting them.
template <int M, int TAG>
__device__ __forceinline__ int swz(int base, int tie) {
  if constexpr (M == 0) return base;
  int r;
  asm("v_xor_b32 %0, %1, %2" : "=v"(r) : "n"(M), "v"(base), "s"(tie), "n"(TAG));
  return r;
}

// K as the A operand of the score MFMAs: rows 16 KB + n of a tile, features 32 KK + 8 g .. +8 (base: see the kernel)
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

// QMODE: what q holds.  0: q as the score MFMAs take it (pre-scaled by the caller).  1: the raw query projection:
// per-(token, head) norm in fp32 while it is loaded, times the softmax scale, one rounding to bf16.  2: unscaled
// bf16 q as the reference's callers pass it: multiplied by the softmax scale while it is loaded (a second rounding
// to bf16: 2^-9 relative per element, the size of the first).
// order in which the feature blocks of V^T are visited: 0, 4, 1, 5, 2, 6, 3, 7
constexpr int v_block(int i) { return (i >> 1) + 4 * (i & 1); }

// Q_CHECK: unscaled bf16 q as it is, the scores multiplied by the softmax scale in fp32 (as the online-softmax kernel does),
// and nobody's promise that they are bounded: see CHECK.
// Q_EITHER: as it is, or raw where the call has norm parameters (a launch of two calls).
constexpr int Q_AS_IS = 0, Q_NORM = 1, Q_SCALE = 2, Q_CHECK = 3, Q_EITHER = 4;


// CHECK (QMODE Q_CHECK): nobody has promised that the scores are bounded.  The kernel computes as if they were, and each wavefront
// leaves a verdict on its 64 rows in a.verdict[4 * item + wavefront]: they are good where SUM_MIN <= row sum <= SUM_MAX
// (then no score is above 64, and the terms that underflow are below 2^-90 of the sum; an overflow leaves inf or NaN in
// it) and every accumulator is finite (2^64 times a value above 2^63 is not).  The lower end keeps products with values
// down to 2^-110 normal numbers.  attn_fwd_bf16_redo_kernel, launched behind it,
// computes the others again with a running maximum.
//
// A launch whose last round of workgroups leaves slots (two per CU) empty has the keys of that round's items shared by
// several workgroups each (a.split_*, split_plan in api.cpp).  Without a running maximum the pieces simply add up: each leaves its
// unnormalised accumulators and row sums in fp32, attn_fwd_bf16_merge_kernel adds them in the order of the keys.
__device__ __forceinline__ void store_partial_zero(float* out, int w, int l) {
  f32x4v* const dst = (f32x4v*)out + w * 2048 + l;
#pragma unroll
  for (int i = 0; i < 32; ++i) dst[i * 64] = f32x4v{0.f, 0.f, 0.f, 0.f};
  out[256 * 128 + 64 * w + l] = 0.f;
}

// QB: query blocks of 16 rows per wavefront: 4, or 2 for launches that are better dealt in smaller pieces (tile_rows in api.cpp).
// A row's result does not depend on it, bit for bit.
#define X16_BLOCK blockIdx.x
template <int QMODE, int QB = 4>
__global__ __launch_bounds__(256, 2) void attn_fwd_bf16_x16_kernel(const AttnKernArgs a) {
#include "attn_fwd_bf16_x16_body.h"
}
#undef X16_BLOCK

// Two calls that do not depend on each other: the workgroups of the second, a text attention of a few tiles each, behind those of the first.
// A launch of the core attention alone ends with slots empty one after the other for the length of a workgroup, and the text's launch, which
// waits for all of it, with a round of its own that starts and ends together: in one launch the short workgroups fill the end of the long ones.
// 24 query and 8 key heads, 100 to 400 text rows, core and text one by one -> together, the layer around them included: 6240 rows 1125 -> 1098 us,
// 6480 rows 2216 -> 2184, 16200 rows 7670 -> 7426, 21600 rows x 2 chunks 29695 -> 29522.  Both ways of taking q in one kernel cost
// 250 registers and no scratch (the single ones: 253 and 255).
#define X16_BLOCK (second ? (pos - ahead) << 3 | (blockIdx.x & 7u) : blockIdx.x)
__global__ __launch_bounds__(256, 2) void attn_fwd_bf16_x16_pair_kernel(const AttnPairArgs) {
  constexpr int QMODE = Q_EITHER, QB = 4;
  const AttnPairArgs& pair = *(const AttnPairArgs*)__builtin_amdgcn_kernarg_segment_ptr();  // (see attn_fwd_bf16_waves.hip)
  const unsigned pos = blockIdx.x >> 3, ahead = pair.ahead;
  const bool second = pos >= ahead;
  const AttnKernArgs& a = pair.job[second ? 1 : 0];
#include "attn_fwd_bf16_x16_body.h"
}
#undef X16_BLOCK

// (see attn_bf16_merge.h)
template <bool CHECK>
__global__ __launch_bounds__(256) void attn_fwd_bf16_merge_kernel(const AttnKernArgs a) {
  __shared__ int s_sel[LOCATE_WORDS];
  if (gate_closed(a)) return;
  merge_pieces<CHECK>(a, blockIdx.x, s_sel);
}

// The rows that a CHECK launch of the kernels above could not be trusted with, again, with a running maximum: same ranges,
// tiles and items.  A workgroup goes through every gridDim.x-th block of that launch, 64 verdicts at a time, and does the
// flagged ones (usually none: the launch then costs one look at 16 bytes per 256 rows and head).  32 rows per wavefront
// at a time, the two halves of its 64 one after the other.  The maximum of a row is raised only when a score comes out
// more than RAISE above it: within that sums and products keep their full precision (values up to 2^110 do not
// overflow them), and rescaling the accumulators is rare.
__global__ __launch_bounds__(256, 2) void attn_fwd_bf16_redo_kernel(const AttnKernArgs a) {
  constexpr int NW = 4, BM = 64 * NW, LOADS = BN / (4 * NW);
  constexpr float RAISE = 8.f;
  __shared__ __attribute__((aligned(1024))) unsigned char sK0[K_TILE_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char sV0[V_TILE_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char sK1[K_TILE_BYTES];
  __shared__ __attribute__((aligned(1024))) unsigned char sV1[V_TILE_BYTES];
  __shared__ int s_sel[LOCATE_WORDS];
  const int tid = threadIdx.x, l = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned blocks = 8u * a.per_xcd;
  for (unsigned base = blockIdx.x; base < blocks; base += 64u * gridDim.x) {
    const unsigned mine = base + (unsigned)l * gridDim.x;
    unsigned kvh, hg, rslot, tile_;
    bool flagged = false;
    if (mine < blocks && decode_block(a, mine, kvh, hg, rslot, tile_)) {
      const u32x4 v = *(const u32x4*)(a.verdict + 4 * (long)item_of(a, kvh, hg, rslot, tile_));
      flagged = (v[0] | v[1] | v[2] | v[3]) != 0;
    }
    for (unsigned long todo = __builtin_amdgcn_ballot_w64(flagged); todo; todo &= todo - 1) {
      __syncthreads();  // (s_sel and the tile slots are free again)
      const WorkItem wi = locate_work(a, BM, tid, s_sel, base + (unsigned)__builtin_ctzl(todo) * gridDim.x);
      if (!wi.valid || wi.ke <= wi.ks) continue;  // (a tile beyond its range has no verdict; one without keys is done)
      const int qe = wi.qe, ks = wi.ks, ke = wi.ke, n_tiles = (ke - ks + BN - 1) / BN;
      const int row0 = wi.q0 + 64 * w;
      const bool wave_on = row0 < qe && __builtin_amdgcn_readfirstlane(a.verdict[4 * (long)wi.item + w]) != 0;
      // one row per 16 lanes, four rows per load, each row through the segment it lives in, clamped to the last key
      auto issue_mat = [&](int k0, unsigned char* tile_base, bool is_v) __attribute__((always_inline)) {
        const long st = is_v ? a.vs_t : a.ks_t;
        const char* const col = is_v ? a.v + (long)wi.kvh * a.vs_h : a.k + (long)wi.kvh * a.ks_h;
        const char* const col2 = is_v ? a.v2 + (long)wi.kvh * a.vs_h : a.k2 + (long)wi.kvh * a.ks_h;
        const int group = is_v ? V_GROUP : K_GROUP, lr = l >> 4, sl = l & 15;
        const int chunk = is_v ? (sl ^ (lr << 1)) : (sl ^ lr);
#pragma unroll
        for (int j = 0; j < LOADS; ++j) {
          const int row = min(k0 + 4 * w + lr + 4 * NW * j, ke - 1);
          const char* p = row < a.k_split ? col + (long)row * st : col2 + (long)(row - a.k_split) * st;
          __builtin_amdgcn_global_load_lds(GLOBAL_PTR(p + chunk * 16), LDS_PTR(void, tile_base + (w + NW * j) * group), 16, 0, 0);
        }
      };
#pragma nounroll
      for (int half = 0; half < 2; ++half) {
        const int rh = row0 + 32 * half;
        const bool on = wave_on && rh < qe;
        const int n = l & 15, g = l >> 4;
        const int base_k = (n >> 2) * K_GROUP + (n & 3) * ROW_BYTES + ((g ^ (n & 3)) << 4);
        const int base_v = g * V_GROUP + (n >> 2) * ROW_BYTES + ((n >> 2) << 5) + ((n & 3) << 3);
        bf16x8 q2[2][4];
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
          const int qr = min(rh + 16 * qb + n, qe - 1);
          const char* qp = a.q + row_offset(a, qr, a.qs_t, a.qs_b) + (long)wi.h * a.qs_h + g * 16;
#pragma unroll
          for (int kk = 0; kk < 4; ++kk) q2[qb][kk] = *(const bf16x8*)(qp + kk * 64);
        }
        f32x4v o2[8][2];
#pragma unroll
        for (int db = 0; db < 8; ++db)
#pragma unroll
          for (int qb = 0; qb < 2; ++qb) o2[db][qb] = f32x4v{0.f, 0.f, 0.f, 0.f};
        float sum2[2] = {0.f, 0.f}, m2[2] = {0.f, 0.f};
        bool first = true;
        auto tile = [&](const unsigned char* Kt, const unsigned char* Vt, int k0) __attribute__((always_inline)) {
          static_for<0, 2>([&](auto tc) __attribute__((always_inline)) {
            constexpr int t = decltype(tc)::value;
            if (k0 + 32 * t >= ke) return;
            f32x4v s2[2][2];
            static_for<0, 2>([&](auto kc) __attribute__((always_inline)) {
              constexpr int kb = decltype(kc)::value;
#pragma unroll
              for (int qb = 0; qb < 2; ++qb) s2[kb][qb] = f32x4v{0.f, 0.f, 0.f, 0.f};
              static_for<0, 4>([&](auto kkc) __attribute__((always_inline)) {
                const bf16x8 kf = read_k<2 * t + kb, decltype(kkc)::value>(Kt, base_k);
#pragma unroll
                for (int qb = 0; qb < 2; ++qb)
                  s2[kb][qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, q2[qb][decltype(kkc)::value], s2[kb][qb], 0, 0, 0);
              });
            });
            float mx[2];
            bool up = first;
#pragma unroll
            for (int qb = 0; qb < 2; ++qb) {
              mx[qb] = -__builtin_inff();
#pragma unroll
              for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                  s2[kb][qb][r] = s2[kb][qb][r] * a.scale_log2 - m2[qb];
                  if (k0 + 32 * t + 16 * kb + 4 * g + r >= ke) s2[kb][qb][r] = -__builtin_inff();  // (the ragged end)
                  mx[qb] = fmaxf(mx[qb], s2[kb][qb][r]);
                }
              up |= __builtin_amdgcn_ballot_w64(mx[qb] > RAISE) != 0;
            }
            if (up) {
#pragma unroll
              for (int qb = 0; qb < 2; ++qb) {
                float m = fmaxf(mx[qb], __shfl_xor(mx[qb], 16));  // (the four lanes of a query)
                m = fmaxf(m, __shfl_xor(m, 32));
                const float delta = (first || m > RAISE) ? m : 0.f;
                const float alpha = first ? 1.f : __builtin_amdgcn_exp2f(-delta);
                m2[qb] += delta;
                sum2[qb] *= alpha;
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) s2[kb][qb] -= delta;
#pragma unroll
                for (int db = 0; db < 8; ++db) o2[db][qb] *= alpha;
              }
              first = false;
            }
            u32x4 p2[2];
#pragma unroll
            for (int qb = 0; qb < 2; ++qb)
#pragma unroll
              for (int kb = 0; kb < 2; ++kb) {
                float p[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) p[r] = __builtin_amdgcn_exp2f(s2[kb][qb][r]);
                sum2[qb] += (p[0] + p[1]) + (p[2] + p[3]);
                p2[qb][2 * kb] = pack_bf16x2(p[0], p[1]);
                p2[qb][2 * kb + 1] = pack_bf16x2(p[2], p[3]);
              }
            __builtin_amdgcn_sched_barrier(0);
            static_for<0, 8>([&](auto dbc) __attribute__((always_inline)) {
              const bf16x8 vf = read_v<t, decltype(dbc)::value>(Vt, base_v, k0);
#pragma unroll
              for (int qb = 0; qb < 2; ++qb)
                o2[decltype(dbc)::value][qb] =
                    __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, __builtin_bit_cast(bf16x8, p2[qb]), o2[decltype(dbc)::value][qb], 0, 0, 0);
            });
          });
        };
        __syncthreads();  // (every wave is done with the tile slots of the half before)
        issue_mat(ks, sK0, false);
        issue_mat(ks, sV0, true);
        for (int j = 0; j < n_tiles; j += 2) {
          wait_vmcnt<0>();
          __syncthreads();
          if (j + 1 < n_tiles) {
            issue_mat(ks + (j + 1) * BN, sK1, false);
            issue_mat(ks + (j + 1) * BN, sV1, true);
          }
          if (on) tile(sK0, sV0, ks + j * BN);
          if (j + 1 >= n_tiles) break;
          wait_vmcnt<0>();
          __syncthreads();
          if (j + 2 < n_tiles) {
            issue_mat(ks + (j + 2) * BN, sK0, false);
            issue_mat(ks + (j + 2) * BN, sV0, true);
          }
          if (on) tile(sK1, sV1, ks + (j + 1) * BN);
        }
        if (!on) continue;
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
          float sum = sum2[qb];
          sum += __shfl_xor(sum, 16);
          sum += __shfl_xor(sum, 32);
          const float inv = 1.f / sum;
          const int q_row = rh + 16 * qb + n;
          if (q_row >= qe) continue;
          char* const op = a.out + row_offset(a, q_row, a.os_t, a.os_b) + wi.o_head + 8 * g;
#pragma unroll
          for (int db = 0; db < 8; ++db)
            *(u32x2*)(op + 32 * db) = u32x2{pack_bf16x2(o2[db][qb][0] * inv, o2[db][qb][1] * inv),
                                            pack_bf16x2(o2[db][qb][2] * inv, o2[db][qb][3] * inv)};
          if (a.lse && g == 0) a.lse[(long)wi.h * a.total_q + q_row] = (m2[qb] + __builtin_amdgcn_logf(sum)) * 0.6931471805599453f;
        }
      }
    }
  }
}

}  // namespace

namespace {
template <bool CHECK>
void launch_merge(const AttnKernArgs& a, hipStream_t stream) {
  if (const unsigned items = split_items(a)) {
    AttnKernArgs m = a;
    m.flags &= ~ATTN_ZERO_GAPS;  // (the rows no range covers are clear by now)
    hipLaunchKernelGGL(attn_fwd_bf16_merge_kernel<CHECK>, dim3(8u * items * MERGE_SHARES<CHECK>), dim3(256), 0, stream, m);
  }
}
}  // namespace

hipError_t launch_attn_fwd_bf16_x16(const AttnKernArgs& a, hipStream_t stream, bool merge) {
  const dim3 grid(split_grid(a));
  if (a.block_m == 128) {
    if (a.q_norm_gamma)
      hipLaunchKernelGGL((attn_fwd_bf16_x16_kernel<Q_NORM, 2>), grid, dim3(256), 0, stream, a);
    else if (a.flags & ATTN_SCALE_Q)
      hipLaunchKernelGGL((attn_fwd_bf16_x16_kernel<Q_SCALE, 2>), grid, dim3(256), 0, stream, a);
    else
      hipLaunchKernelGGL((attn_fwd_bf16_x16_kernel<Q_AS_IS, 2>), grid, dim3(256), 0, stream, a);
    return hipGetLastError();
  }
  if (a.q_norm_gamma)  // raw q, normalised while it is loaded (cross attention)
    hipLaunchKernelGGL(attn_fwd_bf16_x16_kernel<Q_NORM>, grid, dim3(256), 0, stream, a);
  else if (a.flags & ATTN_SCALE_Q)  // unscaled q, scaled while it is loaded (the reference-shaped callables)
    hipLaunchKernelGGL(attn_fwd_bf16_x16_kernel<Q_SCALE>, grid, dim3(256), 0, stream, a);
  else
    hipLaunchKernelGGL(attn_fwd_bf16_x16_kernel<Q_AS_IS>, grid, dim3(256), 0, stream, a);
  if (merge) launch_merge<false>(a, stream);
  return hipGetLastError();
}

hipError_t launch_attn_fwd_bf16_merge(const AttnKernArgs& a, hipStream_t stream) {
  launch_merge<false>(a, stream);
  return hipGetLastError();
}

hipError_t launch_attn_fwd_bf16_x16_pair(const AttnPairArgs& p, hipStream_t stream) {
  AttnPairArgs pair = p;
  pair.ahead = split_grid(p.job[0]) / 8u;
  hipLaunchKernelGGL(attn_fwd_bf16_x16_pair_kernel, dim3(split_grid(p.job[0]) + 8u * p.job[1].per_xcd), dim3(256), 0, stream, pair);
  launch_merge<false>(p.job[0], stream);
  return hipGetLastError();
}

hipError_t launch_attn_fwd_bf16_checked(const AttnKernArgs& a, int compute_units, hipStream_t stream) {
  const dim3 grid(split_grid(a));
  // (two workgroups per CU, a multiple of eight so that a block keeps its XCD)
  const unsigned most = (unsigned)(compute_units / 4) * 8u;
  const unsigned blocks = 8u * a.per_xcd;
  const dim3 again(blocks < most || most == 0 ? blocks : most);
  hipLaunchKernelGGL(attn_fwd_bf16_x16_kernel<Q_CHECK>, grid, dim3(256), 0, stream, a);
  launch_merge<true>(a, stream);
  AttnKernArgs r = a;
  r.flags &= ~ATTN_ZERO_GAPS;  // (as in launch_merge)
  hipLaunchKernelGGL(attn_fwd_bf16_redo_kernel, again, dim3(256), 0, stream, r);
  return hipGetLastError();
}

}  // namespace magi
