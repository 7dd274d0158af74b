// Device-side pieces shared by the range-attention kernels (gfx950): vector types, the mapping from a
// workgroup to its piece of work, and small helpers.  Every kernel that includes this file decomposes the
// launch the same way, so the host side (api.cpp) sizes one grid for all of them.
#pragma once
#include "kernels.h"
#include "wave_ops.h"

#include <type_traits>

namespace magi {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

#define LDS_PTR(T, p) ((T __attribute__((address_space(3)))*)(p))
#define GLOBAL_PTR(p) ((const __attribute__((address_space(1))) void*)(p))

constexpr int MAX_SORT = 256;  // ranges are ranked by key span inside the kernel up to this many

__device__ __forceinline__ unsigned pack_bf16x2(float a, float b) {
  f32x2 x = {a, b};
  bf16x2 r = __builtin_convertvector(x, bf16x2);
  return __builtin_bit_cast(unsigned, r);
}

// range i of a device-side range list (pairs or cumulative), clamped to [0, total]
__device__ __forceinline__ void load_range(const int* r, int mode, int i, int total, int& s, int& e) {
  if (mode == 0) {
    s = r[2 * i];
    e = r[2 * i + 1];
  } else {
    s = r[i];
    e = r[i + 1];
  }
  s = max(0, min(s, total));
  e = max(s, min(e, total));
}

// f(integral_constant<int, I>) for I = B .. E-1, unrolled at compile time
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// s_waitcnt vmcnt(N), leaving the other counters alone
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
  asm volatile("" ::: "memory");
}

// Workgroup barrier that leaves this wavefront's direct loads into LDS in flight (__syncthreads() waits for every one of them,
// s_waitcnt vmcnt(0)); its LDS reads and writes are over.
__device__ __forceinline__ void barrier_loads_in_flight() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// p0 + p1 + acc for a packed pair of bf16 values
__device__ __forceinline__ float pair_sum(unsigned pk, float acc) {
  const bf16x2 one = {(__bf16)1.0f, (__bf16)1.0f};
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pk), one, acc, false);
}

// A launch behind a measured score bound: true when this kernel is not the one the bound selects (every thread of
// the grid sees the same two values, so the whole launch returns).  NaN lengths fail the comparison and select the
// online-softmax kernel.
__device__ __forceinline__ bool gate_closed(const AttnKernArgs& a) {
  if (!a.gate) return false;
  const float b = __builtin_sqrtf(a.gate[0] * a.gate[1]) * a.scale_log2 * 1.01f;
  const bool fits = b <= 64.0f;  // MAGI_SCORE_BOUND_MAX
  return fits != (a.gate_want != 0);
}

// What one workgroup works on: q rows [q0, min(q0 + BM, qe)) of head h against keys [ks, ke) of kv head kvh.
struct WorkItem {
  int h, kvh;
  int q0, qe, ks, ke;
  long o_head;  // byte offset of head h inside a row of `out`
  int item;     // (h, range slot, q tile) in that order: the same work in every launch over the same ranges and tiles
  bool valid;   // false: nothing to do (grid padding, or the q tile lies beyond the range)
};

// byte offset of q row r (stride s_t between rows, s_b between blocks of batch_rows of them)
__device__ __forceinline__ long row_offset(const AttnKernArgs& a, int r, long s_t, long s_b) {
  if (a.batch_rows == 0) return (long)r * s_t;
  const int b = (int)((unsigned)r / (unsigned)a.batch_rows);
  return (long)(r - b * a.batch_rows) * s_t + (long)b * s_b;
}

// This workgroup's share (one of tiles_per_range) of the rows [r0, r1) of its head that no q range covers: zeros, lse =
// -inf.  Done here, by the launch that writes the other rows, the caller needs no clearing pass over the whole output
// (93600 x 24 heads of text cross attention: 596 -> 528 us; two passes per layer forward otherwise).
__device__ __forceinline__ void zero_rows(const AttnKernArgs& a, const WorkItem& wi, int r0, int r1, int tile, int tid) {
  const int per = (r1 - r0 + a.tiles_per_range - 1) / a.tiles_per_range;
  const int b = min(r1, r0 + tile * per), e = min(r1, b + per);
  for (int r = b + (tid >> 4); r < e; r += (int)(blockDim.x >> 4)) {
    *(u32x4*)(a.out + row_offset(a, r, a.os_t, a.os_b) + wi.o_head + 16 * (tid & 15)) = u32x4{0, 0, 0, 0};
    if (a.lse && (tid & 15) == 0) a.lse[(long)wi.h * a.total_q + r] = -__builtin_inff();
  }
}

// blockIdx -> (kv head, range slot, q tile, q head within the GQA group), laid out so that the workgroups an
// XCD receives (blockIdx % 8) share a KV head and walk the same keys at about the same time (each XCD has its
// own L2).  XCD x owns the heads x * (Hkv / 8) .. of the first 8 * (Hkv / 8); the Hkv % 8 heads that are left are
// shared, their (range, tile, q head) items dealt to the XCDs one by one: cut into contiguous pieces instead, an XCD got
// one range's tiles and the last XCDs ran dry.  Ranges are visited longest key span first (ties
// by index), ranked here from the device-side list.
// Every thread of the workgroup must call this (it contains a barrier); s_sel is LOCATE_WORDS ints of LDS.
constexpr int LOCATE_WORDS = 8;

// the arithmetic part: workgroup `block` -> heads, range slot, tile; false for the padding of the grid
__device__ __forceinline__ bool decode_block(const AttnKernArgs& a, unsigned block, unsigned& kvh, unsigned& hg, unsigned& rslot,
                                             unsigned& tile) {
  const unsigned xcd = block & 7u;
  unsigned i = block >> 3;  // position in this XCD's list
  const unsigned G = (unsigned)a.G, tiles = (unsigned)a.tiles_per_range, groups = (unsigned)a.n_ranges * tiles;
  const unsigned whole = (unsigned)a.Hkv >> 3, left = (unsigned)a.Hkv & 7u;
  unsigned u;  // position in the list of one head: (range slot, tile, q head)
  const unsigned per_head = groups * G;
  if (i < whole * per_head) {
    const unsigned n = i / per_head;
    kvh = xcd * whole + n;
    u = i - n * per_head;
  } else {
    i -= whole * per_head;
    if (left == 0u) return false;
    if ((8u % left) == 0u) {  // 8 / left XCDs share a head
      const unsigned share = 8u / left;
      kvh = 8u * whole + xcd / share;
      u = xcd % share + share * i;
    } else {
      u = xcd + 8u * i;
      kvh = u / per_head;
      u -= kvh * per_head;
      kvh += 8u * whole;
    }
    if (u >= per_head || kvh >= (unsigned)a.Hkv) return false;
  }
  const unsigned grp = u / G;
  hg = u - grp * G;
  rslot = grp / tiles;
  tile = grp - rslot * tiles;
  return true;
}
__device__ __forceinline__ int item_of(const AttnKernArgs& a, unsigned kvh, unsigned hg, unsigned rslot, unsigned tile) {
  return (int)(((kvh * a.G + hg) * (unsigned)a.n_ranges + rslot) * (unsigned)a.tiles_per_range + tile);
}

__device__ __forceinline__ WorkItem locate_work(const AttnKernArgs& a, int BM, int tid, int* s_sel, unsigned block) {
  WorkItem wi;
  wi.valid = false;
  unsigned kvh, hg, rslot, tile;
  if (!decode_block(a, block, kvh, hg, rslot, tile)) return wi;
  wi.kvh = (int)kvh;
  wi.h = (int)(kvh * a.G + hg);
  wi.item = item_of(a, kvh, hg, rslot, tile);
  wi.o_head = a.out_group > 0 ? (long)(wi.h / a.out_group) * a.os_g + (long)(wi.h % a.out_group) * a.os_h
                              : (long)wi.h * a.os_h;
  int qs;
  if (a.n_ranges <= 64) {
    // Lane t of the first wave holds range t: one memory latency for all of them, the ranking and the gaps between the
    // q ranges come from registers.
    if (tid < 64) {
      const int t = tid;
      const bool mine = t < a.n_ranges;
      int s = 0, e = 0, q_s = a.total_q, q_e = a.total_q;
      if (mine) {
        load_range(a.k_ranges, a.ranges_mode, t, a.total_k, s, e);
        load_range(a.q_ranges, a.ranges_mode, t, a.total_q, q_s, q_e);
      }
      // rows the launch computes of this range (max_seqlen_q may be smaller than the range)
      const int q_end = min(q_e, q_s + a.tiles_per_range * BM);
      const int my = e - s;
      int rank = 0, gap_e = a.total_q, lead = a.total_q;
      for (int j = 0; j < a.n_ranges; ++j) {
        const int lj = __builtin_amdgcn_readlane(my, j), sj = __builtin_amdgcn_readlane(q_s, j), ej = __builtin_amdgcn_readlane(q_end, j);
        rank += (lj > my) || (lj == my && j < t);
        if (sj < ej) {
          // the gap behind range t ends where the next range starts, and is none if another range covers its start
          gap_e = min(gap_e, sj >= q_end ? sj : ej > q_end ? q_end : a.total_q);
          lead = min(lead, sj);
        }
      }
      if (mine && rank == (int)rslot) {
        s_sel[0] = q_s;
        s_sel[1] = q_e;
        s_sel[2] = s;
        s_sel[3] = e;
        s_sel[4] = q_end;
        s_sel[5] = gap_e;
        s_sel[6] = rank == 0 ? lead : 0;  // rows ahead of the first range
      }
    }
    __syncthreads();
    qs = __builtin_amdgcn_readfirstlane(s_sel[0]);
    wi.qe = __builtin_amdgcn_readfirstlane(s_sel[1]);
    wi.ks = __builtin_amdgcn_readfirstlane(s_sel[2]);
    wi.ke = __builtin_amdgcn_readfirstlane(s_sel[3]);
    if (a.flags & ATTN_ZERO_GAPS) {
      const int g0 = __builtin_amdgcn_readfirstlane(s_sel[4]), g1 = __builtin_amdgcn_readfirstlane(s_sel[5]);
      const int lead = __builtin_amdgcn_readfirstlane(s_sel[6]);
      if (g1 > g0) zero_rows(a, wi, g0, g1, (int)tile, tid);
      if (lead > 0) zero_rows(a, wi, 0, lead, (int)tile, tid);
    }
  } else if (a.n_ranges <= MAX_SORT) {
    // thread t ranks range t; the one whose rank is this workgroup's slot publishes the range itself
    if (tid < a.n_ranges) {
      int s, e, q_s, q_e;
      load_range(a.k_ranges, a.ranges_mode, tid, a.total_k, s, e);
      load_range(a.q_ranges, a.ranges_mode, tid, a.total_q, q_s, q_e);
      const int my = e - s;
      int rank = 0;
      for (int j = 0; j < a.n_ranges; ++j) {
        int sj, ej;
        load_range(a.k_ranges, a.ranges_mode, j, a.total_k, sj, ej);
        const int lj = ej - sj;
        rank += (lj > my) || (lj == my && j < tid);
      }
      if (rank == (int)rslot) {
        s_sel[0] = q_s;
        s_sel[1] = q_e;
        s_sel[2] = s;
        s_sel[3] = e;
      }
    }
    __syncthreads();
    qs = __builtin_amdgcn_readfirstlane(s_sel[0]);
    wi.qe = __builtin_amdgcn_readfirstlane(s_sel[1]);
    wi.ks = __builtin_amdgcn_readfirstlane(s_sel[2]);
    wi.ke = __builtin_amdgcn_readfirstlane(s_sel[3]);
  } else {
    const int ridx = a.n_ranges - 1 - (int)rslot;
    load_range(a.q_ranges, a.ranges_mode, ridx, a.total_q, qs, wi.qe);
    load_range(a.k_ranges, a.ranges_mode, ridx, a.total_k, wi.ks, wi.ke);
  }
  wi.q0 = qs + (int)tile * BM;
  wi.valid = wi.q0 < wi.qe;
  return wi;
}

// Items whose keys are shared by several workgroups (a.split_*): what this workgroup has of its item.
struct SplitPiece {
  float* out;  // nullptr: a whole item
  unsigned piece;
};
// workgroup `block` of the grid with split items -> `block` of the grid without, and the piece of it
template <int FLOATS>
__device__ __forceinline__ SplitPiece split_piece(const AttnKernArgs& a, unsigned& block) {
  const unsigned pos = block >> 3, xcd = block & 7u;
  if (pos < a.split_from) return {nullptr, 0u};
  const unsigned items = a.per_xcd - a.split_from;  // (the longer first pieces of all items ahead of the others)
  const unsigned piece = (pos - a.split_from) / items, i = (pos - a.split_from) - piece * items;
  block = ((a.split_from + i) << 3) | xcd;
  return {a.partial + (long)((i * 8u + xcd) * a.split_pieces + piece) * FLOATS, piece};
}
__device__ __forceinline__ unsigned split_cut(const AttnKernArgs& a, unsigned tiles, unsigned piece) {
  return piece == 0u ? 0u : (unsigned)((unsigned long long)tiles * (a.split_num + piece - 1u) / a.split_den);
}
// A q row whose range has no keys: zeros, lse = -inf.  Lane (row, g) writes half g of the 256-byte row.
__device__ __forceinline__ void store_empty_row(const AttnKernArgs& a, const WorkItem& wi, int q_row, int g) {
  char* op = a.out + row_offset(a, q_row, a.os_t, a.os_b) + wi.o_head + g * 128;
#pragma unroll
  for (int c = 0; c < 8; ++c) *(u32x4*)(op + c * 16) = u32x4{0, 0, 0, 0};
  if (a.lse && g == 0) a.lse[(long)wi.h * a.total_q + q_row] = -__builtin_inff();
}

}  // namespace
}  // namespace magi
