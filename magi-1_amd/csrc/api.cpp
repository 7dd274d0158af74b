// C-ABI layer of libmagi_attn: argument validation, error reporting, kernel dispatch.
#include <hip/hip_runtime.h>
#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstddef>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>

#include "kernels.h"
#include "magi_attn.h"

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int hip_fail(hipError_t e, const char* what) {
  return fail(MAGI_EHIP, "%s: %s", what, hipGetErrorString(e));
}

std::atomic<uint64_t> g_launches{0};

// Counts n launches, and touches thread-local storage of this library.  The C library's table of a thread's storage (the DTV) is brought up to
// date only by an access to a module that was loaded behind the last update, and until then every access of every older module, torch's and HIP's
// on each call, takes the long way.  This library is among the last to be loaded.  Issued calls, 240 rows of rotary 7.14 -> 6.30 us, online softmax of
// 128 rows 13.9 -> 12.0, of one text segment 12.1 -> 10.4.  (Bounded launches touched it before, by their kept plans.)
thread_local volatile unsigned g_touched = 0;
void count_launches(uint64_t n) {
  g_touched = 1;
  g_launches.fetch_add(n, std::memory_order_relaxed);
}

// the caller's view of an argument struct must be this library's
template <class T>
bool same_layout(const T* p) { return p->struct_size == sizeof(T); }
#define MAGI_CHECK_LAYOUT(fn, p)                                                                            \
  if (!same_layout(p))                                                                                      \
    return fail(MAGI_EINVAL, fn ": struct_size %u, this library expects %zu (header / library version mismatch)", \
                (unsigned)(p)->struct_size, sizeof(*(p)))

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// compute units of the current device (asked once per device; 256 when the query fails)
int compute_units() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cached[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}

// Scratch memory of magi_attn_fwd_static_scratch: the two words of the measured score bound (and room to spare).  One
// copy per GPU, held until the process ends; every call on a GPU shares it.
constexpr int SCRATCH_BYTES = 256;
static __device__ __align__(256) unsigned char scratch[SCRATCH_BYTES];

// Device address of `scratch` on the current device (in host code the array's name is a stand-in, not an address):
// asked once per device with that device current, then kept.
std::mutex g_scratch_mutex;
void* g_scratch_ptr[64] = {nullptr};
int static_scratch(void** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
  if (dev < 0 || dev >= 64) return fail(MAGI_ENOSYS, "device index %d beyond the 64 this library keeps scratch pointers for", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
    if (!ptr) return fail(MAGI_EHIP, "hipGetSymbolAddress(scratch) returned no address");
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return MAGI_OK;
}

// Workgroups of one XCD's list (attn_common.h, locate_work): its Hkv / 8 whole heads, and its share of the rest.
unsigned items_per_xcd(int Hq, int Hkv, int n_ranges, int tiles_per_range) {
  const long left = Hkv % 8, per_head = (long)n_ranges * tiles_per_range * (Hq / Hkv);
  return (unsigned)((Hkv / 8) * per_head + (left * per_head + 7) / 8);
}

// tiles of 64 keys; unsigned, since the stated max_seqlen_k may be anything up to 2^31 - 1
unsigned key_tiles(int keys) { return ((unsigned)keys + 63) / 64; }

// Which items of a 256-row launch without a running maximum have their keys shared by several workgroups (AttnKernArgs::split_*).
struct SplitPlan {
  unsigned from, pieces, num, den;
  bool fp8;
  int64_t piece_bytes() const { return 4ll * (fp8 ? magi::SPLIT_FLOATS_FP8 : magi::SPLIT_FLOATS); }
  int64_t bytes(unsigned per_xcd) const { return from < per_xcd ? piece_bytes() * 8 * (per_xcd - from) * pieces : 0; }
};
// The last round of a launch has `left` items for `slots` places (two workgroups per CU) on each XCD.  At most half of them: equal pieces, as
// many as the places allow.  More: two pieces, the first so much longer that the others' second pieces fill the places
// left over in the time it takes (at 47 of 64, 3/4: three quarters on one slot take as long as a slot's three quarters).  A tile
// of 64 keys takes a workgroup about 3 us, 1.9 us alone on its CU (0.62; behind two rounds and more, out of step by then, 1.5); what the shorter round saves is put at half of that
// beside other workgroups (they slow down: the chip is power limited) and has to exceed the price, two launches' latency and
// the partial sums written and read at about 3.3 TB/s.  Measured, whole / split (profiles/shared_keys_sweep.txt, drawn sizes with the
// rule set aside): 148 launches that it splits 0.999 to 3.8, 1.38 on average; 92 that it does not 0.76 to 1.11, 0.97 on
// average; fp8 behind a whole round, 53 that it splits 0.984 to 1.3, 1.04 on average.  At 24 / 8 heads: 18 of 64 items over 7680 keys 208 / 144 us, 9 over 6300 keys 169 / 84, 47 over
// 46800 keys behind one whole round 4463 / 4099, over 9360 keys 876 / 849; not split, 48 over 4016 keys 173 / 187, 42 over 1766
// keys 81 / 98.  Behind eight and more the round is a small part of the launch.
// fp8: three workgroups of 128 rows per CU; a tile takes 1.4 us, 0.46 of that alone on a CU, 0.73 two by two.  Measured, whole /
// split, with items in the last round: 30 of 96 over 46800 keys 2788 / 2733 us, 24 over 25000 keys 905 / 830, 18 over 14400 keys 534
// / 474.  The probabilities are rounded to e4m3 relative to the maximum so far, which a piece sees only its part of: rows that
// are split differ from whole ones by as much as those two roundings do (3e-2 of the result).  Their error against float64 is
// 0.92 to 1.002 of the whole rows' over 30 drawn sizes, 0.974 on average.  Only launches whose rows are mostly whole are
// split all the same, behind one whole round at least.
// Several ranges: the items go longest range first, so the last ones belong to the shortest range, and
// the others' unequal lengths have filled most of the last round already.  The host does not know the lengths; of ranges
// that end a chunk of max_seqlen_q keys apart the shortest is max_seqlen_k less all but one of these (others are only split
// or not split where the other would have been as good or a few per cent better).  bf16 behind a whole round, whole / split where
// that is below half of the longest: four ranges of 1500 to 3750 keys 160 / 188 us, of 2800 to 7015 277 / 308, 10368 rows x 48
// heads over 2592 to 10368 keys a layer of 2896 / 2999 (but six heads over 13000 to 32440 keys 1458 / 1339); two ranges
// of one and two chunks of 7070 keys 1317 / 1334; at half and above: four of 5600 to 9800 500 / 462, two of 32526 to 37947
// 4089 / 3539.  Ranges of a chunk or less each (a batch) do not differ that way.  bf16 without a whole round: up to 5/8 of
// the slots gain (36 of 64 over two ranges of 2766 and 4149 keys 133 / 126), more of them from about 150 tiles on (42 over
// 14308 keys 408 / 352, 45 over 30708 979 / 935; but 42 over 5268 keys 173 / 185, 45 over 6215 203 / 211, 48 over 7216 245 / 258).
// fp8: a few items of a range of half the longest or less fit beside the first round (of 96 slots 3 over 4185 to 16740 keys 299 /
// 315 us, 3 over 5505 to 16515 357 / 377, 6 over 2131 and 4262 116 / 127, 9 over 11852 to 35556 748 / 776; but 9 over 8766 to
// 21915 525 / 454); 14 and more gain 2.5 % on average and lose 1.3 % at the most.
SplitPlan split_plan(unsigned items, int n_ranges, int max_seqlen_q, int max_seqlen_k, bool fp8) {
  SplitPlan s = {UINT32_MAX, 1, 1, 1, fp8};
  const unsigned cus = (unsigned)compute_units() / 8, slots = cus * (fp8 ? 3 : 2);  // of one XCD
  if (slots == 0 || max_seqlen_k <= 0) return s;
  const unsigned rounds = items / slots, left = items % slots, tiles = key_tiles(max_seqlen_k);
  if (left == 0 || rounds >= 8 || (fp8 && rounds == 0)) return s;
  if (n_ranges > 1 && max_seqlen_k > max_seqlen_q) {
    const int64_t shortest = max_seqlen_k - (int64_t)(n_ranges - 1) * max_seqlen_q;
    if (fp8 ? left * 8 <= slots && 2 * shortest <= max_seqlen_k
            : rounds > 0 && (2 * shortest < max_seqlen_k || shortest <= max_seqlen_q))
      return s;
  }
  if (!fp8 && rounds == 0 && n_ranges > 1 && left * 8 > slots * 5 && tiles < 150) return s;
  unsigned num, den;
  if (left * 2 > slots) {
    num = (left + slots - left - 1) / (slots - left);
    den = num + 1;
  } else {
    num = 1;
    den = slots / left < 8 ? slots / left : 8;
    if (den > tiles / 8) den = tiles / 8;
  }
  if (den < 2 || num > 4 || tiles < 4 * den) return s;
  const double piece = (double)num / den, cost_us = 8.0 + 0.3 * 8e-6 * left * (den - num + 1) * s.piece_bytes();
  double saved_us;
  if (fp8) {
    const double round = left <= cus ? 0.46 : left <= 2 * cus ? 0.73 : 1.0;
    saved_us = (round - piece) * 1.4 * tiles / 1.5;
  } else {
    saved_us = (left * 2 > slots ? 0.5 * (1.0 - piece) : (rounds >= 2 ? 0.5 : 0.62) - piece) * 3.0 * tiles;
  }
  if (saved_us < cost_us) return s;
  s.from = rounds * slots;
  s.pieces = den - num + 1;
  s.num = num;
  s.den = den;
  return s;
}

// Whether and how a launch of the online softmax in 128-row workgroups shares the keys of its items (AttnKernArgs::share_*): every
// item in pieces of the same number of tiles, a workgroup each, and a launch behind it that brings them together.
struct SharePlan {
  unsigned pieces, tiles;  // of the longest item, of a piece
  int64_t bytes(unsigned per_xcd) const { return pieces > 1 ? 4ll * magi::ONLINE_PARTIAL_FLOATS * 8 * per_xcd * pieces : 0; }
};
// A kernel's pace: us that a tile of 64 keys takes a workgroup alone on its CU, beside another, beside two; workgroups that run on a CU at a
// time; us of a launch besides.
struct Pace {
  double one, two, three;
  unsigned most;
  double launch_us;
};
constexpr Pace PACE_ONLINE = {1.36, 1.9, 2.55, 3, 9.0};      // 128 rows, 32 per wavefront, online softmax
constexpr Pace PACE_R32 = {1.13, 1.6, 2.4, 3, 6.5};          // the same without a running maximum
constexpr Pace PACE_X16_128 = {1.10, 1.6, 1.6, 2, 6.0};      // 128 rows, two slots for K and for V
constexpr Pace PACE_X16_256 = {1.75, 2.75, 2.75, 2, 7.0};    // 256 rows
// What a launch in pieces of `cut` tiles takes, in us: bringing pieces together takes 5 us and 18 ns each (their way through
// memory).  Workgroups that fit the chip at once run side by side until the shortest are done, and so on; more of them keep it full but
// for the end.
// even: pieces of nearly the same length end together, so a CU that has one more than the others keeps it to the end.
double share_us(const Pace& p, unsigned items, const unsigned* lengths, int n_ranges, unsigned cut, unsigned cus, bool even = false) {
  unsigned len[2 * 16], count[2 * 16];  // the pieces, by length
  int kinds = 0;
  auto add = [&](unsigned l, unsigned c) {
    int i = 0;
    while (i < kinds && len[i] < l) ++i;
    if (i < kinds && len[i] == l) {
      count[i] += c;
      return;
    }
    for (int k = kinds++; k > i; --k) len[k] = len[k - 1], count[k] = count[k - 1];
    len[i] = l, count[i] = c;
  };
  const unsigned each = items / (unsigned)n_ranges;
  double all = 0, parts = 0, work = 0;
  for (int r = 0; r < n_ranges; ++r) {
    const unsigned whole = lengths[r] / cut, rest = lengths[r] % cut;
    if (whole) add(cut, whole * each);
    if (rest) add(rest, each);
    const unsigned n = whole + (rest != 0);
    all += (double)n * each;
    work += (double)lengths[r] * each;
    if (n > 1) parts += (double)n * each;
  }
  auto tile_us = [&](double on_a_cu) {
    if (on_a_cu <= 1) return p.one;
    if (on_a_cu <= 2) return p.one + (p.two - p.one) * (on_a_cu - 1);
    return on_a_cu <= 3 ? p.two + (p.three - p.two) * (on_a_cu - 2) : p.three;
  };
  double t = p.launch_us;
  if (all > (double)p.most * cus) {
    t += p.three * (work / ((double)p.most * cus) + 0.25 * cut);
  } else {
    double left = all;
    for (int i = 0; i < kinds; left -= count[i++])
      t += (len[i] - (i ? len[i - 1] : 0)) * tile_us(i + 1 < kinds && !(even && 8 * len[i] >= 7 * len[kinds - 1]) ? left / cus : std::ceil(left / cus));
  }
  return parts > 0 ? t + 5.0 + 0.018 * parts : t;
}
// key tiles of each range, as far as sizes tell; false where they do not
bool range_tiles(int n_ranges, int max_seqlen_q, int max_seqlen_k, unsigned* lengths) {
  if (max_seqlen_k <= 0 || n_ranges < 1 || n_ranges > 16) return false;
  const bool apart = max_seqlen_k > (int64_t)(n_ranges - 1) * max_seqlen_q;
  for (int r = 0; r < n_ranges; ++r) lengths[r] = key_tiles(max_seqlen_k - (apart ? r * max_seqlen_q : 0));
  return true;
}
// the best of the launches in pieces that take less than `us`
SharePlan best_pieces(const Pace& p, unsigned items, const unsigned* lengths, int n_ranges, double us, bool one_round = false) {
  SharePlan best = {1, 0};
  const unsigned cus = (unsigned)compute_units(), longest = lengths[0];
  static const unsigned char tried[] = {2, 3, 4, 5, 6, 8, 10, 12, 16};
  for (unsigned pieces : tried) {
    const unsigned cut = (longest + pieces - 1) / pieces;
    if (cut < 3 || (double)items * pieces > 8.0 * cus) break;
    unsigned parts = 0;
    for (int r = 0; r < n_ranges; ++r) parts += (lengths[r] + cut - 1) / cut;
    if (one_round && (double)items / n_ranges * parts > (double)p.most * cus) continue;
    const double t = share_us(p, items, lengths, n_ranges, cut, cus, one_round);
    if (t < us) {
      us = t;
      best = {(longest + cut - 1) / cut, cut};
    }
  }
  return best;
}
// Measured, whole / in pieces: 24 items over 127 tiles 181 / 41 us, 126 over 332 455 / 186, 180 over 592 and less 795 / 428, 240 over 180 257
// / 195, 336 over 136 265 / 210, 576 over 378 981 / 846; not cut, 384 over 16 and 32 57 / 62, 528 over 44 and 66 151 / 159, 864 over 24 to
// 72 178 / 193, 1728 over 54 to 108 543 / 565.  The host does not know the ranges' lengths: taken are ranges that end a chunk of
// max_seqlen_q keys apart, or all of max_seqlen_k keys where that does not go.  Only where the estimate is 6 % shorter, 10 % behind a whole round
// (864 items over 86 to 111 tiles 402 / 410), and from 20 tiles on: max_seqlen_k of text is the padded length, of which a call may fill a fraction.  Ranges far
// shorter than stated lose 3 to 4 us (24 heads, 240 rows over 60 keys, 2000 stated: 6.9 / 11.0).  All drawn launches: profiles/launches_below_a_round_sweep.txt.
SharePlan share_plan(unsigned per_xcd, int n_ranges, int max_seqlen_q, int max_seqlen_k) {
  const unsigned cus = (unsigned)compute_units(), items = 8 * per_xcd;
  unsigned lengths[16];
  if (items == 0 || items > 6 * cus || !range_tiles(n_ranges, max_seqlen_q, max_seqlen_k, lengths) || lengths[0] < 20) return {1, 0};
  return best_pieces(PACE_ONLINE, items, lengths, n_ranges,
                     (items > 3 * cus ? 0.90 : 0.94) * share_us(PACE_ONLINE, items, lengths, n_ranges, lengths[0], cus));
}

// How a launch of the 64-rows-per-wavefront kernel without a running maximum is cut: workgroups of 256 rows, their last round's
// items sharing keys where that pays and the caller has brought the memory, or workgroups of 128 rows
// (32 per wavefront; a row's bits are the same).  Those fetch and read every tile for half the rows, so they are only for launches
// that leave two of them per CU a CU of their own or nearly: a tile of 64 keys then takes 1.15 us alone on its CU, 1.75 beside
// another, against 1.75 and 2.5 to 3.0 of 256 rows.  Measured, 24 / 8 heads, 256 rows whole / in pieces / 128 rows: up to one
// workgroup per CU 240 rows over 960 keys 32.1 / - / 21.5 us, 900 over 2000 61 / 45 / 42, text of 183 rows for 468 15.1 / - / 10.5;
// up to two 1300 over 1300 43.5 / - / 37.3, 2600 over 13000 502 / 404 / 366, four ranges of 288 over 1152 to 2016 61 / - / 45; beyond
// 972 x 4 over 972 to 3888 130 / - / 123, but 3800 over 3800 168 / - / 172 and 1000 x 3 over 3000 to 5000 161 / 148 / 173.  Few items
// with long keys are better off in pieces, which cost about 12 us and 0.3 per piece of an XCD: 240 rows over 3000 keys 86 / 33 / 56,
// 1300 over 4000 113 / 81 / 97.
int tile_rows(int Hq, int Hkv, int n_ranges, int max_seqlen_q, int max_seqlen_k, int64_t split_bytes) {
  auto items = [&](int rows) { return items_per_xcd(Hq, Hkv, n_ranges, max_seqlen_q / rows + (max_seqlen_q % rows != 0)); };
  const unsigned cus = (unsigned)compute_units() / 8, whole = items(256), half = items(128);
  if (half > 2 * cus) return 256;
  if (split_bytes <= 0) return 128;
  const SplitPlan s = split_plan(whole, n_ranges, max_seqlen_q, max_seqlen_k, false);
  if (s.from >= whole || s.bytes(whole) > split_bytes) return 128;
  // (without a whole round ahead of them: all items are in pieces)
  const unsigned pieces = whole * s.pieces;
  const double tiles = key_tiles(max_seqlen_k), in_pieces = tiles * s.num / s.den * (pieces <= cus ? 1.75 : 2.6) + 12.0 + 0.3 * pieces;
  return in_pieces <= tiles * (half <= cus ? 1.15 : 1.75) ? 256 : 128;
}

// Whether a launch without a running maximum runs in workgroups of 128 rows, three per CU (attn_fwd_bf16_r32.hip): whole items, which
// have the bits of the other forms' whole items, or pieces of all of them.
struct R32Plan {
  bool use;
  SharePlan share;
};
// Whole: where 256 rows to a workgroup, whole, are what split_plan and tile_rows leave, and one round of the smaller ones (more than two
// per CU, which tile_rows takes care of) holds them all.  Measured, 24 heads, 256 rows / 128: 2700 rows over 2700 keys 125 / 107 us, 3354
// over 3354 152 / 136, 3744 over 3744 168 / 156, four ranges of 792 over 1584 to 3960 138 / 114, three of 1200 over 1200 to 3600 125 / 103;
// but behind that round 2250 x 2 over 2250 and 4500 164 / 185, 2340 x 2 168 / 211.
// Pieces: the estimates of both launches, and at least 5 % less, where all pieces run at a time; pieces of one length
// take as long as the CU that has most of them (264 items in two each, three on 16 CUs: 1386 rows over 6930 and 13860 keys 121 / 140, 197 / 236).  Measured, before / in pieces: 6 heads, 270 rows over 1350 keys 30 / 17, three
// ranges of 312 over 1248 to 1872 31 / 22, four of 252 33 / 20; 24 heads, 432 over 1728 36 / 29, 720 over 2880 49 / 42, three of 612 over
// 5508 to 6732 178 / 144; not so 1080 over 5400 86 / 86, 720 over 720 21 / 25, 660 over 5940 63 / 70, 48 heads 105 / 123,
// two of 660 over 5280 and 5940 113 / 123, four over 1980 to 3960 112 / 116 (256 rows in pieces all: their time by the mean length of the ranges).  Error against float64 over that of whole items 1.0000 to 1.0001 (27 drawn sizes).
// (From 16 tiles on: max_seqlen_k of text is the padded length, 800, of which a call may fill a fraction; 15 tiles would gain 4 to 6 us.)
R32Plan make_r32_plan(int Hq, int Hkv, int n_ranges, int max_seqlen_q, int max_seqlen_k, unsigned cus, int64_t& split_bytes) {
  R32Plan plan = {false, {1, 0}};
  auto items = [&](int rows) { return items_per_xcd(Hq, Hkv, n_ranges, max_seqlen_q / rows + (max_seqlen_q % rows != 0)); };
  const unsigned half = items(128), whole = items(256);
  unsigned lengths[16];
  if (half == 0 || 8 * half > 3 * cus || (split_bytes <= 0 && half <= cus / 4) || !range_tiles(n_ranges, max_seqlen_q, max_seqlen_k, lengths)) return plan;
  // what tile_rows and split_plan make of this much memory
  bool small;
  SplitPlan split;
  auto others = [&](int64_t bytes) {
    small = tile_rows(Hq, Hkv, n_ranges, max_seqlen_q, max_seqlen_k, bytes) == 128;
    split = {UINT32_MAX, 1, 1, 1, false};
    if (!small && bytes > 0) split = split_plan(whole, n_ranges, max_seqlen_q, max_seqlen_k, false);
    if (split.bytes(whole) > bytes) split.from = UINT32_MAX;
    return !small && split.from >= whole && half > cus / 4;  // whole items of 256 rows, more than two of 128 per CU
  };
  if (split_bytes > 0 && lengths[0] >= 16) {
    const bool whole_items = others(INT64_MAX);
    double us, tiles = 0;  // (tiles: of all ranges)
    for (int r = 0; r < n_ranges; ++r) tiles += lengths[r];
    if (split.from < whole)  // (at most one round here: all items are in pieces)
      us = 16.0 + tiles / n_ranges * (double)split.num / split.den * (8 * whole * split.pieces <= cus ? 1.75 : 2.6) + 0.18 * whole * split.pieces;
    else
      us = share_us(whole_items ? PACE_R32 : small ? PACE_X16_128 : PACE_X16_256, 8 * (whole_items || small ? half : whole), lengths, n_ranges,
                    lengths[0], cus);
    plan.share = best_pieces(PACE_R32, 8 * half, lengths, n_ranges, 0.95 * us, true);
    plan.use = plan.share.pieces > 1;
    if (plan.use && plan.share.bytes(half) > split_bytes) {  // (too little memory: whole items)
      plan = {false, {1, 0}};
      split_bytes = 0;
    }
  }
  if (!plan.use) plan.use = others(split_bytes);
  return plan;
}

// (Asked for twice or three times for a launch, for its memory and for itself, and again by the next layer; 1 to 2 us each, which layers that
// wait for the host have not got.  A thread's last eight are kept by their sizes.)
R32Plan r32_plan(int Hq, int Hkv, int n_ranges, int max_seqlen_q, int max_seqlen_k, int64_t& split_bytes) {
  struct Kept {
    int sizes[5];
    unsigned cus;
    int64_t given, left;
    R32Plan plan;
  };
  static thread_local Kept kept[8];  // (cus 0: none)
  static thread_local unsigned next = 0;
  const unsigned cus = (unsigned)compute_units();
  for (const Kept& e : kept)
    if (e.cus == cus && e.given == split_bytes && e.sizes[0] == Hq && e.sizes[1] == Hkv && e.sizes[2] == n_ranges && e.sizes[3] == max_seqlen_q &&
        e.sizes[4] == max_seqlen_k) {
      split_bytes = e.left;
      return e.plan;
    }
  Kept& e = kept[next++ % 8];
  const int64_t given = split_bytes;
  e.plan = make_r32_plan(Hq, Hkv, n_ranges, max_seqlen_q, max_seqlen_k, cus, split_bytes);
  e = {{Hq, Hkv, n_ranges, max_seqlen_q, max_seqlen_k}, cus, given, split_bytes, e.plan};
  return e.plan;
}

// the memory of its pieces, 0 where it takes whole items or none
int64_t r32_bytes(int Hq, int Hkv, int n_ranges, int max_seqlen_q, int max_seqlen_k) {
  int64_t any = INT64_MAX;
  return r32_plan(Hq, Hkv, n_ranges, max_seqlen_q, max_seqlen_k, any)
      .share.bytes(items_per_xcd(Hq, Hkv, n_ranges, max_seqlen_q / 128 + (max_seqlen_q % 128 != 0)));
}

// Whether a launch without a running maximum whose caller permits it (MAGI_ATTN_SHARE_WAVES) has the keys of 32 rows shared by the wavefronts of
// a workgroup (attn_fwd_bf16_waves.hip): how many wavefronts, 0: not.
// Eight, a workgroup per CU, or four, two of them.  Measured, 128 and 256 rows to a workgroup (in pieces where that was the better) / this form, drawn
// sizes (those it takes: profiles/launches_below_a_round_sweep.txt): up to one workgroup of 32 rows per CU, from 65 keys on, 77 launches 0.95 to 1.72
// times as fast, 1.23 on average (12 workgroups over 423 keys 12.1 / 9.7 us, 48 over 480 13.4 / 9.1, 240 over 1113 18.2 / 12.7, 228 over 5930 41.1 /
// 34.5); four wavefronts up to 1024 keys and for more than a workgroup per CU: 288 over 600 15.8 / 12.3, 480 over 1460 30.3 / 22.7, 360 over 4570
// 41.5 / 40.6, but 288 over 5085 40.8 / 47.1, 312 over 8100 52.7 / 72.6; beyond two per CU 576 over 1050 23.6 / 27.3.  max_seqlen_k of text is the
// padded length: 288 workgroups over 39 of 800 keys 7.6 / 8.0, 504 over 184 10.4 / 12.5, so cumulative lengths only up to one per CU.
// Below a SLAB of keys there is nothing to share: by itself such a launch takes the other forms (21 drawn ones of 1 to 31 keys 0.86 to 1.02 of their time in this
// one, 0.94 on average; the same bits), beside another small call this one, a launch less (31 and 20 keys 11.6 us one by one, 7.2 together).  Above,
// by themselves: 32 keys 1.00 to 1.12, 33 to 64 0.90 to 1.04, 0.97 on average (their sums are in another order here, which a call beside another one
// has too).
constexpr int SLAB = 32;
int waves_plan(int Hq, int Hkv, int n_ranges, int ranges_mode, int max_seqlen_q, int max_seqlen_k) {
  if ((double)Hq * n_ranges * (max_seqlen_q / 32 + 1) > 2.0e9) return 0;
  const double items = 8.0 * items_per_xcd(Hq, Hkv, n_ranges, max_seqlen_q / 32 + (max_seqlen_q % 32 != 0));
  const int cus = compute_units();
  if (max_seqlen_k <= 0 || items > (ranges_mode == MAGI_RANGES_CU ? 1 : 2) * cus) return 0;
  if (max_seqlen_k <= 1024) return 4;
  if (items <= cus) return max_seqlen_k <= 8192 ? 8 : 0;
  return max_seqlen_k <= 4096 ? 4 : 0;
}

// HELD: the call takes a form that may share a launch with another, `held` has its arguments and nothing is launched; ALONE: it does not, and
// nothing is launched either.  FIRST, SECOND of two alike: wavefronts that share keys, or 256-row workgroups; a first call of another form is
// launched (MAGI_OK), a second one is ALONE, as it must not run ahead of the first.  TEXT, a second call beside something else: every form of raw q
// with bounded scores, but those whose keys are shared.  BEGIN: of 256-row items some with shared keys leave their pieces, and a launch of whole
// ones waits for the second call (HELD both times); others are launched; END: the arguments of such a call.
constexpr int HELD = 1, ALONE = 2;
enum Held { NOW, FIRST, SECOND, TEXT, BEGIN, END };
int attn_fwd_impl(const magi_attn_args* p, void* stream, float* workspace, magi::AttnKernArgs* held = nullptr, Held how = NOW);
int launch_waves(const magi::AttnKernArgs& a, void* stream);
int attn_fwd_two(const magi_attn_args* first, const magi_attn_args* second, void* stream);
int attn_fwd_end(const magi_attn_args* first, const magi_attn_args* second, void* stream);

// the caller's struct as this version lays it out: itself, or `full` filled from the shorter one of version 103
const magi_attn_args* current_layout(const magi_attn_args* p, magi_attn_args* full) {
  constexpr size_t v103 = offsetof(magi_attn_args, q_batch_rows);
  if (p->struct_size != v103) return p;
  std::memset(full, 0, sizeof(*full));
  std::memcpy(full, p, v103);
  full->struct_size = sizeof(*full);
  return full;
}

}  // namespace

extern "C" {

int magi_version(void) { return 107; }

uint64_t magi_launch_count(void) { return g_launches.load(std::memory_order_relaxed); }

const char* magi_last_error(void) { return g_err; }

int64_t magi_attn_split_bytes(int32_t Hq, int32_t Hkv, int32_t n_ranges, int32_t max_seqlen_q, int32_t max_seqlen_k,
                              int32_t dtype) {
  if (Hq <= 0 || Hkv <= 0 || Hq % Hkv || n_ranges <= 0 || max_seqlen_q <= 0) return 0;
  const bool fp8 = dtype == MAGI_DTYPE_FP8_E4M3;
  const int rows = fp8 ? 128 : 256, tiles = max_seqlen_q / rows + (max_seqlen_q % rows != 0);
  if ((double)Hq * n_ranges * tiles > 2.0e9) return 0;
  const unsigned items = items_per_xcd(Hq, Hkv, n_ranges, tiles);
  const int64_t split = split_plan(items, n_ranges, max_seqlen_q, max_seqlen_k, fp8).bytes(items);
  const int64_t pieces = fp8 ? 0 : r32_bytes(Hq, Hkv, n_ranges, max_seqlen_q, max_seqlen_k);
  return split > pieces ? split : pieces;
}

int64_t magi_attn_split_bytes_256(int32_t Hq, int32_t Hkv, int32_t n_ranges, int32_t max_seqlen_q, int32_t max_seqlen_k) {
  if (Hq <= 0 || Hkv <= 0 || Hq % Hkv || n_ranges <= 0 || max_seqlen_q <= 0) return 0;
  const int tiles = max_seqlen_q / 256 + (max_seqlen_q % 256 != 0);
  if ((double)Hq * n_ranges * tiles > 2.0e9) return 0;
  const unsigned items = items_per_xcd(Hq, Hkv, n_ranges, tiles);
  return split_plan(items, n_ranges, max_seqlen_q, max_seqlen_k, false).bytes(items);
}

int64_t magi_attn_pieces_bytes(int32_t Hq, int32_t Hkv, int32_t n_ranges, int32_t max_seqlen_q, int32_t max_seqlen_k, int32_t bounded) {
  if (Hq <= 0 || Hkv <= 0 || Hq % Hkv || n_ranges <= 0 || max_seqlen_q <= 0) return 0;
  if ((double)Hq * n_ranges * (max_seqlen_q / 128 + 1) > 2.0e9) return 0;
  const unsigned items = items_per_xcd(Hq, Hkv, n_ranges, max_seqlen_q / 128 + (max_seqlen_q % 128 != 0));
  if (bounded) return r32_bytes(Hq, Hkv, n_ranges, max_seqlen_q, max_seqlen_k);
  return share_plan(items, n_ranges, max_seqlen_q, max_seqlen_k).bytes(items);
}

int32_t magi_attn_waves(int32_t Hq, int32_t Hkv, int32_t n_ranges, int32_t ranges_mode, int32_t max_seqlen_q, int32_t max_seqlen_k) {
  if (Hq <= 0 || Hkv <= 0 || Hq % Hkv || n_ranges <= 0 || max_seqlen_q <= 0) return 0;
  return waves_plan(Hq, Hkv, n_ranges, ranges_mode, max_seqlen_q, max_seqlen_k);
}

int32_t magi_attn_tile_rows(int32_t Hq, int32_t Hkv, int32_t n_ranges, int32_t max_seqlen_q, int32_t max_seqlen_k,
                            int64_t split_workspace_bytes) {
  if (Hq <= 0 || Hkv <= 0 || Hq % Hkv || n_ranges <= 0 || max_seqlen_q <= 0) return 256;
  if ((double)Hq * n_ranges * (max_seqlen_q / 128 + 1) > 2.0e9) return 256;
  return tile_rows(Hq, Hkv, n_ranges, max_seqlen_q, max_seqlen_k, split_workspace_bytes);
}

int magi_attn_fwd(const magi_attn_args* p, void* stream) {
  if (!p) return fail(MAGI_EINVAL, "magi_attn_fwd: args is NULL");
  magi_attn_args full;
  p = current_layout(p, &full);
  MAGI_CHECK_LAYOUT("magi_attn_fwd", p);
  return attn_fwd_impl(p, stream, p->workspace);
}

int magi_attn_fwd_two(const magi_attn_args* first, const magi_attn_args* second, void* stream) {
  if (!first || !second) return fail(MAGI_EINVAL, "magi_attn_fwd_two: args is NULL");
  MAGI_CHECK_LAYOUT("magi_attn_fwd_two", first);
  MAGI_CHECK_LAYOUT("magi_attn_fwd_two", second);
  return attn_fwd_two(first, second, stream);
}

int magi_attn_fwd_begin(const magi_attn_args* p, void* stream) {
  if (!p) return fail(MAGI_EINVAL, "magi_attn_fwd_begin: args is NULL");
  MAGI_CHECK_LAYOUT("magi_attn_fwd_begin", p);
  magi::AttnKernArgs left;
  return attn_fwd_impl(p, stream, p->workspace, &left, BEGIN);
}

int magi_attn_fwd_end(const magi_attn_args* first, const magi_attn_args* second, void* stream) {
  if (!first) return fail(MAGI_EINVAL, "magi_attn_fwd_end: args is NULL");
  MAGI_CHECK_LAYOUT("magi_attn_fwd_end", first);
  if (second) MAGI_CHECK_LAYOUT("magi_attn_fwd_end", second);
  return attn_fwd_end(first, second, stream);
}

int magi_attn_fwd_static_scratch(const magi_attn_args* p, void* stream) {
  if (!p) return fail(MAGI_EINVAL, "magi_attn_fwd_static_scratch: args is NULL");
  magi_attn_args full;
  p = current_layout(p, &full);
  MAGI_CHECK_LAYOUT("magi_attn_fwd_static_scratch", p);
  if (p->flags & MAGI_ATTN_CHECKED)
    return fail(MAGI_ENOSYS, "magi_attn_fwd_static_scratch: the workspace of MAGI_ATTN_CHECKED grows with the problem");
  static_assert(4 * sizeof(float) <= SCRATCH_BYTES, "the measured score bound needs four words");
  void* ws = nullptr;
  const int rc = static_scratch(&ws);
  if (rc != MAGI_OK) return rc;
  return attn_fwd_impl(p, stream, static_cast<float*>(ws));
}

}  // extern "C"

namespace {

// a call of wavefronts that share keys by itself
int launch_waves(const magi::AttnKernArgs& a, void* stream) {
  magi::AttnPairArgs pair;
  pair.job[0] = a;
  pair.job[1].per_xcd = 0;
  const hipError_t e = magi::launch_attn_fwd_bf16_waves(pair, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return hip_fail(e, "magi_attn_fwd launch");
  count_launches(1);
  return MAGI_OK;
}

// two held calls of one form in one launch: 32 rows to a workgroup, whose wavefronts share keys; or 256 rows of q as it is or raw
int launch_alike(const magi::AttnPairArgs& pair, void* stream) {
  const hipStream_t st = static_cast<hipStream_t>(stream);
  const magi::AttnKernArgs& a = pair.job[0];
  const hipError_t e = a.block_m == 32 ? magi::launch_attn_fwd_bf16_waves(pair, st) : magi::launch_attn_fwd_bf16_x16_pair(pair, st);
  if (e != hipSuccess) return hip_fail(e, "magi_attn_fwd launch");
  count_launches(1 + (a.block_m != 32 && a.split_from < a.per_xcd));
  return MAGI_OK;
}

// Whether so many workgroups of 256 threads are a launch: HIP takes less than 2^32 threads.  (Two calls may fit apart and not together: ranges of
// a long max_seqlen_q have most of their tiles beyond their rows.)
bool fits(uint64_t workgroups) { return workgroups * 256 <= UINT32_MAX; }

// a held text call in tiles of 128 (as attn_text_rows.h takes it) or 256 rows, whole items, beside so many other workgroups; false, and b as it was,
// where the launch would not fit
bool text_in_rows(magi::AttnKernArgs& b, int max_seqlen_q, int rows, uint64_t others) {
  const int tiles = max_seqlen_q / rows + (max_seqlen_q % rows != 0);
  if ((double)b.Hq * b.n_ranges * tiles > 2.0e9) return false;
  const unsigned per_xcd = items_per_xcd(b.Hq, b.Hkv, b.n_ranges, tiles);
  if (!fits(others + 8ull * per_xcd)) return false;
  b.block_m = rows;
  b.tiles_per_range = tiles;
  b.per_xcd = per_xcd;
  b.split_from = UINT32_MAX;
  return true;
}

// a second call that did not go with the first, which has been launched: `two` is what attn_fwd_impl returned for it
int launch_behind(int two, const magi_attn_args* second, void* stream) {
  return two == HELD || two == ALONE ? attn_fwd_impl(second, stream, second->workspace) : two;
}

// the second half of magi_attn_fwd_begin(first), beside second
int attn_fwd_end(const magi_attn_args* first, const magi_attn_args* second, void* stream) {
  const hipStream_t st = static_cast<hipStream_t>(stream);
  magi::AttnPairArgs pair;
  magi::AttnKernArgs &a = pair.job[0], &b = pair.job[1];
  const int one = attn_fwd_impl(first, stream, first->workspace, &a, END);
  if (one != HELD) return one < 0 ? one : fail(MAGI_EINVAL, "magi_attn_fwd_end: an empty call leaves nothing");
  const bool whole = a.split_from >= a.per_xcd;
  const int two = second ? attn_fwd_impl(second, stream, second->workspace, &b, TEXT) : MAGI_OK;
  // (beside the workgroups of the first, or the four of each of its items that bring the pieces together)
  const uint64_t others = whole ? split_grid(a) : 32ull * split_items(a);
  const bool together = two == HELD && text_in_rows(b, second->max_seqlen_q, whole ? 256 : 128, others);
  const hipError_t e = whole ? (together ? magi::launch_attn_fwd_bf16_x16_pair(pair, st) : magi::launch_attn_fwd_bf16_x16(a, st))
                             : (together ? magi::launch_attn_text_merge(pair, st) : magi::launch_attn_fwd_bf16_merge(a, st));
  if (e != hipSuccess) return hip_fail(e, "magi_attn_fwd_end launch");
  count_launches(1);
  return together ? MAGI_OK : launch_behind(two, second, stream);
}

// first, then second, which do not depend on each other: in one launch where both take the form for it
int attn_fwd_two(const magi_attn_args* first, const magi_attn_args* second, void* stream) {
  magi::AttnPairArgs pair;
  magi::AttnKernArgs &a = pair.job[0], &b = pair.job[1];
  const int one = attn_fwd_impl(first, stream, first->workspace, &a, FIRST);
  if (one != HELD) return one < 0 ? one : attn_fwd_impl(second, stream, second->workspace);
  if (first->dtype == MAGI_DTYPE_FP8_E4M3) {
    const hipStream_t st = static_cast<hipStream_t>(stream);
    const int two = attn_fwd_impl(second, stream, second->workspace, &b, TEXT);
    const bool together = two == HELD && text_in_rows(b, second->max_seqlen_q, 128, split_grid(a));
    const hipError_t e = together ? magi::launch_attn_fwd_fp8_text(pair, st) : magi::launch_attn_fwd_fp8(a, st);
    if (e != hipSuccess) return hip_fail(e, "magi_attn_fwd launch");
    count_launches(1 + (a.split_from < a.per_xcd));
    return together ? MAGI_OK : launch_behind(two, second, stream);
  }
  const int two = attn_fwd_impl(second, stream, second->workspace, &b, SECOND);
  // (of 32 rows there is at most a workgroup or two per CU)
  if (two == HELD && a.block_m == b.block_m && (b.block_m == 32 || (b.split_from >= b.per_xcd && fits(split_grid(a) + 8ull * b.per_xcd))))
    return launch_alike(pair, stream);
  const int rc = attn_fwd_impl(first, stream, first->workspace);
  return rc < 0 ? rc : launch_behind(two, second, stream);
}

int not_begun() { return fail(MAGI_EINVAL, "magi_attn_fwd_end: not a call that magi_attn_fwd_begin leaves anything of"); }

int attn_fwd_impl(const magi_attn_args* p, void* stream, float* workspace, magi::AttnKernArgs* held, Held how) {
  if (p->D != 128) return fail(MAGI_ENOSYS, "magi_attn_fwd: head_dim %d not implemented (128 only)", p->D);
  if (p->dtype != MAGI_DTYPE_BF16 && p->dtype != MAGI_DTYPE_FP8_E4M3)
    return fail(MAGI_EINVAL, "magi_attn_fwd: unknown dtype %d", p->dtype);
  if (p->Hq <= 0 || p->Hkv <= 0 || p->Hq % p->Hkv != 0)
    return fail(MAGI_EINVAL, "magi_attn_fwd: Hq=%d must be a positive multiple of Hkv=%d", p->Hq, p->Hkv);
  if (p->total_q < 0 || p->total_k < 0 || p->n_ranges < 0 || p->max_seqlen_q < 0)
    return fail(MAGI_EINVAL, "magi_attn_fwd: negative size");
  if (p->ranges_mode != MAGI_RANGES_PAIRS && p->ranges_mode != MAGI_RANGES_CU)
    return fail(MAGI_EINVAL, "magi_attn_fwd: unknown ranges_mode %d", p->ranges_mode);
  static_assert(MAGI_ATTN_ZERO_UNCOVERED == magi::ATTN_ZERO_GAPS, "flag bits of the header and the kernels");
  if ((p->flags & MAGI_ATTN_ZERO_UNCOVERED) && (p->n_ranges < 1 || p->n_ranges > 64 || (p->total_q > 0 && p->max_seqlen_q == 0)))
    return fail(MAGI_ENOSYS, "magi_attn_fwd: MAGI_ATTN_ZERO_UNCOVERED needs 1 to 64 ranges and max_seqlen_q > 0");
  if (p->n_ranges == 0 || p->total_q == 0 || p->max_seqlen_q == 0) return MAGI_OK;
  if (!p->q || !p->out || !p->q_ranges || !p->k_ranges) return fail(MAGI_EINVAL, "magi_attn_fwd: NULL q/out/ranges");
  const bool all_in_second = p->k2 && p->v2 && p->k_split == 0;  // an empty first segment may be NULL
  if (p->total_k > 0 && (!p->k || !p->v) && !all_in_second)
    return fail(MAGI_EINVAL, "magi_attn_fwd: NULL k/v with total_k > 0");
  const int esz = p->dtype == MAGI_DTYPE_BF16 ? 2 : 1;
  const int64_t row_elems = 16 / esz;  // 16-byte vectors
  if (p->q_stride_h % row_elems || p->q_stride_t % row_elems || p->k_stride_h % row_elems ||
      p->k_stride_t % row_elems || p->v_stride_h % row_elems || p->v_stride_t % row_elems || p->o_stride_h % 8 ||
      p->o_stride_t % 8)
    return fail(MAGI_EINVAL, "magi_attn_fwd: strides must keep rows 16-byte aligned");
  if (!aligned16(p->q) || !aligned16(p->k) || !aligned16(p->v) || !aligned16(p->out) || !aligned16(p->k2) ||
      !aligned16(p->v2))
    return fail(MAGI_EINVAL, "magi_attn_fwd: q/k/v/out must be 16-byte aligned");
  if (p->q_stride_h < p->D || p->k_stride_h < p->D || p->v_stride_h < p->D || p->o_stride_h < p->D)
    return fail(MAGI_EINVAL, "magi_attn_fwd: head stride smaller than head_dim");
  if (p->q_stride_t < p->D || p->k_stride_t < p->D || p->v_stride_t < p->D || p->o_stride_t < p->D)
    return fail(MAGI_EINVAL, "magi_attn_fwd: token stride smaller than head_dim (rows may not overlap or run backwards)");
  // (the kernels address a 64-key tile with 32-bit byte offsets from its first row)
  if (p->k_stride_t > (1 << 23) || p->v_stride_t > (1 << 23))
    return fail(MAGI_ENOSYS, "magi_attn_fwd: k / v token strides above 2^23 elements are not implemented");
  if (p->dtype == MAGI_DTYPE_FP8_E4M3 && (p->flags & MAGI_ATTN_Q_PRESCALED))
    return fail(MAGI_EINVAL, "magi_attn_fwd: MAGI_ATTN_Q_PRESCALED is a bf16 flag (fp8: MAGI_ATTN_FP8_POW2_PRESCALED)");
  if ((p->flags & MAGI_ATTN_FP8_FAST_EXP2) && !(p->dtype == MAGI_DTYPE_FP8_E4M3 && (p->flags & MAGI_ATTN_FP8_POW2_PRESCALED)))
    return fail(MAGI_EINVAL, "magi_attn_fwd: MAGI_ATTN_FP8_FAST_EXP2 goes with fp8 and MAGI_ATTN_FP8_POW2_PRESCALED");
  if (p->dtype == MAGI_DTYPE_BF16 && (p->flags & MAGI_ATTN_FP8_POW2_PRESCALED))
    return fail(MAGI_EINVAL, "magi_attn_fwd: MAGI_ATTN_FP8_POW2_PRESCALED is an fp8 flag");
  if (!(p->score_bound >= 0.f)) return fail(MAGI_EINVAL, "magi_attn_fwd: score_bound must be >= 0");
  const bool q_norm = p->q_norm_gamma != nullptr;
  if (q_norm) {
    if (p->dtype != MAGI_DTYPE_BF16 || (p->flags & MAGI_ATTN_Q_PRESCALED))
      return fail(MAGI_EINVAL, "magi_attn_fwd: q_norm takes raw bf16 q (no MAGI_ATTN_Q_PRESCALED)");
    if (!(p->score_bound > 0.f && p->score_bound <= MAGI_SCORE_BOUND_MAX))
      return fail(MAGI_ENOSYS, "magi_attn_fwd: q_norm is implemented for bounded scores (0 < score_bound <= %g)",
                  (double)MAGI_SCORE_BOUND_MAX);
    if (p->q_norm_kind != MAGI_NORM_LAYERNORM_1P && p->q_norm_kind != MAGI_NORM_RMSNORM_1P)
      return fail(MAGI_EINVAL, "magi_attn_fwd: q_norm_kind %d", p->q_norm_kind);
    if (!(p->q_norm_eps >= 0.f)) return fail(MAGI_EINVAL, "magi_attn_fwd: q_norm_eps");
    if (!aligned16(p->q_norm_gamma) || !aligned16(p->q_norm_beta))
      return fail(MAGI_EINVAL, "magi_attn_fwd: q_norm parameters must be 16-byte aligned");
  }
  if (p->score_bound > 0.f && p->dtype != MAGI_DTYPE_BF16)
    return fail(MAGI_EINVAL, "magi_attn_fwd: score_bound is a promise about bf16 inputs");
  const bool auto_bound = (p->flags & MAGI_ATTN_AUTO_BOUND) != 0;
  if (auto_bound) {
    if (p->dtype != MAGI_DTYPE_BF16 || p->score_bound > 0.f || q_norm || p->q_tile_rows != 0 ||
        (p->flags & MAGI_ATTN_BOUNDED_MFMA32))
      return fail(MAGI_EINVAL, "magi_attn_fwd: MAGI_ATTN_AUTO_BOUND goes with bf16 and without score_bound, q_norm, "
                               "q_tile_rows and MAGI_ATTN_BOUNDED_MFMA32 (it measures the bound and picks the kernel itself)");
    if (!workspace || !aligned16(workspace))
      return fail(MAGI_EINVAL, "magi_attn_fwd: MAGI_ATTN_AUTO_BOUND needs a 16-byte workspace on the device, 16-byte aligned");
  }
  if ((p->flags & MAGI_ATTN_ROW_BITS) && (p->flags & MAGI_ATTN_SHARE_WAVES))
    return fail(MAGI_EINVAL, "magi_attn_fwd: MAGI_ATTN_ROW_BITS and MAGI_ATTN_SHARE_WAVES exclude each other");
  if ((p->flags & MAGI_ATTN_ROW_BITS) && (p->split_workspace || p->dtype != MAGI_DTYPE_BF16))
    return fail(MAGI_EINVAL, "magi_attn_fwd: MAGI_ATTN_ROW_BITS goes with bf16 and without split_workspace");
  const bool checked = (p->flags & MAGI_ATTN_CHECKED) != 0;
  if (checked) {
    if (p->dtype != MAGI_DTYPE_BF16 || p->score_bound > 0.f || q_norm || p->q_tile_rows != 0 ||
        (p->flags & (MAGI_ATTN_BOUNDED_MFMA32 | MAGI_ATTN_AUTO_BOUND)))
      return fail(MAGI_EINVAL, "magi_attn_fwd: MAGI_ATTN_CHECKED goes with bf16 and without score_bound, q_norm, q_tile_rows, "
                               "MAGI_ATTN_BOUNDED_MFMA32 and MAGI_ATTN_AUTO_BOUND");
    if (!workspace || !aligned16(workspace))
      return fail(MAGI_EINVAL, "magi_attn_fwd: MAGI_ATTN_CHECKED needs a workspace on the device, 16-byte aligned, of 16 bytes "
                               "per q head, range and 256 rows of max_seqlen_q");
  }
  if (p->split_workspace && (!aligned16(p->split_workspace) || p->split_workspace_bytes < 0))
    return fail(MAGI_EINVAL, "magi_attn_fwd: split_workspace must be 16-byte aligned");
  if (p->out_group_heads < 0 || (p->out_group_heads > 0 && (p->Hq % p->out_group_heads || p->o_stride_g % 8)))
    return fail(MAGI_EINVAL, "magi_attn_fwd: out_group_heads must divide Hq and o_stride_g keep rows 16-byte aligned");
  int k_split = p->total_k;
  if (p->k2 || p->v2) {
    if (!p->k2 || !p->v2) return fail(MAGI_EINVAL, "magi_attn_fwd: k2 and v2 must be given together");
    if (p->k_split < 0 || p->k_split > p->total_k)
      return fail(MAGI_EINVAL, "magi_attn_fwd: k_split %d outside [0, total_k=%d]", p->k_split, p->total_k);
    k_split = p->k_split;
  }
  if (p->dtype == MAGI_DTYPE_FP8_E4M3) {
    if (!p->q_scale || !p->k_scale || !p->v_scale || p->scale_chunk_tokens <= 0)
      return fail(MAGI_EINVAL, "magi_attn_fwd: fp8 needs q/k/v scales and scale_chunk_tokens > 0");
    if ((p->k2_scale != nullptr) != (p->v2_scale != nullptr))
      return fail(MAGI_EINVAL, "magi_attn_fwd: k2_scale and v2_scale come together");
    if (p->k2_scale && (!p->k2 || p->k_split % p->scale_chunk_tokens))
      return fail(MAGI_EINVAL, "magi_attn_fwd: k2_scale / v2_scale need k2 / v2 and k_split on a scale-chunk boundary");
  }

  magi::AttnKernArgs a;
  std::memset(&a, 0, sizeof(a));
  a.q = static_cast<const char*>(p->q);
  a.k = static_cast<const char*>(p->k);
  a.v = static_cast<const char*>(p->v);
  a.k2 = static_cast<const char*>(p->k2);
  a.v2 = static_cast<const char*>(p->v2);
  a.out = static_cast<char*>(p->out);
  a.lse = p->lse;
  a.q_ranges = p->q_ranges;
  a.k_ranges = p->k_ranges;
  a.q_norm_gamma = p->q_norm_gamma;
  a.q_norm_beta = p->q_norm_beta;
  a.q_norm_eps = p->q_norm_eps;
  a.q_norm_kind = p->q_norm_kind;
  a.q_scale = p->q_scale;
  a.k_scale = p->k_scale;
  a.v_scale = p->v_scale;
  a.qs_t = p->q_stride_t * esz;
  a.qs_h = p->q_stride_h * esz;
  a.ks_t = p->k_stride_t * esz;
  a.ks_h = p->k_stride_h * esz;
  a.vs_t = p->v_stride_t * esz;
  a.vs_h = p->v_stride_h * esz;
  a.os_t = p->o_stride_t * 2;
  a.os_h = p->o_stride_h * 2;
  a.os_g = p->o_stride_g * 2;
  a.out_group = p->out_group_heads;
  a.total_q = p->total_q;
  a.total_k = p->total_k;
  a.k_split = k_split;
  a.n_ranges = p->n_ranges;
  a.ranges_mode = p->ranges_mode;
  // Kernel choice for bf16.
  //  * Scores with a promised bound (score_bound): the kernels without a running maximum that hold 64 query rows per
  //    wavefront; 256-row workgroups (4 waves, two per CU: the two waves of a SIMD belong to different workgroups
  //    and drift out of step, so one computes scores while the other is in its softmax) on v_mfma_f32_16x16x32
  //    (the part is power limited and that shape takes less energy per FLOP; measured +3 % on the 720p layer,
  //    between 0 and +6 % from box to box), 128-row ones with 32 rows per wavefront where that leaves at most two of them per CU
  //    (tile_rows), three of those per CU where one round of them holds the launch or its keys are better shared (r32_plan); the
  //    32x32x16 form on request and for 512-row workgroups.
  //  * Otherwise 32 rows per wavefront with the online softmax: 384-row workgroups (12 waves, one workgroup per CU,
  //    every K / V tile fetched once for three times as many rows and one barrier per tile) pay on grids of many
  //    rounds with long key ranges (measured: +3 % at 43 rounds, +1 % at 9.4, -3 % at 5.3); small grids and short
  //    key ranges (cross attention) keep 128 rows (4 waves, three workgroups per CU).
  if (p->dtype == MAGI_DTYPE_FP8_E4M3 && p->q_tile_rows != 0 && p->q_tile_rows != 128)
    return fail(MAGI_EINVAL, "magi_attn_fwd: q_tile_rows %d (fp8: 128)", p->q_tile_rows);
  const bool promised = p->dtype == MAGI_DTYPE_BF16 && p->score_bound > 0.f && p->score_bound <= MAGI_SCORE_BOUND_MAX;
  const bool mfma32 = (p->flags & MAGI_ATTN_BOUNDED_MFMA32) != 0;
  if (p->q_batch_rows != 0) {
    if (p->q_batch_rows < 0 || p->total_q % p->q_batch_rows)
      return fail(MAGI_EINVAL, "magi_attn_fwd: q_batch_rows %d must divide total_q=%d", p->q_batch_rows, p->total_q);
    if (p->dtype != MAGI_DTYPE_BF16 || !(p->score_bound > 0.f) || mfma32 || (promised && p->q_tile_rows != 0 && p->q_tile_rows != 256))
      return fail(MAGI_ENOSYS, "magi_attn_fwd: q_batch_rows is implemented for bf16 with a score_bound, 256-row tiles where it is in force");
    if (p->q_stride_b % 8 || p->o_stride_b % 8)
      return fail(MAGI_EINVAL, "magi_attn_fwd: batch strides must keep rows 16-byte aligned");
    a.batch_rows = p->q_batch_rows;
    a.qs_b = p->q_stride_b * 2;
    a.os_b = p->o_stride_b * 2;
  }
  if (mfma32 && !(promised && (p->flags & MAGI_ATTN_Q_PRESCALED)))
    return fail(MAGI_EINVAL, "magi_attn_fwd: MAGI_ATTN_BOUNDED_MFMA32 goes with bf16, MAGI_ATTN_Q_PRESCALED and a score_bound in force");
  a.Hq = p->Hq;
  a.Hkv = p->Hkv;
  a.G = p->Hq / p->Hkv;
  a.scale_chunk_tokens = p->scale_chunk_tokens;
  a.scale_split_chunk = 0x7fffffff;
  if (p->dtype == MAGI_DTYPE_FP8_E4M3 && p->k2_scale) {
    a.scale_split_chunk = p->k_split / p->scale_chunk_tokens;
    a.k2_scale_delta = (p->k2_scale - p->k_scale) - (long)a.scale_split_chunk * p->Hkv;
    a.v2_scale_delta = (p->v2_scale - p->v_scale) - (long)a.scale_split_chunk * p->Hkv;
  }
  const float scale = p->softmax_scale > 0.f ? p->softmax_scale : 1.0f / std::sqrt((float)p->D);
  a.scale_log2 = scale * 1.4426950408889634f;
  if (p->dtype == MAGI_DTYPE_BF16 && (p->flags & MAGI_ATTN_Q_PRESCALED)) a.scale_log2 = 1.f;  // q . k is the exp2 exponent
  // (with q_norm, or a score bound on unscaled q, the kernel multiplies q by scale_log2 itself while loading it, after
  // which the same holds)

  // One launch of `a` as the bounded-score kernel (bounded) or as the kernel without a promise about the scores; with
  // MAGI_ATTN_CHECKED the bounded-score kernel and the launch that repeats what it could not be trusted with.
  auto launch = [&](bool bounded) -> int {
    // a bound stated for unscaled q (what the reference's callers pass): the kernel applies the softmax scale while
    // it loads q, after which the scores are exp2 exponents as with MAGI_ATTN_Q_PRESCALED
    int64_t split_bytes = p->split_workspace ? p->split_workspace_bytes : 0;  // (0 where it is too little for the launch's pieces)
    const bool scale_q = bounded && !q_norm && !checked && !(p->flags & MAGI_ATTN_Q_PRESCALED);
    a.block_m = 128;
    R32Plan r32 = {false, {1, 0}};
    if (p->dtype == MAGI_DTYPE_BF16) {
      const double wg384 = (double)p->Hq * p->n_ranges * ((p->max_seqlen_q + 383) / 384);
      const bool long_keys = p->max_seqlen_k == 0 || p->max_seqlen_k >= 4096;  // (0 = not stated)
      if (bounded && !checked && !auto_bound && !mfma32 && p->q_tile_rows == 0 && (p->flags & MAGI_ATTN_SHARE_WAVES))
        a.waves = p->max_seqlen_k >= SLAB || how == FIRST || how == SECOND
                      ? waves_plan(p->Hq, p->Hkv, p->n_ranges, p->ranges_mode, p->max_seqlen_q, p->max_seqlen_k)
                      : 0;
      if (bounded && !checked && !mfma32 && p->q_tile_rows == 0 && !a.waves)
        r32 = r32_plan(p->Hq, p->Hkv, p->n_ranges, p->max_seqlen_q, p->max_seqlen_k, split_bytes);
      if (a.waves)
        a.block_m = 32;
      else if (r32.use)
        a.block_m = 128;
      else if (bounded && !checked && !mfma32)
        a.block_m = tile_rows(p->Hq, p->Hkv, p->n_ranges, p->max_seqlen_q, p->max_seqlen_k, split_bytes);
      else if (bounded)
        a.block_m = 256;  // (512-row workgroups fetch half the tiles and measure 1 % slower: their two waves per SIMD march in step)
      else if (wg384 >= 9.0 * compute_units() && long_keys)
        a.block_m = 384;
      if (p->q_tile_rows != 0) {
        const int r = p->q_tile_rows;
        if ((q_norm || scale_q) && r != 256)
          return fail(MAGI_EINVAL, "magi_attn_fwd: q_tile_rows %d (with q_norm, or a score bound on unscaled q: 256)", r);
        if (bounded ? (r != 256 && r != 512) : (r != 128 && r != 384))
          return fail(MAGI_EINVAL, "magi_attn_fwd: q_tile_rows %d (bf16: 128 or 384; with a score bound: 256 or 512)", r);
        a.block_m = r;
      }
    }
    a.tiles_per_range = (p->max_seqlen_q + a.block_m - 1) / a.block_m;
    a.flags = p->flags | (bounded ? magi::ATTN_BOUNDED : 0) | (scale_q ? magi::ATTN_SCALE_Q : 0);
    const double total = (double)p->Hq * p->n_ranges * a.tiles_per_range;
    if (total > 2.0e9) return fail(MAGI_EINVAL, "magi_attn_fwd: grid too large (%.3g workgroups)", total);
    a.per_xcd = items_per_xcd(p->Hq, p->Hkv, p->n_ranges, a.tiles_per_range);
    a.split_from = UINT32_MAX;
    const bool fp8 = p->dtype == MAGI_DTYPE_FP8_E4M3;
    auto pieces = [&](const SharePlan& s) {
      a.share_pieces = s.pieces;
      a.share_tiles = s.tiles;
      if (s.pieces > 1) a.partial = static_cast<float*>(p->split_workspace);
    };
    a.share_pieces = 1;
    if (a.waves) {
      if (how == END) return not_begun();
      if (how == TEXT) return ALONE;
      if (!held || how == BEGIN) return launch_waves(a, stream);
      *held = a;
      return HELD;
    }
    if (r32.use) pieces(r32.share);
    if ((fp8 || (bounded && a.block_m == 256 && !mfma32)) && split_bytes > 0) {
      const SplitPlan s = split_plan(a.per_xcd, p->n_ranges, p->max_seqlen_q, p->max_seqlen_k, fp8);
      if (s.from < a.per_xcd && s.bytes(a.per_xcd) <= split_bytes) {
        a.partial = static_cast<float*>(p->split_workspace);
        a.split_from = s.from;
        a.split_pieces = s.pieces;
        a.split_num = s.num;
        a.split_den = s.den;
      }
    }
    // The online softmax on unscaled q, 128 rows a workgroup: the 16x16x32 form for launches of more workgroups than run at a time
    // (three per CU) and for shared keys, the 32x32x16 form for the others.  Measured, 32x32x16 / 16x16x32: 9360 rows x 2
    // chunks x 24 heads over 28080 and 37440 keys 6604 / 6407 us, 93600 x 24 text cross attention 612 / 600, over 20 keys 223 / 202,
    // 4580 x 48 over 3435 to 6870 555 / 545; 700 x 24 over 700 22.3 / 23.2, 700 x 48 over 1400 48.5 / 50.7, 2000 x 24 57 / 58.
    // (MAGI_ATTN_ROW_BITS: the 32x32x16 forms in all sizes, whose order of the keys is one.)
    const bool online128 = !fp8 && !bounded && a.block_m == 128 && !(p->flags & (MAGI_ATTN_Q_PRESCALED | MAGI_ATTN_ROW_BITS));
    if (online128 && !a.gate && split_bytes > 0) {
      const SharePlan s = share_plan(a.per_xcd, p->n_ranges, p->max_seqlen_q, p->max_seqlen_k);
      if (s.bytes(a.per_xcd) <= split_bytes) pieces(s);
    }
    // (of the other forms the one of large launches: in the smaller ones the core's rows or keys are dealt out over the whole chip as it is)
    const bool x16 = bounded && a.block_m == 256 && !checked && !mfma32 && !auto_bound;
    const bool plain = x16 && !scale_q;
    // (raw q is bounded, in 128- or 256-row workgroups)
    const bool hold = how == FIRST  ? plain || (fp8 && (p->flags & MAGI_ATTN_FP8_POW2_PRESCALED))
                      : how == TEXT ? q_norm && a.share_pieces <= 1
                                    : how != NOW && plain;
    if (hold) {
      *held = a;
      if (how == BEGIN && a.split_from < a.per_xcd) {
        const hipError_t e = magi::launch_attn_fwd_bf16_x16(a, static_cast<hipStream_t>(stream), false);
        if (e != hipSuccess) return hip_fail(e, "magi_attn_fwd_begin launch");
        count_launches(1);
      }
      return HELD;
    }
    if (how == END) return not_begun();
    if (how == SECOND || how == TEXT) return ALONE;
    hipError_t e;
    if (p->dtype != MAGI_DTYPE_BF16)
      e = magi::launch_attn_fwd_fp8(a, static_cast<hipStream_t>(stream));
    else if (checked)
      e = magi::launch_attn_fwd_bf16_checked(a, compute_units(), static_cast<hipStream_t>(stream));
    else if (r32.use || (online128 && (a.share_pieces > 1 || 8.0 * a.per_xcd > 3.0 * compute_units())))
      e = magi::launch_attn_fwd_bf16_r32(a, static_cast<hipStream_t>(stream));
    else if (bounded && a.block_m <= 256 && !mfma32)
      e = magi::launch_attn_fwd_bf16_x16(a, static_cast<hipStream_t>(stream));
    else if (bounded)
      e = magi::launch_attn_fwd_bf16_w64(a, static_cast<hipStream_t>(stream));
    else
      e = magi::launch_attn_fwd_bf16(a, static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return hip_fail(e, "magi_attn_fwd launch");
    count_launches((checked ? 2 : 1) + (a.split_from < a.per_xcd) + (a.share_pieces > 1));
    return MAGI_OK;
  };

  if (checked) {
    a.verdict = reinterpret_cast<int*>(workspace);
    return launch(true);
  }
  if (!auto_bound) return launch(promised);
  if (how == SECOND || how == TEXT) return ALONE;
  if (how == END) return not_begun();

  // No promise about the scores: measure one.  Two streaming passes leave the largest squared length of a q row and
  // of a k row in the workspace (|q . k| <= |q| |k|); both attention kernels are launched behind them, each tests
  // the bound on the device and only the one it selects runs (the other returns at once).  No host synchronisation.
  hipStream_t st = static_cast<hipStream_t>(stream);
  unsigned* ws = reinterpret_cast<unsigned*>(workspace);
  hipError_t e = magi::launch_gate_init(ws, st);
  if (e == hipSuccess) e = magi::launch_row_norm_max(a.q, a.qs_t, a.qs_h, p->total_q, p->Hq, ws, st);
  if (e == hipSuccess && k_split > 0) e = magi::launch_row_norm_max(a.k, a.ks_t, a.ks_h, k_split, p->Hkv, ws + 1, st);
  if (e == hipSuccess && p->total_k > k_split)
    e = magi::launch_row_norm_max(a.k2, a.ks_t, a.ks_h, p->total_k - k_split, p->Hkv, ws + 1, st);
  if (e != hipSuccess) return hip_fail(e, "magi_attn_fwd bound measurement");
  count_launches(2 + (k_split > 0) + (p->total_k > k_split));
  a.gate = workspace;
  a.gate_want = 1;
  int rc = launch(true);
  if (rc != MAGI_OK) return rc;
  a.gate_want = 0;
  return launch(false);
}

}  // namespace

namespace {

// magi_small_projections, and with `e4m3` magi_small_projections_e4m3
struct SmallProjE4m3 {
  float q_scale, k_scale;
  void* v_out;
};
int small_projections_impl(const magi_small_proj_args* p, const SmallProjE4m3* e4m3, void* stream) {
  if (!p) return fail(MAGI_EINVAL, "magi_small_projections: args is NULL");
  MAGI_CHECK_LAYOUT("magi_small_projections", p);
  if (p->S < 0 || p->T < 0 || p->Hq < 0 || p->Hkv < 0 || p->Hqx < 0 || p->batch < 0)
    return fail(MAGI_EINVAL, "magi_small_projections: negative size");
  const bool hidden = p->S > 0 && p->Hq + p->Hkv + p->Hqx > 0, text = p->T > 0 && p->Hkv > 0;
  if (!hidden && !text) return MAGI_OK;
  if ((double)(p->S / 32 + 1) * (p->Hq + 2.0 * p->Hkv + p->Hqx) + (double)(p->T / 32 + 1) * 2 * p->Hkv > 2.0e9)
    return fail(MAGI_ENOSYS, "magi_small_projections: too many rows");
  if (!(p->eps >= 0.f)) return fail(MAGI_EINVAL, "magi_small_projections: eps");
  magi::SmallProjKernArgs a;
  std::memset(&a, 0, sizeof(a));
  a.Hq = p->Hq;
  a.Hkv = p->Hkv;
  a.Hqx = p->Hqx;
  a.eps = p->eps;
  a.batch = p->batch > 1 ? p->batch : 1;
  if (hidden) {
    if (p->K <= 0 || p->K % 64) return fail(MAGI_ENOSYS, "magi_small_projections: K=%d is not a multiple of 64", p->K);
    if (!p->x || !p->w) return fail(MAGI_EINVAL, "magi_small_projections: NULL x / w");
    if (p->x_stride < p->K || p->x_stride % 8 || !aligned16(p->x) || !aligned16(p->w))
      return fail(MAGI_EINVAL, "magi_small_projections: rows of x and w must be 16-byte aligned and at least K long");
    // (32-bit byte offsets within the descriptors' 2^31 - 1: row 63 of a workgroup's 64 rows of x, 2^25 bytes apart at most, which nearly
    // fills them; the 128 weight rows of a head)
    if (p->x_stride > (1 << 24) || p->K > (1 << 22)) return fail(MAGI_ENOSYS, "magi_small_projections: rows above 2^22 elements are not implemented");
    if (p->ln_w && (p->K > 1024 || (text && p->Kt > 1024)))
      return fail(MAGI_ENOSYS, "magi_small_projections: the input norm is implemented for K (and Kt) up to 1024");
    if ((p->ln_w != nullptr) != (p->ln_b != nullptr) || !aligned16(p->ln_w) || !aligned16(p->ln_b) || (p->ln_w && !(p->ln_eps >= 0.f)))
      return fail(MAGI_EINVAL, "magi_small_projections: ln_w and ln_b come together, 16-byte aligned, with ln_eps >= 0");
    if (p->R2 < 0 || p->R2 % 8 || 2 * p->R2 > 128) return fail(MAGI_EINVAL, "magi_small_projections: R2=%d must be a multiple of 8 up to 64", p->R2);
    if ((p->Hq > 0 && (!p->q_out || !p->gq)) || (p->Hkv > 0 && !p->gk) || (p->Hqx > 0 && !p->qx_out))
      return fail(MAGI_EINVAL, "magi_small_projections: NULL output or norm parameter");
    if (p->n_cache_rows < 0 || p->n_cache_rows > p->S)
      return fail(MAGI_EINVAL, "magi_small_projections: n_cache_rows %d outside [0, S=%d]", p->n_cache_rows, p->S);
    if (p->Hkv > 0 && ((p->n_cache_rows > 0 && !p->kv_out) || (p->n_cache_rows < p->S && !p->kv_tail)))
      return fail(MAGI_EINVAL, "magi_small_projections: NULL kv_out / kv_tail");
    if (p->kv_stride_t % 8 || p->kv_tail_stride_t % 8 || !aligned16(p->q_out) || !aligned16(p->kv_out) || !aligned16(p->kv_tail) ||
        !aligned16(p->qx_out) || !aligned16(p->rope) || !aligned16(p->gq) || !aligned16(p->bq) || !aligned16(p->gk) || !aligned16(p->bk))
      return fail(MAGI_EINVAL, "magi_small_projections: buffers must be 16-byte aligned");
    if (!std::isfinite(p->q_premul)) return fail(MAGI_EINVAL, "magi_small_projections: q_premul is not finite");
    a.x = static_cast<const char*>(p->x);
    a.w = static_cast<const char*>(p->w);
    a.ln_w = static_cast<const char*>(p->ln_w);
    a.ln_b = static_cast<const char*>(p->ln_b);
    a.x_stride = p->x_stride * 2;
    a.S = p->S;
    a.K = p->K;
    a.ln_fp32 = p->ln_params_fp32 != 0;
    a.ln_eps = p->ln_eps;
    a.rope = p->R2 > 0 ? p->rope : nullptr;
    a.R2 = a.rope ? p->R2 : 0;
    a.gq = p->gq;
    a.bq = p->bq;
    a.gk = p->gk;
    a.bk = p->bk;
    a.q_premul = p->q_premul == 0.f ? 1.f : p->q_premul;
    a.n_cache_rows = p->n_cache_rows;
    a.q_out = static_cast<char*>(p->q_out);
    a.kv_out = static_cast<char*>(p->kv_out);
    a.kv_tail = static_cast<char*>(p->kv_tail);
    a.kv_stride_t = p->kv_stride_t * 2;
    a.kv_tail_stride_t = p->kv_tail_stride_t * 2;
    a.qx_out = static_cast<char*>(p->qx_out);
    if (e4m3) {
      if ((p->Hq > 0 && !(e4m3->q_scale > 0.f && std::isfinite(e4m3->q_scale))) ||
          (p->Hkv > 0 && (!(e4m3->k_scale > 0.f && std::isfinite(e4m3->k_scale)) || !e4m3->v_out || !aligned16(e4m3->v_out))))
        return fail(MAGI_EINVAL, "magi_small_projections_e4m3: q_quant_scale and k_quant_scale must be positive and finite, v_out 16-byte aligned");
      a.out_fp8 = 1;
      a.q_inv_scale = 1.f / e4m3->q_scale;
      a.k_inv_scale = 1.f / e4m3->k_scale;
      a.v_out = static_cast<char*>(e4m3->v_out);
      a.kv_stride_t = p->kv_stride_t;
      a.kv_tail_stride_t = p->kv_tail_stride_t;
    }
  }
  if (text) {
    if (p->Kt <= 0 || p->Kt % 64) return fail(MAGI_ENOSYS, "magi_small_projections: Kt=%d is not a multiple of 64", p->Kt);
    if (!p->text || !p->w_text || !p->text_out || !p->gkx) return fail(MAGI_EINVAL, "magi_small_projections: NULL text / w_text / text_out / gkx");
    if (p->text_stride < p->Kt || p->text_stride % 8 || !aligned16(p->text) || !aligned16(p->w_text) || !aligned16(p->text_out) ||
        !aligned16(p->gkx) || !aligned16(p->bkx))
      return fail(MAGI_EINVAL, "magi_small_projections: rows of text and w_text must be 16-byte aligned and at least Kt long");
    if (p->text_stride > (1 << 24) || p->Kt > (1 << 22)) return fail(MAGI_ENOSYS, "magi_small_projections: rows above 2^22 elements are not implemented");
    a.text = static_cast<const char*>(p->text);
    a.w_text = static_cast<const char*>(p->w_text);
    a.text_stride = p->text_stride * 2;
    a.T = p->T;
    a.Kt = p->Kt;
    a.gkx = p->gkx;
    a.bkx = p->bkx;
    a.text_out = static_cast<char*>(p->text_out);
  }
  hipError_t e = magi::launch_small_proj(a, compute_units(), static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return hip_fail(e, "magi_small_projections launch");
  count_launches(1);
  return MAGI_OK;
}

}  // namespace

static int prologue_impl(const magi_prologue_args* p, void* v_row_max, void* stream) {
  if (!p) return fail(MAGI_EINVAL, "magi_qk_prologue: args is NULL");
  MAGI_CHECK_LAYOUT("magi_qk_prologue", p);
  if (p->D != 128) return fail(MAGI_ENOSYS, "magi_qk_prologue: head_dim %d not implemented (128 only)", p->D);
  if (p->S < 0 || p->Hq < 0 || p->Hkv < 0) return fail(MAGI_EINVAL, "magi_qk_prologue: negative size");
  if (p->S == 0 || p->Hq + p->Hkv == 0) return MAGI_OK;
  if (p->R2 < 0 || p->R2 % 8 || 2 * p->R2 > p->D)
    return fail(MAGI_EINVAL, "magi_qk_prologue: R2=%d must be a multiple of 8 with 2*R2 <= D", p->R2);
  if (p->norm_kind < 0 || p->norm_kind > 2) return fail(MAGI_EINVAL, "magi_qk_prologue: norm_kind %d", p->norm_kind);
  if (p->batch < 0) return fail(MAGI_EINVAL, "magi_qk_prologue: negative batch");
  if (p->Hq > 0 && (!p->q_raw || !p->q_out)) return fail(MAGI_EINVAL, "magi_qk_prologue: NULL q_raw/q_out");
  const bool out8 = p->out_dtype == MAGI_DTYPE_FP8_E4M3;
  if (p->out_dtype != MAGI_DTYPE_BF16 && !out8) return fail(MAGI_EINVAL, "magi_qk_prologue: out_dtype %d", p->out_dtype);
  if (p->Hkv > 0 && (!p->k_raw || (!p->v_raw && !out8))) return fail(MAGI_EINVAL, "magi_qk_prologue: NULL k_raw/v_raw");
  if (out8 && ((p->Hq > 0 && !(p->q_quant_scale > 0.f && std::isfinite(p->q_quant_scale))) ||
               (p->Hkv > 0 && !(p->k_quant_scale > 0.f && std::isfinite(p->k_quant_scale)))))
    return fail(MAGI_EINVAL, "magi_qk_prologue: e4m3 outputs need positive finite q_quant_scale / k_quant_scale");
  if (p->n_cache_rows < 0 || p->n_cache_rows > p->S)
    return fail(MAGI_EINVAL, "magi_qk_prologue: n_cache_rows %d outside [0, S=%d]", p->n_cache_rows, p->S);
  if (p->Hkv > 0 && p->n_cache_rows > 0 && !p->kv_out) return fail(MAGI_EINVAL, "magi_qk_prologue: NULL kv_out");
  if (p->Hkv > 0 && p->n_cache_rows < p->S && !p->kv_tail)
    return fail(MAGI_EINVAL, "magi_qk_prologue: kv_tail needed for rows >= n_cache_rows");
  if (p->norm_kind != MAGI_NORM_NONE && ((p->Hq > 0 && !p->gq) || (p->Hkv > 0 && !p->gk)))
    return fail(MAGI_EINVAL, "magi_qk_prologue: NULL gamma");
  if (p->R2 > 0 && p->rope && (reinterpret_cast<uintptr_t>(p->rope) & 15u))
    return fail(MAGI_EINVAL, "magi_qk_prologue: rope must be 16-byte aligned");
  if (p->q_raw_stride_t % 8 || p->k_raw_stride_t % 8 || p->v_raw_stride_t % 8 || p->kv_stride_t % 8 ||
      p->kv_tail_stride_t % 8)
    return fail(MAGI_EINVAL, "magi_qk_prologue: strides must keep rows 16-byte aligned");
  if (!aligned16(p->q_raw) || !aligned16(p->k_raw) || ((!out8 || v_row_max) && !aligned16(p->v_raw)) || !aligned16(p->q_out) ||
      !aligned16(p->kv_out) || !aligned16(p->kv_tail))
    return fail(MAGI_EINVAL, "magi_qk_prologue: buffers must be 16-byte aligned");

  magi::PrologueKernArgs a;
  std::memset(&a, 0, sizeof(a));
  a.q_raw = static_cast<const char*>(p->q_raw);
  a.k_raw = static_cast<const char*>(p->k_raw);
  a.v_raw = static_cast<const char*>(p->v_raw);
  a.rope = p->R2 > 0 ? p->rope : nullptr;
  a.gq = p->gq;
  a.bq = p->bq;
  a.gk = p->gk;
  a.bk = p->bk;
  a.q_out = static_cast<char*>(p->q_out);
  a.kv_out = static_cast<char*>(p->kv_out);
  a.kv_tail = static_cast<char*>(p->kv_tail);
  a.q_raw_stride_t = p->q_raw_stride_t * 2;
  a.k_raw_stride_t = p->k_raw_stride_t * 2;
  a.v_raw_stride_t = p->v_raw_stride_t * 2;
  a.kv_stride_t = p->kv_stride_t * (out8 ? 1 : 2);
  a.kv_tail_stride_t = p->kv_tail_stride_t * (out8 ? 1 : 2);
  a.out_fp8 = out8;
  a.q_inv_scale = out8 && p->Hq > 0 ? 1.f / p->q_quant_scale : 1.f;
  a.k_inv_scale = out8 && p->Hkv > 0 ? 1.f / p->k_quant_scale : 1.f;
  a.S = p->S;
  a.n_cache_rows = p->n_cache_rows;
  a.Hq = p->Hq;
  a.Hkv = p->Hkv;
  a.R2 = a.rope ? p->R2 : 0;
  a.norm_kind = p->norm_kind;
  a.eps = p->eps;
  a.batch = p->batch > 1 ? p->batch : 1;
  if (!(p->q_premul == p->q_premul) || std::fabs(p->q_premul) > 1e30f)
    return fail(MAGI_EINVAL, "magi_qk_prologue: q_premul is not finite");
  a.q_premul = p->q_premul == 0.f ? 1.f : p->q_premul;
  a.v_row_max = static_cast<unsigned short*>(v_row_max);
  hipError_t e = magi::launch_prologue(a, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return hip_fail(e, "magi_qk_prologue launch");
  count_launches(1);
  return MAGI_OK;
}

extern "C" {

int magi_qk_prologue(const magi_prologue_args* p, void* stream) { return prologue_impl(p, nullptr, stream); }

int magi_qk_prologue_row_max(const magi_prologue_args* p, void* v_row_max, void* stream) {
  if (p && p->struct_size == sizeof(*p) && p->S > 0 && p->Hkv > 0) {  // (the rest is prologue_impl's to refuse)
    if (p->out_dtype != MAGI_DTYPE_FP8_E4M3) return fail(MAGI_EINVAL, "magi_qk_prologue_row_max: e4m3 outputs only");
    if (!p->v_raw || !v_row_max) return fail(MAGI_EINVAL, "magi_qk_prologue_row_max: NULL v_raw/v_row_max");
  }
  return prologue_impl(p, v_row_max, stream);
}

int magi_qkv_proj_prologue(const magi_qkv_proj_args* p, void* stream) {
  if (!p) return fail(MAGI_EINVAL, "magi_qkv_proj_prologue: args is NULL");
  MAGI_CHECK_LAYOUT("magi_qkv_proj_prologue", p);
  if (p->D != 128) return fail(MAGI_ENOSYS, "magi_qkv_proj_prologue: head_dim %d not implemented (128 only)", p->D);
  if (p->S < 0 || p->K <= 0 || p->Hq < 0 || p->Hkv < 0 || p->Hqx < 0)
    return fail(MAGI_EINVAL, "magi_qkv_proj_prologue: bad size");
  const int heads = p->Hq + 2 * p->Hkv + p->Hqx;
  if (p->S == 0 || heads == 0) return MAGI_OK;
  if (p->K % 64) return fail(MAGI_ENOSYS, "magi_qkv_proj_prologue: K=%d is not a multiple of 64", p->K);
  if (heads % 2) return fail(MAGI_ENOSYS, "magi_qkv_proj_prologue: an odd number of heads (%d) is not implemented", heads);
  if (p->rope && p->R2 != 48 && p->R2 != 0)
    return fail(MAGI_ENOSYS, "magi_qkv_proj_prologue: R2=%d not implemented (48, or 0 / NULL rope for none)", p->R2);
  if (p->norm_kind < 0 || p->norm_kind > 2) return fail(MAGI_EINVAL, "magi_qkv_proj_prologue: norm_kind %d", p->norm_kind);
  if (p->batch < 0) return fail(MAGI_EINVAL, "magi_qkv_proj_prologue: negative batch");
  if (!p->x || !p->w) return fail(MAGI_EINVAL, "magi_qkv_proj_prologue: NULL x / w");
  if (p->x_stride < p->K || p->w_stride < p->K) return fail(MAGI_EINVAL, "magi_qkv_proj_prologue: row stride below K");
  if (p->Hq > 0 && !p->q_out) return fail(MAGI_EINVAL, "magi_qkv_proj_prologue: NULL q_out");
  if (p->Hqx > 0 && !p->qx_out) return fail(MAGI_EINVAL, "magi_qkv_proj_prologue: NULL qx_out");
  if (p->n_cache_rows < 0 || p->n_cache_rows > p->S)
    return fail(MAGI_EINVAL, "magi_qkv_proj_prologue: n_cache_rows %d outside [0, S=%d]", p->n_cache_rows, p->S);
  if (p->Hkv > 0 && p->n_cache_rows > 0 && !p->kv_out) return fail(MAGI_EINVAL, "magi_qkv_proj_prologue: NULL kv_out");
  if (p->Hkv > 0 && p->n_cache_rows < p->S && !p->kv_tail)
    return fail(MAGI_EINVAL, "magi_qkv_proj_prologue: kv_tail needed for rows >= n_cache_rows");
  if (p->norm_kind != MAGI_NORM_NONE && ((p->Hq > 0 && !p->gq) || (p->Hkv > 0 && !p->gk)))
    return fail(MAGI_EINVAL, "magi_qkv_proj_prologue: NULL gamma");
  if (p->x_stride % 8 || p->w_stride % 8 || p->kv_stride_t % 8 || p->kv_tail_stride_t % 8)
    return fail(MAGI_EINVAL, "magi_qkv_proj_prologue: strides must keep rows 16-byte aligned");
  if (!aligned16(p->x) || !aligned16(p->w) || !aligned16(p->q_out) || !aligned16(p->kv_out) || !aligned16(p->kv_tail) ||
      !aligned16(p->qx_out) || !aligned16(p->rope) || !aligned16(p->gq) || !aligned16(p->bq) || !aligned16(p->gk) ||
      !aligned16(p->bk))
    return fail(MAGI_EINVAL, "magi_qkv_proj_prologue: buffers must be 16-byte aligned");
  // (the loader addresses a workgroup's 256 rows with 32-bit byte offsets)
  if (p->x_stride > (1 << 21) || p->w_stride > (1 << 21))
    return fail(MAGI_ENOSYS, "magi_qkv_proj_prologue: row strides above 2^21 elements are not implemented");
  if (!(p->q_premul == p->q_premul) || std::fabs(p->q_premul) > 1e30f)
    return fail(MAGI_EINVAL, "magi_qkv_proj_prologue: q_premul is not finite");
  magi::QkvGemmKernArgs a;
  std::memset(&a, 0, sizeof(a));
  a.x = static_cast<const char*>(p->x);
  a.w = static_cast<const char*>(p->w);
  a.rope = (p->rope && p->R2 == 48) ? p->rope : nullptr;
  a.gq = p->gq;
  a.bq = p->bq;
  a.gk = p->gk;
  a.bk = p->bk;
  a.q_out = static_cast<char*>(p->q_out);
  a.kv_out = static_cast<char*>(p->kv_out);
  a.kv_tail = static_cast<char*>(p->kv_tail);
  a.qx_out = static_cast<char*>(p->qx_out);
  a.x_stride = p->x_stride * 2;
  a.w_stride = p->w_stride * 2;
  a.kv_stride_t = p->kv_stride_t * 2;
  a.kv_tail_stride_t = p->kv_tail_stride_t * 2;
  a.S = p->S;
  a.K = p->K;
  a.n_cache_rows = p->n_cache_rows;
  a.Hq = p->Hq;
  a.Hkv = p->Hkv;
  a.Hqx = p->Hqx;
  a.norm_kind = p->norm_kind;
  a.eps = p->eps;
  a.batch = p->batch > 1 ? p->batch : 1;
  a.q_premul = p->q_premul == 0.f ? 1.f : p->q_premul;
  hipError_t e = magi::launch_qkv_gemm_prologue(a, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return hip_fail(e, "magi_qkv_proj_prologue launch");
  count_launches(1);
  return MAGI_OK;
}

int magi_small_projections(const magi_small_proj_args* p, void* stream) { return small_projections_impl(p, nullptr, stream); }

int magi_small_projections_e4m3(const magi_small_proj_args* p, float q_quant_scale, float k_quant_scale, void* v_out, void* stream) {
  const SmallProjE4m3 e4m3 = {q_quant_scale, k_quant_scale, v_out};
  return small_projections_impl(p, &e4m3, stream);
}

int magi_small_layer(const magi_small_layer_args* p, void* stream) {
  if (!p) return fail(MAGI_EINVAL, "magi_small_layer: args is NULL");
  MAGI_CHECK_LAYOUT("magi_small_layer", p);
  if (p->parts < 1 || p->parts > 3) return fail(MAGI_EINVAL, "magi_small_layer: parts %d", p->parts);
  auto at = [](void* base, int64_t elements) -> const void* { return base ? static_cast<char*>(base) + 2 * elements : nullptr; };
  magi_attn_args a;
  std::memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.q_stride_t = (int64_t)p->Hq * 128;
  a.q_stride_h = a.o_stride_h = a.D = 128;
  a.k_stride_h = a.v_stride_h = 256;
  a.total_q = p->S;
  a.Hq = p->Hq;
  a.Hkv = p->Hkv;
  a.dtype = MAGI_DTYPE_BF16;
  a.o_stride_t = p->o_stride_t;
  a.o_stride_g = p->o_stride_g;
  a.out_group_heads = p->out_group_heads;
  if (p->parts & 1) {
    magi_small_proj_args s;
    std::memset(&s, 0, sizeof(s));
    s.struct_size = sizeof(s);
    s.x = p->x;
    s.w = p->w;
    s.ln_w = p->ln_w;
    s.ln_b = p->ln_b;
    s.x_stride = s.K = p->K;
    s.S = p->S;
    s.ln_params_fp32 = p->ln_params_fp32;
    s.ln_eps = p->ln_eps;
    s.Hq = s.Hqx = p->Hq;
    s.Hkv = p->Hkv;
    s.R2 = p->R2;
    s.rope = p->rope;
    s.gq = p->gq;
    s.bq = p->bq;
    s.gk = p->gk;
    s.bk = p->bk;
    s.eps = p->eps;
    s.batch = 1;
    s.q_premul = p->q_premul;
    s.n_cache_rows = p->kept;
    s.q_out = p->q;
    s.kv_out = p->kv_new;
    s.kv_tail = p->kv_side;
    s.kv_stride_t = s.kv_tail_stride_t = p->kv_row;
    s.qx_out = p->qx;
    s.text = p->text;
    s.w_text = p->w_text;
    s.text_stride = p->text_stride;
    s.T = p->T;
    s.Kt = p->Kt;
    s.gkx = p->gkx;
    s.bkx = p->bkx;
    s.text_out = p->text_kv;
    if (const int rc = small_projections_impl(&s, nullptr, stream)) return rc;
    a.q = p->q;
    a.k = p->kv;
    a.v = at(p->kv, 128);
    a.k2 = p->kv_side;
    a.v2 = at(p->kv_side, 128);
    a.k_stride_t = a.v_stride_t = p->kv_row;
    a.total_k = p->total_k;
    a.k_split = p->k_split;
    a.q_ranges = p->q_ranges;
    a.k_ranges = p->k_ranges;
    a.n_ranges = p->n_core;
    a.ranges_mode = MAGI_RANGES_PAIRS;
    a.max_seqlen_q = p->max_core_q;
    a.max_seqlen_k = p->max_core_k;
    a.flags = MAGI_ATTN_Q_PRESCALED | MAGI_ATTN_SHARE_WAVES | p->core_flags;
    a.score_bound = p->core_bound;
    a.out = p->core_out;
    a.split_workspace = p->core_split;
    a.split_workspace_bytes = p->core_split_bytes;
    if (p->parts == 1) return attn_fwd_impl(&a, stream, nullptr);
  }
  const magi_attn_args core = a;
  if (p->parts & 2) {
    a.q = p->qx;
    a.k = p->text_kv;
    a.v = at(p->text_kv, 128);
    a.k2 = a.v2 = nullptr;
    a.k_stride_t = a.v_stride_t = (int64_t)p->Hkv * 256;
    a.total_k = a.k_split = p->T;
    a.q_ranges = p->cu_q;
    a.k_ranges = p->cu_k;
    a.n_ranges = p->n_cross;
    a.ranges_mode = MAGI_RANGES_CU;
    a.max_seqlen_q = p->max_cross_q;
    a.max_seqlen_k = p->max_cross_k;
    a.flags = MAGI_ATTN_SHARE_WAVES | p->cross_flags;
    a.score_bound = p->cross_bound;
    a.out = p->cross_out;
    a.split_workspace = p->cross_split;
    a.split_workspace_bytes = p->cross_split_bytes;
    a.q_norm_gamma = p->gqx;
    a.q_norm_beta = p->bqx;
    a.q_norm_eps = p->eps;
    a.q_norm_kind = MAGI_NORM_LAYERNORM_1P;
    return p->parts == 3 ? attn_fwd_two(&core, &a, stream) : attn_fwd_impl(&a, stream, nullptr);
  }
  return MAGI_OK;
}

int magi_layer_norm(const void* x, int64_t x_stride, const void* weight, const void* bias, int32_t params_fp32,
                    void* y, int64_t y_stride, int64_t rows, int32_t cols, float eps, void* stream) {
  if (rows < 0 || cols < 0) return fail(MAGI_EINVAL, "magi_layer_norm: negative size");
  if (rows == 0 || cols == 0) return MAGI_OK;
  if (cols % 8 || cols > 8192)
    return fail(MAGI_ENOSYS, "magi_layer_norm: cols %d not implemented (multiples of 8 up to 8192)", cols);
  if (!x || !y) return fail(MAGI_EINVAL, "magi_layer_norm: NULL x/y");
  if (x_stride < cols || y_stride < cols) return fail(MAGI_EINVAL, "magi_layer_norm: row stride below cols");
  if (x_stride % 8 || y_stride % 8 || !aligned16(x) || !aligned16(y))
    return fail(MAGI_EINVAL, "magi_layer_norm: rows must be 16-byte aligned");
  if (!(eps >= 0.f)) return fail(MAGI_EINVAL, "magi_layer_norm: eps");
  if (rows > 0x7fffffffLL * 4) return fail(MAGI_ENOSYS, "magi_layer_norm: more than 2^33 rows");  // (4 rows per workgroup)
  hipError_t e = magi::launch_layer_norm(static_cast<const char*>(x), x_stride * 2, weight, bias, params_fp32 != 0,
                                         static_cast<char*>(y), y_stride * 2, rows, cols, eps,
                                         static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return hip_fail(e, "magi_layer_norm launch");
  count_launches(1);
  return MAGI_OK;
}

int magi_layer_norm_e4m3(const void* x, int64_t x_stride, const void* weight, const void* bias, int32_t params_fp32,
                         const float* const* scales, void* const* ys, int32_t n_out, int64_t rows, int32_t cols, float eps,
                         void* stream) {
  if (rows < 0 || cols < 0 || n_out < 0) return fail(MAGI_EINVAL, "magi_layer_norm_e4m3: negative size");
  if (rows == 0 || cols == 0 || n_out == 0) return MAGI_OK;
  if (n_out > 4) return fail(MAGI_ENOSYS, "magi_layer_norm_e4m3: %d outputs (at most 4)", n_out);
  if (cols % 8 || cols > 8192)
    return fail(MAGI_ENOSYS, "magi_layer_norm_e4m3: cols %d not implemented (multiples of 8 up to 8192)", cols);
  if (!x || !scales || !ys) return fail(MAGI_EINVAL, "magi_layer_norm_e4m3: NULL pointer");
  if (x_stride < cols) return fail(MAGI_EINVAL, "magi_layer_norm_e4m3: row stride below cols");
  if (x_stride % 8 || !aligned16(x) || !aligned16(weight) || !aligned16(bias))
    return fail(MAGI_EINVAL, "magi_layer_norm_e4m3: rows and parameters must be 16-byte aligned");
  if (!(eps >= 0.f)) return fail(MAGI_EINVAL, "magi_layer_norm_e4m3: eps");
  magi::LnQuantKernArgs a;
  std::memset(&a, 0, sizeof(a));
  for (int k = 0; k < n_out; ++k) {
    if (!scales[k] || !ys[k]) return fail(MAGI_EINVAL, "magi_layer_norm_e4m3: NULL scale / output %d", k);
    if (!aligned16(scales[k]) || (reinterpret_cast<uintptr_t>(ys[k]) & 7u))
      return fail(MAGI_EINVAL, "magi_layer_norm_e4m3: scales must be 16-byte aligned, outputs 8-byte");
    a.scale[k] = scales[k];
    a.y[k] = static_cast<char*>(ys[k]);
  }
  a.x = static_cast<const char*>(x);
  a.xs = x_stride * 2;
  a.w = static_cast<const char*>(weight);
  a.b = static_cast<const char*>(bias);
  a.rows = rows;
  a.cols = cols;
  a.n_out = n_out;
  a.eps = eps;
  hipError_t e = magi::launch_layer_norm_quant(a, params_fp32 != 0, compute_units(), static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return hip_fail(e, "magi_layer_norm_e4m3 launch");
  count_launches(1);
  return MAGI_OK;
}

int magi_div_clamp_to_e4m3(const void* x, int64_t x_stride, const float* scale, int32_t scale_len, void* y,
                           int64_t y_stride, int64_t rows, int32_t cols, void* stream) {
  if (rows < 0 || cols < 0) return fail(MAGI_EINVAL, "magi_div_clamp_to_e4m3: negative size");
  if (rows == 0 || cols == 0) return MAGI_OK;
  if (cols % 8) return fail(MAGI_ENOSYS, "magi_div_clamp_to_e4m3: cols %d is not a multiple of 8", cols);
  if (!x || !y || !scale) return fail(MAGI_EINVAL, "magi_div_clamp_to_e4m3: NULL pointer");
  if (scale_len != 1 && scale_len != cols)
    return fail(MAGI_EINVAL, "magi_div_clamp_to_e4m3: scale_len %d (1, or cols = %d)", scale_len, cols);
  if (x_stride < cols || y_stride < cols) return fail(MAGI_EINVAL, "magi_div_clamp_to_e4m3: row stride below cols");
  if (x_stride % 8 || y_stride % 8 || !aligned16(x) || (reinterpret_cast<uintptr_t>(y) & 7u) || !aligned16(scale))
    return fail(MAGI_EINVAL, "magi_div_clamp_to_e4m3: rows of x must be 16-byte aligned, rows of y 8-byte, scale 16-byte");
  if (rows * (int64_t)(cols / 8) > 0x7fffffffLL * 256)
    return fail(MAGI_ENOSYS, "magi_div_clamp_to_e4m3: more than 2^39 groups of eight elements");
  hipError_t e = magi::launch_div_clamp(static_cast<const char*>(x), x_stride * 2, scale, scale_len != 1,
                                        static_cast<char*>(y), y_stride, rows, cols, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return hip_fail(e, "magi_div_clamp_to_e4m3 launch");
  count_launches(1);
  return MAGI_OK;
}

int magi_head_norm(const void* x, int64_t x_stride_t, int64_t x_stride_h, const float* gamma, const float* beta,
                   void* y, int32_t S, int32_t H, int32_t D, int32_t norm_kind, float eps, void* stream) {
  if (D != 128) return fail(MAGI_ENOSYS, "magi_head_norm: head_dim %d not implemented (128 only)", D);
  if (S < 0 || H < 0) return fail(MAGI_EINVAL, "magi_head_norm: negative size");
  if (S == 0 || H == 0) return MAGI_OK;
  if (!x || !y) return fail(MAGI_EINVAL, "magi_head_norm: NULL x/y");
  if (norm_kind < 0 || norm_kind > 2) return fail(MAGI_EINVAL, "magi_head_norm: norm_kind %d", norm_kind);
  if (norm_kind != MAGI_NORM_NONE && !gamma) return fail(MAGI_EINVAL, "magi_head_norm: NULL gamma");
  if (x_stride_t % 8 || x_stride_h % 8 || !aligned16(x) || !aligned16(y))
    return fail(MAGI_EINVAL, "magi_head_norm: rows must be 16-byte aligned");
  hipError_t e = magi::launch_head_norm(static_cast<const char*>(x), x_stride_t * 2, x_stride_h * 2, gamma, beta,
                                        static_cast<char*>(y), S, H, norm_kind, eps, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return hip_fail(e, "magi_head_norm launch");
  count_launches(1);
  return MAGI_OK;
}

int magi_apply_rotary(const void* x, const float* cos, const float* sin, void* y, int32_t B, int32_t S, int32_t H,
                      int32_t D, int32_t R2, int32_t is_bf16, void* stream) {
  if (B < 0 || S < 0 || H < 0 || D <= 0 || D % 2) return fail(MAGI_EINVAL, "magi_apply_rotary: bad shape");
  if (R2 < 0 || 2 * R2 > D) return fail(MAGI_EINVAL, "magi_apply_rotary: rotary_dim %d > head_dim %d", 2 * R2, D);
  if ((long)B * S * H == 0) return MAGI_OK;
  if (!x || !y || (R2 > 0 && (!cos || !sin))) return fail(MAGI_EINVAL, "magi_apply_rotary: NULL pointer");
  hipError_t e = magi::launch_rotary(x, cos, sin, y, B, S, H, D, R2, is_bf16, static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return hip_fail(e, "magi_apply_rotary launch");
  count_launches(1);
  return MAGI_OK;
}

static int quantize_impl(const magi_quantize_args* p, void* stream, bool always_one_launch, const void* row_max = nullptr) {
  if (!p) return fail(MAGI_EINVAL, "magi_quantize_fp8: args is NULL");
  MAGI_CHECK_LAYOUT("magi_quantize_fp8", p);
  if (p->D != 128) return fail(MAGI_ENOSYS, "magi_quantize_fp8: head_dim %d not implemented (128 only)", p->D);
  if (p->T < 0 || p->H < 0 || p->chunk_tokens <= 0) return fail(MAGI_EINVAL, "magi_quantize_fp8: bad size");
  if (!(p->premul == p->premul) || p->premul == 0.f)
    return fail(MAGI_EINVAL, "magi_quantize_fp8: premul must be finite and non-zero");
  if (p->n_rows_first < 0 || p->n_rows_first > p->T)
    return fail(MAGI_EINVAL, "magi_quantize_fp8: n_rows_first %d outside [0, T=%d]", p->n_rows_first, p->T);
  if (p->n_rows_first < p->T && p->n_rows_first % p->chunk_tokens)
    return fail(MAGI_EINVAL, "magi_quantize_fp8: n_rows_first must be a multiple of chunk_tokens");
  if (p->T == 0 || p->H == 0) return MAGI_OK;
  if (p->H > 65535) return fail(MAGI_ENOSYS, "magi_quantize_fp8: more than 65535 heads");
  if (!p->x) return fail(MAGI_EINVAL, "magi_quantize_fp8: NULL pointer");
  if (p->n_rows_first > 0 && (!p->y || !p->scales)) return fail(MAGI_EINVAL, "magi_quantize_fp8: NULL pointer");
  if (p->n_rows_first < p->T && (!p->y2 || !p->scales2))
    return fail(MAGI_EINVAL, "magi_quantize_fp8: y2 / scales2 needed for rows >= n_rows_first");
  if (p->x_stride_t % 8 || p->x_stride_h % 8 || !aligned16(p->x) || !aligned16(p->y) || !aligned16(p->y2))
    return fail(MAGI_EINVAL, "magi_quantize_fp8: rows must be 16-byte aligned");
  if (row_max) {
    hipError_t e = magi::launch_quantize_fp8_row_max(static_cast<const char*>(p->x), p->x_stride_t * 2, p->x_stride_h * 2,
                                                     static_cast<char*>(p->y), p->scales, p->T, p->H, p->chunk_tokens, p->premul,
                                                     p->pow2_scales, p->n_rows_first, static_cast<char*>(p->y2), p->scales2,
                                                     static_cast<const unsigned short*>(row_max), compute_units(),
                                                     static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return hip_fail(e, "magi_quantize_fp8_row_max launch");
    count_launches(1);
    return MAGI_OK;
  }
  int n_launches = 0;
  hipError_t e = magi::launch_quantize_fp8(static_cast<const char*>(p->x), p->x_stride_t * 2, p->x_stride_h * 2,
                                           static_cast<char*>(p->y), p->scales, p->T, p->H, p->chunk_tokens, p->premul,
                                           p->pow2_scales, p->n_rows_first, static_cast<char*>(p->y2), p->scales2,
                                           always_one_launch, compute_units(), static_cast<hipStream_t>(stream), &n_launches);
  if (e != hipSuccess) return hip_fail(e, "magi_quantize_fp8 launch");
  count_launches((uint64_t)n_launches);
  return MAGI_OK;
}

int magi_quantize_fp8_split(const magi_quantize_args* p, void* stream) { return quantize_impl(p, stream, true); }

int magi_quantize_fp8_row_max(const magi_quantize_args* p, const void* row_max, void* stream) {
  if (!row_max) return fail(MAGI_EINVAL, "magi_quantize_fp8_row_max: NULL row_max");
  return quantize_impl(p, stream, true, row_max);
}

int magi_quantize_fp8(const void* x, int64_t x_stride_t, int64_t x_stride_h, void* y, float* scales, int32_t T,
                      int32_t H, int32_t D, int32_t chunk_tokens, float premul, int32_t pow2_scales, void* stream) {
  magi_quantize_args q;
  std::memset(&q, 0, sizeof(q));
  q.struct_size = sizeof(q);
  q.x = x;
  q.x_stride_t = x_stride_t;
  q.x_stride_h = x_stride_h;
  q.T = T;
  q.H = H;
  q.D = D;
  q.chunk_tokens = chunk_tokens;
  q.premul = premul;
  q.pow2_scales = pow2_scales;
  q.y = y;
  q.scales = scales;
  q.n_rows_first = T;
  return quantize_impl(&q, stream, false);
}

}  // extern "C"
