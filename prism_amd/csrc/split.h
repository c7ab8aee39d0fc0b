// Split launches of the pair kernels: launches whose pairs do not fill the GPU
// evenly cut the lists of some pairs into parts that run side by side.
//
// An attention launch of P pairs runs on R workgroups at once, so it takes
// ceil(P / R) rounds of a whole pair's list: 80 pairs (2,000 audio queries of
// five heads over a clip's keys) leave 432 of 512 slots idle for the length of
// one list, 2,160 pairs take five rounds where 4.2 would do.  Pairs below
// `whole` (whole rounds) keep one work item each; every later pair is `splits`
// items, item i of which walks the listed tiles t with (t / 8) mod splits == i
// (prism_part_union).  Each leaves its float32 accumulators in a workspace, in
// the attention kernel's own register layout (coalesced float4 stores), and a
// merge kernel adds a pair's items in item order and writes the result:
// deterministic, and no less precise than one long sum.
//
// Which tiles belong together depends on their index alone, and whole is a
// boundary of the pairing's groups, so a tile's result does not depend on how
// tiles were paired, nor on entries that contribute exact zeros (padded
// queries).  Groups of eight tiles are dealt in turn because lists are
// clustered: contiguous ranges would give some items most of the entries.
// Measured (D = 128, merge included): dQ of 80 pairs of 1,030 entries 1,673 ->
// 490 us, dK/dV of 80 pairs of 180 entries 659 -> 255 us, dQ of 2,160 pairs of
// 180 entries 2,002 -> 1,875 us.
//
// The workspace lives for the two launches: items x 128 x D floats for dQ, twice
// that for dK/dV; by the rule below at most 237 MB at D = 128 (the last 514 of
// 4,095 pairs of dQ, 258 of 1,791 of dK/dV, in seven items each).
//
// The forward is not split: its O would differ in its last bits, and delta =
// rowsum(O dO) carries such a bit into a whole row of dQ.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.h"

struct SplitArgs {
  int whole, splits;
  float4* acc;  // [slots] accumulators of an item
};
// pair and workspace slot (-1: a whole list) of work item `it`
struct SplitItem {
  int pair, slot;
};

__host__ __device__ __forceinline__ SplitItem split_item(int whole, int splits, int it) {
  if (it < whole) return SplitItem{it, -1};
  return SplitItem{whole + (it - whole) / splits, it - whole};
}

// Entries that an item of a split pair can hold: its groups of eight of the
// col_tiles listed tiles.  (The pairs' items together: little more than the
// pair's own row, not `splits` rows.)
__host__ __device__ __forceinline__ int64_t split_item_cap(int64_t col_tiles, int splits) {
  const int64_t cap = (col_tiles + 8 * splits - 1) / (8 * splits) * 8;
  return cap < col_tiles ? cap : col_tiles;
}

// Which pairs to split, and into how many items, for heads * per_head pairs on
// `slots` workgroups.  Launches of eight rounds or more keep whole lists: the
// work queue already ends them within an eighth of their time, usually much
// less.  Otherwise the pairs past the last full round (from a group boundary:
// four pairs of a head) are cut into the number of items with the fewest
// rounds' worth of time, ceil(rest s / slots) / s, plus 0.02 per item for what
// an item costs beside its entries (its prologue, the workspace written and
// read).  Lists of fewer than 512 possible entries are not cut: the merge
// launch and the workspace then cost what the idle slots do (1,024 pairs of 49
// entries, D = 64: 168 us whole, 184 cut; 64 pairs of 5: 24 against 42).
inline void split_plan(int64_t heads, int64_t per_head, int64_t max_entries, int64_t slots, int64_t* whole,
                       int* splits) {
  const int64_t pairs = heads * per_head;
  *whole = pairs;
  *splits = 1;
  if (pairs >= 8 * slots || max_entries < 512) return;
  int64_t full = pairs / slots * slots;
  full = full / per_head * per_head + (full % per_head) / 4 * 4;
  const int64_t rest = pairs - full;
  double best = (double)((rest + slots - 1) / slots);
  for (int64_t s = 2; s <= 16; ++s) {
    const double t = (double)((rest * s + slots - 1) / slots) / (double)s + 0.02 * (double)s;
    if (t < best) {
      best = t;
      *splits = (int)s;
    }
  }
  if (*splits > 1) *whole = full;
}

inline int split_check(const char* who, int64_t total, int64_t whole, int splits, const void* acc) {
  PRISM_REQUIRE(splits >= 1 && splits <= 64, "%s: splits must be in [1, 64]", who);
  PRISM_REQUIRE(whole >= 0 && whole <= total, "%s: whole must be in [0, pairs]", who);
  PRISM_REQUIRE(whole + (total - whole) * splits < (1ll << 31), "%s: grid too large", who);
  PRISM_REQUIRE(whole == total || acc, "%s: null workspace", who);
  return PRISM_OK;
}
