// How the flash kernel's items (four 64-row query blocks of one head against all key tiles) are
// dealt out to workgroups.  Host code only.
#pragma once

#include <algorithm>
#include <cstdint>

#define FA_WAVES 8
#define FA_QBLK_PER_WG (FA_WAVES / 2)
#define FA_PART_WAVE (64 * 64 + 2 * 64)                      // floats of one wave's partial: O, m, l
#define FA_PART_FLOATS (FA_WAVES * FA_PART_WAVE)

#define FA_XCDS 8

// Items [0, n_whole) run whole, up to `bundle` of them per workgroup (n_bundle workgroups on each
// XCD); the tiles of the others are cut into n_chunk equal ranges, one per workgroup, and combined.
struct FlashPlan { int n_whole, bundle, n_bundle, n_chunk; int64_t part_bytes; };

// The whole items of workgroup wg < FA_XCDS * n_bundle: first, first + n_bundle, ... (count of
// them, maybe 0).  Workgroup wg runs on XCD wg % 8, and each XCD has a contiguous range of the
// items, its workgroups side by side in it: the items of one head run at the same time and read
// its K and V from that XCD's L2.  With consecutive items in a workgroup instead, a head's
// second item came after its first had moved on (320 heads, 320 queries, 4,096 keys: 499 us a
// call, now 438; 432 with one item a workgroup).
struct FlashRun { int first, count; };
constexpr FlashRun flash_whole_run(int wg, int n_whole, int n_bundle) {
  const int per = (n_whole + FA_XCDS - 1) / FA_XCDS, x = wg % FA_XCDS;
  const int first = x * per + wg / FA_XCDS;
  const int end = (x + 1) * per < n_whole ? (x + 1) * per : n_whole;
  return FlashRun{first, first < end ? (end - first + n_bundle - 1) / n_bundle : 0};
}

// One workgroup fills a CU's LDS, so the chip runs FA_CUS of them at a time, and a last round
// of r < FA_CUS items takes as long as a full one.
//  * Those r items are cut into FA_CUS chunks of r n_tiles / FA_CUS tiles when that saves
//    more than FA_COMBINE_TILES tiles: the sums' kernel takes 9-13 us and a tile 1.7 us of a
//    workgroup, and a chunk's workgroup has a start of its own (about 5 us).  Chunks are not
//    shorter than FA_MIN_CHUNK tiles.
//  * Whole items go several to a workgroup, up to FA_BUNDLE_TILES tiles: beyond that a
//    workgroup's start no longer counts and many workgroups even out the CUs (220 tiles an
//    item, 8.6 rounds: 4,710 us with bundles of 1 or 2 items, 4,870 us with 8; 8 tiles an item,
//    40 rounds: 1 % between 14, 20 and 40 items).  Of these counts the one whose
//    rounds are shortest, a start costing FA_START_TILES tiles: bundles that do not fill the
//    last round cost more than the starts they save (768 items of 256 tiles: in pairs 1,541 us,
//    one by one 1,350; 1,792 of 147: in threes 2,093, one by one 1,804).
#define FA_CUS 256
#define FA_MIN_CHUNK 4
#define FA_COMBINE_TILES 12
#define FA_BUNDLE_TILES 512
#define FA_START_TILES 3

inline FlashPlan flash_plan(int64_t n_work, int n_tiles, bool may_split) {
  FlashPlan f;
  const int64_t rounds = n_work / FA_CUS, rest = n_work % FA_CUS;
  f.n_whole = (int)n_work;
  f.n_chunk = 0;
  f.bundle = 1;
  int64_t per_xcd = 0;
  if (n_tiles > 0) {                     // 0: a size query for a call without keys (refused later)
    if (may_split && rest > 0) {
      const int64_t g = std::min<int64_t>(FA_CUS, std::max<int64_t>(rest, rest * n_tiles / FA_MIN_CHUNK));
      if (n_tiles - (rest * n_tiles + g - 1) / g > FA_COMBINE_TILES) {
        f.n_whole = (int)(rounds * FA_CUS);
        f.n_chunk = (int)g;
      }
    }
    per_xcd = ((int64_t)f.n_whole + FA_XCDS - 1) / FA_XCDS;
    const int64_t cus = FA_CUS / FA_XCDS, per_cu = (per_xcd + cus - 1) / cus;
    int64_t best = INT64_MAX;
    for (int64_t m = 1; m <= std::max<int64_t>(1, std::min<int64_t>(per_cu, FA_BUNDLE_TILES / n_tiles)); ++m) {
      const int64_t n = (per_xcd + m - 1) / m;
      const int64_t cost = (n + cus - 1) / cus * (m * n_tiles + FA_START_TILES);
      if (cost < best) {
        best = cost;
        f.bundle = (int)m;
      }
    }
  }
  f.n_bundle = (int)((per_xcd + f.bundle - 1) / f.bundle);
  f.part_bytes = f.n_chunk ? (int64_t)(f.n_chunk + rest) * FA_PART_FLOATS * 4 : 0;
  return f;
}

inline int64_t flash_items(int BH, int n_qblk) {
  return (int64_t)BH * ((n_qblk + FA_QBLK_PER_WG - 1) / FA_QBLK_PER_WG);
}

// over any number of items
inline int64_t flash_part_bytes_max(int n_tiles) {
  return n_tiles > FA_COMBINE_TILES ? (int64_t)(2 * FA_CUS - 1) * FA_PART_FLOATS * 4 : 0;
}
