// How the flash kernel's items (four 64-row query blocks of one head against all key tiles) are
// dealt out to workgroups.  Host code only.
#pragma once

#include <algorithm>
#include <cstdint>

#define FA_WAVES 8
#define FA_QBLK_PER_WG (FA_WAVES / 2)
#define FA_PART_WAVE (64 * 64 + 2 * 64)                      // floats of one wave's partial: O, m, l
#define FA_PART_FLOATS (FA_WAVES * FA_PART_WAVE)

// Items [0, n_whole) run whole, `bundle` consecutive ones per workgroup (n_bundle workgroups); the
// tiles of the others are cut into n_chunk equal ranges, one per workgroup, and combined.
struct FlashPlan { int n_whole, bundle, n_bundle, n_chunk; int64_t part_bytes; };

// One workgroup fills a CU's LDS, so the chip runs FA_CUS of them at a time, and a last round
// of r < FA_CUS items takes as long as a full one.
//  * Those r items are cut into FA_CUS chunks of r n_tiles / FA_CUS tiles when that saves
//    more than FA_COMBINE_TILES tiles: the sums' kernel takes 9-13 us and a tile 1.7 us of a
//    workgroup, and a chunk's workgroup has a start of its own (about 5 us).  Chunks are not
//    shorter than FA_MIN_CHUNK tiles.
//  * Whole items go several to a workgroup, up to FA_BUNDLE_TILES tiles: beyond that a
//    workgroup's start no longer counts and many workgroups even out the CUs (220 tiles an
//    item, 8.6 rounds: 4,710 us with bundles of 1 or 2 items, 4,870 us with 8; 8 tiles an item,
//    40 rounds: 783, 775 and 773 us with 14, 20 and 40 items).  Of these counts the one whose
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
  if (n_tiles > 0) {                     // 0: a size query for a call without keys (refused later)
    if (may_split && rest > 0) {
      const int64_t g = std::min<int64_t>(FA_CUS, std::max<int64_t>(rest, rest * n_tiles / FA_MIN_CHUNK));
      if (n_tiles - (rest * n_tiles + g - 1) / g > FA_COMBINE_TILES) {
        f.n_whole = (int)(rounds * FA_CUS);
        f.n_chunk = (int)g;
      }
    }
    const int64_t per_cu = ((int64_t)f.n_whole + FA_CUS - 1) / FA_CUS;
    int64_t best = INT64_MAX;
    for (int64_t m = 1; m <= std::max<int64_t>(1, std::min<int64_t>(per_cu, FA_BUNDLE_TILES / n_tiles)); ++m) {
      const int64_t n = (f.n_whole + m - 1) / m;
      const int64_t cost = (n + FA_CUS - 1) / FA_CUS * (m * n_tiles + FA_START_TILES);
      if (cost < best) {
        best = cost;
        f.bundle = (int)m;
      }
    }
  }
  f.n_bundle = (f.n_whole + f.bundle - 1) / f.bundle;
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
