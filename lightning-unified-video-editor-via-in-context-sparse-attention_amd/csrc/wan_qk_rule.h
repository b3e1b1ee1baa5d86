// Which q / k producer serves a call.  Host code only.
#pragma once

#include <algorithm>
#include <cstdint>

#define WQ_MAX_CH 10

// 8-dim chunks a lane of the one-pass kernel holds of a row, per 512 dims (4 heads)
constexpr int wan_row_chunks(int H) { return H <= 12 ? 3 : (H <= 20 ? 5 : WQ_MAX_CH); }

// The one-pass kernel for n_wg 64-token blocks of q and k (each a workgroup)?  It saves the second
// read of the projections, but few workgroups leave most CUs idle for its four rounds, and chunks
// that a row does not fill are paid for.  blocks = n_wg H, 64-token blocks of one head; times in
// us, two passes / one:
//  * up to 5 heads never: a third of the lanes at most hold anything.  3 heads 136 / 200 at 12,288
//    blocks, 4 heads 169 / 195 at 16,384, 5 heads 198 / 199 at 19,500; 6 heads 127 / 125 at 12,876.
//  * 3 and 5 chunks, three and more workgroups a CU: from 12,000 blocks.  12 heads 113 / 109 at
//    9,360, 119 / 105 at 12,408; 8 heads 132 / 115 at 13,664; 13 heads 132 / 122 at 13,572; 20 heads
//    118 / 101 at 12,320.
//  * 10 chunks, 512 workgroups at a time: a round of them takes about 92 us however many heads the
//    rows hold, the two passes about 10 us per 1,000 blocks, so from 9,600 blocks a round (8,000
//    without block sums, which spare a barrier a chunk), and at least 14,000.  40 heads 119 / 126 at
//    12,480, 142 / 131 at 14,080 (one round), 225 / 216 at 21,120 (two); 24 heads 155 / 188 at 14,976,
//    199 / 192 at 18,720, 242 / 207 at 23,424 (two), 265 / 265 at 25,776 (three); 21 heads 116 / 157
//    at 12,306, 240 / 264 at 24,570, 400 / 385 at 43,008 (four).
constexpr bool wan_one_pass(int64_t n_wg, int H, bool sums) {
  const int64_t blocks = n_wg * H;
  if (H <= 5 || H > 4 * WQ_MAX_CH) return false;
  if (wan_row_chunks(H) < WQ_MAX_CH) return blocks >= 12000;
  return blocks >= std::max<int64_t>(14000, (n_wg + 511) / 512 * (sums ? 9600 : 8000));
}
