// The split grid of a k2b or RTN decode call: S splits of a sequence, its heads in
// `blocks` blocks of hpb (grid z), and win_wgs workgroups (grid x, after the
// splits) that score the window and do nothing else.  Host code only.
//   S: one workgroup per CU over the batch, or what split_tokens asks for; at
//     most one per 64-token group.
//   blocks: a range with few groups leaves CUs idle while the 8 waves of a
//     workgroup, two per SIMD, share its issue slots; its heads are spread over
//     2, 4 or 8 workgroups as long as all of them, and the window's, have a CU.
//   win_wgs: as many as give every (tile, head) pair a wave, 4 pairs a workgroup
//     where there is room; none where there is not enough: the splits then score
//     the window after their groups, and, where they are fewer than its tiles,
//     are as many as those (one per CU at most).  Heads that are spread always
//     have them: the splits of every block would score the window again.
// Measured, us a call at h_kv 8, G 4 (with neither, and with both): k2b rank 16,
// 256 tokens and a 60-row window 17.4 -> 12.1 (the query loads together in both:
// see load_q4); 8,576 tokens, bf16, a 161-row window (no room to spread) 17.7 ->
// 15.5; RTN 128 tokens 16.9 -> 12.4.
// Everything follows from the bounds (max_len, tail_cap), not from a call's own
// window length, so a bound call's workspace fits it at any length.
#pragma once

#include <algorithm>
#include <cstdint>

namespace bmx {

struct SplitPlan {
  int S, blocks, hpb, win_wgs;
};

inline SplitPlan plan_splits(int batch, int h_kv, int groups, int max_len, int split_tokens, int tail_cap, int cus) {
  SplitPlan p;
  const int per_seq = std::max(1, cus / batch);
  const int tiles = (tail_cap + 15) / 16, pairs = tiles * h_kv;
  auto window = [&](int blocks) { return (pairs + 4 * blocks - 1) / (4 * blocks); };   // workgroups of one block
  p.S = split_tokens > 0 ? (max_len + split_tokens - 1) / split_tokens : per_seq;
  p.S = std::max(1, std::min(p.S, groups));
  p.blocks = 1;
  p.win_wgs = 0;
  if (split_tokens == 0) {
    while (2 * p.blocks <= h_kv && 2 * p.blocks * ((int64_t)p.S + window(2 * p.blocks)) <= per_seq) p.blocks *= 2;
    p.win_wgs = std::max(0, std::min(per_seq / p.blocks - p.S, window(p.blocks)));
    if (p.win_wgs * p.blocks * 8 < pairs) p.win_wgs = 0;   // blocks == 1: spread heads have window(blocks)
  }
  if (p.win_wgs == 0 && p.S < tiles) p.S = std::min(tiles, std::max(p.S, per_seq));
  p.hpb = (h_kv + p.blocks - 1) / p.blocks;
  return p;
}

}  // namespace bmx
