// Which workgroup tile a dense map takes, and in how many parts the head's K loop runs: host rules, free of GPU calls.
// Times are of one MI355X, on the 17,937-row encoder (14 stages of K) and the 4,299-row head.
#pragma once

#include <algorithm>
#include <cstdint>

#include "common.hpp"

namespace fly {

constexpr int GBK = 64;   // K per LDS stage

// The workgroup tile, 10 TM + TN for 32 TM x 32 TN, of a product over `stages` stages of K.  The gemm_tile tuning key
// forces one: 1 = 64 x 64, 2 = 128 x 64, 3 = 128 x 128, or 10 TM + TN with TM in {2, 3, 4} and TN in {2, 4, 5}.
// Otherwise, measured (us):
// * 128 x 128 from 1,024 tiles on: encoder of 1120 boards 106 against 121 (64 x 64) and 112 (64 x 160);
// * 64 x 160 where its columns cover the batch with no more padding than 64 do and its tiles fill at least 82% of their
//   rounds of 512 workgroups (two per CU): head of 1120 boards 125 against 129 (64 x 64), encoder of 480 60 against 68;
//   with rounds less full it loses (head of 640: 103 against 87, of 1280: 167 against 147);
// * 128 x 128 from 400 tiles on that pad at most 10% more columns than 64 and fill at least 60% of their rounds, or
//   have 32 stages or more: head of 1500 boards 141 against 163, of 2048 (53% of two rounds) 208 against 225, encoder
//   of 640 59 against 64; but encoder of 500 (55% of two rounds) 58 against 54, of 400 (512 columns against 448) 65
//   against 60.  Not below 8 stages, where the tile's own start and end weigh more than its operand reads (4,299 rows,
//   3000 boards: 1 stage 63 against 58, 5 stages 87 against 77, 10 stages 114 against 115);
// * else 64 x 64.
inline int gemm_shape(int64_t arows, int64_t brows, int64_t stages, int tile_key) {
  int shape = tile_key;
  if (shape == 1) shape = 22;
  else if (shape == 2) shape = 42;
  else if (shape == 3) shape = 44;
  const int tm = shape / 10, tn = shape % 10;
  if ((tm == 2 || tm == 3 || tm == 4) && (tn == 2 || tn == 4 || tn == 5)) return shape;
  const int64_t large = ((arows + 127) / 128) * ((brows + 127) / 128);
  if (large >= 1024) return 44;
  const int64_t wide = ((arows + 63) / 64) * ((brows + 159) / 160);
  if (round_up(brows, 160) <= round_up(brows, 64) && wide * 100 >= round_up(wide, 512) * 82) return 25;
  const bool full = large * 100 >= round_up(large, 512) * 60 || stages >= 32;
  return large >= 400 && stages >= 8 && full && round_up(brows, 128) * 10 <= round_up(brows, 64) * 11 ? 44 : 22;
}

inline int64_t gemm_tiles(int64_t arows, int64_t brows, int shape) {
  const int bm = 32 * (shape / 10), bn = 32 * (shape % 10);
  return ((arows + bm - 1) / bm) * ((brows + bn - 1) / bn);
}

// Parts of the head GEMM's K loop of `stages` stages, when no tuning forces a number.  The full-size head's 4,299 rows
// make few tiles (68 for up to 64 boards), each a chain of 37 stages; parts of K fill the other CUs, at the cost of a
// share of C each (k_assemble adds them).  The fewest parts, up to 3, within 15% of the least rounds of 512 workgroups
// (two per CU) per part; none past 640 tiles, where the shares' bytes cost what the rounds gain.  Measured, us of the
// head for 1, 2 and 3 parts: 1 board 39 / 27 / 24, 128 boards 44 / 39 / 34, 256 boards 59 / 49 / 48, 480 boards 77 / 69 /
// 72, 640 boards 78 / 83 / 84, 1120 boards 113 / 125 / 146.
// A chain of fewer stages is over sooner, and its shares cost the same: 19 stages gain (128 boards 29.7 / 28.3 / 27.6, 320
// boards 39.0 / 35.5 / 37.4, 500 boards 48.6 / 46.8 / 49.9), 16 not everywhere (128 boards 25.9 in one part and 26.9 in
// three, 500 boards 43.5 and 44.9 in two), 8 no more (128 boards 20.4 / 20.5 / 22.7, 256 boards 25.7 / 27.3 / 31.3),
// except in 2 parts while those are at most one workgroup per CU (64 boards: 4 stages 16.1 / 15.8 / 18.1, 8 stages
// 19.4 / 17.2 / 19.0, 16 stages 25.5 / 20.3 / 21.1).  2 stages gain nothing (64 boards 14.9 / 14.9, 128 boards 15.5 /
// 17.9).
inline int head_parts(int64_t tiles, int64_t stages) {
  const int most = tiles > 640 ? 1 : stages >= 18 ? 3 : stages >= 4 && tiles <= 128 ? 2 : 1;
  auto cost = [&](int s) { return (double)((tiles * s + 511) / 512) / s; };
  double least = cost(1);
  for (int s = 2; s <= most; ++s) least = std::min(least, cost(s));
  int s = 1;
  while (cost(s) > 1.15 * least) ++s;
  return s;
}

}  // namespace fly
