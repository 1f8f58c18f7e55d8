// How a launch of prompt attention (prefill_flash.h) divides its keys.
#pragma once

#include <algorithm>

namespace rlli {

// Scratch of tiles whose keys several workgroups share: f32 sums and (maximum,
// sum of weights) of every part, row and query head.
struct PrefillParts {
  float* o;                 // [splits, rows, n_q, D]
  float* ml;                // [splits, rows, n_q, 2]
  int splits;               // 1: no scratch
  int rows;
};

// Two waves per head; why the line lies there is in by_group.
inline bool two_waves(int n_tiles, int n_kv, int group, int keys) {
  return group % 4 == 0 && n_tiles * n_kv * (group / 4) <= 400 && keys >= 384;
}

// Parts of up to a workgroup per CU in all, where tiles alone leave half of
// them idle: a tile is a chain of steps of 128 keys, 2 to 2.4 us each.  The
// parts and the launch that puts them together cost 7 us, so a part has four
// steps at least, which the device sees to (tables may be wider than the
// sequences in them), and what they spare eight.  (us, 32/8 heads of 128,
// undivided first: 128 rows behind 4000 tokens 76 and 43, 256 behind 7000 128
// and 60, 512 behind 7000 137 and 94, 64 behind 1500 35 and 29; but 512 behind
// 1500, 44, gain nothing by two parts that read twice as much out of an XCD's
// L2 at a time, and 512 behind none, 17, lose 7.)
inline int prefill_splits(int n_tiles, int n_kv, int group, int keys) {
  if (n_tiles == 0 || !two_waves(n_tiles, n_kv, group, keys)) return 1;
  const int blocks = n_tiles * n_kv * (group / 4);
  const int n = std::max(1, std::min({16, 256 / blocks, keys / 512}));
  return keys - keys / n >= 1024 ? n : 1;
}

}  // namespace rlli
