// How decode attention divides sequences into parts, for those who write and
// read them.
#pragma once

#include "common.h"

namespace rlli {
namespace decode {

constexpr float kNegInf = -1e30f;
constexpr int UNIT = 32;          // tokens
constexpr int MIN_UNITS = 8;      // of a part: two per wave
// of a single sequence, which leaves most CUs idle: one per wave (behind 1000
// tokens 9.3 -> 7.4 us)
constexpr int MIN_ONE = 4;

DEV_INLINE int units_of(int len) { return (len + UNIT - 1) / UNIT; }

// Units of a part, of ``units`` in all sequences.
DEV_INLINE int part_size_of(int units, int shares, int batch) {
  return max((units + shares - 1) / shares,
             batch == 1 ? MIN_ONE : MIN_UNITS);
}

DEV_INLINE int parts_of(int len, int size) {
  return (units_of(len) + size - 1) / size;
}

}  // namespace decode
}  // namespace rlli
