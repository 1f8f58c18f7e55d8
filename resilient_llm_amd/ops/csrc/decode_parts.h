// How decode attention divides sequences into parts, for those who write and
// read them.
#pragma once

#include "common.h"

namespace rlli {
namespace decode {

constexpr float kNegInf = -1e30f;
constexpr int UNIT = 32;          // tokens
constexpr int MIN_UNITS = 8;      // of a part: two per wave

DEV_INLINE int units_of(int len) { return (len + UNIT - 1) / UNIT; }

// Units of a part, of ``units`` in all sequences.
DEV_INLINE int part_size_of(int units, int shares) {
  return max((units + shares - 1) / shares, MIN_UNITS);
}

DEV_INLINE int parts_of(int len, int size) {
  return (units_of(len) + size - 1) / size;
}

}  // namespace decode
}  // namespace rlli
