// What a matrix-core wave's stream pieces take in the LDS.  One formula for the kernel that stages them, the
// validator of a tiling and the planner's count: none of them may reserve less than another uses.
#pragma once
#include <stdint.h>

namespace grf {

constexpr uint32_t kPieceWindow = 8;  // bytes the refill reads from the aligned cursor on

// 16-byte units of one of a wave's sixteen slots.  `held`: the slot has a row, whose piece is the stream's
// bytes first .. past (from the 16-byte aligned start, as the copy takes them).  A slot without one takes
// a unit whatever range it was handed (the kernel reads the index's first entry for it, at any phase), so
// that every row begins at a unit of its own.  constexpr: the host's and the device's alike.
template <class T>
constexpr T piece_units(bool held, T first, T past) {
  return held ? (past - (first & ~(T)15) + kPieceWindow + 15) >> 4 : 1;
}

}  // namespace grf
