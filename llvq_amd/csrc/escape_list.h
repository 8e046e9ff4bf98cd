// How many places a tile's list of escapes has, and the way a wavefront walks a tile's codes where they were too few: plain
// arithmetic, compiled for gfx950 and for the host.
#pragma once
#include <cmath>
#include <cstdint>

#include "decode_core.h"
#include "step_sums.h"

namespace llvq {

// Of uniformly drawn points of shells 2..12 0.078 % are escapes, of shells 2..13 0.316 % (2 M draws of each).
constexpr double kEscapeShare = 0.78e-3, kEscapeShare13 = 3.16e-3;
// Places, a multiple of eight: as many as a tile of such points has but for one in 30 000, whose codes are read.  (At 2560 columns
// the eight places are too few for one tile in 80 000, of which a 4B model has 58 000; sixteen would be 0.7 % more to read, in
// every product.)  Shell 13 takes no batched products, whose kernels have room for 32.
constexpr double kListMisses = 1. / 30000;
constexpr uint32_t kMaxListSlots = 32, kMaxListSlots13 = 96;
constexpr uint32_t kMaxListBlocks = 1u << 19;  // what an entry has bits for; rows of more have no list, and their codes are read
inline uint32_t list_slots(uint32_t nb, bool shell13) {
  if (nb == 0 || nb > kMaxListBlocks) return 0u;
  const double mean = (double)kTileRows * nb * (shell13 ? kEscapeShare13 : kEscapeShare);
  const uint32_t most = shell13 ? kMaxListSlots13 : kMaxListSlots;
  double term = std::exp(-mean), within = term;
  for (uint32_t k = 1; k < most; ++k) {  // within: the chance of fewer than k
    if (k % 8u == 1u && k > 8u && 1. - within <= kListMisses) return k - 1u;
    term *= mean / k;
    within += term;
  }
  return most;
}

// A tile's codes: eight units to a step and lane (l, q) = (lane % 8, lane / 8) at piece l of the step's unit q, which has four
// blocks each of rows l and l + 8.  Their meta dwords give a mask with bit 8 k for block k of row l and bit 8 k + 1 for row l + 8;
// taken lane after lane and bit after bit, a row's blocks come in their order.
LLVQ_HD uint32_t walk_mask(uint32_t meta_lo, uint32_t meta_hi) {  // (bytes of kBlockEscape = 192 or more: the two top bits)
  return (meta_lo & meta_lo << 1 & 0x80808080u) >> 7 | (meta_hi & meta_hi << 1 & 0x80808080u) >> 6;
}
LLVQ_HD uint32_t walk_key(uint32_t step, uint32_t lane, uint32_t bit) {  // row << 28 | block
  return ((lane & 7u) | (bit & 1u) << 3) << 28 | ((step * kStepUnits + (lane >> 3)) * 4u + (bit >> 3));
}

}  // namespace llvq
