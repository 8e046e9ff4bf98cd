// Where the sums of a tile's steps lie in LDS between the wavefronts that leave them there and the one that adds them up
// (gemv_tiles_kernel): plain integer arithmetic, compiled for gfx950 and for the host.
#pragma once
#include <cstdint>

#include "decode_core.h"

namespace llvq {

constexpr uint32_t kStepUnits = 8;
constexpr uint32_t kStepBlocks = 4 * kStepUnits;
LLVQ_HD uint32_t tile_steps(uint32_t nb) { return (nb + kStepBlocks - 1u) / kStepBlocks; }

constexpr uint32_t kGemvMaxWaves = 16;
constexpr uint32_t kGemvWideSteps = 2;  // steps of a wavefront where a row has more than sixteen
constexpr uint32_t kGemvRounds = 8;     // tiles per team between two sums over the team's wavefronts, at the most
constexpr uint32_t kGemvMaxBlocks = kStepBlocks * kGemvMaxWaves * kGemvWideSteps;

// A tile's steps go to a team of wavefronts, one each (two each past sixteen).  A row is added up in an order that does not
// depend on that: the lanes of a step (rows_sum), the steps of equal number mod 4 one behind the other, those four sums;
// so a matrix gives the same bits whatever it shares a launch with.
LLVQ_HD uint32_t gemv_team(uint32_t nb) {
  const uint32_t steps = tile_steps(nb);
  return steps > kGemvMaxWaves ? kGemvMaxWaves : steps ? steps : 1u;
}
LLVQ_HD bool gemv_wide(uint32_t nb) { return nb > kStepBlocks * kGemvMaxWaves; }
// ... and so that there is a wavefront for each of the workgroup's
LLVQ_HD uint32_t gemv_batch(uint32_t team) { return team < kGemvRounds ? team : kGemvRounds; }

// The array: kGemvRounds rounds of as many steps as a workgroup's teams take together.  Tile `team_index` of a round begins here.
LLVQ_HD uint32_t sums_steps(bool wide) { return kGemvMaxWaves * (wide ? kGemvWideSteps : 1u); }
LLVQ_HD uint32_t sums_at(uint32_t round, uint32_t team_index, uint32_t team, bool wide) { return round * sums_steps(wide) + team_index * team; }
// The step of a tile of `steps` that a lane of class c reads as its i-th: past the tile's last that one again (a row may have none).
LLVQ_HD uint32_t sums_read(uint32_t i, uint32_t c, uint32_t steps) {
  const uint32_t s = 4u * i + c, last = steps ? steps - 1u : 0u;
  return s < last ? s : last;
}

}  // namespace llvq
