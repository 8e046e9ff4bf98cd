// What a batch-1 product keeps in LDS (step_sums.h): how wide a row may be, and every place that its sums over a tile's steps are read
// from, for every row length, round and team of a workgroup: in the array, and the steps of a tile where its wavefronts left them.  And how a list of products is
// shared out.  Prints the first that is not so and returns 1.
#include "step_sums.h"

#include <cstdio>

using namespace llvq;

int main() {
  for (uint32_t nb = 0; nb <= kGemvMaxBlocks; ++nb) {
    const bool wide = gemv_wide(nb);
    const uint32_t steps = tile_steps(nb), team = gemv_team(nb), teams = kGemvMaxWaves / team;
    for (uint32_t round = 0; round < gemv_batch(team); ++round)
      for (uint32_t t = 0; t < teams; ++t)
        for (uint32_t i = 0; i < sums_steps(wide) / 4u; ++i)
          for (uint32_t c = 0; c < 4u; ++c) {
            const uint32_t begin = sums_at(round, t, team, wide), at = begin + sums_read(i, c);
            if (at >= sums_room(wide) || begin + steps > sums_room(wide) || (4u * i + c < steps && at != begin + 4u * i + c)) {
              std::printf("%u blocks, round %u, team %u: read %u of %u\n", nb, round, t, at, sums_room(wide));
              return 1;
            }
          }
    // The same of a list of products: places of tiles whose sums are pending, and reads of as many steps as the widest row has.
    for (uint32_t task_steps : {1u, kSeqShortTaskSteps, kSeqTaskSteps}) {
      const uint32_t tasks = seq_tasks(steps, task_steps);
      if (tasks > 1u && (seq_slots(tasks) > kSeqMaxSlots || (seq_slots(tasks) - 1u) * steps + sums_read(kGemvMaxBlocks / kStepBlocks / 4u - 1u, 3u) >= kSeqPartSteps)) {
        std::printf("%u blocks, tasks of %u steps: %u places\n", nb, task_steps, seq_slots(tasks));
        return 1;
      }
    }
  }
  // A decoder's widest row: gate and up as one result fit, rows of one step to a wavefront.
  if (gemv_wide(8192 / kDim) || gemv_tiles_lds_bytes(8192 / kDim, 8192, false, false, true) > 160u * 1024u) return 1;
  // The rotated rows that are rotated in their product's launch, which has 160 KB: of the widths a rotation can have these are the widest.
  const struct { uint32_t width; bool f32, fits; } rotated[] = {{19456, true, true},  {20480, true, true},  {21504, true, false},
                                                                {23552, false, true}, {24576, false, true}, {17408, true, true}};
  for (const auto& r : rotated)
    if ((gemv_tiles_lds_bytes(r.width / kDim, r.width, r.f32, true) <= 160u * 1024u) != r.fits) {
      std::printf("%u columns rotated: %u bytes\n", r.width, (unsigned)gemv_tiles_lds_bytes(r.width / kDim, r.width, r.f32, true));
      return 1;
    }
  // A layer of a 4B model as one launch of 256 workgroups: each has tasks for its wavefronts (but for two), whichever matrix its share is of.
  const struct { uint32_t rows, width; } layer[] = {{6144, 2560}, {2560, 4096}, {19456, 2560}, {2560, 9728}};
  uint64_t bytes = 0;
  for (const auto& m : layer) bytes += (uint64_t)m.rows / 16 * ((m.width / kDim + 3) / 4) * kUnitBytes;
  for (const auto& m : layer) {
    const uint64_t tiles = bytes / 256 / ((uint64_t)(m.width / kDim + 3) / 4 * kUnitBytes);
    const uint32_t tasks = seq_tasks(tile_steps(m.width / kDim), seq_task_steps(bytes, 256));
    if (tiles * tasks < kSeqWaves - 2) {
      std::printf("%u columns: %u tasks of a workgroup\n", m.width, (unsigned)tiles * tasks);
      return 1;
    }
  }
  if (seq_task_steps(36 * bytes, 256) != kSeqTaskSteps) return 1;
  return 0;
}
