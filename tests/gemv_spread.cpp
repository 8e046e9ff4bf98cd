// How a batch-1 launch of rows past sixteen steps shares out its steps (GemvSpread of step_sums.h), walked as tiles_product walks it: every step
// of every tile computed once, where its tile's sum is read from, in the array, and every tile finished once.  Prints the first that is
// not so and returns 1.
#include "step_sums.h"

#include <cstdio>
#include <vector>

using namespace llvq;

static const char* spread_fault(uint32_t nb, uint32_t tiles, uint32_t cus) {
  GemvGrid g = gemv_grid(nb, tiles, cus, false, true, false);
  spread_into(g, gemv_spread(nb, tiles, g.grid));
  const GemvSpread s = spread_of(g);
  const uint32_t steps = tile_steps(nb);
  if (g.waves != kGemvMaxWaves || s.batch < 1u || s.batch > kGemvMaxWaves) return "wavefronts";
  std::vector<uint32_t> finished(tiles);
  for (uint32_t wg = 0; wg < g.grid; ++wg) {
    const uint32_t slots = s.slots - (wg < s.full ? 0u : 1u);
    uint32_t slot[kGemvMaxWaves], step[kGemvMaxWaves];
    for (uint32_t w = 0; w < kGemvMaxWaves; ++w) {
      const uint32_t team = (w * g.inv_team) >> 16;
      if (team) return "a wavefront's first step";
      slot[w] = 0;
      step[w] = w - team * g.team;
    }
    for (uint32_t r0 = 0; r0 < slots; r0 += s.batch) {
      const uint32_t r1 = r0 + s.batch < slots ? r0 + s.batch : slots;
      std::vector<uint32_t> left(sums_room(true));
      for (uint32_t w = 0; w < kGemvMaxWaves; ++w)
        while (slot[w] < r1) {
          const uint32_t at = (slot[w] - r0) * steps + step[w];
          if (slot[w] < r0 || step[w] >= steps || at >= sums_room(true) || left[at]++) return "a step's place";
          if ((step[w] += kGemvMaxWaves) >= steps) {
            step[w] -= steps;
            ++slot[w];
          }
        }
      for (uint32_t fin = 0; fin < kGemvMaxWaves; ++fin) {
        if (fin >= s.batch || r0 + fin >= slots) continue;
        for (uint32_t i = 0; i < kGemvMaxBlocks / kStepBlocks / 4u; ++i)
          for (uint32_t c = 0; c < 4u; ++c) {
            const uint32_t at = fin * steps + sums_read(i, c);
            if (at >= sums_room(true)) return "a read past the array";
            if (4u * i + c < steps && left[at] != 1u) return "a step not computed";
          }
        const uint32_t tile = (r0 + fin) * g.grid + wg;
        if (tile >= tiles) return "a tile that is not there";
        ++finished[tile];
      }
    }
    if (slots * g.grid + wg < tiles) return "a tile left over";
  }
  for (uint32_t t = 0; t < tiles; ++t)
    if (finished[t] != 1u) return "a tile finished other than once";
  return nullptr;
}

int main() {
  for (uint32_t steps = kGemvMaxWaves + 1u; steps <= kGemvMaxBlocks / kStepBlocks; ++steps)
    for (uint32_t cus : {1u, 7u, 64u, 256u, 304u})
      for (uint32_t tiles : {1u, 2u, 6u, 7u, 8u, 15u, 63u, 64u, 65u, 100u, 255u, 256u, 257u, 320u, 511u, 513u, 1000u, 2049u, 3585u, 4097u, 7169u})
        for (uint32_t nb : {(steps - 1u) * kStepBlocks + 1u, steps * kStepBlocks})
          if (const char* what = spread_fault(nb, tiles, cus)) {
            std::printf("%u blocks, %u tiles on %u CUs: %s\n", nb, tiles, cus, what);
            return 1;
          }
  return 0;
}
