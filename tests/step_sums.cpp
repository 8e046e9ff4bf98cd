// What a batch-1 product keeps in LDS (step_sums.h): how wide a row may be, and every place that its sums over a tile's steps are read
// from, for every row length, round and team of a workgroup: in the array, and the steps of a tile where its wavefronts left them.  How a list of
// products is shared out.  And how a batch-1 launch's tiles are: each is computed and finished once, gate with its up, and a row's norm is summed in
// one order.  Prints the first that is not so and returns 1.
#include "step_sums.h"

#include <cstdio>
#include <vector>

using namespace llvq;

// What is wrong with the layout of a launch over `tiles` tiles (gated: pairs of them) of rows of nb blocks, if anything is (tiles_product, slot by slot).
static const char* layout_fault(uint32_t nb, uint32_t tiles, uint32_t cus, bool gated, bool full, bool norm) {
  const GemvGrid g = gemv_grid(nb, tiles, cus, gated, full, norm);
  const uint32_t batch = gemv_batch(g.team), each = gated ? 2u : 1u;
  if (g.team != gemv_team(nb) || !g.teams || g.waves > kGemvMaxWaves || g.waves < g.team * g.teams || !g.grid || g.grid > cus) return "wavefronts";
  if (g.passes > (gemv_wide(nb) ? 4u : 2u) || g.passes * g.waves * 16u < tile_steps(nb) * kStepBlocks) return "passes";
  for (uint32_t i = 0; i <= kGemvMaxWaves; ++i)
    if ((i * g.inv_team) >> 16 != i / g.team || (i * g.inv_teams) >> 16 != i / g.teams) return "a division";
  if (norm && g.waves != kGemvMaxWaves && g.passes > 1u) return "the order of a norm";
  const auto tile_of = [&](uint32_t slot, uint32_t wg) { return slot / each * g.grid + wg; };
  std::vector<uint8_t> computed(tiles * each), finished(tiles * each);
  for (uint32_t wg = 0; wg < g.grid; ++wg) {
    for (uint32_t r0 = 0; r0 < g.rounds; r0 += batch) {
      const uint32_t r1 = r0 + batch < g.rounds ? r0 + batch : g.rounds;
      for (uint32_t t = 0; t < g.teams; ++t)
        for (uint32_t r = r0; r < r1; ++r) {
          const uint32_t slot = r * g.teams + t, tile = tile_of(slot, wg);
          if (tile >= tiles) break;
          ++computed[tile * each + slot % each];
        }
      for (uint32_t fin = 0; fin < g.waves; ++fin) {
        const uint32_t round = fin / g.teams, slot = r0 * g.teams + fin, tile = tile_of(slot, wg);
        if (round >= batch || tile >= tiles) continue;
        if (r0 + round >= r1 || slot % each != fin % each) return "a finisher's round";  // (an odd one is of an up tile)
        if (gated && fin % 2u == 0u && (fin + 1u >= g.waves || (fin + 1u) / g.teams >= batch || ((fin + 1u) * kTileRows + kTileRows) * 2u > kGatedFloats)) return "a pair apart";
        if (++finished[tile * each + slot % each] > computed[tile * each + slot % each]) return "finished before it is computed";
      }
    }
    const uint32_t past = tile_of(g.rounds * g.teams, wg);
    if (past < tiles) return "rounds";
  }
  for (uint32_t i = 0; i < tiles * each; ++i)
    if (computed[i] != 1u || finished[i] != 1u) return "a tile computed or finished other than once";
  return nullptr;
}

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
  // Every number of steps, tiles around what a card's CUs take in a round and what teams take in a batch of them, cards of few CUs
  std::vector<uint32_t> counts;
  for (uint32_t i = 1; i <= 70; ++i) counts.push_back(i);
  for (uint32_t i : {127u, 255u, 256u, 257u, 384u, 511u, 512u, 513u, 608u, 767u, 1024u, 1088u, 2047u, 2049u, 2176u, 4096u, 4097u, 9496u}) counts.push_back(i);
  for (uint32_t steps = 0; steps <= kGemvMaxBlocks / kStepBlocks; ++steps)
    for (uint32_t cus : {1u, 7u, 64u, 256u, 304u})
      for (uint32_t tiles : counts)
        for (uint32_t kind = 0; kind < 4u; ++kind) {
          const uint32_t nb = steps * kStepBlocks;
          const bool gated = kind == 1u, norm = kind == 1u || kind == 2u, full = gemv_wide(nb) || kind == 3u;
          if (gated && (gemv_wide(nb) || !nb)) continue;
          if (const char* what = layout_fault(nb, tiles, cus, gated, full, norm)) {
            std::printf("%u steps, %u tiles%s on %u CUs, kind %u: %s\n", steps, tiles, gated ? " in pairs" : "", cus, kind, what);
            return 1;
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
