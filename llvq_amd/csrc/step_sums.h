// What a batch-1 product keeps in LDS (gemv_tiles_kernel): the activation's planes, and the sums of a tile's steps between the
// wavefronts that leave them there and the one that adds them up.  Plain integer arithmetic, compiled for gfx950 and for the host.
#pragma once
#include <cstdint>

#include "decode_core.h"

namespace llvq {

constexpr uint32_t kTileRows = 16;
constexpr uint32_t kUnitBytes = 640;
constexpr uint32_t kStepUnits = 8;
constexpr uint32_t kStepBlocks = 4 * kStepUnits;
LLVQ_HD uint32_t tile_steps(uint32_t nb) { return (nb + kStepBlocks - 1u) / kStepBlocks; }

constexpr uint32_t kGemvMaxWaves = 16;
constexpr uint32_t kGemvWideSteps = 2;  // steps of a wavefront where a row has more than sixteen
constexpr uint32_t kGemvRounds = 8;     // tiles per team between two sums over the team's wavefronts, at the most
constexpr uint32_t kGemvMaxBlocks = kStepBlocks * kGemvMaxWaves * kGemvWideSteps;

// A tile's steps go to a team of wavefronts, one each (past sixteen: GemvSpread).  A row is added up in an order that does not
// depend on that: the lanes of a step (rows_sum), the steps of equal number mod 4 one behind the other, those four sums;
// so a matrix gives the same bits whatever it shares a launch with.
LLVQ_HD uint32_t gemv_team(uint32_t nb) {
  const uint32_t steps = tile_steps(nb);
  return steps > kGemvMaxWaves ? kGemvMaxWaves : steps ? steps : 1u;
}
// How often the quads of that many wavefronts pass over a row's blocks, whole steps of them.
LLVQ_HD uint32_t stage_passes(uint32_t nb, uint32_t waves) { return (tile_steps(nb) * kStepBlocks + waves * 16u - 1u) / (waves * 16u); }
LLVQ_HD bool gemv_wide(uint32_t nb) { return nb > kStepBlocks * kGemvMaxWaves; }
// ... and so that there is a wavefront for each of the workgroup's
LLVQ_HD uint32_t gemv_batch(uint32_t team) { return team < kGemvRounds ? team : kGemvRounds; }

// Wavefronts of a workgroup with `tiles` tiles: those with steps, and one for each tile that is finished at a time.  (Eight tokens of a 4B
// model: 12 060 us with those with steps only, 11 910; as many besides as it takes to quantise the activation in one pass, 12 050.)
LLVQ_HD uint32_t gemv_waves(uint32_t team, uint32_t teams, uint32_t tiles) {
  const uint32_t at_a_time = gemv_batch(team) * teams, finish = tiles < at_a_time ? tiles : at_a_time;
  return team * teams + finish < kGemvMaxWaves ? team * teams + finish : kGemvMaxWaves;
}
// Wavefronts below which a launch that norms its row does not go.  A row's squares are added a wavefront at a time, each over its sixteen blocks
// of every pass, and the wavefronts' sums in order: with a wavefront for every sixteen blocks, or with all sixteen, as sequences have them, that
// is one order whatever shares the launch.  (With fewer, 2560 columns in five wavefronts for instance, one row in eight had another norm than in
// a sequence, in its last bit.)
LLVQ_HD uint32_t gemv_norm_waves(uint32_t nb) { return 2u * tile_steps(nb) < kGemvMaxWaves ? 2u * tile_steps(nb) : kGemvMaxWaves; }

// The array: kGemvRounds rounds of as many steps as a workgroup's teams take together, and room behind them for what a sum reads past
// its tile's steps and does not use: the places to read are then the same for every tile.  (Each held back by the number of steps,
// which is twelve instructions in front of the first product, took 0.08 us of every launch.)  Tile `team_index` of a round begins here.
LLVQ_HD uint32_t sums_steps(bool wide) { return kGemvMaxWaves * (wide ? kGemvWideSteps : 1u); }
LLVQ_HD uint32_t sums_at(uint32_t round, uint32_t team_index, uint32_t team, bool wide) { return round * sums_steps(wide) + team_index * team; }
LLVQ_HD uint32_t sums_room(bool wide) { return kGemvRounds * sums_steps(wide) + (wide ? 0u : kGemvMaxWaves); }
// Gate and up as one result (tiles_product, GATED): where the scales and extras of a wavefront's sixteen rows are, and how many teams a
// workgroup has for `slots` tiles.  A pair's two tiles are finished together, so the teams' tiles of a batch of rounds are an even number.
LLVQ_HD uint32_t gated_at(bool wide) { return sums_room(wide) * kTileRows; }
constexpr uint32_t kGatedFloats = kGemvMaxWaves * kTileRows * 2;
LLVQ_HD uint32_t gated_teams(uint32_t slots, uint32_t team) {
  const uint32_t most = kGemvMaxWaves / team, teams = slots < most ? slots : most;
  if (!((gemv_batch(team) * teams) & 1u)) return teams;
  return teams < most ? teams + 1u : teams - 1u;  // (such a team is of seven wavefronts at the most: most >= 2)
}
// A launch's workgroups, their teams and wavefronts, as the host lays them out.  Slot i of a workgroup is tile i * grid + its number (gated: of
// pairs of slots); round r of team t is slot r * teams + t.
struct GemvGrid {
  uint32_t team, teams;          // wavefronts of a team, teams of a workgroup
  uint32_t waves, grid, passes;  // wavefronts (those that no team has only stage the activation); workgroups; how often the former pass over the activation
  uint32_t inv_team, inv_teams;  // 2^16 / team and 2^16 / teams, rounded up: exact for the seventeen numbers that are divided
  uint32_t rounds;               // tiles of a team, at the most
};
// tiles: of all matrices, or pairs of them (gated).  full: sixteen wavefronts whatever there is for them.  norm: the launch norms its row.
// Teams go to as many CUs as there are tiles for, then to the same CU, up to sixteen wavefronts: a small launch
// is short because every CU has a part of it, a large one because a CU keeps sixteen wavefronts' loads in flight.
inline GemvGrid gemv_grid(uint32_t nb, uint32_t tiles, uint32_t cus, bool gated, bool full, bool norm) {
  GemvGrid g{};
  g.team = gemv_team(nb);
  uint32_t slots;  // tiles of the fullest workgroup
  if (gated) {
    g.grid = cus < tiles ? cus : tiles;
    slots = 2u * ((tiles + g.grid - 1u) / g.grid);
    g.teams = gated_teams(slots, g.team);
  } else {
    const uint32_t each = (tiles + cus - 1u) / cus, most = kGemvMaxWaves / g.team;
    g.teams = each < most ? each : most;
    const uint32_t filled = (tiles + g.teams - 1u) / g.teams;
    g.grid = cus < filled ? cus : filled;
    slots = (tiles + g.grid - 1u) / g.grid;
  }
  g.rounds = (slots + g.teams - 1u) / g.teams;
  g.waves = full ? kGemvMaxWaves : gemv_waves(g.team, g.teams, slots);
  if (norm && g.waves < gemv_norm_waves(nb)) g.waves = gemv_norm_waves(nb);
  g.passes = stage_passes(nb, g.waves);
  g.inv_team = (65536u + g.team - 1u) / g.team;
  g.inv_teams = (65536u + g.teams - 1u) / g.teams;
  return g;
}
// Rows of more than sixteen steps: a workgroup's steps, its slots' one behind the other, go to its sixteen wavefronts in turn, one at a time.
// (As a team that takes a tile's steps two at a time: of the 23 steps of a 14B down_proj nine wavefronts then have no second one.)
struct GemvSpread {
  uint32_t slots, full;  // tiles of a workgroup, one fewer from workgroup `full` on
  uint32_t batch;        // tiles whose sums are in LDS together and finished together, a wavefront each
};
LLVQ_HD uint32_t spread_batch(uint32_t steps) {  // (of the last one as many places are read as the widest row has steps)
  const uint32_t most = (sums_room(true) - sums_steps(true)) / steps + 1u;
  return most < kGemvMaxWaves ? most : kGemvMaxWaves;
}
inline GemvSpread gemv_spread(uint32_t nb, uint32_t tiles, uint32_t grid) {
  const uint32_t more = tiles % grid;
  return {tiles / grid + (more ? 1u : 0u), more ? more : grid, spread_batch(tile_steps(nb))};
}
// The arguments of a launch are four lines of memory and no more: such a launch has its numbers in the places of those that only teams use.
inline void spread_into(GemvGrid& g, const GemvSpread& s) {
  g.rounds = s.slots;
  g.teams = s.full;
  g.inv_teams = s.batch;
}
LLVQ_HD GemvSpread spread_of(const GemvGrid& g) { return {g.rounds, g.teams, g.inv_teams}; }
// The step that a lane of class c reads as its i-th.
LLVQ_HD uint32_t sums_read(uint32_t i, uint32_t c) { return 4u * i + c; }
// In LDS the four blocks of a unit lie together: 3 dwords per digit and block, then each block's sum of its integers
// (v = 2 n + b: sum v x = 2 sum n x + b sum x) and scale.  The pad spreads the eight units of a step over the banks.
template <int DIG> struct XPlanes {
  static constexpr uint32_t kBlock = 3 * DIG, kSums = 4 * kBlock, kDwords = kSums + 8 + (DIG == 6 ? 4 : 0);
};
// Units of the planes in LDS: whole steps, and a step of zeros behind them for the wavefronts whose steps end early.
LLVQ_HD uint32_t gemv_plane_units(uint32_t nb) { return (tile_steps(nb) + 1u) * kStepUnits; }

LLVQ_HD uint32_t gemv_lds_fixed() { return 128u + 64u; }
// The rotated activation and the sums share their place: rows of 20480 columns with f32 results, 24576 with binary16, are the widest that
// fit (160 KB).  One behind the other, 19456 and 20480 columns with f32 results and 23552 with binary16 took a launch more, 3.6 to 4 us.
inline uint64_t gemv_tiles_lds_bytes(uint32_t nb, uint32_t d_in, bool f32_out, bool rotated, bool gated = false) {
  const uint64_t planes = (uint64_t)gemv_plane_units(nb) * (f32_out ? XPlanes<6>::kDwords : XPlanes<4>::kDwords) * 4;
  const uint64_t sums = sums_room(gemv_wide(nb)) * kTileRows * 4 + (gated ? kGatedFloats * 4 : 0), values = rotated ? ((uint64_t)d_in * 4 + 31) / 16 * 16 : 0;
  return gemv_lds_fixed() + planes + (sums > values ? sums : values);
}

// ---- lists of products as one launch (gemv_seq.h) ----
constexpr uint32_t kSeqWaves = 16;
// Steps of a task of independent items, `bytes` of tiles on `grid` workgroups.  Two where a wavefront has sixteen steps or fewer: with few
// tiles to a workgroup tasks of four leave wavefronts without one, and with many the sums through LDS cost more than that.  One layer of a 4B
// model (2 steps a wavefront) 17.1 us with four, 14.8 with two, 14.6 with one; four layers (9) 38.1, 37.4, 38.0; six (13) 51.7, 50.2,
// 52.0; twelve (26) 91.2, 93.2, 97.4.
constexpr uint32_t kSeqTaskSteps = 4, kSeqShortTaskSteps = 2, kSeqShortSteps = 16;
LLVQ_HD uint32_t seq_task_steps(uint64_t bytes, uint32_t grid) {
  return bytes > (uint64_t)kSeqShortSteps * kSeqWaves * kStepUnits * kUnitBytes * grid ? kSeqTaskSteps : kSeqShortTaskSteps;
}
LLVQ_HD uint32_t seq_tasks(uint32_t steps, uint32_t task_steps) { return steps ? (steps + task_steps - 1u) / task_steps : 1u; }

constexpr uint32_t kSeqDrift = 4;      // tasks of a wavefront between two barriers, where tiles are shared
// Tiles whose sums may be pending between two barriers, when a tile is `tasks` >= 2 tasks: those that begin there, and one
// that is cut at either end.
LLVQ_HD uint32_t seq_slots(uint32_t tasks) { return kSeqDrift * kSeqWaves / tasks + 2u; }
// Sixteen rows of sums for each of their steps: at the most 4 tasks (64 / tasks + 2) with tasks <= 8.
constexpr uint32_t kSeqPartSteps = 4 * (kSeqDrift * kSeqWaves + 2 * 8), kSeqMaxSlots = kSeqDrift * kSeqWaves / 2 + 2;

}  // namespace llvq
