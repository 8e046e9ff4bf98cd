// A tile's list of escapes (escape_list.h) on the host, built and run by tests/test_escape_list.py: its places are as many as uniform
// codes need but for one tile in 30 000, by the share of escapes that draws show; and the walk over a tile's codes that replaces
// a list meets each block once, a row's in their order.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "block_code.h"
#include "escape_list.h"

using namespace llvq;

static void fail(const char* what, uint32_t a, double b) {
  std::printf("%s: %u, %g\n", what, a, b);
  std::exit(1);
}

int main() {
  for (int cap = 12; cap <= 13; ++cap) {
    const uint64_t top = cap == 12 ? 111043117458000ULL : kN13;
    const double share = cap == 12 ? kEscapeShare : kEscapeShare13;
    uint64_t z = 88172645463325252ULL, seen = 0;
    const int draws = 1000000;
    for (int i = 0; i < draws; ++i) {
      z ^= z << 13; z ^= z >> 7; z ^= z << 17;
      int8_t p[24];
      int shell = 0;
      if (!host_decode(z % (top + 1), p, &shell)) fail("no such rank", (uint32_t)i, 0);
      uint32_t n[3] = {0, 0, 0};
      for (int c = 0; c < 24; ++c) n[c / 8] |= ((uint32_t)(p[c] >> 1) & 15u) << (4 * (c % 8));
      BlockCode code{};
      if (!block_encode(n, (uint32_t)p[0] & 1u, 0, (uint32_t)shell, code)) fail("no code", (uint32_t)i, 0);
      seen += code.meta >= kBlockEscape;
    }
    // (four deviations of a count: 4 sqrt(780) of 780 at the worst)
    if (std::fabs((double)seen / (draws * share) - 1.) > 4. / std::sqrt(draws * share)) fail("share", (uint32_t)cap, (double)seen / draws);
    for (uint32_t nb = 1; nb <= kGemvMaxBlocks; ++nb) {
      const uint32_t slots = list_slots(nb, cap == 13);
      const double mean = 16. * nb * share;
      const auto above = [&](uint32_t places) {
        double sum = 0;
        for (uint32_t k = places + 1; k < places + 400; ++k) sum += std::exp(k * std::log(mean) - mean - std::lgamma(k + 1.));
        return sum;
      };
      if (slots % 8 || slots == 0 || slots > (cap == 12 ? kMaxListSlots : kMaxListSlots13)) fail("places", nb, slots);
      if (above(slots) > kListMisses * 1.0001) fail("too few places", nb, above(slots) * 30000);
      if (slots > 8 && above(slots - 8) < kListMisses * 0.9999) fail("too many places", nb, above(slots - 8) * 30000);
    }
  }
  if (list_slots(0, false) || list_slots(0, true)) fail("places of no block", 0, 0);
  for (uint32_t nb : {1u << 19, (1u << 19) + 1u})  // (an entry has 19 bits for the block)
    if (list_slots(nb, false) != (nb >> 19 << 19 == nb ? kMaxListSlots : 0u)) fail("places of the widest rows", nb, list_slots(nb, false));
  for (uint32_t byte = 0; byte < 256; ++byte)
    for (uint32_t k = 0; k < 4; ++k) {
      const uint32_t lo = byte << (8 * k) | (0x7F7F7F7Fu & ~(255u << (8 * k))), want = byte >= kBlockEscape ? 1u << (8 * k) : 0u;
      if (walk_mask(lo, 0x7F7F7F7Fu) != want || walk_mask(0xBFBFBFBFu, lo) != want << 1) fail("mask", byte, k);
    }
  for (uint32_t nb = 1; nb <= kGemvMaxBlocks; ++nb) {
    const uint32_t units = (nb + 3) / 4;
    std::vector<uint32_t> next(16, 0);
    for (uint32_t step = 0; step < tile_steps(nb); ++step)
      for (uint32_t lane = 0; lane < 64; ++lane) {
        if (step * kStepUnits + (lane >> 3) >= units) continue;
        for (uint32_t bit = 0; bit < 32; ++bit) {
          if ((bit & 7u) > 1u) continue;
          const uint32_t key = walk_key(step, lane, bit);
          if ((key & 0xFFFFFFFu) != next[key >> 28]++) fail("order", nb, key);
        }
      }
    for (uint32_t row = 0; row < 16; ++row)
      if (next[row] != 4 * units) fail("blocks", nb, row);
  }
  std::printf("ok\n");
  return 0;
}
