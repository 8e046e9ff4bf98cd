// The 80-bit block code on the host, built and run by tests/test_block_code.py: every point has a code, and the code gives
// back the point, its gain and its shell.
//   1. Shapes: every multiset of 24 coordinates of one parity whose squares add up to 16 m <= 208, whose sum is 0 (even)
//      or 4 (odd) mod 8 and whose coordinates of either residue mod 4 are as many as a Golay word has bits.  Whether a point
//      has a code depends on nothing else, and every point of the lattice is of such a shape.
//   2. Points of the lattice: class boundaries are passed on the command line, random ranks are drawn here.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <utility>

#include "../llvq_amd/csrc/block_code.h"

using namespace llvq;

static size_t shapes = 0, escapes = 0, ranks = 0;

static bool round_trip(const int (&v)[24], uint32_t gain, uint32_t shell) {
  const uint32_t odd = (uint32_t)v[0] & 1u;
  uint32_t n[3] = {0, 0, 0};
  for (int i = 0; i < 24; ++i) n[i / 8] |= ((uint32_t)(v[i] >> 1) & 15u) << (4 * (i % 8));
  BlockCode c{};
  if (!block_encode(n, odd, gain, shell, c)) return false;
  if (c.meta > 255u || (c.s & ~0x11111111u)) return false;
  escapes += c.meta >= kBlockEscape;
  uint32_t w[3], win = c.meta & 7u, slot = c.meta >> 3, negative = 0, far = 24, picks[3] = {0, 0, 0};
  EscapePick pick{8, 0};
  block_octets(c.d0, c.d1, c.s << 3, w);
  if (c.meta >= kBlockEscape) {
    const BlockEscape e = block_escape(w, c.meta);
    w[0] = e.w0;
    win = e.win;
    slot = e.slot;
    negative = e.negative;
    far = e.at;
    std::memcpy(picks, w, sizeof w);
    pick = escape_pick(picks, e);
    if (far < 24 ? pick.index > 7 : pick.index != 8) return false;
  } else {
    std::memcpy(picks, w, sizeof w);
  }
  for (uint32_t i = 0; i < 24; ++i) {
    const int got = nibble_at(w[i / 8], i % 8) + (int)win - 3 - (i == far ? 16 : 0);
    if ((negative ? -got : got) != v[i]) return false;
    const uint32_t index = (picks[i / 8] >> (4 * (i % 8) + 1)) & 7u;  // the same looked up
    const int looked = index == pick.index ? pick.value : 2 * ((int)index < 4 ? (int)index : (int)index - 8) + (int)win - 3;
    if ((negative ? -looked : looked) != v[i] || (picks[i / 8] & 0x11111111u)) return false;
  }
  return shell == 0 || slot == gain * 12u + shell - 2u;
}

static void fail(const int (&v)[24], const char* what) {
  std::fprintf(stderr, "%s:", what);
  for (int x : v) std::fprintf(stderr, " %d", x);
  std::fprintf(stderr, "\n");
  std::exit(1);
}

// Places coordinates of magnitude m, m + 2, ... from `at` on; `left` of the norm is to be spent.
static void walk(int (&v)[24], int at, int m, int left) {
  if (at == 24) {
    int sum = 0, weight = 0;
    for (int x : v) {
      sum += x;
      weight += (x & 2) != 0;
    }
    if (left % 16 || left == 192 || (sum & 7) != (v[0] & 1 ? 4 : 0)) return;
    if (weight != 0 && weight != 8 && weight != 12 && weight != 16 && weight != 24) return;
    ++shapes;
    for (uint32_t gain = 0; gain < 2; ++gain)
      for (int first = 0; first < 24; first += 23) {  // (the hidden bits change the first coordinate)
        std::swap(v[0], v[first]);
        if (!round_trip(v, gain, (208u - (uint32_t)left) / 16u)) fail(v, "shape");
        std::swap(v[0], v[first]);
      }
    return;
  }
  if (m * m > left) return;
  for (int count = 0; count <= 24 - at && count * m * m <= left; ++count)
    for (int negative = 0; negative <= (m ? count : 0); ++negative) {
      for (int i = 0; i < count; ++i) v[at + i] = i < negative ? -m : m;
      if (at + count == 24) walk(v, 24, 0, left - count * m * m);
      else walk(v, at + count, m + 2, left - count * m * m);
    }
}

int main(int argc, char** argv) {
  int v[24];
  walk(v, 0, 0, 208);
  walk(v, 0, 1, 208);
  const size_t seen = escapes;
  escapes = 0;
  auto rank = [&](uint64_t idx) {
    int8_t p[24];
    int shell = 0;
    if (!host_decode(idx, p, &shell)) {
      std::fprintf(stderr, "rank %llu has no point\n", (unsigned long long)idx);
      std::exit(1);
    }
    for (int i = 0; i < 24; ++i) v[i] = p[i];
    for (uint32_t gain = 0; gain < 2; ++gain)
      if (!round_trip(v, gain, (uint32_t)shell)) fail(v, "rank");
    ++ranks;
  };
  for (int a = 1; a < argc; ++a) rank(std::strtoull(argv[a], nullptr, 10));
  uint64_t z = 88172645463325252ULL;
  for (int i = 0; i < 400000; ++i) {
    z ^= z << 13; z ^= z >> 7; z ^= z << 17;
    rank(z % (kN13 + 1));
  }
  if (shapes == 0 || seen == 0 || escapes == 0 || ranks != 400000 + (size_t)(argc - 1)) {
    std::fprintf(stderr, "%zu shapes, %zu of them escapes; %zu ranks, %zu escapes\n", shapes, seen / 4, ranks, escapes / 2);
    return 1;
  }
  std::printf("ok: %zu shapes, %zu of them escapes; %zu ranks, %zu escapes\n", shapes, seen / 4, ranks, escapes / 2);
  return 0;
}
