// A lattice point of 24 coordinates, its gain bit and its shell in 80 bits that unpack into operands of the 4-bit dot
// product with a few logical instructions.  Compiled for gfx950 and for the host.
//
// The coordinates v of a point are all even or all odd and lie, but for 0.08 % of uniformly drawn points of shells 2..12
// (0.32 % of shells 2..13), in a window [b, b + 14] with -11 <= b <= -4 of their parity: v = 2 j + b with j of 3 bits.
// Nothing is rounded.
//
// An octet of coordinates is a dword of eight nibbles, two's complement, 2 (j - 4) in each: their lowest bits are free.
//   d0, d1  the first two octets' nibbles; in the free bits, bit 1 (d0) or 2 (d1) of the third octet's
//   s       bit 3 of the third octet's: the eight bits of four blocks share a dword, block k's in bit k of the nibbles
//   meta    below kBlockEscape: (gain * 12 + shell - 2) << 3 | win with win = b + 11.  The origin is any of these with v = 0.
// so v = nibble + win - 3.
//
// Any other point (meta >= kBlockEscape) is the point or its negative with all coordinates but one in a window that the
// code names, the one 16 below its place there (or, escape 48, with none such).  Which coordinate takes the code's room,
// so the gain bit and whether it is the negative are hidden where a point has room to spare: its coordinates add up to 0
// (even) or 4 (odd) mod 8, hence the j's to 0 or 2 mod 4, and k = gain + 2 negative is added to the first of them.  The
// shell is what the coordinates' squares add up to.
//   kBlockEscape +  0 + p: b = -6, coordinate p (in nibble order) 16 below
//   kBlockEscape + 24 + p: b = -5, the same
//   kBlockEscape + 48:     b = -11, none
// That these reach every point of shells up to 13 is a matter of magnitudes alone (a point's squares add up to 208 at the
// most); tests/block_code.cpp walks all of them.
#pragma once
#include <cstdint>

#include "decode_core.h"

namespace llvq {

constexpr uint32_t kBlockEscape = 192;  // byte >= 192: its two top bits are set
constexpr uint32_t kScaleSlots = 32;    // block scales, at gain * 12 + shell - 2

struct BlockCode {
  uint32_t d0, d1, s, meta;
};

LLVQ_HD int nibble_at(uint32_t w, uint32_t q) { return (int)(w << (28u - 4u * q)) >> 28; }

// n: the nibbles of v = 2 n + odd, any order of columns.  False: no code (no point of shells 0..13 is like that).
LLVQ_HD bool block_encode(const uint32_t (&n)[3], uint32_t odd, uint32_t gain, uint32_t shell, BlockCode& out) {
  int lo = 127, hi = -127;
#pragma unroll
  for (int o = 0; o < 3; ++o)
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) {
      const int v = 2 * nibble_at(n[o], q) + (int)odd;
      lo = v < lo ? v : lo;
      hi = v > hi ? v : hi;
    }
  const int top = odd ? -5 : -4, bottom = odd ? -11 : -10;
  int b = lo < top ? lo : top, sign = 1;
  uint32_t meta, k = 0;
  bool ok = true;
  if (b >= bottom && hi <= b + 14) {
    meta = (gain * 12u + (shell ? shell - 2u : 0u)) << 3 | (uint32_t)(b + 11);
  } else {
    b = odd ? -5 : -6;
    int below[2] = {0, 0}, at[2] = {0, 0};  // of the point and of its negative
#pragma unroll
    for (int o = 0; o < 3; ++o)
#pragma unroll
      for (uint32_t q = 0; q < 8; ++q) {
        const int v = 2 * nibble_at(n[o], q) + (int)odd;
        if (v < b) { ++below[0]; at[0] = o * 8 + (int)q; }
        if (-v < b) { ++below[1]; at[1] = o * 8 + (int)q; }
      }
    const bool plain = below[0] == 1 && lo >= b - 16 && hi <= b + 14;
    const bool negated = below[1] == 1 && -hi >= b - 16 && -lo <= b + 14;
    if (plain || negated) {
      sign = plain ? 1 : -1;
      meta = kBlockEscape + (odd ? 24u : 0u) + (uint32_t)(plain ? at[0] : at[1]);
    } else {
      ok = odd && -hi >= -11 && -lo <= 3;
      b = -11;
      sign = -1;
      meta = kBlockEscape + 48u;
    }
    k = gain + (sign < 0 ? 2u : 0u);
  }
  uint32_t j[3] = {0, 0, 0};
#pragma unroll
  for (int o = 0; o < 3; ++o)
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) j[o] |= (uint32_t)(((2 * nibble_at(n[o], q) + (int)odd) * sign - b) >> 1 & 7) << (4 * q);
  j[0] = (j[0] & ~7u) | ((j[0] + k) & 7u);
#pragma unroll
  for (int o = 0; o < 3; ++o) j[o] = (j[o] ^ 0x44444444u) << 1;
  out.d0 = j[0] | ((j[2] >> 1) & 0x11111111u);
  out.d1 = j[1] | ((j[2] >> 2) & 0x11111111u);
  out.s = (j[2] >> 3) & 0x11111111u;
  out.meta = meta;
  return ok;
}

LLVQ_HD int dot8(uint32_t a, uint32_t b, int c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_sdot8((int)a, (int)b, c, false);
#else
  for (uint32_t q = 0; q < 8; ++q) c += nibble_at(a, q) * nibble_at(b, q);
  return c;
#endif
}

// The octets' nibbles; s3: the block's bits of s as the nibbles' top bits (whatever the others are).
LLVQ_HD void block_octets(uint32_t d0, uint32_t d1, uint32_t s3, uint32_t (&w)[3]) {
  w[0] = d0 & 0xEEEEEEEEu;
  w[1] = d1 & 0xEEEEEEEEu;
  w[2] = ((((d1 & 0x11111111u) << 1) | (d0 & 0x11111111u)) << 1) | (s3 & 0x88888888u);
}

// What a code of kBlockEscape or more stands for: the first octet's nibbles with nothing hidden in them, the window, the
// scale's slot, whether it is the negative, and the coordinate that is 16 below (0..23, more: none).  About 45 instructions; who
// puts the coordinates back into a form of its own needs as many again or more (gemm_kernel.h: 120 in gemm_escape, 200 in code_block).
struct BlockEscape {
  uint32_t w0, win, slot, negative, at;
};
LLVQ_HD BlockEscape block_escape(const uint32_t (&w)[3], uint32_t meta) {
  const uint32_t f = meta - kBlockEscape, odd = f >= 24u ? 1u : 0u;
  const bool none = f >= 48u;
  const uint32_t p = f - 24u * odd;
  const uint32_t sum = (uint32_t)dot8(w[0], 0x11111111u, dot8(w[1], 0x11111111u, dot8(w[2], 0x11111111u, 0))) >> 1;  // (of j - 4: mod 4 that of j)
  const uint32_t k = (sum - 2u * odd) & 3u;
  BlockEscape x;
  x.w0 = bfi32(0xEu, w[0] - 2u * k, w[0]);
  x.win = none ? 0u : odd ? 6u : 5u;
  x.at = p;
  x.negative = k >> 1;
  // Coordinates n + c with the one at p 16 less; the squares' sum is 16 times the shell.
  const int c = (int)x.win - 3, total = dot8(x.w0, 0x11111111u, dot8(w[1], 0x11111111u, dot8(w[2], 0x11111111u, 0)));
  const int squares = dot8(x.w0, x.w0, dot8(w[1], w[1], dot8(w[2], w[2], 0)));
  const int far = nibble_at(p < 8u ? x.w0 : p < 16u ? w[1] : w[2], p & 7u) + c;
  const int norm = squares + 2 * c * total + 24 * c * c + (none ? 0 : 256 - 32 * far);
  x.slot = (k & 1u) * 12u + ((uint32_t)norm >> 4) - 2u;
  return x;
}

// For who looks a coordinate's three bits up in eight values, at i (as a signed number) 2 i + win - 3: an index that none of
// the others has, in the nibbles now in the far one's place, and the far one's value (24 places on: no index, 8).  There is one:
// no point of shells up to 13 has more than eight different coordinates (nine of one parity have squares that add up to 240
// or more), and the far one is unlike all others.  About 70 instructions.  w: the octets, the first with nothing hidden in it.
struct EscapePick {
  uint32_t index;
  int value;
};
LLVQ_HD EscapePick escape_pick(uint32_t (&w)[3], const BlockEscape& e) {
  uint32_t used = 0;
  int far = 0;
#pragma unroll
  for (uint32_t o = 0; o < 3; ++o) {
    const bool here = e.at >> 3 == o;
    const uint32_t at = here ? 15u << (4u * (e.at & 7u)) : 0u;
    far = here ? nibble_at(w[o], e.at & 7u) : far;
    const uint32_t others = bfi32(at, w[o] >> 4 | w[o] << 28, w[o]);  // its neighbour's instead
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) used |= 1u << ((others >> (4u * q + 1u)) & 7u);
  }
  EscapePick p{8u, far + (int)e.win - 19};
  if (e.at < 24u) p.index = (uint32_t)__builtin_ctz(~used & 0x1FFu);
#pragma unroll
  for (uint32_t o = 0; o < 3; ++o)
    if (e.at >> 3 == o) w[o] = bfi32(15u << (4u * (e.at & 7u)), (p.index & 7u) << (4u * (e.at & 7u) + 1u), w[o]);
  return p;
}

}  // namespace llvq
