// The batched product Y[M, d_out] = X[M, d_in] W^T on the matrix cores (M >= 2), over the tiles of tiles.h.  Included by
// llvq_hip.hip after it.  The reference runs a row loop of matrix-vector products (llvq-llm/src/model.rs:521-529).
//
// Weights are multiplied as binary16: v centroid[gain] / sqrt(16 shell) rounded once; sums are f32; row scale and tail
// columns are applied in f32 at the end.  The PAIR variants of the kernels multiply what that rounding took as well and keep
// their sums in f64 (of f32 sums over 32 or 48 columns), for the rows whose results are f32 exact (llvq_hip.hip,
// gemm_same_basis).  Relative error of f32 results in norm, 2561 x 1000 at 65 rows: 2.1e-4 with one term, 1.01e-7 with two,
// 0.97e-7 for rows one by one; 13000 columns: 2.2e-4, 1.37e-7, 1.38e-7.  Two terms alone, summed in f32, left up to 6e-7.  A dword of a block's nibbles is eight consecutive columns of a row, which is
// exactly what a lane hands to a 16-deep (32 x 32) or 32-deep (16 x 16) product step, so a wavefront turns the ten bytes
// of a block that its lanes load into its own fragments: no weights pass through LDS, and the order in which the products walk the
// columns is the order the blocks lie in (the lane groups of a fragment hold the same octet of two or four neighbouring
// blocks).  17 instructions per eight weights, and 8 per block to put its three octets together; 12 and 4 in the wide kernels,
// which look the weights up.
//
// The activations come as octets: xt[c][m] = columns 8 c .. 8 c + 7 of row m, 16 bytes, m_pad rows to a column octet, so
// that the fragments of 16 or 32 rows are runs of 256 or 512 bytes (tile_activations_kernel; in x they would be 16-byte
// pieces 2 d_in bytes apart, and a load of them would touch as many cache lines as it has lanes).
#pragma once

namespace llvq {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float acc4_t __attribute__((ext_vector_type(4)));
typedef float acc16_t __attribute__((ext_vector_type(16)));

constexpr int kGemmMaxGroup = 4;
constexpr uint32_t kGemmSmallRows = 64;     // activation rows up to which the split kernel (gemm_tiles_kernel) runs
constexpr uint32_t kGemmTileRowsSmall = 16; // weight rows of a fragment there

// ---- activations as column octets ----------------------------------------------------------------
// One lane per octet; a wavefront takes eight octets of eight rows: 128 consecutive bytes of a row read, 128 of the copy
// written.  Rows from M on and columns from kcols on are zero.  gate: the activations are f16(silu(gate)) x, and their tail columns
// go to `rows` (octets past the copy's have lanes of their own).
__global__ __launch_bounds__(256) void tile_activations_kernel(const __half* __restrict__ x, const __half* __restrict__ gate, __half* __restrict__ rows,
                                                               uint32_t M, uint32_t ldx, uint32_t kcols, uint32_t m_pad, uint32_t n_oct, uint4* __restrict__ xt) {
  const uint32_t lane = threadIdx.x & 63u, wave = blockIdx.x * 4u + (threadIdx.x >> 6);
  const uint32_t groups_m = m_pad >> 3;
  const uint32_t gc = wave / groups_m, gm = wave - gc * groups_m;
  const uint32_t c = gc * 8u + (lane & 7u), m = gm * 8u + (lane >> 3);
  uint4 v = make_uint4(0, 0, 0, 0);
  if (m < M && c * 8u < (gate ? ldx : kcols)) {
    HalfOctet o = *reinterpret_cast<const HalfOctet*>(x + (size_t)m * ldx + c * 8u);
    if (gate) {
      const HalfOctet g = *reinterpret_cast<const HalfOctet*>(gate + (size_t)m * ldx + c * 8u);
#pragma unroll
      for (int j = 0; j < 4; ++j) o.w[j] = pack_halves(silu_mul(half_lo(g.w[j]), half_lo(o.w[j])), silu_mul(half_hi(g.w[j]), half_hi(o.w[j])));
    }
    if (c * 8u < kcols) v = make_uint4(o.w[0], o.w[1], o.w[2], o.w[3]);
    else *reinterpret_cast<HalfOctet*>(rows + (size_t)m * ldx + c * 8u) = o;
  }
  // the copy wants eight rows of one octet together: lane (octet, row) <- lane (row, octet)
  const int from = (int)(((lane & 7u) * 8u + (lane >> 3)) * 4u);
  v.x = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)v.x);
  v.y = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)v.y);
  v.z = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)v.z);
  v.w = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)v.w);
  const uint32_t oc = gc * 8u + (lane >> 3), om = gm * 8u + (lane & 7u);
  if (oc < n_oct) xt[(size_t)oc * m_pad + om] = v;
}

// ---- weights ---------------------------------------------------------------------------------------
// The matrix's table of scales for dequant_octet: a lane keeps its entry (scale_table) as the sum of two binary16 numbers
// (low half: the entry rounded, high half: what that left), a power of two taken out first that puts the largest entry into
// [8, 16), so that neither number nor a sixteenth of it leaves the normal range by more than the precision can spare.
// `unit` is that power of two; it goes back in with the row scales.
__device__ __forceinline__ float table_unit(float entry) {
  int e = (int)(__float_as_uint(entry) & 0x7F800000u);  // (two lanes to an entry, eight to a row of lanes)
  e = max(e, __builtin_amdgcn_update_dpp(0, e, 0x122, 0xF, 0xF, false));  // row_ror 2, 4, 8
  e = max(e, __builtin_amdgcn_update_dpp(0, e, 0x124, 0xF, 0xF, false));
  e = max(e, __builtin_amdgcn_update_dpp(0, e, 0x128, 0xF, 0xF, false));
  e = max(max(__builtin_amdgcn_readlane(e, 0), __builtin_amdgcn_readlane(e, 16)), max(__builtin_amdgcn_readlane(e, 32), __builtin_amdgcn_readlane(e, 48)));
  return ldexpf(1.f, min(max((e >> 23) - 130, -100), 100));  // (a table of zeros or with an infinity in it: any power will do)
}
__device__ __forceinline__ uint32_t split_table(float entry, float unit) {
  const float v = entry * (1.f / unit);
  const _Float16 hi = (_Float16)v;
  const _Float16 lo = (_Float16)(v - (float)hi);
  return __builtin_bit_cast(uint32_t, half2_t{hi, lo});
}
// A block's octets as the unpacking wants them: v = nibble + 16 (the lowest bit of the next nibble around) + win - 3, that
// bit for the blocks with one coordinate 16 below (block_code.h), where all others get it and the window goes down by 16.
// And the two parts of the block's scale.
struct GemmBlock {
  uint32_t w[3], parts, meta;
  int win;
};
__device__ __forceinline__ uint32_t scale_parts(uint32_t meta, uint32_t table) {
  return (uint32_t)__builtin_amdgcn_ds_bpermute((int)meta, (int)table);
}
// s, m: the {s, meta} dwords of the block's row; k: the block in its unit.
__device__ __forceinline__ GemmBlock gemm_block(uint32_t d0, uint32_t d1, uint32_t s, uint32_t m, uint32_t k, uint32_t table) {
  GemmBlock b;
  block_octets(d0, d1, s << (3u - k), b.w);
  const uint32_t meta = m >> (8u * k);
  b.meta = meta & 255u;
  b.parts = scale_parts(meta, table);
  b.win = (int)(meta & 7u);
  return b;
}
__device__ __forceinline__ bool is_escape(const GemmBlock& b) { return b.meta >= kBlockEscape; }
// For all lanes (the scales are in all of them), where any has an escape.
__device__ __forceinline__ void gemm_escape(GemmBlock& b, uint32_t table) {
  const bool escape = is_escape(b);
  const BlockEscape e = block_escape(b.w, b.meta);
  const uint32_t parts = scale_parts(e.slot << 3, table) ^ (e.negative ? 0x80008000u : 0u);
  const uint32_t q = e.at & 7u, bit = 1u << (4u * (q == 7u ? 0u : q + 1u));
  const bool one = e.at < 24u;
  b.w[0] = escape ? e.w0 : b.w[0];
#pragma unroll
  for (uint32_t o = 0; o < 3; ++o) b.w[o] |= escape && one ? 0x11111111u & ~((e.at >> 3) == o ? bit : 0u) : 0u;
  b.win = escape ? (int)e.win - (one ? 16 : 0) : b.win;
  b.parts = escape ? parts : b.parts;
}
// An escape of a tile's list in the same form, from lane `of` of `e` to lane `to`: a nibble n is 8 less, of which the bit above
// has 16 and the window the rest.
__device__ __forceinline__ void gemm_listed(GemmBlock& b, const u32x4_t& e, uint32_t of, uint32_t to, uint32_t lane, uint32_t table) {
  const bool mine = lane == to;
#pragma unroll
  for (int o = 0; o < 3; ++o) {
    const uint32_t n = (uint32_t)__builtin_amdgcn_readlane((int)e[o], of), up = ~(n >> 3) & 0x11111111u;
    const uint32_t w = (((n & 0x77777777u) ^ 0x44444444u) << 1) | (up << 4 | up >> 28);
    b.w[o] = mine ? w : b.w[o];
  }
  const uint32_t key = (uint32_t)__builtin_amdgcn_readlane((int)e.w, of);
  const uint32_t parts = (uint32_t)__builtin_amdgcn_readlane((int)table, (key & 31u) * 2u);
  b.parts = mine ? parts : b.parts;
  b.win = mine ? (int)((key >> 8) & 1u) - 5 : b.win;
}
// The parts of a block's scale (and a sixteenth of them), and what takes a nibble's offset off (dequant_octet), in pairs.
struct BlockScale {
  half2_t c, c16;
  uint32_t b, b16;
};
__device__ __forceinline__ BlockScale block_scale(int win, uint32_t parts) {
  const half2_t c = __builtin_bit_cast(half2_t, parts);
  // -(1024 + 11 - win) and -(1024 + 16 (11 - win)) as binary16
  const uint32_t b = (uint32_t)mad24(win, -0x00010001, (int)0xE40BE40Bu), b16 = (uint32_t)mad24(win, -0x00100010, (int)0xE4B0E4B0u);
  return BlockScale{c, c * half2_t{(_Float16)0.0625f, (_Float16)0.0625f}, b, b16};
}
// One dword of nibbles -> eight weights.  A binary16 number of the form 1024 + k has k in its low bits: a nibble there, its
// top bit turned over, with the lowest bit of the next one on top of it, makes 1024 + 11 - win + v, or 1024 +
// 16 (11 - win) + 16 v where it lies four bits higher.
// v (hi + lo) is rounded once: v lo is small enough for its own rounding to be
// lost in that of the sum.  17 instructions, all of which run beside the matrix cores; the mixed-precision
// multiply-add (two fewer) does not: 4 products and 20 of those took 103 ns of a SIMD, with packed or f32 ones 70.
__device__ __forceinline__ half2_t octet_bits(uint32_t w, int i) {  // nibbles i and i + 4
  const uint32_t u = i < 2 ? w : __builtin_amdgcn_alignbit(w, w, 8);
  return __builtin_bit_cast(half2_t, (i & 1) ? (u & 0x01E001E0u) ^ 0x64806480u : (u & 0x001E001Eu) ^ 0x64086408u);
}
__device__ __forceinline__ half2_t dequant_two(uint32_t w, const BlockScale& s, int i) {
  const half2_t v = octet_bits(w, i) + __builtin_bit_cast(half2_t, (i & 1) ? s.b16 : s.b);
  const half2_t c = (i & 1) ? s.c16 : s.c;
  return __builtin_elementwise_fma(v, half2_t{c.x, c.x}, v * half2_t{c.y, c.y});
}
__device__ __forceinline__ half8_t dequant_octet(uint32_t w, const BlockScale& s) {
  half8_t out;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const half2_t y = dequant_two(w, s, i);
    out[2 * i] = y.x;
    out[2 * i + 1] = y.y;
  }
  return out;
}

// The same with what the rounding took as a second binary16 number each: the two make the weight to 2^-22 of it.  (A nibble
// that lies four bits higher is brought down by the operation that takes the offset off, so both halves are v itself; what is
// left of v hi after the first rounding is exact, and v lo joins it in one more.)  27 instructions.
struct TwoPair {
  half2_t hi, lo;
};
__device__ __forceinline__ TwoPair dequant_two_pair(uint32_t w, const BlockScale& s, int i) {
  const half2_t hi = half2_t{s.c.x, s.c.x}, lo = half2_t{s.c.y, s.c.y}, u = octet_bits(w, i);
  // (a sixteenth of -(1024 + 16 k) is -(64 + k): the exponent four lower)
  const half2_t v = (i & 1) ? __builtin_elementwise_fma(u, half2_t{(_Float16)0.0625f, (_Float16)0.0625f}, __builtin_bit_cast(half2_t, s.b16 - 0x10001000u))
                            : u + __builtin_bit_cast(half2_t, s.b);
  const half2_t y = __builtin_elementwise_fma(v, hi, v * lo);
  return TwoPair{y, __builtin_elementwise_fma(v, lo, __builtin_elementwise_fma(v, hi, -y))};
}
struct WeightPair {
  half8_t hi, lo;
};
__device__ __forceinline__ WeightPair dequant_octet_pair(uint32_t w, const BlockScale& s) {
  WeightPair out;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const TwoPair y = dequant_two_pair(w, s, i);
    out.hi[2 * i] = y.hi.x;
    out.hi[2 * i + 1] = y.hi.y;
    out.lo[2 * i] = y.lo.x;
    out.lo[2 * i + 1] = y.lo.y;
  }
  return out;
}

// The wide kernel unpacks by looking up: the weights of the eight values that a block's coordinates can have, binary16, lie
// in LDS, 16 bytes for each meta byte, in the order of three bits of the coordinates' nibbles, the low bytes of all before
// the high ones; v_perm_b32 picks four at a time.  12 instructions an octet where arithmetic takes 17 (dequant_octet) and one
// dword in place of the scale's four.  Meta bytes below kBlockEscape are windows of the matrix's scales, those from
// there on are of a wavefront's escapes, 16 of them at a time: no point of shells up to 13 has more than eight different coordinates
// (nine of one parity have squares that add up to 240 or more), so each can be written that way.
constexpr uint32_t kValueBytes = 256u * 16u;  // with PAIR a second such table, of what the rounding took
constexpr uint32_t kWaveValues = (256u - kBlockEscape) / 4u;
struct Values {
  u32x4_t hi, lo;
};
__device__ __forceinline__ void value_to(Values& t, int i, float y) {
  const _Float16 hi = (_Float16)y, lo = (_Float16)(y - (float)hi);
  const uint32_t a = __builtin_bit_cast(uint16_t, hi), b = __builtin_bit_cast(uint16_t, lo), at = 8u * ((uint32_t)i & 3u);
  t.hi[i >> 2] |= (a & 255u) << at;
  t.hi[2 + (i >> 2)] |= (a >> 8) << at;
  t.lo[i >> 2] |= (b & 255u) << at;
  t.lo[2 + (i >> 2)] |= (b >> 8) << at;
}
// A block as d0, d1 and its bits of s (in bit 0 of the nibbles) that picks from eight weights of its own.  n: the nibbles of v =
// 2 n + odd.  About 300 instructions.
struct ValueBlock {
  Values t;
  uint32_t d0, d1, s, at;  // at: where it belongs, of who keeps it
};
__device__ __forceinline__ ValueBlock value_block(const uint32_t (&n)[3], uint32_t odd, float scale) {
  uint32_t there = 0, pick[3] = {0, 0, 0};
  const uint32_t u[3] = {n[0] ^ 0x88888888u, n[1] ^ 0x88888888u, n[2] ^ 0x88888888u};  // n + 8
#pragma unroll
  for (int o = 0; o < 3; ++o)
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) there |= 1u << ((u[o] >> (4u * q)) & 15u);
#pragma unroll
  for (int o = 0; o < 3; ++o)
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) pick[o] |= (uint32_t)__builtin_popcount(there & ((1u << ((u[o] >> (4u * q)) & 15u)) - 1u)) << (4u * q);
  ValueBlock b{{{}, {}}, pick[0] << 1 | (pick[2] & 0x11111111u), pick[1] << 1 | ((pick[2] >> 1) & 0x11111111u), (pick[2] >> 2) & 0x11111111u, 0u};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int v = there ? 2 * ((int)__builtin_ctz(there) - 8) + (int)odd : 0;
    there &= there - 1u;
    value_to(b.t, i, (float)v * scale);
  }
  return b;
}
// A quarter of an octet's unpacking: w's three bits at bit SHIFT of its nibbles.  Quarters 0 and 1 leave the pairs of
// nibbles (0, 4) and (2, 6), 2 and 3 the others; a quarter's first half hands its bytes to the second.
struct ValuePick {
  uint32_t at, high;
};
template <uint32_t SHIFT>
__device__ __forceinline__ void pick_values(uint32_t w, const u32x4_t& t, uint32_t quarter, ValuePick& p, u32x4_t& to) {
  if ((quarter & 1u) == 0u) {
    const uint32_t shift = SHIFT + (quarter ? 4u : 0u);
    p.at = (shift ? w >> shift : w) & 0x07070707u;
    p.high = __builtin_amdgcn_perm(t[3], t[2], p.at);
  } else {
    const uint32_t low = __builtin_amdgcn_perm(t[1], t[0], p.at);
    to[quarter >> 1] = __builtin_amdgcn_perm(p.high, low, 0x06020400u);
    to[2 + (quarter >> 1)] = __builtin_amdgcn_perm(p.high, low, 0x07030501u);
  }
}

struct GemmMat {
  const uint8_t* base;  // the matrix (table, then records)
  void* y;
  uint32_t d_out, tile_begin;  // first row tile of this matrix in the launch
  uint32_t stride, slots;      // of its tiles in memory
};
struct GemmArgs {
  const uint4* xt;     // [octets][m_pad]
  const __half* x;     // [M, ldx] the activations in the matrices' basis (the tail columns are read from here)
  float* ws;           // [splits][m_pad][n_tiles * rows of a tile] partial sums (splits > 1)
  GemmMat mat[kGemmMaxGroup];
  uint32_t n_mats, n_tiles;
  uint32_t y_f32;      // output type: binary32, else binary16
  uint32_t ldx, tail_w;
  uint32_t M, m_pad, nb;
  uint32_t m_tiles, splits, steps_per_split;  // the wide kernel's grid
  // Where gemm_tiles_kernel finds octet j of block k of unit q of row m: xs + q * xs_unit + k * xs_block + j * xs_octet + m * xs_row, rows
  // past xs_last being that one.
  const uint8_t* xs;
  uint32_t xs_unit, xs_block, xs_octet, xs_row, xs_last;
};
// All arguments asked for at once (as touch_args does for the batch-1 products').
__device__ __forceinline__ void touch_args(const GemmArgs& a) {
  asm volatile("" ::"s"(a.ws), "s"(a.mat[1].base), "s"(a.mat[3].base), "s"(a.M), "s"(a.xs_last));
}

// What a product whose columns are split leaves for the launch behind it: value r of activation row m of matrix i is the sum, in order, of
// ws[(p m_pad + m) ld + first[i] + r] over the splits p.  No splits: the results are where they belong.  (A prompt's norms and its heads' norms
// read them: a launch of 9 us less for q/k/v, o and down of each layer, and results that do not go through memory a second time.  500 tokens of
// twelve 4B layers 2916 -> 2697 us with it and what is said at the product's end.)
struct GemmSums {
  const float* ws;
  uint32_t splits, m_pad, ld;
  uint32_t first[kGemmMaxGroup];
};
constexpr uint32_t kReduceSplits = 4;  // whose values are asked for together
// N values of row m from place `at` on (at a multiple of four)
template <uint32_t N>
__device__ __forceinline__ void parts_read(const GemmSums& s, uint32_t m, uint32_t at, float (&out)[N]) {
  static_assert(N % 4 == 0, "in sixteens of bytes");
#pragma unroll
  for (uint32_t i = 0; i < N; ++i) out[i] = 0.f;
  const size_t step = (size_t)s.m_pad * s.ld;
  const float* from = s.ws + (size_t)m * s.ld + at;
  for (uint32_t p0 = 0; p0 < s.splits; p0 += kReduceSplits) {
    float4 v[kReduceSplits][N / 4];
#pragma unroll
    for (uint32_t p = 0; p < kReduceSplits; ++p) {  // (past the last: the last again)
      const float4* q = reinterpret_cast<const float4*>(from + min(p0 + p, s.splits - 1u) * step);
#pragma unroll
      for (uint32_t i = 0; i < N / 4; ++i) v[p][i] = q[i];
    }
#pragma unroll
    for (uint32_t p = 0; p < kReduceSplits; ++p) {
      if (p0 + p >= s.splits) break;
#pragma unroll
      for (uint32_t i = 0; i < N / 4; ++i) {
        out[4 * i] += v[p][i].x;
        out[4 * i + 1] += v[p][i].y;
        out[4 * i + 2] += v[p][i].z;
        out[4 * i + 3] += v[p][i].w;
      }
    }
  }
}

struct GemmTile {
  const uint8_t* base;
  void* y;
  uint32_t row0, d_out, stride, slots;
};
__device__ __forceinline__ GemmTile gemm_tile_at(const GemmArgs& a, uint32_t tile, uint32_t rows_per_tile) {
  GemmTile t{a.mat[0].base, a.mat[0].y, 0u, a.mat[0].d_out, a.mat[0].stride, a.mat[0].slots};
  uint32_t begin = 0;
#pragma unroll
  for (uint32_t k = 1; k < (uint32_t)kGemmMaxGroup; ++k)
    if (k < a.n_mats && tile >= a.mat[k].tile_begin) {
      t.base = a.mat[k].base;
      t.y = a.mat[k].y;
      t.d_out = a.mat[k].d_out;
      t.stride = a.mat[k].stride;
      t.slots = a.mat[k].slots;
      begin = a.mat[k].tile_begin;
    }
  t.row0 = (tile - begin) * rows_per_tile;
  return t;
}
__device__ __forceinline__ void store_y(void* y, size_t at, float v, uint32_t f32) {
  if (f32) reinterpret_cast<float*>(y)[at] = v;
  else reinterpret_cast<__half*>(y)[at] = __float2half_rn(v);
}

// A lane offset, made opaque where it is used: widened to 64 bits outside a loop it could no longer be the offset operand
// of a load with a scalar base.
__device__ __forceinline__ uint32_t lane_offset(uint32_t v) {
  asm volatile("" : "+v"(v));
  return v;
}

// ---- up to 64 activation rows -----------------------------------------------------------------------
// What bounds it: bytes in flight and the chain of one launch (4096 x 4096 is 9 MB of tiles); the matrix cores have next
// to nothing to do.  So a workgroup of sixteen wavefronts takes RG x 16 weight rows and all of the batch, the wavefronts
// share the row out (wavefront w: four blocks from 4 w on, then from 4 (w + 16) on, ...), every load of a step is in
// flight while the step before is multiplied, and the sixteen partial sums meet in LDS: no workspace, no second kernel.
// RG = 1, MT = 1: up to 16 rows of activations; RG = 2, MT = 4: up to 64 (two row groups share the activation
// fragments, whose way from L2 would bind otherwise).
// Of few rows the octets are read from the rows themselves (gemm_direct in llvq_hip.hip has the rule, and both sides' times).
// 2560 x 2560 at 5 rows: 35.9 -> 10.4 us (6.7 -> 4.7 with that, between the native calls); rotated q, k, v of 2560 columns at 64 rows, rotation included: 58.1 -> 21.7 us
// (before: codes unranked in the product, partial sums through memory).
// PAIR: both terms of the weights (dequant_octet_pair), 32 columns to a product sum that starts from zero, those added in
// f64; RG = 1 always, two row groups would not fit the registers.  4097 columns, 1024 rows by 64: 16 -> 14 us (twice the
// workgroups), 5000 by 33: 15 -> 22 us.
template <int RG, int MT, bool PAIR>
__global__ __launch_bounds__(1024) void gemm_tiles_kernel(GemmArgs a) {
  extern __shared__ __align__(16) uint8_t smem[];
  touch_args(a);
  constexpr uint32_t kRows = RG * 16, kCols = MT * 16;
  float* part = reinterpret_cast<float*>(smem);           // [16 wavefronts][RG][MT][64 lanes][4]
  float* tw = part + 16 * RG * MT * 256;                  // [kRows][24] tail weights
  float* scale_s = tw + kRows * 24;
  float* tx = scale_s + kRows;                            // [kCols][24] tail activations
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t nb = a.nb, n_quads = (nb + 3u) >> 2;
  const GemmTile t = gemm_tile_at(a, blockIdx.x, kRows);
  const uint32_t stride = t.stride, head = tile_head_bytes(a.tail_w);
  const uint8_t* recs = t.base + kTileTableBytes + (size_t)(t.row0 / kTileRows) * stride;
  const uint32_t last_rec = tile_count(t.d_out) - 1u - t.row0 / kTileRows;  // tiles past the matrix's last repeat it
  const uint32_t g = lane >> 4, m16 = lane & 15u;  // the lane's block of a unit, and its row
  const float entry = __uint_as_float(scale_table(t.base, lane));
  const uint32_t d_off = head + (m16 & 7u) * 16u + ((m16 >> 3) * 2u + (g >> 1)) * 128u + (g & 1u) * 8u;
  const uint32_t m_off = head + (m16 & 7u) * 16u + 512u + (m16 >> 3) * 8u;
  const uint32_t x_row = MT == 1 ? min(m16, a.xs_last) * a.xs_row : m16 * 16u, x_off = x_row + g * a.xs_block;

  struct Words { u32x2_t d, m; } W[RG];
  u32x4_t X[3][MT];
  auto load_w = [&](uint32_t q, bool live) {
    const uint32_t keep = live ? 0xFFFFFFFFu : 0u;
#pragma unroll
    for (uint32_t k = 0; k < (uint32_t)RG; ++k) {
      const uint8_t* p = uniform_global(recs + (size_t)min(k, last_rec) * stride + ((q * kUnitBytes) & keep));
      W[k].d = *reinterpret_cast<const u32x2_t*>(p + lane_offset(d_off & keep));
      W[k].m = *reinterpret_cast<const u32x2_t*>(p + lane_offset(m_off & keep));
    }
  };
  auto load_x = [&](uint32_t j, uint32_t q, bool live) {
    const uint32_t keep = live ? 0xFFFFFFFFu : 0u;
    const uint8_t* p = uniform_global(a.xs + (((size_t)q * a.xs_unit + j * a.xs_octet) & (size_t)(int64_t)(int32_t)keep));
    uint32_t off = x_off;
    if (MT == 1 && 4u * q + 4u > nb) off = x_row + min(g, nb - 1u - min(4u * q, nb - 1u)) * a.xs_block;  // (in the last unit: a block that is there)
    off = lane_offset(off & keep);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const HalfOctet o = *reinterpret_cast<const HalfOctet*>(p + off + (uint32_t)mt * 256u);
      X[j][mt] = u32x4_t{o.w[0], o.w[1], o.w[2], o.w[3]};
    }
  };
  // The row scales and the tail's operands, needed at the end: asked for first.
  const uint32_t op_row = tid % kRows, op_col = tid / kRows;  // column 24: the row's scale
  float op_w = 0.f;
  uint32_t op_x[2] = {};
  {
    const uint8_t* rec = recs + (size_t)min(op_row / kTileRows, last_rec) * stride;
    op_w = reinterpret_cast<const float*>(rec)[op_col < a.tail_w ? tail_at(op_row & 15u, op_col, a.tail_w) : op_row & 15u];
    if (a.tail_w) {
#pragma unroll
      for (uint32_t i = 0; i < 2; ++i) {
        const uint32_t k = tid + i * 1024u, m = k / 24u, c = k - m * 24u;
        op_x[i] = reinterpret_cast<const uint16_t*>(a.x)[(size_t)min(m, a.M - 1u) * a.ldx + nb * kDim + min(c, a.tail_w - 1u)];
      }
    }
  }
  // the tiles' lists of escapes, 32 lanes each
  u32x4_t listed = {};
  if (t.slots && (lane >> 5) < (uint32_t)RG)
    listed = *reinterpret_cast<const u32x4_t*>(recs + (size_t)min(lane >> 5, last_rec) * stride + stride - (t.slots - min(lane & 31u, t.slots - 1u)) * 16u);
  if ((lane & 31u) >= t.slots) listed.w = 0u;
  uint32_t q = wave;
  load_w(q, q < n_quads);
#pragma unroll
  for (uint32_t j = 0; j < 3; ++j) load_x(j, q, q < n_quads);
  // (What needs none of these stands here, and the columns of the tail are found by a division by 24, not by their number: between the
  // last of these loads and the loop every instruction of a SIMD's four wavefronts counts.  1000 x 2000 at 33 rows 11.15 -> 10.9 us,
  // 12288 x 4099 at 9 16.3 -> 15.6, 12288 x 4096 at 64 26.3 -> 25.9.)
  typedef double sum4_t __attribute__((ext_vector_type(4)));
  typename std::conditional<PAIR, sum4_t, acc4_t>::type acc[RG][MT];
#pragma unroll
  for (int k = 0; k < RG; ++k)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[k][mt] = 0;
#pragma unroll
  for (int k = 0; k < RG; ++k)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) asm volatile("" : "+v"(acc[k][mt]));
  __builtin_amdgcn_sched_barrier(0);
  const float unit = table_unit(entry);
  const uint32_t table = split_table(entry, unit);
  const bool read_codes = t.slots == 0u || __builtin_amdgcn_ballot_w64(listed.w == ~0u) != 0u;
  // (before the loop: the registers are needed there)
  if (op_col < a.tail_w) tw[op_row * 24u + op_col] = op_w;
  else if (op_col == 24u) scale_s[op_row] = op_w * unit;
  if (a.tail_w) {
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
      const uint32_t k = tid + i * 1024u;
      if (k < kCols * 24u) tx[k] = __half2float(__ushort_as_half((unsigned short)op_x[i]));
    }
  }
  for (; q < n_quads; q += 16u) {
    if (MT == 1 && 4u * q + 4u > nb) {  // octets of blocks that are not there are zero, and their weights are
      const uint32_t there = 4u * q + g < nb ? 0xFFFFFFFFu : 0u;
#pragma unroll
      for (uint32_t j = 0; j < 3; ++j) X[j][0] &= there;
    }
    const uint32_t qn = q + 16u;
    const bool live = qn < n_quads;
    BlockScale s[RG];
    GemmBlock b[RG];
#pragma unroll
    for (int k = 0; k < RG; ++k) {
      b[k] = gemm_block(W[k].d.x, W[k].d.y, W[k].m.x, W[k].m.y, g, table);
      // Escapes from the tiles' lists, where those count: 30 instructions and not 120 (what the codes take here, block_escape with them).  (One of twenty units has one, but so
      // has nearly every workgroup, and waits for it: 0.1 us of 6.5.)
      if (__builtin_amdgcn_ballot_w64(is_escape(b[k]))) {
        if (read_codes) {
          gemm_escape(b[k], table);
        } else {
          for (uint64_t left = __builtin_amdgcn_ballot_w64(((listed.w >> 11) & 0x1FFFFu) == q && (lane >> 5) == (uint32_t)k && listed.w != 0u); left; left &= left - 1u) {
            const uint32_t of = (uint32_t)__builtin_ctzll(left), key = (uint32_t)__builtin_amdgcn_readlane((int)listed.w, of);
            gemm_listed(b[k], listed, of, ((key >> 9) & 3u) * 16u + (key >> 28), lane, table);
          }
        }
      }
      s[k] = block_scale(b[k].win, b[k].parts);
    }
    // a register is asked for again as soon as its contents are used, and not moved from there
    auto next_words = [&]() __attribute__((always_inline)) {
      __builtin_amdgcn_sched_barrier(0);
      load_w(qn, live);
      __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (RG == 1) next_words();
#pragma unroll
    for (uint32_t j = 0; j < 3; ++j) {
      half8_t w[RG], w2[RG];
#pragma unroll
      for (int k = 0; k < RG; ++k) {
        const uint32_t nibbles = b[k].w[j];
        if constexpr (PAIR) {
          const WeightPair p = dequant_octet_pair(nibbles, s[k]);
          w[k] = p.hi;
          w2[k] = p.lo;
        } else {
          w[k] = dequant_octet(nibbles, s[k]);
        }
      }
      if (RG != 1 && j == 0u) next_words();  // (two groups' words have no registers beside the blocks' octets before)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int k = 0; k < RG; ++k) {
          if constexpr (PAIR) {
            const acc4_t lo = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, X[j][mt]), w2[k], acc4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            const acc4_t one = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, X[j][mt]), w[k], lo, 0, 0, 0);
            acc[k][mt] += __builtin_convertvector(one, sum4_t);
          } else {
            acc[k][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, X[j][mt]), w[k], acc[k][mt], 0, 0, 0);
          }
        }
      __builtin_amdgcn_sched_barrier(0);
      load_x(j, qn, live);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // (From the lane's number anew: nothing of this may occupy registers during the loop.)
  const uint32_t tid_e = lane_offset(threadIdx.x), lane_e = tid_e & 63u;
  // of a fragment a lane's row is a weight row (lane % 16) and its four elements activation rows 4 (lane / 16) + e
#pragma unroll
  for (int k = 0; k < RG; ++k)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      *reinterpret_cast<acc4_t*>(part + (((wave * RG + k) * MT + mt) * 64u + lane_e) * 4u) = __builtin_convertvector(acc[k][mt], acc4_t);
  __syncthreads();
  // A lane takes one or two neighbours of a fragment's four, a row of sixteen lanes' worth of weight rows side by side: the 32 lanes that LDS serves
  // together read 256 bytes that lie together, and what is stored together are the tile's rows.  (By output, a row after the other, the reads
  // were sixteen bytes apart, four to a bank: half of the kernel's LDS cycles.  Rotated q, k, v of 4096 columns at 64 rows 16.8 -> 15.25 us, rotation
  // included, 2560 x 9728 at 60 22.8 -> 21.6, 12288 x 4096 at 33 23.3 -> 22.15; up to 32 rows the same, or 1 % faster.)
  constexpr uint32_t kPer = kRows * kCols > 1024u ? 2u : 1u, kPieces = 4u / kPer;
  for (uint32_t o = tid_e; o < kRows * kCols / kPer; o += 1024u) {
    const uint32_t e = o % kPieces * kPer, row16 = o / kPieces % 16u, above = o / (kPieces * 16u);
    const uint32_t k = above % RG, l4 = above / RG % 4u, mt = above / (RG * 4u);
    const float* p = part + ((k * MT + mt) * 64u + l4 * 16u + row16) * 4u + e;
    typedef typename std::conditional<PAIR, double, float>::type sum_t;
    sum_t s[kPer] = {};
#pragma unroll
    for (uint32_t w = 0; w < 16; ++w)
#pragma unroll
      for (uint32_t i = 0; i < kPer; ++i) s[i] += (sum_t)p[w * RG * MT * 256 + i];
    const uint32_t row = k * 16u + row16;
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) {
      const uint32_t m = mt * 16u + l4 * 4u + e + i;
      if (m >= a.M || t.row0 + row >= t.d_out) continue;
      float tl = 0.f;
      for (uint32_t c = 0; c < a.tail_w; ++c) tl = fmaf(tw[row * 24u + c], tx[m * 24u + c], tl);
      store_y(t.y, (size_t)m * t.d_out + t.row0 + row, fmaf((float)s[i], scale_s[row], tl), a.y_f32);
    }
  }
}
template <int RG, int MT>
__host__ constexpr size_t gemm_small_lds() { return (size_t)(16 * RG * MT * 256 + RG * 16 * 25 + MT * 16 * 24) * 4; }
static_assert(gemm_small_lds<2, 4>() <= 160 * 1024, "partial sums of sixteen wavefronts fit a CU's LDS");

// A fragment's results on their way to y, ld values from an activation row's to the next: a lane has sixteen of one activation row (weight rows
// 8 g + 4 h .. + 3, g < 4).  Where y and its rows lie on 16-byte boundaries they go through LDS (`turn`, a wavefront's own), so that a store
// takes whole lines, eight lanes to a row: as the lanes have them a store is sixteen bytes each of 32 rows, and the partial results of a 4B layer's
// products of 500 rows took 2 us longer each; f32 results without splits 12000 x 1000 at 600 rows 32.1 us and 30.6 so, 13000 x 408 at 600 21.9 and 20.6,
// 12288 x 4096 at 512 and others of long rows the same.  Else one by one.
// wave_lds_order: what a wavefront has read of LDS has come before it writes there, and the other way round.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
template <int RF>
__host__ __device__ constexpr uint32_t turn_bytes() { return 32u * (64u * RF + 16u) > 32u * 144u ? 32u * (64u * RF + 16u) : 32u * 144u; }
// What a store of fragment (k, c) needs: the first activation row of c, rows there are, the wavefront's first weight row in a row of y.
struct StoreAt {
  void* y;
  size_t ld;
  uint32_t m, m_end, row, d_out;  // (d_out: of rows from `row` on, those below it are stored)
  uint8_t* turn;
};
template <int RF>
struct StoreF32 {
  static __device__ __forceinline__ void store(const StoreAt& t, uint32_t k, uint32_t lane, const acc16_t& v) {
    const uint32_t l32 = lane & 31u, h = lane >> 5, r = lane >> 3, q = lane & 7u;
    float* const to = reinterpret_cast<float*>(t.turn) + l32 * 36u + h * 4u;
    wave_lds_order();
#pragma unroll
    for (int g = 0; g < 4; ++g) *reinterpret_cast<float4*>(to + g * 8) = make_float4(v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]);
    wave_lds_order();
#pragma unroll
    for (uint32_t i = 0; i < 4u; ++i) {
      const float4 o = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(t.turn) + (i * 8u + r) * 36u + q * 4u);
      const uint32_t m = t.m + i * 8u + r;
      if (m < t.m_end) *reinterpret_cast<float4*>(reinterpret_cast<float*>(t.y) + (size_t)m * t.ld + t.row + k * 32u + q * 4u) = o;
    }
  }
};
// As the lanes have them, the halves exchanged so that a lane has eight rows in a row: binary16 results with PAIR, whose fragments are not converted and
// stored beside each other's products, and wait for LDS by themselves.  (9728 x 700 at 350 rows 40.0 us through LDS, 39.5 so, at 90 38.8 and 38.2, 12288 x 4099 at 500 175.7
// and 175.1, other shapes the same; f32 results take a whole microsecond more: 1000 x 409 at 600 29.9 and 30.8.)
struct StoreF16Direct {
  static __device__ __forceinline__ void store(const StoreAt& t, uint32_t k, uint32_t lane, const acc16_t& v) {
    const uint32_t m = t.m + (lane & 31u), h = lane >> 5;
    if (m >= t.m_end) return;
    uint32_t p[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) p[i] = __builtin_bit_cast(uint32_t, half2_t{(_Float16)v[2 * i], (_Float16)v[2 * i + 1]});
    _Float16* out = reinterpret_cast<_Float16*>(t.y) + (size_t)m * t.ld + t.row + k * 32u;
#pragma unroll
    for (int g = 0; g < 4; g += 2) {
      const auto a = __builtin_amdgcn_permlane32_swap(p[2 * g], p[2 * g + 2], false, false);
      const auto b = __builtin_amdgcn_permlane32_swap(p[2 * g + 1], p[2 * g + 3], false, false);
      *reinterpret_cast<u32x4_t*>(out + (g + h) * 8u) = u32x4_t{a[0], b[0], a[1], b[1]};
    }
  }
};
template <int RF>
struct StoreF16 {  // (all fragments of an activation row with the last of them)
  static __device__ __forceinline__ void store(const StoreAt& t, uint32_t k, uint32_t lane, const acc16_t& v) {
    constexpr uint32_t kPitch = 64u * RF + 16u, kPieces = 4u * RF;  // bytes of a row in LDS, and 16-byte pieces of it
    const uint32_t l32 = lane & 31u, h = lane >> 5;
    if (k == 0u) wave_lds_order();
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<u32x2_t*>(t.turn + l32 * kPitch + k * 64u + (uint32_t)g * 16u + h * 8u) =
          u32x2_t{__builtin_bit_cast(uint32_t, half2_t{(_Float16)v[4 * g], (_Float16)v[4 * g + 1]}), __builtin_bit_cast(uint32_t, half2_t{(_Float16)v[4 * g + 2], (_Float16)v[4 * g + 3]})};
    if (k + 1u != (uint32_t)RF) return;
    wave_lds_order();
#pragma unroll
    for (uint32_t i = 0; i < 2u * RF; ++i) {
      const uint32_t p = i * 64u + lane, r = p / kPieces, q = p - r * kPieces, m = t.m + r;
      const u32x4_t o = *reinterpret_cast<const u32x4_t*>(t.turn + r * kPitch + q * 16u);
      if (m < t.m_end) *reinterpret_cast<u32x4_t*>(reinterpret_cast<_Float16*>(t.y) + (size_t)m * t.ld + t.row + q * 8u) = o;
    }
  }
};
template <typename Y>
struct StoreEach {
  static __device__ __forceinline__ void store(const StoreAt& t, uint32_t k, uint32_t lane, const acc16_t& v) {
    const uint32_t m = t.m + (lane & 31u);
    Y* out = reinterpret_cast<Y*>(t.y) + (size_t)m * t.ld;
    if (m >= t.m_end) return;
#pragma unroll
    for (uint32_t e = 0; e < 16; ++e) {
      const uint32_t r = t.row + k * 32u + 8u * (e >> 2) + 4u * (lane >> 5) + (e & 3u);
      if (r < t.d_out) out[r] = (Y)v[e];
    }
  }
};

// ---- more activation rows ----------------------------------------------------------------------------
// What bounds it: a wavefront with a SIMD to itself issues an instruction every four cycles at the most, and a step has 270
// beside its 48 products of 32 cycles (RF = 2, CF = 8), not all of which fall between those; what it waits for, nothing
// else fills.  Then power: a loop of nothing but products on random numbers reaches 1650 TFLOP/s, at three quarters of the clock.
// So what counts is the number of instructions, and where they stand.  A workgroup of four wavefronts takes 128 RF weight rows by 32 CF
// activation rows; a wavefront unpacks 32 RF rows (RF fragments) against all of the activation rows (CF fragments).  CF = 8, RF = 2:
// 256 accumulators, half the unpacking for a product (1.21 us a step).  RF = 3, CF = 4 (gemm_tall_kernel): three quarters of
// that tile, half as much unpacking again for a product (1.12 us), for matrices whose tiles of the other leave CUs idle: gate and up of
// an 8B layer at 512 rows are 192 of those and 256 of these, 112.6 and 110.2 us; of a 4B layer at 500 rows 152 and 204, 78 and 73 us.
// CF = 4, RF = 2: two workgroups on a CU (0.76 us a step each) or one (0.80), for batches and matrices that fill neither.
// Octets and tiles go from memory to LDS without passing through registers, two to three steps of 48 columns (two
// blocks) ahead.
// PAIR: both terms of the weights against the same activations, 2 CF more products a round; every step's sums go to f64
// ones (512 registers: CF = 4, RF = 2 and one wavefront on a SIMD).  2.5 us a step, of which moving those sums in and out of the
// accumulator registers is most; 13000 x 5121 at 600 rows 115 -> 252 us.  (With arithmetic for the look-ups that loop was as fast over
// 13 bytes a block, 250 us; small products took 1.5 to 2.5 us less, without lists of escapes to wait for and read: 4096 x 4097 at
// 130 rows 45.3 us, 47.9 now.)
// Launches with too few tiles to fill the chip split the columns (`splits`): partial results go to the workspace and are added in order by
// gemm_sum_kernel or by the launch that takes them (GemmSums), with PAIR partial sums by gemm_reduce_pair_kernel; otherwise the tile is finished here.
// Gate and up of an 8B layer (24576 x 4096) at 512 rows: 116 -> 110 us, 935 TFLOP/s (116 with 17 binary16 operations an octet and
// 13 bytes a block; 121 with those and ten); a plain f16 product of that size by the vendor's library runs at 1159 on this card.
template <int RF>
__host__ __device__ constexpr uint32_t gemm_wide_rows() { return 128u * RF; }
template <int RF>
__host__ __device__ constexpr uint32_t gemm_wide_tiles() { return 2u * RF * 384u; }  // {d0, d1} of two blocks of a wavefront's tiles, 256 bytes each; their {s, meta}
constexpr uint32_t kWideDepth = 4;         // LDS buffers, a step each
template <int CF>
__host__ __device__ constexpr uint32_t gemm_wide_x_bytes() { return 6u * 32u * CF * 16u; }
template <int RF, int CF>
__host__ __device__ constexpr uint32_t gemm_wide_buf() { return gemm_wide_x_bytes<CF>() + 4u * gemm_wide_tiles<RF>(); }
template <int RF, int CF, bool PAIR>
__host__ constexpr size_t gemm_wide_lds() {
  return (PAIR ? 2u * kValueBytes + 256u * sizeof(ValueBlock) : kValueBytes) + (size_t)kWideDepth * gemm_wide_buf<RF, CF>();
}
static_assert(2 * gemm_wide_lds<2, 4, false>() <= 160 * 1024 && gemm_wide_lds<2, 8, false>() <= 160 * 1024 && gemm_wide_lds<3, 4, false>() <= 160 * 1024 &&
              gemm_wide_lds<2, 4, true>() <= 160 * 1024, "two workgroups of the first, one of the others on a CU");
// A wavefront's lists of escapes as they come, and those of its split with the tile's number, where the last buffer will be.
template <int RF>
__host__ __device__ constexpr uint32_t gemm_wide_lists() { return 2u * RF * kMaxListSlots * 16u; }
static_assert(gemm_wide_buf<2, 4>() >= 4u * (gemm_wide_lists<2>() + 64u * 20u) && gemm_wide_buf<3, 4>() >= 4u * (gemm_wide_lists<3>() + 64u * 20u), "the lists fit a buffer");
template <int RF, int CF>
__host__ constexpr bool gemm_wide_tail_fits() { return kWideDepth * gemm_wide_buf<RF, CF>() >= ((gemm_wide_rows<RF>() + 32u * CF) * kDim + gemm_wide_rows<RF>()) * 4u + 4u * turn_bytes<RF>(); }
static_assert(gemm_wide_tail_fits<2, 4>() && gemm_wide_tail_fits<2, 8>() && gemm_wide_tail_fits<3, 4>(), "what the end has in LDS fits the buffers");

// 16 bytes per lane from base + offset to LDS, lane after lane from `lds` on.  In assembly because the compiler, which
// cannot tell the buffers apart, would have every read of LDS wait for all of these; the counting is done by hand
// (wide_wait), and there are no other loads in flight where it is.  M0, where the place in LDS goes, is an operand: the
// compiler writes it, and knows that it did.
__device__ __forceinline__ void load_to_lds(uint32_t lds, uint32_t offset, const uint8_t* base) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "{m0}"(lds), "v"(offset), "s"(base) : "memory");
}
// Three of these, 1024 bytes apart in LDS; and two or three, the last by the first LANES lanes only, 512 bytes for each 16 of
// them behind the first.  An instruction's offset counts in LDS and in memory: the lanes' offsets have it taken off, and
// kLoadBias put on, which the base is without.  (All lanes are active where these are used; a condition would be a branch,
// and what is in front of it and behind it could not be moved across.)
constexpr uint32_t kLoadBias = 4096;
__device__ __forceinline__ void load_three_to_lds(uint32_t lds, uint32_t o0, uint32_t o1, uint32_t o2, const uint8_t* base) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %4\n\tglobal_load_lds_dwordx4 %2, %4 offset:1024\n\tglobal_load_lds_dwordx4 %3, %4 offset:2048"
               : : "{m0}"(lds), "v"(o0), "v"(o1), "v"(o2), "s"(base) : "memory");
}
template <int RF>
__device__ __forceinline__ void load_tiles_to_lds(uint32_t lds, const uint32_t (&o)[RF], const uint8_t* d, const uint8_t* m) {
  if constexpr (RF == 2)
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %3\n\ts_mov_b32 exec_hi, 0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %4 offset:1024\n\ts_mov_b32 exec_hi, -1"
                 : : "{m0}"(lds), "v"(o[0]), "v"(o[1]), "s"(d), "s"(m) : "memory");
  else
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %4\n\ts_mov_b32 exec_hi, 0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %4 offset:1024\n\t"
                 "s_mov_b32 exec_hi, 0xffff\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %3, %5 offset:1536\n\ts_mov_b32 exec_hi, -1"
                 : : "{m0}"(lds), "v"(o[0]), "v"(o[1]), "v"(o[2]), "s"(d), "s"(m) : "memory");
}
// A barrier by itself: what LDS reads of a wavefront are in flight it has not begun to need, and what they read stays.
__device__ __forceinline__ void wide_barrier() {
  asm volatile("" : : : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" : : : "memory");
}
template <int N>
__device__ __forceinline__ void wide_wait() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }

template <int RF, int CF, bool PAIR>
__device__ __forceinline__ void wide_product(const GemmArgs& a) {
  constexpr uint32_t kCols = 32u * CF, kRows = gemm_wide_rows<RF>(), kBuf = gemm_wide_buf<RF, CF>();
  constexpr uint32_t kTileBytes = gemm_wide_tiles<RF>(), kTerms = PAIR ? 2u : 1u;
  constexpr int kLoadsX = 3 * CF / 4, kLoadsW = RF, kLoads = kLoadsX + kLoadsW;  // of a wavefront in a step
  static_assert(RF == 2 || RF == 3, "a wavefront's tiles: four, and two more");
  // (aligned so that an entry's address is its offset or'ed in)
  extern __shared__ __align__(4096) uint8_t wide_smem[];  // weights of the meta bytes, [kWideDepth] x { [6 octets][kCols] 16 bytes, tiles }
  uint8_t* const smem = wide_smem + kTerms * kValueBytes;
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t l32 = lane & 31u, h = lane >> 5;
  // tiles of one row group are neighbours in the grid: they read the same weights
  const uint32_t mt = blockIdx.x % a.m_tiles, rest = blockIdx.x / a.m_tiles;
  const uint32_t tile = rest % a.n_tiles, split = rest / a.n_tiles;
  const GemmTile t = gemm_tile_at(a, tile, kRows);
  const uint32_t nb = a.nb, stride = t.stride, head = tile_head_bytes(a.tail_w);
  const uint32_t row0 = t.row0 + wave * (32u * RF);     // this wavefront's first row
  const uint32_t n_rec = tile_count(t.d_out);
  const float entry_f = __uint_as_float(scale_table(t.base, lane));
  const uint32_t n_steps = (nb + 1u) >> 1;
  const uint32_t s0 = split * a.steps_per_split, s1 = min(s0 + a.steps_per_split, n_steps);
  const uint8_t* rec0 = uniform_global(t.base + kTileTableBytes + (size_t)(t.row0 / kTileRows) * stride);
  // tiles past the matrix's last repeat it: their rows are not stored
  auto record = [&](uint32_t row) __attribute__((always_inline)) { return (min(row / kTileRows, n_rec - 1u) - t.row0 / kTileRows) * stride; };
  // a load of tiles takes the lines of two blocks, of four or two tiles, or those of {s, meta} of all of this wavefront's; a load of octets 64 activation rows of one
  uint32_t w_off[kLoadsW], x_off[kLoadsX];
  w_off[0] = record(row0 + (lane >> 4) * 16u) + head + ((lane >> 3) & 1u) * 256u + (lane & 7u) * 16u;
  if constexpr (RF == 3) w_off[1] = record(row0 + (4u + ((lane >> 4) & 1u)) * 16u) + head + ((lane >> 3) & 1u) * 256u + (lane & 7u) * 16u;
  w_off[RF - 1] = record(row0 + min(lane >> 3, 2u * RF - 1u) * 16u) + head + 512u + (lane & 7u) * 16u;
#pragma unroll
  for (uint32_t i = 0; i < (uint32_t)kLoadsX; ++i) {
    const uint32_t k = wave * kLoadsX + i, o = k / (kCols / 64u), m = k % (kCols / 64u) * 64u + lane;
    x_off[i] = (o * a.m_pad + mt * kCols + m) * 16u + kLoadBias - i % 3u * 1024u;
  }
  w_off[0] += kLoadBias;
  if constexpr (RF == 3) w_off[1] += kLoadBias - 1024u;
  w_off[RF - 1] += kLoadBias - 512u * RF;
  const uint32_t x_step = 6u * a.m_pad * 16u, values_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)wide_smem;
  const uint32_t smem_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  // where the steps come from, one after the other; steps past the last are loaded too, so that the count of loads in flight is
  // always the same
  uint32_t from_left = s1 - 1u - s0, from_odd = (s0 & 1u) * 128u;
  const uint8_t* from_x = uniform_global(reinterpret_cast<const uint8_t*>(a.xt) + (size_t)s0 * x_step - kLoadBias);
  const uint8_t* from_unit = uniform_global(rec0 + (size_t)(s0 >> 1) * kUnitBytes - kLoadBias);
  auto load_x = [&](uint32_t buffer, uint32_t i) __attribute__((always_inline)) {
    load_three_to_lds(smem_at + buffer + (wave * kLoadsX + 3u * i) * 1024u, x_off[3 * i], x_off[3 * i + 1], x_off[3 * i + 2], from_x);
  };
  auto load_w = [&](uint32_t buffer) __attribute__((always_inline)) {
    load_tiles_to_lds<RF>(smem_at + buffer + gemm_wide_x_bytes<CF>() + wave * kTileBytes, w_off, from_unit + from_odd, from_unit);
  };
  auto to_next_step = [&](uint32_t part) __attribute__((always_inline)) {  // (in three: between two products there is room for no more)
    if (part == 0u) from_x += from_left ? x_step : 0u;
    if (part == 1u) from_unit += from_left && from_odd ? kUnitBytes : 0u;
    if (part == 2u) from_odd ^= from_left ? 128u : 0u;
    if (part == 2u) from_left -= from_left ? 1u : 0u;
  };
  auto load = [&](uint32_t buffer) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)kLoadsX / 3u; ++i) load_x(buffer, i);
    load_w(buffer);
#pragma unroll
    for (uint32_t part = 0; part < 3u; ++part) to_next_step(part);
  };
  // What the end needs from the tiles' heads: the row scales, a lane's own, and (so that they are in L2 then) the lines of the tail columns.
  // (Asked for there they were two to three waits for memory in every workgroup.  With that, operands a fragment ahead and stores of whole lines the
  // end takes 6.5 us of a tile of 384 rows and sixteen tail columns where it took 11: 12288 + 12288 x 4096 at 512 rows 111.3 -> 108.8 us.)
  float my_scale[(RF + 1) / 2];
#pragma unroll
  for (uint32_t i = 0; i < (uint32_t)(RF + 1) / 2u; ++i) {
    const uint32_t row = row0 + min(i * 64u + lane, 32u * RF - 1u);
    my_scale[i] = reinterpret_cast<const float*>(rec0 + record(row))[row & 15u];
  }
  uint32_t touched = 0;
  if (a.tail_w) touched = *reinterpret_cast<const uint32_t*>(rec0 + record(t.row0 + min(tid / 9u, kRows / 16u - 1u) * 16u) + min(tid % 9u, (head >> 7) - 1u) * 128u);
  acc16_t acc[RF][CF];
  double sum[PAIR ? RF : 1][PAIR ? CF : 1][16];  // of the steps, with PAIR
  const float unit = table_unit(entry_f), table = entry_f * (1.f / unit);
  const auto scale_of = [&](uint32_t meta) __attribute__((always_inline)) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_ds_bpermute((int)meta, (int)__float_as_uint(table)));
  };
  // One step: three rounds of 2 CF products (an octet of columns of two blocks), in whose shadow everything else runs: the
  // weights of the round after are unpacked, two at a time, and its activations read into the registers of those just used.
  // In the middle of the first every wavefront waits for its loads of the next step and then for the others; the step before
  // has been read by then, and its buffer is filled again during the second, which also reads the next step's tiles and puts
  // their octets together.
  // w: the next round's weights, [1] what the rounding took of them.  B: the block they are unpacked from, T: the weights it
  // picks from.  (With PAIR the sums leave no registers for the next one's beside them.)
  struct Block { uint32_t w[3], meta; };
  u32x4_t w[kTerms][RF] = {}, T[RF][kTerms], Tn[RF];
  half8_t x[CF];
  Block B[RF], Bn[RF];
  u32x2_t words[RF], metas[RF];
  const auto unpack_part = [&](auto octet, uint32_t idx, ValuePick (&pick)[kTerms], u32x4_t (&to)[kTerms][RF]) __attribute__((always_inline)) {
    constexpr uint32_t j = decltype(octet)::value;
    const uint32_t k = idx >> 2;
#pragma unroll
    for (uint32_t p = 0; p < kTerms; ++p) pick_values<j == 2u ? 0u : 1u>(B[k].w[j], T[k][p], idx & 3u, pick[p], to[p][k]);
  };
  const uint32_t x_at = (h * 3u * kCols + l32) * 16u;
  const uint32_t wave_at = gemm_wide_x_bytes<CF>() + wave * kTileBytes;
  const uint32_t w_at = wave_at + (l32 >> 4) * 256u + ((l32 >> 3) & 1u) * 128u + (l32 & 7u) * 16u + h * 8u;
  const uint32_t meta_at = wave_at + 512u * RF + (l32 >> 4) * 128u + (l32 & 7u) * 16u + ((l32 >> 3) & 1u) * 8u;
  auto read_x_part = [&](uint32_t buffer, uint32_t j, uint32_t c) __attribute__((always_inline)) {
    x[c] = __builtin_bit_cast(half8_t, (reinterpret_cast<const u32x4_t*>(smem + (buffer + x_at)) + j * kCols)[c * 32u]);
  };
  auto read_x = [&](uint32_t buffer, uint32_t j) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t c = 0; c < (uint32_t)CF; ++c) read_x_part(buffer, j, c);
  };
  auto read_w = [&](uint32_t buffer) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t k = 0; k < (uint32_t)RF; ++k) {
      words[k] = *reinterpret_cast<const u32x2_t*>(smem + (buffer + w_at) + k * 512u);
      metas[k] = *reinterpret_cast<const u32x2_t*>(smem + (buffer + meta_at) + k * 256u);
    }
  };
  // the lane's block of a step is 2 (step & 1) + h of its unit: by how much its bits of the dwords are turned
  uint32_t turn_s = (2u * (s0 & 1u) + h - 2u) & 31u, turn_m = (8u * (2u * (s0 & 1u) + h) - 4u) & 31u;
  auto read_values = [&](uint32_t k) __attribute__((always_inline)) {
    const uint32_t meta = __builtin_amdgcn_alignbit(metas[k].y, metas[k].y, turn_m);
    Bn[k].meta = meta;
    const uint32_t from = (meta & 0xFF0u) | values_at;
    if constexpr (PAIR) {
#pragma unroll
      for (uint32_t p = 0; p < kTerms; ++p) T[k][p] = *(const __attribute__((address_space(3))) u32x4_t*)(uintptr_t)(from + p * kValueBytes);
    } else {
      Tn[k] = *(const __attribute__((address_space(3))) u32x4_t*)(uintptr_t)from;
    }
  };
  auto assemble = [&](uint32_t k) __attribute__((always_inline)) {
    const uint32_t third = __builtin_amdgcn_alignbit(metas[k].x, metas[k].x, turn_s);  // bit 2 of its three
    Bn[k].w[0] = words[k].x;
    Bn[k].w[1] = words[k].y;
    Bn[k].w[2] = bfi32(0x33333333u, bfi32(0x11111111u, words[k].x, words[k].y << 1), third);
  };
  auto turn = [&]() __attribute__((always_inline)) {
    turn_s ^= 30u;
    turn_m ^= 16u;
  };
  // Escapes (block_code.h): a lane keeps one of this wavefront's, from its tiles' lists, as a block that picks from weights of
  // its own, and puts it in the place of the code in LDS once that has come; where there is none in a step that is one
  // comparison.  (Their codes read as they came, in one of ten steps and so in a third of a workgroup's, cost
  // 6 to 10 % of the time, every wavefront waiting for the slowest; weights exchanged where they are unpacked, 7 %.)
  // at: {d0, d1} and {s, meta} in the wavefront's tiles, 12 bits each, and the block of its unit.  (With PAIR it waits in LDS.)
  uint32_t own_step = ~0u;
  ValueBlock own{};
  ValueBlock* const own_lds = reinterpret_cast<ValueBlock*>(smem + kWideDepth * kBuf) + tid;
  // What no lane keeps, because it is past 64 or of a list that does not count, is read from its code, and left_steps says in which
  // steps that can be: there the codes that no lane keeps go to a lane each, which reads it, some 250 instructions, and puts it in
  // its own place likewise.  Steps with more than kWaveValues are for every lane to read its blocks, 200 instructions a fragment
  // that has one.  Gate and up of a 4B layer at 512 rows, 81 us: with one tile whose list does not count 101 -> 87 us, with one
  // escape in a hundred blocks 191 -> 124 us; 17408 x 17408 with the escapes of uniform codes, past 64 in one wavefront of six,
  // 500 -> 360 us, without any 350 (before: from the first of these on every step was read by every lane, 500 instructions a fragment).
  uint32_t left_steps = t.slots ? 0u : ~0u;  // bit s of the 2048 in the lanes: step s0 + s (+ 2048 ...) may have one of those
  const uint32_t my_tiles = gemm_wide_x_bytes<CF>() + wave * kTileBytes;
  const auto tile_place = [&](uint32_t tile_of, uint32_t row, uint32_t blk) __attribute__((always_inline)) {
    return (tile_of * 256u + (row >> 3) * 128u + (row & 7u) * 16u + (blk & 1u) * 8u) | (512u * RF + tile_of * 128u + (row & 7u) * 16u + (row >> 3) * 8u) << 12 | (blk & 3u) << 24;
  };
  const auto code_block = [&](uint32_t (&o)[3], uint32_t meta) __attribute__((always_inline)) {  // (for all lanes: the scales are in all of them)
    const BlockEscape e = block_escape(o, meta);
    o[0] = e.w0;
    const EscapePick p = escape_pick(o, e);
    ValueBlock b{{{}, {}}, o[0] | ((o[2] >> 1) & 0x11111111u), o[1] | ((o[2] >> 2) & 0x11111111u), (o[2] >> 3) & 0x11111111u, 0u};
    const float scale = scale_of(e.slot << 3);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int v = (uint32_t)i == p.index ? p.value : 2 * (i < 4 ? i : i - 8) + (int)e.win - 3;
      value_to(b.t, i, (float)(e.negative ? -v : v) * scale);
    }
    return b;
  };
  // b of the lanes in `there` into the tiles, its weights from place `first` on of the wavefront's sixteen.
  const auto place = [&](const ValueBlock& b, uint64_t there, uint32_t first, uint8_t* tiles) __attribute__((always_inline)) {
    const uint32_t v = kBlockEscape + wave * kWaveValues + first + __builtin_amdgcn_mbcnt_hi((uint32_t)(there >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)there, 0u));
    *reinterpret_cast<u32x2_t*>(tiles + (b.at & 0xFFFu)) = u32x2_t{b.d0, b.d1};
    uint32_t* const meta = reinterpret_cast<uint32_t*>(tiles + ((b.at >> 12) & 0xFFFu));
    const uint32_t k = b.at >> 24;
    __hip_atomic_fetch_and(meta, ~(0x11111111u << k), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    __hip_atomic_fetch_or(meta, b.s << k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    reinterpret_cast<uint8_t*>(meta + 1)[k] = (uint8_t)v;
    reinterpret_cast<u32x4_t*>(wide_smem)[v] = b.t.hi;
    if constexpr (PAIR) reinterpret_cast<u32x4_t*>(wide_smem + kValueBytes)[v] = b.t.lo;
  };
  auto place_escapes = [&](uint32_t s, uint32_t buffer) __attribute__((always_inline)) {
    const uint64_t mine = __builtin_amdgcn_ballot_w64(own_step == s);
    if (PAIR ? mine != 0u : __builtin_expect(mine != 0u, 0)) {
      asm volatile("");  // (a branch of its own: as one condition with the next it is six instructions more in every step)
      if (own_step == s) {
        if constexpr (PAIR) own = *own_lds;
        place(own, mine, 0, smem + buffer + my_tiles);
      }
    }
  };
  const auto some_left = [&](uint32_t s) __attribute__((always_inline)) {
    return s < s1 && ((uint32_t)__builtin_amdgcn_readlane((int)left_steps, ((s - s0) >> 5) & 63u) >> ((s - s0) & 31u) & 1u) != 0u;
  };
  // A step's codes, and those that place_escapes left: placed too (1), for every lane to read its own if there are more than
  // places (2), or none (0).
  uint32_t codes[RF];
  uint64_t left[RF];
  const auto read_codes = [&](uint32_t s, uint32_t buffer) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t k = 0; k < (uint32_t)RF; ++k) codes[k] = (smem + (buffer + meta_at) + k * 256u + 4u)[2u * (s & 1u) + h];
  };
  const auto place_left = [&](uint32_t s, uint32_t buffer) __attribute__((always_inline)) -> uint32_t {
    uint8_t* const tiles = smem + buffer + my_tiles;
#pragma unroll
    for (uint32_t k = 0; k < (uint32_t)RF; ++k) left[k] = __builtin_amdgcn_ballot_w64(codes[k] >= kBlockEscape);
    const uint64_t mine = __builtin_amdgcn_ballot_w64(own_step == s);
    const uint32_t first = (uint32_t)__builtin_popcountll(mine);
    const uint32_t mine_at = PAIR ? own_lds->at : own.at;
    for (uint64_t m = mine; m; m &= m - 1u) {
      const uint32_t at = (uint32_t)__builtin_amdgcn_readlane((int)mine_at, (uint32_t)__builtin_ctzll(m));
#pragma unroll
      for (uint32_t k = 0; k < (uint32_t)RF; ++k)
        left[k] &= ((at >> 9) & 7u) == k ? ~(1ull << (((at >> 8) & 1u) * 16u + ((at >> 7) & 1u) * 8u + ((at >> 4) & 7u) + ((at >> 3) & 1u) * 32u)) : ~0ull;
    }
    // lane i's the i-th of them: fragment, row and half of a step
    uint32_t n = 0, at = tile_place(0u, 0u, 0u);
#pragma unroll
    for (uint32_t k = 0; k < (uint32_t)RF; ++k)
      for (uint64_t m = left[k]; m; m &= m - 1u) {
        const uint32_t l = (uint32_t)__builtin_ctzll(m);
        at = lane == n ? tile_place(2u * k + ((l & 31u) >> 4), l & 15u, 2u * (s & 1u) + (l >> 5)) : at;
        ++n;
      }
    if (n == 0u || first + n > kWaveValues) return n ? 2u : 0u;
    const u32x2_t d = *reinterpret_cast<const u32x2_t*>(tiles + (at & 0xFFFu)), sm = *reinterpret_cast<const u32x2_t*>(tiles + ((at >> 12) & 0xFFFu));
    const uint32_t k = at >> 24;
    uint32_t o[3];
    block_octets(d.x, d.y, sm.x << (3u - k), o);
    ValueBlock b = code_block(o, (sm.y >> (8u * k)) & 255u);
    b.at = at;
    if (lane < n) place(b, (1ull << n) - 1u, first, tiles);
    return 1u;
  };
  auto decode_escapes = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t k = 0; k < (uint32_t)RF; ++k) {
      if (__builtin_expect(!left[k], 1)) continue;
      uint32_t o[3];
      block_octets(Bn[k].w[0], Bn[k].w[1], Bn[k].w[2] << 1, o);
      const ValueBlock b = code_block(o, (Bn[k].meta >> 4) & 255u);
      if (left[k] >> lane & 1u) {
        Bn[k].w[0] = b.d0;
        Bn[k].w[1] = b.d1;
        Bn[k].w[2] = (b.d0 & 0x11111111u) | (b.d1 & 0x11111111u) << 1 | b.s << 2;
        if constexpr (PAIR) {
          T[k][0] = b.t.hi;
          T[k][kTerms - 1u] = b.t.lo;
        } else {
          Tn[k] = b.t.hi;
        }
      }
    }
  };
  auto round = [&](uint32_t buffer, uint32_t next, uint32_t last, uint32_t s, auto round_j, auto left_t, uint32_t& found) __attribute__((always_inline)) {
    constexpr uint32_t j = decltype(round_j)::value, jn = j < 2u ? j + 1u : 0u;  // of the products, and of what is unpacked
    constexpr uint32_t kParts = (PAIR && j == 1u ? 8u : 4u) * RF / CF;  // (PAIR: T is read anew behind its last use)
    u32x4_t to[kTerms][RF];
    ValuePick pick[kTerms];
    if (j == 1u) {
      read_w(next);
      turn();
    }
    if (j == 2u) {
#pragma unroll
      for (int k = 0; k < RF; ++k) {
        B[k] = Bn[k];
        if constexpr (!PAIR) T[k][0] = Tn[k];
      }
    }
#pragma unroll
    for (uint32_t c = 0; c < (uint32_t)CF; ++c) {
      if (j == 0u && c == (uint32_t)CF / 2u) {
        wide_wait<kLoads>();
        wide_barrier();
        if constexpr (decltype(left_t)::value) read_codes(s + 1u, next);
      }
#pragma unroll
      for (int p = (int)kTerms - 1; p >= 0; --p)
#pragma unroll
        for (int k = 0; k < RF; ++k)
          acc[k][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, w[p][k]), x[c],
                                                              PAIR && j == 0u && p == (int)kTerms - 1 ? acc16_t{} : acc[k][c], 0, 0, 0);  // (PAIR: a step's sum)
      if (j < 2u) read_x_part(buffer, jn, c);
      else read_x_part(next, 0, c);
      const uint32_t first = c * kParts, after = min(first + kParts, 4u * RF);
#pragma unroll
      for (uint32_t i = first; i < after; ++i) unpack_part(std::integral_constant<uint32_t, jn>{}, i, pick, to);
      // (here, not where it is used)
#pragma unroll
      for (uint32_t p = 0; p < kTerms; ++p)
        if (first < after) {
          if (after & 1u) asm volatile("" : "+v"(pick[p].at), "+v"(pick[p].high));
          else asm volatile("" : "+v"(to[p][(after - 1u) >> 2]));
        }
      if (j == 2u && c < 3u) to_next_step(c);
      if (j == 1u) {
        if (c == CF / 2u) {
#pragma unroll
          for (uint32_t k = 0; k < (uint32_t)RF; ++k) read_values(k);
        }
        if (c + RF >= (uint32_t)CF) assemble(c + RF - CF);
        // (three steps ahead)
        if (c % 2u == 0u && c / 2u < (uint32_t)kLoadsX / 3u) load_x(last, c / 2u);
        if (c == 2u * (uint32_t)kLoadsX / 3u) load_w(last);
      }
#pragma unroll
      for (int i = 0; i < (PAIR ? 2 * RF : RF); ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // a product,
        __builtin_amdgcn_sched_group_barrier(0x002, CF == 8 ? 3 : 4, 0);  // vector instructions
        if (i == 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // an LDS read
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (j == 0u) place_escapes(s + 1u, next);
    if constexpr (decltype(left_t)::value && j == 0u) found = some_left(s + 1u) ? place_left(s + 1u, next) : 0u;
    if constexpr (decltype(left_t)::value && j == 1u)
      if (found == 2u) decode_escapes();
#pragma unroll
    for (uint32_t p = 0; p < kTerms; ++p)
#pragma unroll
      for (int k = 0; k < RF; ++k) w[p][k] = to[p][k];
  };
  // the lists first, into the buffer that is filled last: the lanes take theirs while the first step's octets and tiles come
  const uint32_t slots = t.slots, n_listed = 2u * RF * slots;
  const uint32_t lists_at = 3u * kBuf + wave * (gemm_wide_lists<RF>() + 64u * 20u);
  const uint8_t* const lists = uniform_global(rec0 + stride - slots * 16u);
  for (uint32_t e0 = 0; e0 < n_listed; e0 += 64u) {
    const uint32_t e = min(e0 + lane, n_listed - 1u), tile_of = e / slots;
    load_to_lds(smem_at + lists_at + e0 * 16u, record(row0 + tile_of * 16u) + (e - tile_of * slots) * 16u, lists);
  }
  load(0);
  load(kBuf);
  load(2u * kBuf);
  {
    // the weights of meta byte `tid`
    const float v = scale_of(tid & 255u);
    Values values{};
#pragma unroll
    for (int i = 0; i < 8; ++i) value_to(values, i, (float)(2 * (i < 4 ? i : i - 8) + (int)(tid & 7u) - 3) * v);
    if (tid < kBlockEscape) {
      reinterpret_cast<u32x4_t*>(wide_smem)[tid] = values.hi;
      if constexpr (PAIR) reinterpret_cast<u32x4_t*>(wide_smem + kValueBytes)[tid] = values.lo;
    }
  }
  if (slots) {
    wide_wait<3 * kLoads>();
    const u32x4_t* const raw = reinterpret_cast<const u32x4_t*>(smem + lists_at);
    u32x4_t* const kept = reinterpret_cast<u32x4_t*>(smem + lists_at + gemm_wide_lists<RF>());
    uint32_t* const kept_tile = reinterpret_cast<uint32_t*>(kept + 64);
    uint32_t n = 0;
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)RF; ++i) {
      const uint32_t from = min(i * 64u + lane, n_listed - 1u);
      const u32x4_t e = raw[from];
      const uint32_t step = (e.w >> 10) & 0x3FFFFu;
      if (__builtin_amdgcn_ballot_w64(e.w == ~0u)) left_steps = ~0u;
      const bool valid = i * 64u + lane < n_listed && e.w != 0u && e.w != ~0u && step >= s0 && step < s1;
      const uint64_t there = __builtin_amdgcn_ballot_w64(valid);
      const uint32_t at = n + __builtin_amdgcn_mbcnt_hi((uint32_t)(there >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)there, 0u));
      if (valid && at < 64u) {
        kept[at] = e;
        kept_tile[at] = from / slots;
      }
      n += (uint32_t)__builtin_popcountll(there);
      for (uint64_t over = __builtin_amdgcn_ballot_w64(valid && at >= 64u); over; over &= over - 1u) {
        const uint32_t bit = (uint32_t)__builtin_amdgcn_readlane((int)step, (uint32_t)__builtin_ctzll(over)) - s0;
        left_steps |= lane == ((bit >> 5) & 63u) ? 1u << (bit & 31u) : 0u;
      }
    }
    wave_lds_order();
    if (n) {
      const u32x4_t e = kept[lane];
      const uint32_t tile_of = kept_tile[lane], row = e.w >> 28, blk = (e.w >> 9) & 0x7FFFFu, nibbles[3] = {e.x, e.y, e.z};
      own = value_block(nibbles, (e.w >> 8) & 1u, scale_of((e.w & 31u) << 3));
      own.at = tile_place(tile_of, row, blk);
      own_step = lane < n ? blk >> 1 : ~0u;
      if constexpr (PAIR) *own_lds = own;
      if (n > kWaveValues) {  // perhaps more of one step than there is room for
        uint32_t same = 0;
        for (uint32_t i = 0; i < min(n, 64u); ++i) same += (uint32_t)__builtin_amdgcn_readlane((int)own_step, i) == own_step ? 1u : 0u;
        if (__builtin_amdgcn_ballot_w64(lane < n && same > kWaveValues)) left_steps = ~0u;
        if (same > kWaveValues) own_step = ~0u;
      }
    }
  }
  const bool any_left = __builtin_amdgcn_ballot_w64(left_steps != 0u) != 0u;
  // The end's operands, behind the first steps' loads: what waits for the one waits for the other.  (In front of them these came a way from memory later.
  // With that, and the tail operands read where there are none: 2612 x 672 at 96 rows 17.9 us with f32 results, 17.4 so, 1000 x 408 at 600 17.3 with binary16
  // ones and 16.5, 12288 x 4096 at 512 65.3 and 64.7, 9728 x 2560 at 500 43.6 and 43.0.)
#pragma unroll
  for (int i = 0; i < (RF + 1) / 2; ++i) asm volatile("" : "+v"(my_scale[i]));
  asm volatile("" ::"v"(touched));
  wide_wait<2 * kLoads>();
  lds_barrier();
  // A step from its tiles in LDS: the first, and with PAIR those that something was left of, whose first octet is unpacked already.
  auto begin = [&](uint32_t buffer, bool all, auto first) __attribute__((always_inline)) {
    read_w(buffer);
    if constexpr (decltype(first)::value) read_x(buffer, 0);
#pragma unroll
    for (uint32_t k = 0; k < (uint32_t)RF; ++k) {
      read_values(k);
      assemble(k);
    }
    if (__builtin_expect(all, 0)) decode_escapes();
#pragma unroll
    for (uint32_t k = 0; k < (uint32_t)RF; ++k) {
      B[k] = Bn[k];
      if constexpr (!PAIR) T[k][0] = Tn[k];
      ValuePick pick[kTerms];
#pragma unroll
      for (uint32_t i = 0; i < 4u; ++i) unpack_part(std::integral_constant<uint32_t, 0>{}, 4u * k + i, pick, w);
    }
  };
  // (What is rare is said to be: it then stands behind the rest of the kernel, and 6000 x 1000 at 130 rows takes 28.9 us, not 29.5.)
  place_escapes(s0, 0);
  uint32_t found = 0;
  if (__builtin_expect(any_left && some_left(s0), 0)) {
    read_codes(s0, 0);
    found = place_left(s0, 0);
  }
  begin(0, found == 2u, std::true_type{});
#pragma unroll
  for (int k = 0; k < RF; ++k)
#pragma unroll
    for (int c = 0; c < CF; ++c)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[k][c][e] = 0.f;
  if constexpr (PAIR) {
#pragma unroll
    for (int k = 0; k < RF; ++k)
#pragma unroll
      for (int c = 0; c < CF; ++c)
#pragma unroll
        for (int e = 0; e < 16; ++e) sum[k][c][e] = 0.;
  }
  uint32_t buffer = 0, next = kBuf, last = 3u * kBuf, s = s0;
  auto steps_to = [&](uint32_t end, auto left_t) __attribute__((always_inline)) {
    do {  // (a split has at least one step)
      round(buffer, next, last, s, std::integral_constant<uint32_t, 0>{}, left_t, found);
      round(buffer, next, last, s, std::integral_constant<uint32_t, 1>{}, left_t, found);
      round(buffer, next, last, s, std::integral_constant<uint32_t, 2>{}, left_t, found);
      last = buffer;
      buffer = next;
      next = next + kBuf == kWideDepth * kBuf ? 0u : next + kBuf;
      if constexpr (PAIR) {
#pragma unroll
        for (int k = 0; k < RF; ++k)
#pragma unroll
          for (int c = 0; c < CF; ++c) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
              sum[k][c][e] += (double)acc[k][c][e];
            }
          }
      }
    } while (++s < end);
  };
  // (What the rare steps need costs the others 2 to 3 % where it stands in the same loop.  A second loop with PAIR would not fit the
  // registers, 36 too many: there the loop ends in front of such a step and begins again with it.  12288 x 4099 at 500 rows 199 -> 194 us,
  // 13000 x 5121 at 600 rows 259 -> 252; two loops without PAIR are as fast as that and need half the time for a rare step.)
  if constexpr (PAIR) {
    for (;;) {
      uint32_t end = any_left ? s + 1u : s1;
      while (end < s1 && !some_left(end)) ++end;
      steps_to(end, std::false_type{});
      if (s == s1) break;
      read_codes(s, buffer);
      found = place_left(s, buffer);
      if (found) begin(buffer, found == 2u, std::false_type{});
    }
  } else if (__builtin_expect(!any_left, 1)) {
    steps_to(s1, std::false_type{});
  } else {
    steps_to(s1, std::true_type{});
  }
  if constexpr (PAIR) {
#pragma unroll
    for (int k = 0; k < RF; ++k)
#pragma unroll
      for (int c = 0; c < CF; ++c)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[k][c][e] = (float)sum[k][c][e];
  }
  wide_wait<0>();
  if constexpr (CF == 8) {
#pragma unroll
    for (int k = 0; k < RF; ++k)
#pragma unroll
      for (int c = 0; c < CF; ++c) asm volatile("" : "+a"(acc[k][c]));  // one by one from here: all of them would not fit the vector registers
  }
  // A lane's activation row is l32 of a fragment; element e is weight row 8 (e / 4) + 4 h + e % 4 of it.
  // (From the lane's number anew: nothing of this may occupy registers during the loop.)
  const uint32_t lane_e = lane_offset(lane), l32e = lane_e & 31u, he = lane_e >> 5;
  const bool in_parts = RF == 2 && a.splits > 1u;  // (gemm_plan splits no tiles of 384 rows)
  const uint32_t n_rows = a.n_tiles * kRows;
  float* const parts = a.ws + (size_t)split * a.m_pad * n_rows;
  uint8_t* const turn_at = smem + ((kRows + 32u * CF) * kDim + kRows) * 4u + wave * turn_bytes<RF>();
  if (PAIR && in_parts) {
    __syncthreads();
#pragma unroll
    for (uint32_t c = 0; c < (uint32_t)CF; ++c)
#pragma unroll
      for (uint32_t k = 0; k < (uint32_t)RF; ++k)
        StoreF32<RF>::store(StoreAt{parts, n_rows, mt * kCols + c * 32u, a.M, tile * kRows + wave * (32u * RF), 0u, turn_at}, k, lane_e, acc[k][c] * unit);
    return;
  }
  // The tail columns this workgroup adds: of a split its share of them, in pairs.
  const uint32_t tail_w = a.tail_w, tail_parts = in_parts ? a.splits : 1u, tail_part = in_parts ? split : 0u;
  const uint32_t tail0 = PAIR ? 0u : (tail_w / 2u * tail_part / tail_parts) * 2u, tail1 = PAIR ? tail_w : (tail_w / 2u * (tail_part + 1u) / tail_parts) * 2u;
  // The tail's operands to LDS: a lane would wait for each of its loads in turn.
  float* const scales = reinterpret_cast<float*>(smem) + wave * (32u * RF);
  float* w_tail = reinterpret_cast<float*>(smem) + kRows;
  float* x_tail = w_tail + kRows * kDim;
  __syncthreads();
#pragma unroll
  for (uint32_t i = 0; i < (uint32_t)(RF + 1) / 2u; ++i)
    if (i * 64u + lane < 32u * RF) scales[i * 64u + lane] = my_scale[i] * unit;
  if constexpr (PAIR) {
    for (uint32_t c0 = 0; c0 < tail_w; c0 += 8u) {
      float v[8];
      const uint32_t m = mt * kCols + tid % kCols;
      const __half* tx = a.x + (size_t)min(m, a.M - 1u) * a.ldx + nb * kDim;
#pragma unroll
      for (uint32_t r0 = 0; r0 < kRows; r0 += 256u) {
        const uint32_t row = min(r0 + tid, kRows - 1u);
        const float* rec = reinterpret_cast<const float*>(rec0 + record(t.row0 + row));
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) v[i] = rec[tail_at(row & 15u, min(c0 + i, tail_w - 1u), tail_w)];
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i)
          if (r0 + tid < kRows && c0 + i < tail_w) w_tail[(c0 + i) * kRows + row] = v[i];
      }
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) v[i] = __half2float(tx[min(c0 + i, tail_w - 1u)]);
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i)
        if (tid < kCols && c0 + i < tail_w) x_tail[(c0 + i) * kCols + tid] = v[i];
    }
  } else if (tail0 != tail1) {
    // Eight or sixteen columns: the heads as they are, 16 bytes a lane, and the activations by octets.
    constexpr uint32_t kW = (kRows + 255u) / 256u * 4u, kX = 2u * kCols / 256u;
    const uint32_t pieces = tail_depth(tail_w) * 16u;  // of a tile
    u32x4_t w[kW];
    HalfOctet x[kX];
#pragma unroll
    for (uint32_t i = 0; i < kW; ++i) {
      const uint32_t k = min(i * 256u + tid, kRows / 16u * pieces - 1u), of = k / pieces;
      w[i] = *reinterpret_cast<const u32x4_t*>(rec0 + record(t.row0 + of * 16u) + 128u + (k - of * pieces) * 16u);
    }
#pragma unroll
    for (uint32_t i = 0; i < kX; ++i) {
      const uint32_t k = i * 256u + tid, m = mt * kCols + k % kCols, c = k / kCols * 8u;
      x[i] = *reinterpret_cast<const HalfOctet*>(a.x + (size_t)min(m, a.M - 1u) * a.ldx + nb * kDim + (c < tail_w ? c : 0u));
    }
#pragma unroll
    for (uint32_t i = 0; i < kW; ++i) reinterpret_cast<u32x4_t*>(w_tail)[min(i * 256u + tid, kRows / 16u * pieces - 1u)] = w[i];
#pragma unroll
    for (uint32_t i = 0; i < kX; ++i) {
      const uint32_t k = i * 256u + tid, c = k / kCols * 8u;
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) {
        x_tail[(c + 2u * j) * kCols + k % kCols] = half_lo(x[i].w[j]);
        x_tail[(c + 2u * j + 1u) * kCols + k % kCols] = half_hi(x[i].w[j]);
      }
    }
  }
  __syncthreads();
  // ld, from: values from one of the results' activation rows to the next, and where this wavefront's first weight row is in one.
  // A fragment's tail columns, two at a time (the halves hold one each), are a chain of f32 products of 64 cycles, beside which the fragment in
  // front of it is converted and stored; its operands are read a fragment ahead.
  auto finish = [&](auto to, void* y, size_t ld, uint32_t from) __attribute__((always_inline)) {
    constexpr uint32_t kPairs = PAIR ? 1u : 8u, kFragments = RF * CF;  // pairs of tail columns
    const uint32_t pairs = (tail1 - tail0) >> 1;
    float scale[RF][16], tw[RF][kPairs], tx[kPairs];
#pragma unroll
    for (uint32_t k = 0; k < (uint32_t)RF; ++k) {
#pragma unroll
      for (uint32_t g = 0; g < 4u; ++g) {
        const float4 v = *reinterpret_cast<const float4*>(scales + k * 32u + g * 8u + he * 4u);
        scale[k][4 * g] = v.x;
        scale[k][4 * g + 1] = v.y;
        scale[k][4 * g + 2] = v.z;
        scale[k][4 * g + 3] = v.w;
      }
      if (!PAIR && pairs) {
        const uint32_t row = wave * (32u * RF) + k * 32u + l32e;
        const float* at = w_tail + (row >> 4) * 64u * tail_depth(tail_w);
#pragma unroll
        for (uint32_t i = 0; i < kPairs; ++i) tw[k][i] = at[tail_at(row & 15u, min(tail0 + 2u * i + he, 15u), tail_w) - 32u];  // (past the last: not used)
      }
    }
    auto read_c = [&](uint32_t c) __attribute__((always_inline)) {
#pragma unroll
      for (uint32_t i = 0; i < kPairs; ++i) tx[i] = x_tail[min(tail0 + 2u * i + he, 15u) * kCols + c * 32u + l32e];
    };
    auto put = [&](uint32_t i, const acc16_t& v) __attribute__((always_inline)) {
      decltype(to)::store(StoreAt{y, ld, mt * kCols + i / RF * 32u, a.M, from, t.d_out, turn_at}, i % RF, lane_e, v);
    };
    acc16_t before;
    if (!PAIR && pairs) read_c(0);
#pragma unroll
    for (uint32_t i = 0; i < kFragments; ++i) {
      const uint32_t k = i % RF, c = i / RF;
      acc16_t v;
      if constexpr (PAIR) {
        // (One by one on top of the blocks' sum each column costs that a rounding: they are summed by themselves and meet it last.  A column past
        // the last is zero in both operands: zero times the last one again is not zero where that is infinite.)
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = 0.f;
        for (uint32_t j = 0; j < tail_w; j += 2u) {
          const uint32_t col = min(j + he, tail_w - 1u);
          const float w = w_tail[col * kRows + wave * (32u * RF) + k * 32u + l32e], x1 = x_tail[col * kCols + c * 32u + l32e];
          v = __builtin_amdgcn_mfma_f32_32x32x2f32(j + he < tail_w ? w : 0.f, j + he < tail_w ? x1 : 0.f, v, 0, 0, 0);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          float r = fmaf(acc[k][c][e], scale[k][e], v[e]);
          asm("" : "+v"(r));  // (an f32 value in every store: where they convert one by one it would be one operation, rounded once)
          v[e] = r;
        }
        put(i, v);
        __builtin_amdgcn_sched_barrier(0);
      } else {
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = acc[k][c][e] * scale[k][e];
#pragma unroll
        for (uint32_t j = 0; j < kPairs; ++j)
          if (j < pairs) v = __builtin_amdgcn_mfma_f32_32x32x2f32(tw[k][j], tx[j], v, 0, 0, 0);
        if (pairs && k + 1u == (uint32_t)RF && c + 1u < (uint32_t)CF) read_c(c + 1u);
        if (i) put(i - 1u, before);
        before = v;
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (!PAIR) put(kFragments - 1u, before);
  };
  const bool whole = row0 + 32u * RF <= t.d_out && ((reinterpret_cast<uintptr_t>(t.y) | t.d_out * (a.y_f32 ? 4u : 2u)) & 15u) == 0;
  if (!PAIR && in_parts) {
    finish(StoreF32<RF>{}, parts, n_rows, tile * kRows + wave * (32u * RF));
  } else if (a.y_f32) {
    if (whole) finish(StoreF32<RF>{}, t.y, t.d_out, row0);
    else finish(StoreEach<float>{}, t.y, t.d_out, row0);
  } else {
    if (whole) finish(typename std::conditional<PAIR, StoreF16Direct, StoreF16<RF>>::type{}, t.y, t.d_out, row0);
    else finish(StoreEach<_Float16>{}, t.y, t.d_out, row0);
  }
}
template <int CF, bool PAIR>
__global__ __launch_bounds__(256, CF == 8 || PAIR ? 1 : 2) void gemm_wide_kernel(GemmArgs a) { wide_product<2, CF, PAIR>(a); }
__global__ __launch_bounds__(256, 1) void gemm_tall_kernel(GemmArgs a) { wide_product<3, 4, false>(a); }

// PAIR: the partial sums of the column splits, added in order; row scale and tail columns.  A lane takes one weight row and
// kReduceM activation rows, so that the row's tail is read once for them.
// What bounds it is how many round trips to memory a lane makes: the sums and the tail columns are read four splits and
// eight columns at a time, the activations' tail comes to LDS with the first of them.  (One by one 11.3 us for 500
// rows of 2560 with 8 or 16 tail columns and 14.9 for 6144; so 9.0 and 10.3; and a microsecond less with a workgroup's lanes a tile's rows,
// which needs no division, and loads of the splits there are alone.)
constexpr uint32_t kReduceM = 8;
// The splits are added in f64 and the tail by itself.  Grid (tiles of 256 weight rows, the only ones that are split; kReduceM
// activation rows).
constexpr uint32_t kReduceRows = 256;
static_assert(kReduceRows == gemm_wide_rows<2>(), "a workgroup's lanes are a tile's rows");
__global__ __launch_bounds__(256) void gemm_reduce_pair_kernel(GemmArgs a) {
  __shared__ float x_tail[kReduceM][32];
  static_assert(kReduceM * 32u == 256u && kDim <= 32, "a value of the activations' tail per lane");
  touch_args(a);
  const uint32_t n_rows = a.n_tiles * kReduceRows, m0 = blockIdx.y * kReduceM, out_row = blockIdx.x * kReduceRows + threadIdx.x;
  const GemmTile t = gemm_tile_at(a, blockIdx.x, kReduceRows);
  const uint32_t my_row = t.row0 + threadIdx.x, row = min(my_row, t.d_out - 1u);  // lanes past the last row repeat it
  const uint32_t stride = t.stride;
  const uint8_t* rec = t.base + kTileTableBytes + (size_t)(row / kTileRows) * stride;
  const uint32_t r = row & 15u, tail_w = a.tail_w;
  if (tail_w) {
    const uint32_t m = min(m0 + threadIdx.x / 32u, a.M - 1u), c = min(threadIdx.x % 32u, tail_w - 1u);
    x_tail[threadIdx.x / 32u][threadIdx.x % 32u] = __half2float(a.x[(size_t)m * a.ldx + a.nb * kDim + c]);
  }
  const float scale = reinterpret_cast<const float*>(rec)[r];
  // (a class's columns lie together: four of each at a time, the first of them asked for before the sums; what is behind the
  // last is not used)
  struct __attribute__((packed, aligned(4))) F4 { float v[4]; } tw[4];
  const auto read_tail = [&](uint32_t i0) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t c = 0; c < 4u; ++c) tw[c] = *reinterpret_cast<const F4*>(reinterpret_cast<const float*>(rec) + tail_at(r, 4u * i0 + c, tail_w));
  };
  if (tail_w) read_tail(0);
  double s[kReduceM];
#pragma unroll
  for (uint32_t k = 0; k < kReduceM; ++k) s[k] = 0;
  for (uint32_t p0 = 0; p0 < a.splits; p0 += kReduceSplits) {
    float v[kReduceSplits][kReduceM];
#pragma unroll
    for (uint32_t p = 0; p < kReduceSplits; ++p) {
      if (p0 + p >= a.splits) break;
#pragma unroll
      for (uint32_t k = 0; k < kReduceM; ++k) v[p][k] = uniform_global(a.ws + ((size_t)(p0 + p) * a.m_pad + min(m0 + k, a.M - 1u)) * n_rows)[out_row];
    }
#pragma unroll
    for (uint32_t p = 0; p < kReduceSplits; ++p) {
      if (p0 + p >= a.splits) break;
#pragma unroll
      for (uint32_t k = 0; k < kReduceM; ++k) s[k] += (double)v[p][k];
    }
  }
  float out[kReduceM];
#pragma unroll
  for (uint32_t k = 0; k < kReduceM; ++k) out[k] = 0.f;
  if (tail_w) {
    lds_barrier();
    const uint32_t depth = tail_depth(tail_w);
    for (uint32_t i0 = 0; i0 < depth; i0 += 4u) {
      if (i0) read_tail(i0);
#pragma unroll
      for (uint32_t i = 0; i < 4u; ++i)
#pragma unroll
        for (uint32_t c = 0; c < 4u; ++c)
          if (4u * (i0 + i) + c < tail_w) {
#pragma unroll
            for (uint32_t k = 0; k < kReduceM; ++k) out[k] = fmaf(tw[c].v[i], x_tail[k][4u * (i0 + i) + c], out[k]);
          }
    }
  }
  if (my_row < t.d_out) {
#pragma unroll
    for (uint32_t k = 0; k < kReduceM; ++k)
      if (m0 + k < a.M) store_y(t.y, (size_t)(m0 + k) * t.d_out + row, fmaf((float)s[k], scale, out[k]), a.y_f32);
  }
}

// The partial results of the column splits (each has its row scale and its share of the tail columns), added in order, where no launch behind the
// product takes them as they are (GemmSums).  A lane takes four weight rows of kSumM activation rows, kReduceSplits splits at a time.  (The launch that
// also had scales and tails to see to took 8.8 us for 500 rows of 2560; 6000 x 1000 at 130 rows 28.1 -> 25.4 us, 4096 x 4096 at 300 33.8 -> 32.1.)
constexpr uint32_t kSumM = 2;
__device__ __forceinline__ void add_four(float (&s)[4], const float4& v) {
  s[0] += v.x;
  s[1] += v.y;
  s[2] += v.z;
  s[3] += v.w;
}
__global__ __launch_bounds__(256) void gemm_sum_kernel(GemmArgs a) {
  touch_args(a);
  const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const GemmTile t = gemm_tile_at(a, blockIdx.x, kReduceRows);
  const uint32_t n_rows = a.n_tiles * kReduceRows, m0 = (blockIdx.y * 4u + wave) * kSumM, row = t.row0 + lane * 4u;
  if (m0 >= a.M) return;
  float s[kSumM][4] = {};
  for (uint32_t p0 = 0; p0 < a.splits; p0 += kReduceSplits) {
    float4 v[kReduceSplits][kSumM];
#pragma unroll
    for (uint32_t p = 0; p < kReduceSplits; ++p) {
      if (p0 + p >= a.splits) break;
#pragma unroll
      for (uint32_t k = 0; k < kSumM; ++k)
        v[p][k] = reinterpret_cast<const float4*>(uniform_global(a.ws + ((size_t)(p0 + p) * a.m_pad + min(m0 + k, a.M - 1u)) * n_rows + blockIdx.x * kReduceRows))[lane];
    }
#pragma unroll
    for (uint32_t p = 0; p < kReduceSplits; ++p) {
      if (p0 + p >= a.splits) break;
#pragma unroll
      for (uint32_t k = 0; k < kSumM; ++k) add_four(s[k], v[p][k]);
    }
  }
  const bool whole = row + 4u <= t.d_out && ((reinterpret_cast<uintptr_t>(t.y) | (size_t)t.d_out * (a.y_f32 ? 4u : 2u)) & (a.y_f32 ? 15u : 7u)) == 0;
#pragma unroll
  for (uint32_t k = 0; k < kSumM; ++k) {
    if (m0 + k >= a.M) break;
    const size_t at = (size_t)(m0 + k) * t.d_out + row;
    if (whole && a.y_f32) *reinterpret_cast<float4*>(reinterpret_cast<float*>(t.y) + at) = make_float4(s[k][0], s[k][1], s[k][2], s[k][3]);
    else if (whole) *reinterpret_cast<uint2*>(reinterpret_cast<__half*>(t.y) + at) = make_uint2(pack_halves(s[k][0], s[k][1]), pack_halves(s[k][2], s[k][3]));
    else
      for (uint32_t i = 0; i < 4u; ++i)
        if (row + i < t.d_out) store_y(t.y, at + i, s[k][i], a.y_f32);
  }
}

}  // namespace llvq
