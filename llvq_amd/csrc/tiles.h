// The weight layout the products read, the kernel that writes it at upload, and the batch-1 product over it.
//
// A code stream is unranked once, on the device, when its matrix is uploaded: unranking costs about 500 vector
// instructions per block, and a product that repeats it is bound by them at 5 % of what HBM delivers (2.26 ms for the
// 150.7 M blocks of a 4B model, 434 GB/s of codes).  What is kept of a block are the ten bytes of block_code.h, the
// integer point itself; 13 (4-bit coordinates and a byte) were 23 % more to read.
//
//   matrix: 32 floats (the block scales, centroid / sqrt(16 shell), in the order of block_code.h's slots, zeros behind
//           them), then one tile per 16 rows:
//             16 row scales (f32), the number of escapes in it and 60 bytes of nothing; the tail columns (tail_at), 64 lanes
//             of (tail_w + 3) / 4 floats; the units of four blocks; the list of escapes
//   unit:   640 bytes, five 128-byte lines of eight 16-byte pieces, piece l of a line being of rows l and l + 8:
//             {d0, d1} of blocks 0 and 1 of row l; of blocks 2 and 3; the same two lines of row l + 8;
//             {s, meta} of row l, {s, meta} of row l + 8, four blocks in a dword
//           nibble q of a dword holds column 8 j + {0, 2, 4, 6, 1, 3, 5, 7}[q]: nibbles q and q + 4 are neighbouring
//           columns in the two halves of the dword, which is what a packed binary16 unpack wants, and a dword is the
//           operand of an 8-wide 4-bit dot product.
//
//   escape: a block whose code says kBlockEscape or more (block_code.h), as 16 bytes: the nibbles n of v = 2 n + odd, and
//           row << 28 | block << 9 | odd << 8 | slot, in the order of these, zeros behind them.  The products, in which a
//           wavefront would take block_escape's path for one of its lanes at a time, take such blocks for zero where they
//           meet them (their slot's scale is) and make up for it from the list.  Where a tile has more of them than
//           list_slots (all of them, or by chance) its list does not count and they read the codes.
//
// Eight units are a step of a wavefront, 5120 consecutive bytes: lane (l, q) = (lane % 8, lane / 8) loads the five pieces l
// of unit q.  Every line of memory is asked for by one load, whole, and marked as not to be kept: read like that the card
// delivers 6.9 TB/s (a loop of nothing else, 8 or 16 wavefronts on a CU), without the mark 6.1, and 5.9 where 12-byte
// pieces and their bytes of meta are asked for by two loads that share lines (there the mark makes it 5.4).  A 4B model as one
// launch takes 257 us with the mark and 291 without; four layers by themselves, which the 256 MB cache holds, 38.0 and 36.2.
#pragma once

#include "block_code.h"
#include "escape_list.h"
#include "step_sums.h"

namespace llvq {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr uint32_t kTileTableBytes = kScaleSlots * 4;

// Floats of a row's tail columns that a lane of its four holds: column c is the (c / 4)-th of lane class c % 4.
__host__ __device__ inline uint32_t tail_depth(uint32_t tail_w) { return (tail_w + 3u) >> 2; }
__host__ __device__ inline uint32_t tile_head_bytes(uint32_t tail_w) { return 128u + 256u * tail_depth(tail_w); }
__host__ __device__ inline uint32_t tile_units(uint32_t nb) { return (nb + 3u) >> 2; }
// bytes of one tile of sixteen rows, a multiple of 128
__host__ __device__ inline uint32_t tile_stride(uint32_t nb, uint32_t tail_w, uint32_t slots) {
  return tile_head_bytes(tail_w) + tile_units(nb) * kUnitBytes + slots * 16u;
}
__host__ __device__ inline uint32_t list_at(uint32_t nb, uint32_t tail_w) { return tile_head_bytes(tail_w) + tile_units(nb) * kUnitBytes; }
constexpr uint32_t kCountAt = 64;  // byte of a tile at which the number of its escapes is
__host__ __device__ inline uint32_t tile_count(uint32_t d_out) { return (d_out + kTileRows - 1u) / kTileRows; }
// The lane that holds row r's class c, wherever sixteen rows meet four classes: what two exchanges, across 8 and 16 lanes,
// add up are the classes of one row.
__host__ __device__ inline uint32_t row_lane(uint32_t r, uint32_t c) { return (r & 7u) | c << 3 | (r >> 3) << 5; }
__host__ __device__ inline uint32_t lane_row(uint32_t lane) { return (lane & 7u) | (lane >> 5) << 3; }
__host__ __device__ inline uint32_t lane_class(uint32_t lane) { return (lane >> 3) & 3u; }
// float of a tile that holds tail column c of row r
__host__ __device__ inline uint32_t tail_at(uint32_t r, uint32_t c, uint32_t tail_w) { return 32u + row_lane(r, c & 3u) * tail_depth(tail_w) + (c >> 2); }

// ---- upload: code stream -> tiles ---------------------------------------------------------------
// One lane per block, a wavefront a unit: lane % 4 is the block in it, lane / 4 the row.  The lanes of a wavefront take
// both coset programs (about 800 instructions per block, and 250 for the code, 4 ms for a 4B model's blocks): an upload is
// bound by the copy of the codes over PCIe, fifteen times that.
// `rows` rows; codes and tiles are those rows' own.
__device__ __forceinline__ uint32_t quad_or(uint32_t v) {
  v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false);
  return v | (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, false);
}
template <bool WIDE>
__global__ __launch_bounds__(512) void transcode_kernel(GlobalTables g, const uint8_t* __restrict__ codes, uint8_t* __restrict__ tiles,
                                                        uint32_t rows, uint32_t nb, uint32_t tail_w, uint32_t slots) {
  extern __shared__ __align__(16) uint8_t smem[];
  const DecodeTables T = stage_tables<WIDE>(smem, g);
  __syncthreads();
  const uint32_t stride = tile_stride(nb, tail_w, slots), head = tile_head_bytes(tail_w), per_tile = tile_units(nb);
  const uint32_t units = tile_count(rows) * per_tile;  // (the host keeps a launch's blocks below 2^32)
  const uint32_t lane = threadIdx.x & 63u, k = lane & 3u, r = lane >> 2, waves = blockDim.x >> 6;
  for (uint32_t u = blockIdx.x * waves + (threadIdx.x >> 6); u < units; u += gridDim.x * waves) {
    const uint32_t tile = u / per_tile, in_tile = u - tile * per_tile;
    const uint32_t row = tile * kTileRows + r, b = in_tile * 4u + k;
    uint32_t w[3] = {0, 0, 0}, par = 0, gain = 0, shell = 0;
    if (row < rows && b < nb) {
      const uint64_t at = (uint64_t)row * nb + b;
      uint64_t rec;
      if constexpr (WIDE) {  // block `at` is the 49 bits from bit 49 at on; the staged stream has slack behind it
        const uint64_t bit = at * kDenseBits;
        const uint32_t sh = (uint32_t)(bit & 7u);
        uint64_t acc = 0;
        for (uint32_t i = 0; i < 7u; ++i) acc = (acc << 8) | codes[(bit >> 3) + i];
        rec = (acc >> (56u - sh - kDenseBits)) & ((1ULL << kDenseBits) - 1u);
      } else {
        rec = read_record(codes, 6 * at);
      }
      const int ci = decode_index(T, rec >> 1, [&](int p, int v) {
        const uint32_t nib = ((uint32_t)(v >> 1) & 15u) << (4u * (((uint32_t)p & 7u) >> 1) + 16u * ((uint32_t)p & 1u));
        par = (uint32_t)v & 1u;
        if (p < 8) w[0] |= nib;
        else if (p < 16) w[1] |= nib;
        else w[2] |= nib;
      });
      if (ci >= 0) {
        gain = (uint32_t)rec & 1u;
        shell = T.cls[ci].shell;
      }
    }
    BlockCode c;
    block_encode(w, par, gain, shell, c);
    const uint32_t s = quad_or(c.s << k), meta = quad_or(c.meta << (8u * k));
    if (c.meta >= kBlockEscape && slots) {
      uint8_t* t = tiles + (size_t)tile * stride;
      const uint32_t e = atomicAdd(reinterpret_cast<uint32_t*>(t + kCountAt), 1u);
      if (e < slots) *reinterpret_cast<uint4*>(t + stride - slots * 16u + e * 16u) = make_uint4(w[0], w[1], w[2], r << 28 | b << 9 | par << 8 | (gain * 12u + shell - 2u));
    }
    uint8_t* out = tiles + (size_t)tile * stride + head + (size_t)in_tile * kUnitBytes + (r & 7u) * 16u;
    *reinterpret_cast<uint2*>(out + ((r >> 3) * 2u + (k >> 1)) * 128u + (k & 1u) * 8u) = make_uint2(c.d0, c.d1);
    if (k == 0) *reinterpret_cast<uint2*>(out + 512u + (r >> 3) * 8u) = make_uint2(s, meta);
  }
}

// The lists in order, behind transcode_kernel, whose lanes put an escape wherever there was room: a wavefront per tile, an
// escape a lane, or two where there are places for more, which go where as many lie before them.
static_assert(kMaxListSlots13 <= 128 && kMaxListSlots <= kMaxListSlots13, "two places of a list to a lane");
__global__ __launch_bounds__(256) void sort_lists_kernel(uint8_t* __restrict__ tiles, uint32_t n_tiles, uint32_t stride, uint32_t slots) {
  const uint32_t tile = blockIdx.x * 4u + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
  if (tile >= n_tiles) return;
  uint8_t* t = tiles + (size_t)tile * stride;
  const uint32_t count = *reinterpret_cast<const uint32_t*>(t + kCountAt);
  uint4* list = reinterpret_cast<uint4*>(t + stride - slots * 16u);
  if (count > slots) {
    if (lane == 0) list[0].w = 0xFFFFFFFFu;  // for those who read the list alone
    return;
  }
  if (slots <= 64u) {
    const uint4 mine = list[min(lane, slots - 1u)];
    uint32_t before = 0;
    for (uint32_t e = 0; e < count; ++e) before += (uint32_t)__shfl((int)mine.w, (int)e) < mine.w ? 1u : 0u;
    if (lane < count) list[before] = mine;
    else if (lane < slots) list[lane] = make_uint4(0, 0, 0, 0);
    return;
  }
  uint4 mine[2];
  uint32_t before[2] = {0, 0};
#pragma unroll
  for (uint32_t i = 0; i < 2; ++i) mine[i] = list[min(i * 64u + lane, slots - 1u)];
  for (uint32_t e = 0; e < count; ++e) {
    const uint32_t key = (uint32_t)__shfl((int)(e < 64u ? mine[0].w : mine[1].w), (int)(e & 63u));
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) before[i] += key < mine[i].w ? 1u : 0u;
  }
#pragma unroll
  for (uint32_t i = 0; i < 2; ++i) {
    const uint32_t at = i * 64u + lane;
    if (at < count) list[before[i]] = mine[i];
    else if (at < slots) list[at] = make_uint4(0, 0, 0, 0);
  }
}

// Row scales, the escapes' counters (zero) and tail columns into the tiles' heads (zeros for rows past the last and columns that are not there), the
// matrix's block scales to `table_out` where that is given (as an argument: a copy of 128 bytes from the host costs an
// upload 15 us).
struct TileTable { float v[kScaleSlots]; };
__global__ __launch_bounds__(256) void tile_heads_kernel(TileTable table, float* table_out, const float* __restrict__ rscale, const float* __restrict__ tail, uint8_t* __restrict__ tiles,
                                                         uint32_t rows, uint32_t nb, uint32_t tail_w, uint32_t slots) {
  if (table_out && blockIdx.x == 0 && threadIdx.x < kScaleSlots) table_out[threadIdx.x] = table.v[threadIdx.x];
  const uint32_t per = kTileRows * (1u + 4u * tail_depth(tail_w)), stride = tile_stride(nb, tail_w, slots);
  const uint32_t total = tile_count(rows) * per;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
    const uint32_t tile = i / per, k = i - tile * per, r = k & 15u, j = k >> 4;  // j = 0: the scale, j > 0: tail column j - 1
    const uint32_t row = tile * kTileRows + r;
    float v = 0.f;
    if (row < rows) v = !j ? rscale[row] : j <= tail_w ? tail[(size_t)row * tail_w + j - 1u] : 0.f;
    reinterpret_cast<float*>(tiles + (size_t)tile * stride)[j ? tail_at(r, j - 1u, tail_w) : r] = v;
    if (k == 0) *reinterpret_cast<uint32_t*>(tiles + (size_t)tile * stride + kCountAt) = 0u;
  }
}

// A pointer that is the same in every lane and points into device memory, made scalar and typed global: loads through it
// take a scalar base and a 32-bit lane offset.  Pointers that a kernel reads out of a table in memory need it most: they
// carry no address space, and loads through them would be generic ("flat") ones, which count on two wait counters out of
// order, so that every wait behind one drains all loads in flight.
template <typename T>
__device__ __forceinline__ T* uniform_global(T* p) {
  typedef T __attribute__((address_space(1))) global_t;
  const uint64_t bits = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)bits), hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(bits >> 32));
  return (T*)reinterpret_cast<global_t*>(((uint64_t)hi << 32) | lo);
}

// ---- the activation as 4-bit digit planes -------------------------------------------------------
// Block-scaled fixed point: per 24-column block a power-of-two scale 2^s and an integer per value, cut into balanced
// 4-bit digits.  Four digits for results stored as binary16 (|x| <= 2^14: a value is rounded at 2^-15 of its block's
// largest, a sixteenth of the half ulp such a result carries anyway), six for f32 results (2^22: every binary16 value
// within 2^12 of its block's largest is exact).  An 8-wide 4-bit dot product then takes one digit of eight columns
// against a dword of weights, exactly.
template <int DIG>
__device__ __forceinline__ uint32_t plane_at(uint32_t blk) { return (blk >> 2) * XPlanes<DIG>::kDwords + (blk & 3u) * XPlanes<DIG>::kBlock; }
template <int DIG>
__device__ __forceinline__ uint32_t plane_sum_at(uint32_t blk) { return (blk >> 2) * XPlanes<DIG>::kDwords + XPlanes<DIG>::kSums + (blk & 3u) * 2u; }

// An inclusive maximum of the lanes' |f32| bit patterns over a quad (integers: a NaN is larger than anything).
__device__ __forceinline__ uint32_t quad_max(uint32_t v) {
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false));
  return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, false));
}
__device__ __forceinline__ int quad_sum(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, false);
  return v + __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, false);
}

// Eight values of a block (columns 8 sub .. 8 sub + 7 of it), sub = lane % 4; the quad's fourth lane passes zeros and
// only takes part in the exchange.  m: what the f32 bits of the quad's values have for a largest magnitude (a NaN is larger than
// anything); value(j, up, magic): value j times up plus magic, fused.  Writes the block's planes at xb, its sum and scale at xs.
// Every wavefront of a workgroup quantises and every workgroup does it for itself, so that its instructions count: about 50 from binary16 values
// (converted as they are multiplied), 60 from f32 ones; with a value at a time 100, and a token of a 4B model 1535 us, not 1516.
template <int DIG, class Value>
__device__ __forceinline__ void quantize_scaled(uint32_t m, Value&& value, uint32_t sub, uint32_t* xb, uint32_t* xs) {
  constexpr int kBits = DIG == 4 ? 14 : 22;
  constexpr uint32_t kMagic = 0x4B400000u;  // 1.5 2^23: adding it leaves the rounded integer in the low mantissa bits
  // Biased exponent of the block's largest, at least the one below which `scale` would leave the normal range (2^-105 with
  // six digits, 2^-113 with four): smaller blocks are quantised at that scale.
  const uint32_t e = max(m >> 23, (uint32_t)kBits);
  const bool bad = m >= 0x7F800000u;     // inf or NaN: the block's products are NaN, whatever the digits
  const float up = __uint_as_float((253u + (uint32_t)kBits - e) << 23);
  const float scale = bad ? __builtin_nanf("") : __uint_as_float((e + 1u - (uint32_t)kBits) << 23);
  uint32_t t[8], total = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    t[j] = __float_as_uint(value(j, up, __uint_as_float(kMagic)));
    total += t[j];
  }
  const int sum = quad_sum((int)(total - 8u * kMagic));
  uint32_t lo[DIG / 2], hi[DIG / 2];  // byte k of the values in slots 0..3 and 4..7: columns 0, 4, 1, 5 and 2, 6, 3, 7
  if constexpr (DIG == 4) {
    uint32_t p[4];  // two 16-bit values each; adding 8 to every digit and flipping its top bit makes the digits balanced
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t w = __builtin_amdgcn_perm(t[2 * j + 1], t[2 * j], 0x05040100u);
      typedef unsigned short us2 __attribute__((ext_vector_type(2)));
      const us2 s = __builtin_bit_cast(us2, w) + __builtin_bit_cast(us2, 0x88888888u);
      p[j] = __builtin_bit_cast(uint32_t, s) ^ 0x88888888u;
    }
    lo[0] = __builtin_amdgcn_perm(p[2], p[0], 0x06020400u);
    lo[1] = __builtin_amdgcn_perm(p[2], p[0], 0x07030501u);
    hi[0] = __builtin_amdgcn_perm(p[3], p[1], 0x06020400u);
    hi[1] = __builtin_amdgcn_perm(p[3], p[1], 0x07030501u);
  } else {
    uint32_t u[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) u[j] = (t[j] - kMagic + 0x888888u) ^ 0x888888u;
    const int first[2][4] = {{0, 4, 1, 5}, {2, 6, 3, 7}};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t a = u[first[h][0]], b = u[first[h][1]], c = u[first[h][2]], d = u[first[h][3]];
      const uint32_t ab = __builtin_amdgcn_perm(b, a, 0x05010400u), cd = __builtin_amdgcn_perm(d, c, 0x05010400u);  // bytes 0, 0, 1, 1
      uint32_t* dst = h ? hi : lo;
      dst[0] = __builtin_amdgcn_perm(cd, ab, 0x05040100u);
      dst[1] = __builtin_amdgcn_perm(cd, ab, 0x07060302u);
      dst[2] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(d, c, 0x0C0C0602u), __builtin_amdgcn_perm(b, a, 0x0C0C0602u), 0x05040100u);
    }
  }
  if (sub < 3u) {
#pragma unroll
    for (int k = 0; k < DIG / 2; ++k) {
      xb[(2 * k) * 3 + sub] = bfi32(0x0F0F0F0Fu, lo[k], hi[k] << 4);
      xb[(2 * k + 1) * 3 + sub] = bfi32(0x0F0F0F0Fu, lo[k] >> 4, hi[k]);
    }
  } else {
    xs[0] = (uint32_t)sum;
    xs[1] = __float_as_uint(scale);
  }
}

// f32 values.  kAny: they may be any; else one of them is not finite only if none of the lane's is (a rotation's).
template <int DIG, bool kAny>
__device__ __forceinline__ void quantize_octet(const float (&v)[8], uint32_t sub, uint32_t* xb, uint32_t* xs) {
  uint32_t m = 0;
  if constexpr (kAny) {
#pragma unroll
    for (int j = 0; j < 8; ++j) m = max(m, __float_as_uint(v[j]) & 0x7FFFFFFFu);
  } else {
    float f;  // (of a NaN and another value these give the other)
    asm("v_max_f32 %0, |%1|, |%2|" : "=v"(f) : "v"(v[0]), "v"(v[1]));
#pragma unroll
    for (int j = 2; j < 8; j += 2) asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(f) : "v"(v[j]), "v"(v[j + 1]));
    m = __float_as_uint(f);
  }
  quantize_scaled<DIG>(quad_max(m), [&](int j, float up, float magic) { return fmaf(v[j], up, magic); }, sub, xb, xs);
}
// binary16 values, in pairs
template <int DIG>
__device__ __forceinline__ void quantize_halves(const uint32_t (&w)[4], uint32_t sub, uint32_t* xb, uint32_t* xs) {
  typedef unsigned short us2 __attribute__((ext_vector_type(2)));
  us2 two = __builtin_bit_cast(us2, w[0] & 0x7FFF7FFFu);
#pragma unroll
  for (int j = 1; j < 4; ++j) two = __builtin_elementwise_max(two, __builtin_bit_cast(us2, w[j] & 0x7FFF7FFFu));
  const uint32_t m = quad_max(max((uint32_t)two.x, (uint32_t)two.y));
  quantize_scaled<DIG>(__float_as_uint(half_lo(m)), [&](int j, float up, float magic) { return fmaf(j & 1 ? half_hi(w[j >> 1]) : half_lo(w[j >> 1]), up, magic); }, sub, xb, xs);
}

// ---- batch-1 product ------------------------------------------------------------------------------
// What a launch's activation is made from.
enum : int { kSrcF16 = 0, kSrcRotated = 1, kSrcSiluMul = 2, kSrcAddRmsNorm = 3, kSrcFinished = 4 };  // (the last: f32 values, in.x_f32)

struct TileMat {
  const uint8_t* base;  // the matrix (table, then records)
  void* y;
  uint32_t d_out;
  uint32_t tile_begin;  // first tile of this matrix in the launch
  uint32_t stride, slots;
};
struct GemvArgs {
  ActivationIn in;
  uint32_t nb, tail_w, n_mats, n_tiles;
  GemvGrid g;  // what the host knows as well, so that no wavefront works it out
  TileMat m[kMaxGroup];
};
// Asks for all of a launch's arguments at once: each of their cache lines is a miss of its own, and the compiler would load
// them one behind the other, where they are used.  (With this, and no blockDim, which is a load from memory behind another one, and no
// division in front of the first load of a row, a launch of a decode step takes 0.2 us less: 1565 -> 1535 us a token of a 4B model.)
__device__ __forceinline__ void touch_args(const GemvArgs& a) {
  static_assert(offsetof(GemvArgs, m) + sizeof(TileMat) * kMaxGroup <= 256, "four lines");
  asm volatile("" ::"s"(a.in.norm_w), "s"(a.nb), "s"(a.m[1].d_out), "s"(a.m[3].slots));
}

struct GemvLds {
  float* xtail;      // [32]
  float* red;        // [16]
  uint32_t* planes;  // [plane units][XPlanes::kDwords]
  float* part;       // [sums_room][16 rows]
  float* xf;         // [d_in] f32 values of a rotated activation, in the same place: they are in the planes before there are sums
};
template <int DIG>
__device__ __forceinline__ GemvLds gemv_lds(uint8_t* smem, uint32_t plane_units) {
  GemvLds L;
  L.xtail = reinterpret_cast<float*>(smem);
  L.red = L.xtail + 32;
  L.planes = reinterpret_cast<uint32_t*>(L.red + 16);
  L.part = reinterpret_cast<float*>(L.planes + (size_t)plane_units * XPlanes<DIG>::kDwords);
  L.xf = L.part;
  return L;
}

__device__ __forceinline__ uint32_t pack_halves(float lo, float hi) {
  return (uint32_t)__half_as_ushort(__float2half_rn(lo)) | (uint32_t)__half_as_ushort(__float2half_rn(hi)) << 16;
}
__device__ __forceinline__ float round_half(float v) { return __half2float(__float2half_rn(v)); }
__device__ __forceinline__ float silu_mul(float gate, float up) { return round_half(round_half(gate / (1.0f + __expf(-gate))) * up); }

// Activations that another workgroup of the same launch stores (gemv_seq.h) are loaded at device scope, dword by dword.
template <bool kDeviceScope>
__device__ __forceinline__ void load_halves(const __half* p, uint32_t (&w)[4]) {
  if constexpr (kDeviceScope) {
    if ((reinterpret_cast<uintptr_t>(p) & 3u) == 0) {
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = __hip_atomic_load(reinterpret_cast<const uint32_t*>(p) + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        w[j] = (uint32_t)__half_as_ushort(load_half<true>(p + 2 * j)) | (uint32_t)__half_as_ushort(load_half<true>(p + 2 * j + 1)) << 16;
    }
  } else {
    const HalfOctet o = *reinterpret_cast<const HalfOctet*>(p);
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = o.w[j];
  }
}

// Fills the planes and the tail values in LDS from `in`, by every lane of the workgroup.
// `request` is called once, behind the loads of the activation's operands: the first weights go out there.  (With a
// barrier in front, so that no wavefront's operands come behind the others' weights, a decode step took 3 % longer.  A
// rotation in octets has it behind the levels in registers: loads come back in order, and with the weights right behind the
// operands the first wavefronts' weights kept the last ones' operands waiting.  2560 x 9728 on the card: 11.35 us, and 11.1
// so; a rotated 14B decode of 8 tokens 4365 and 4265 us; behind the first barrier of rotate_rest, 4335.)
// PMAX: how often the workgroup's quads pass over the padded blocks, at most; `waves`, `passes`: its wavefronts and how often that is
// (stage_passes).  store_resid: this workgroup is the one that stores the new residual.  Ends without a barrier.
template <int DIG, int SRC, int PMAX, bool kDeviceScope = false, class Request>
__device__ __forceinline__ void stage_x(const ActivationIn& in, uint32_t nb, uint32_t tail_w, uint32_t waves, uint32_t passes, const GemvLds& L,
                                        bool store_resid, Request&& request) {
  const uint32_t tid = threadIdx.x, n_thr = waves * 64u, lane = tid & 63u, wave = tid >> 6;
  const uint32_t sub = tid & 3u, quad = tid >> 2, quads = n_thr >> 2;
  const uint32_t pad = tile_steps(nb) * kStepBlocks, d_in = nb * kDim + tail_w;
  auto zeros = [&]() {  // past the tail, and the step of zeros
    if (tid < 32u) L.xtail[tid] = 0.f;
    for (uint32_t i = tid; i < kStepUnits * XPlanes<DIG>::kDwords; i += n_thr) L.planes[plane_at<DIG>(pad) + i] = 0u;
  };
  if constexpr (SRC == kSrcRotated) {
    // The activation is rotated into LDS and quantised from there (what it is made of is binary16).
    // A launch in a rotated basis has 1024 lanes.
    float* xf = L.xf;
    zeros();
    const RotTable* table = reinterpret_cast<const RotTable*>(in.rot_fragments);
    const bool norm = in.prologue == kPrologueAddRmsNorm, silu = in.prologue == kPrologueSiluMul;
    auto norm_scale = [&](float ss) {
      ss = wave_sum(ss);
      if (lane == 0) L.red[wave] = ss;
      lds_barrier();
      float total = 0.f;
      for (uint32_t w = 0; w < 16u; ++w) total += L.red[w];
      return 1.0f / sqrtf(total / (float)d_in + in.eps);
    };
    if (in.rot_m >= kRotOctetM) {
      // Every operand of a wavefront's tile is requested before the first is used.
      // (Rows past sixteen tiles: a second turn.  Those have no norm in front: a decoder's hidden size ends at 8192.)
      const uint8_t* signs = reinterpret_cast<const uint8_t*>(in.rot_signbits);
      HalfOctet a[2] = {}, b[2] = {}, g[2] = {};
      uint32_t sg[2] = {0, 0};
      rot_h8_t h[2] = {};
      auto load_tile = [&](uint32_t tile) {
#pragma unroll
        for (uint32_t i = 0; i < 2u; ++i) {
          const uint32_t from = rot_octet_at(tile, i) < d_in ? rot_octet_at(tile, i) : 0u;
          if (norm) g[i] = *reinterpret_cast<const HalfOctet*>(in.norm_w + from);
          if (in.x2) b[i] = *reinterpret_cast<const HalfOctet*>(in.x2 + from);
          a[i] = *reinterpret_cast<const HalfOctet*>(in.x + from);
          sg[i] = signs[from >> 3];
        }
      };
      // (A wavefront without a tile asks for none: loads of sixteen wavefronts that nobody uses are a microsecond in front of the weights'.)
      const bool has_tile = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave) * kRotTile < d_in;
      if (has_tile) {
        load_tile(wave);
        h[0] = table->lane[lane].h[0];
        h[1] = table->lane[lane].h[1];
      }
      __builtin_amdgcn_sched_barrier(0);
      float inv = 0.f;
      if (norm) {
        float ss = 0.f;
#pragma unroll
        for (uint32_t i = 0; i < 2u; ++i) {
          if (rot_octet_at(wave, i) >= d_in) continue;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            float lo = half_lo(a[i].w[j]), hi = half_hi(a[i].w[j]);
            if (in.x2) {
              lo = round_half(lo + half_lo(b[i].w[j]));
              hi = round_half(hi + half_hi(b[i].w[j]));
            }
            a[i].w[j] = pack_halves(lo, hi);
            ss = fmaf(lo, lo, fmaf(hi, hi, ss));
          }
          if (in.resid_out && store_resid) *reinterpret_cast<HalfOctet*>(in.resid_out + rot_octet_at(wave, i)) = a[i];
        }
        inv = norm_scale(ss);
      }
#pragma unroll 1
      for (uint32_t tile = wave; tile * kRotTile < d_in; tile += 16u) {
        uint32_t x[2][4];
#pragma unroll
        for (uint32_t i = 0; i < 2u; ++i) {
          if (silu) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
              a[i].w[j] = pack_halves(silu_mul(half_lo(b[i].w[j]), half_lo(a[i].w[j])), silu_mul(half_hi(b[i].w[j]), half_hi(a[i].w[j])));
          } else if (norm) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
              a[i].w[j] = pack_halves(half_lo(a[i].w[j]) * inv * half_lo(g[i].w[j]), half_hi(a[i].w[j]) * inv * half_hi(g[i].w[j]));
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) x[i][j] = rot_octet_at(tile, i) < d_in ? flip_signs(a[i].w[j], sg[i], j) : 0u;
        }
        if ((tile + 16u) * kRotTile < d_in) load_tile(tile + 16u);  // (on their way beside this tile's levels)
        rotate_tile_to<false>(xf, x[0], x[1], h, tile, d_in, in.rot_m, in.rot_k, in.rot_inv);
      }
      request();
    } else {
      auto put = [&](uint32_t i, float v) { xf[i] = flip_sign(v, in.rot_signbits[i >> 5] >> (i & 31u), 0); };
      if (norm) {
        float ss = 0.f;
        for (uint32_t i = tid; i < d_in; i += n_thr) {
          float r = __half2float(in.x[i]);
          if (in.x2) r = round_half(r + __half2float(in.x2[i]));
          if (in.resid_out && store_resid) in.resid_out[i] = __float2half_rn(r);
          xf[i] = r;
          ss += r * r;
        }
        request();
        const float inv = norm_scale(ss);
        for (uint32_t i = tid; i < d_in; i += n_thr) put(i, round_half(xf[i] * inv * __half2float(in.norm_w[i])));
      } else {
        for (uint32_t i = tid; i < d_in; i += n_thr)
          put(i, silu ? silu_mul(__half2float(in.x2[i]), __half2float(in.x[i])) : __half2float(in.x[i]));
        request();
      }
    }
    const RotBlock block = rot_block(table, in.rot_m, in.rot_k);
    lds_barrier();
    rotate_rest<false>(xf, d_in, in.rot_m, in.rot_k, in.rot_inv, table, block, in.rot_m < kRotOctetM);
    lds_barrier();
#pragma unroll 1
    for (uint32_t p = 0; p < passes; ++p) {
      const uint32_t blk = quad + p * quads;
      if (blk >= pad) break;
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = 0.f;
      if (blk < nb && sub < 3u) {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = xf[blk * kDim + sub * 8u + j];
      }
      quantize_octet<DIG, false>(v, sub, L.planes + plane_at<DIG>(blk), L.planes + plane_sum_at<DIG>(blk));
    }
    if (tid < tail_w) L.xtail[tid] = xf[nb * kDim + tid];
  } else if constexpr (SRC == kSrcFinished) {
    // Every value is asked for in front of the weights: loads come back in order.
    struct __attribute__((packed, aligned(4))) Four { float v[4]; };
    float v[PMAX][8] = {};
    if (nb) {
#pragma unroll
      for (int p = 0; p < PMAX; ++p) {
        const uint32_t blk = quad + (uint32_t)p * quads, at = blk < nb && sub < 3u ? blk * kDim + sub * 8u : 0u;
        const Four a = *reinterpret_cast<const Four*>(in.x_f32 + at), b = *reinterpret_cast<const Four*>(in.x_f32 + at + 4u);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[p][j] = a.v[j];
          v[p][4 + j] = b.v[j];
        }
      }
    }
    const float t = in.x_f32[min(nb * kDim + tid, d_in - 1u)];
    __builtin_amdgcn_sched_barrier(0);
    request();
    __builtin_amdgcn_sched_barrier(0);
    zeros();
#pragma unroll
    for (int p = 0; p < PMAX; ++p) {
      const uint32_t blk = quad + (uint32_t)p * quads;
      if (blk >= pad) break;
#pragma unroll
      for (int j = 0; j < 8; ++j) v[p][j] = blk < nb && sub < 3u ? v[p][j] : 0.f;
      quantize_octet<DIG, true>(v[p], sub, L.planes + plane_at<DIG>(blk), L.planes + plane_sum_at<DIG>(blk));
    }
    if (tid < tail_w) L.xtail[tid] = t;
  } else {
    // One or two passes at a time, every operand requested before the first is used; a lane without columns reads the
    // row's first.  The norm's sum comes between two walks: the first leaves the summed values, as binary16, where the
    // second puts the block's planes (or, when two passes are all, in the registers).
    constexpr int kChunk = PMAX > 2 && DIG == 6 ? 1 : 2;
    const __half* second = SRC == kSrcAddRmsNorm ? (in.x2 ? in.x2 : in.x) : in.x2;
    uint32_t a[kChunk][4], b[kChunk][4], g[kChunk][4];
    auto block_of = [&](uint32_t p) { return quad + p * quads; };
    auto load_operands = [&](uint32_t p0) {
#pragma unroll
      for (int k = 0; k < kChunk; ++k) {
        const uint32_t blk = block_of(p0 + (uint32_t)k);
        const uint32_t at = (blk < nb && sub < 3u) ? blk * kDim + sub * 8u : 0u;
#pragma unroll
        for (int j = 0; j < 4; ++j) a[k][j] = b[k][j] = g[k][j] = 0u;
        if (p0 + (uint32_t)k < passes && nb) {
          load_halves<kDeviceScope>(in.x + at, a[k]);
          if constexpr (SRC != kSrcF16) load_halves<kDeviceScope>(second + at, b[k]);
          if constexpr (SRC == kSrcAddRmsNorm && PMAX <= kChunk) load_halves<false>(in.norm_w + at, g[k]);
        }
      }
    };
    auto emit = [&](int k, uint32_t blk, float inv) {  // a[k] (and b, g) -> the planes of block blk
      const bool ok = blk < nb && sub < 3u;
      uint32_t w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float lo = half_lo(a[k][j]), hi = half_hi(a[k][j]);
        w[j] = a[k][j];
        if constexpr (SRC == kSrcSiluMul) w[j] = pack_halves(silu_mul(half_lo(b[k][j]), lo), silu_mul(half_hi(b[k][j]), hi));
        if constexpr (SRC == kSrcAddRmsNorm) w[j] = pack_halves(lo * inv * half_lo(g[k][j]), hi * inv * half_hi(g[k][j]));
        w[j] = ok ? w[j] : 0u;
      }
      quantize_halves<DIG>(w, sub, L.planes + plane_at<DIG>(blk), L.planes + plane_sum_at<DIG>(blk));
    };
    load_operands(0);
    const uint32_t t_at = min(nb * kDim + tid, d_in - 1u);
    float t0 = __half2float(load_half<kDeviceScope>(in.x + t_at)), t1 = 0.f, tg = 0.f;
    if constexpr (SRC != kSrcF16) t1 = __half2float(load_half<kDeviceScope>(second + t_at));
    if constexpr (SRC == kSrcAddRmsNorm) tg = __half2float(in.norm_w[t_at]);
    request();
    __builtin_amdgcn_sched_barrier(0);
    zeros();
    float inv = 0.f;
    if constexpr (SRC == kSrcAddRmsNorm) {
      float ss = 0.f;
      auto add_up = [&](uint32_t p0) {
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
          const uint32_t blk = block_of(p0 + (uint32_t)k);
          if (blk < nb && sub < 3u) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              float lo = half_lo(a[k][j]), hi = half_hi(a[k][j]);
              if (in.x2) {
                lo = round_half(lo + half_lo(b[k][j]));
                hi = round_half(hi + half_hi(b[k][j]));
              }
              a[k][j] = pack_halves(lo, hi);
              ss = fmaf(lo, lo, fmaf(hi, hi, ss));
            }
            if (in.resid_out && store_resid) {
              __half* dst = in.resid_out + blk * kDim + sub * 8u;
              if constexpr (kDeviceScope) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                  store_half<true>(dst + 2 * j, __ushort_as_half((unsigned short)(a[k][j] & 0xFFFFu)));
                  store_half<true>(dst + 2 * j + 1, __ushort_as_half((unsigned short)(a[k][j] >> 16)));
                }
              } else {
                HalfOctet o;
#pragma unroll
                for (int j = 0; j < 4; ++j) o.w[j] = a[k][j];
                *reinterpret_cast<HalfOctet*>(dst) = o;
              }
            }
            if constexpr (PMAX > kChunk) {
              uint32_t* keep = L.planes + plane_at<DIG>(blk) + sub * 4u;
#pragma unroll
              for (int j = 0; j < 4; ++j) keep[j] = a[k][j];
            }
          }
        }
      };
      add_up(0);
      if constexpr (PMAX > kChunk) {
#pragma unroll 1
        for (uint32_t p0 = kChunk; p0 < passes; p0 += kChunk) {
          load_operands(p0);
          add_up(p0);
        }
      }
      if (tid < tail_w) {
        if (in.x2) t0 = round_half(t0 + t1);
        if (in.resid_out && store_resid) store_half<kDeviceScope>(in.resid_out + nb * kDim + tid, __float2half_rn(t0));
        ss = fmaf(t0, t0, ss);
      }
      ss = wave_sum(ss);
      if (lane == 0) L.red[wave] = ss;
      lds_barrier();
      float total = 0.f;
      for (uint32_t w = 0; w < waves; ++w) total += L.red[w];
      inv = 1.0f / sqrtf(total / (float)d_in + in.eps);
    }
    if constexpr (SRC == kSrcAddRmsNorm && PMAX > kChunk) {
#pragma unroll 1
      for (uint32_t p = 0; p < passes; ++p) {
        const uint32_t blk = block_of(p);
        if (blk >= pad) break;
        const bool ok = blk < nb && sub < 3u;
        const uint32_t* kept = L.planes + plane_at<DIG>(blk) + sub * 4u;
#pragma unroll
        for (int j = 0; j < 4; ++j) a[0][j] = ok ? kept[j] : 0u;
        load_halves<false>(in.norm_w + (ok ? blk * kDim + sub * 8u : 0u), g[0]);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the quad's four lanes have read what they now overwrite
        emit(0, blk, inv);
      }
    } else {
#pragma unroll
      for (int k = 0; k < kChunk; ++k)
        if (block_of((uint32_t)k) < pad) emit(k, block_of((uint32_t)k), inv);
      if constexpr (PMAX > kChunk) {
#pragma unroll 1
        for (uint32_t p0 = kChunk; p0 < passes; p0 += kChunk) {
          load_operands(p0);
#pragma unroll
          for (int k = 0; k < kChunk; ++k)
            if (block_of(p0 + (uint32_t)k) < pad) emit(k, block_of(p0 + (uint32_t)k), inv);
        }
      }
    }
    if (tid < tail_w) {
      if constexpr (SRC == kSrcSiluMul) t0 = silu_mul(t1, t0);
      if constexpr (SRC == kSrcAddRmsNorm) t0 = round_half(t0 * inv * tg);
      L.xtail[tid] = t0;
    }
  }
}

// A lane's share of a step: five pieces of a unit, two rows by four blocks.
struct StepWords {
  u32x4_t p[5];
};
// What a lane adds to a tile's address for its unit of a step (units past the last repeat it: they meet zeros in the planes).
__device__ __forceinline__ uint32_t step_offset(uint32_t step, uint32_t units, uint32_t head, uint32_t lane) {
  const uint32_t u = min(step * kStepUnits + (lane >> 3), max(units, 1u) - 1u);
  return head + u * kUnitBytes + (lane & 7u) * 16u;
}
// A scalar base the compiler cannot take apart again: loads through it add a 32-bit lane offset.
__device__ __forceinline__ const uint8_t* scalar_base(const uint8_t* p) {
  typedef const uint8_t __attribute__((address_space(1))) global_u8;
  uint64_t bits = reinterpret_cast<uint64_t>(uniform_global(p));
  asm("" : "+s"(bits));
  return (const uint8_t*)reinterpret_cast<global_u8*>(bits);
}
template <int P>
__device__ __forceinline__ void load_piece(StepWords& W, const uint8_t* base, uint32_t off) {
  W.p[P] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(base + off + P * 128u));
}
__device__ __forceinline__ void load_step(StepWords& W, const uint8_t* base, uint32_t off) {
  load_piece<0>(W, base, off);
  load_piece<1>(W, base, off);
  load_piece<2>(W, base, off);
  load_piece<3>(W, base, off);
  load_piece<4>(W, base, off);
}

// The block scales, two lanes to each: a block's meta byte is the address of its own in them (a lane's register is at four
// times its number, and the two lowest bits don't count).
__device__ __forceinline__ uint32_t scale_table(const uint8_t* base, uint32_t lane) {
  return reinterpret_cast<const uint32_t*>(base)[lane >> 1];
}
__device__ __forceinline__ float scale_at(uint32_t meta, uint32_t table) {
  return __int_as_float(__builtin_amdgcn_ds_bpermute((int)meta, (int)table));
}

// first + the sum of a block's digit products, exact, from the top digit down.  (One chain: each step of it waits a little
// for the one before, which the other wavefronts of a SIMD fill; two side by side take two more instructions.)
template <int DIG>
__device__ __forceinline__ int digits_sum(const uint32_t (&w)[3], const int (&x)[3 * DIG], int first) {
  int t = 0;
#pragma unroll
  for (int k = DIG - 1; k >= 0; --k) {
    if (k != DIG - 1) t = (t << 4) + (k ? 0 : first);
#pragma unroll
    for (int o = 0; o < 3; ++o) t = __builtin_amdgcn_sdot8((int)w[o], x[3 * k + o], t, false);
  }
  return t;
}
// a * b + c, a and b of 24 bits
__device__ __forceinline__ int mad24_lanes(int a, int b, int c) {
  int r;  // (the compiler would extend the factors first)
  asm("v_mad_i32_i24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// One block's part in a product: acc + sum of (n + win - 3) x, exact but for the f32 conversion, scaled by the block's weight
// scale and the activation's.  12 or 18 dot products and about 18 more instructions.
struct BlockTerm {
  uint32_t w[3], win;
  float c;
};
// K: the block in its unit; s, m: its row's {s, meta} dwords.  (An escape's scale is zero here: tile_extras sees to it.)
template <int DIG, int K>
__device__ __forceinline__ BlockTerm block_term(uint32_t d0, uint32_t d1, uint32_t s, uint32_t m, uint32_t table) {
  BlockTerm b;
  block_octets(d0, d1, s << (3 - K), b.w);
  const uint32_t meta = m >> (8 * K);
  b.win = meta & 7u;
  b.c = scale_at(meta, table);
  return b;
}
// sum, less: the sum of the block's integers x, and -3 times that (four digits' sums have 20 bits).
template <int DIG>
__device__ __forceinline__ float block_sum(const BlockTerm& b, const int (&x)[3 * DIG], int sum, int less, float scale, float acc) {
  const int t = digits_sum<DIG>(b.w, x, DIG == 4 ? mad24_lanes((int)b.win, sum, less) : (int)b.win * sum + less);
  return fmaf((float)t, b.c * scale, acc);
}

// A block's digit planes.
template <int DIG>
__device__ __forceinline__ void load_planes(const uint32_t* xb, int (&x)[3 * DIG]) {
  if constexpr (DIG == 4) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(xb + 4 * i);
#pragma unroll
      for (int j = 0; j < 4; ++j) x[4 * i + j] = (int)v[j];
    }
  } else {
#pragma unroll
    for (int i = 0; i < 3 * DIG / 2; ++i) {
      const u32x2_t v = *reinterpret_cast<const u32x2_t*>(xb + 2 * i);
      x[2 * i] = (int)v.x;
      x[2 * i + 1] = (int)v.y;
    }
  }
}

// A step's products, rows l and l + 8 of the tile: what the lane's four blocks add up to.  xq: the unit's planes.
// `reload(p)` is called for every piece as soon as its registers are free: what is to be loaded next goes out there.
template <int DIG, class Reload>
__device__ __forceinline__ void step_product(const StepWords& W, const uint32_t* xq, uint32_t table, float& lo, float& hi, Reload&& reload) {
  lo = hi = 0.f;
  auto block = [&](auto block_k) __attribute__((always_inline)) {
    constexpr int K = decltype(block_k)::value;
    int x[3 * DIG];
    load_planes<DIG>(xq + K * XPlanes<DIG>::kBlock, x);
    const u32x2_t ss = *reinterpret_cast<const u32x2_t*>(xq + XPlanes<DIG>::kSums + 2 * K);
    const int sum = (int)ss.x, less = DIG == 4 ? __mul24(sum, -3) : sum * -3;
    const float scale = __uint_as_float(ss.y);
    const BlockTerm a = block_term<DIG, K>(W.p[K >> 1][2 * (K & 1)], W.p[K >> 1][2 * (K & 1) + 1], W.p[4].x, W.p[4].y, table);
    const BlockTerm b = block_term<DIG, K>(W.p[2 + (K >> 1)][2 * (K & 1)], W.p[2 + (K >> 1)][2 * (K & 1) + 1], W.p[4].z, W.p[4].w, table);
    lo = block_sum<DIG>(a, x, sum, less, scale, lo);
    hi = block_sum<DIG>(b, x, sum, less, scale, hi);
    __builtin_amdgcn_sched_barrier(0);  // the registers are free again only now: the loads need no others, and the products of several blocks at once would not fit
  };
  block(std::integral_constant<int, 0>{});
  block(std::integral_constant<int, 1>{});
  reload(std::integral_constant<int, 0>{});
  reload(std::integral_constant<int, 2>{});
  __builtin_amdgcn_sched_barrier(0);
  block(std::integral_constant<int, 2>{});
  block(std::integral_constant<int, 3>{});
  reload(std::integral_constant<int, 1>{});
  reload(std::integral_constant<int, 3>{});
  reload(std::integral_constant<int, 4>{});
  __builtin_amdgcn_sched_barrier(0);
}

// The sum over the four classes of a row (row_lane), in every lane of it.
__device__ __forceinline__ float classes_sum(float v) {
  v += dpp_move<0x128>(v);  // row_ror:8
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}
// The sums over a step's units of rows l (lo) and l + 8 (hi): row lane_row(lane)'s in every lane.
__device__ __forceinline__ float rows_sum(float lo, float hi) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(lo), __float_as_uint(hi), false, false);
  return classes_sum(__uint_as_float(p[0]) + __uint_as_float(p[1]));
}

// What a tile adds to its rows besides its steps, as one wavefront loads it: the row scales, the tail columns (a lane's
// share, the neighbours' behind it), the escapes.
struct TileExtras {
  float scale;
  u32x4_t tail;
  u32x2_t tail2;
  uint32_t count;
  u32x4_t escape;
};
// (not live: not to be used, and one cache line)
__device__ __forceinline__ TileExtras load_extras(const uint8_t* rec, uint32_t nb, uint32_t tail_w, uint32_t slots, bool live, uint32_t lane) {
  struct __attribute__((packed, aligned(4))) W4 { u32x4_t w; };
  struct __attribute__((packed, aligned(4))) W2 { u32x2_t w; };
  const uint32_t depth = tail_depth(tail_w), at = live & (depth != 0u) ? 128u + lane * depth * 4u : 0u;
  TileExtras x;
  x.scale = reinterpret_cast<const float*>(rec)[live ? lane_row(lane) : 0u];
  x.count = *reinterpret_cast<const uint32_t*>(rec + kCountAt);
  x.tail = reinterpret_cast<const W4*>(rec + at)->w;
  x.tail2 = reinterpret_cast<const W2*>(rec + at + (live & (depth > 4u) ? 16u : 0u))->w;
  x.escape = *reinterpret_cast<const u32x4_t*>(rec + (live & (slots != 0u) ? list_at(nb, tail_w) + min(lane, slots - 1u) * 16u : 0u));
  return x;
}
// The rows' tail columns and escapes, the latter by the row scales: row lane_row(lane)'s in every lane.  A lane takes an
// escape of the list, and a row adds up its own in their order.
template <int DIG>
__device__ __forceinline__ float tile_extras(const TileExtras& X, const uint8_t* rec, uint32_t nb, uint32_t tail_w, uint32_t slots, uint32_t table,
                                             const GemvLds& L, uint32_t lane) {
  const uint32_t depth = tail_depth(tail_w);
  float t = 0.f;
#pragma unroll
  for (uint32_t i = 0; i < 6; ++i)
    if (i < depth) t = fmaf(__uint_as_float(i < 4u ? X.tail[i & 3u] : X.tail2[i & 1u]), L.xtail[4u * i + lane_class(lane)], t);
  t = classes_sum(t);
  const uint32_t count = (uint32_t)__builtin_amdgcn_readfirstlane((int)X.count);
  if (count == 0u) return t;
  float sum = 0.f;
  auto to_rows = [&](float f, uint32_t key, uint32_t n) {  // those of lanes 0 .. n - 1
    for (uint32_t e = 0; e < n; ++e) {
      const uint32_t row = (uint32_t)__builtin_amdgcn_readlane((int)key, (int)e) >> 28;
      const float p = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), (int)e));
      sum += lane_row(lane) == row ? p : 0.f;
    }
  };
  if (__builtin_expect(count <= slots, 1)) {
    auto listed = [&](const u32x4_t& e, uint32_t n) __attribute__((always_inline)) {
      const uint32_t key = lane < n ? e.w : 0u, blk = (key >> 9) & 0x7FFFFu, w[3] = {e.x, e.y, e.z};  // (the others: any block that is there)
      int x[3 * DIG];
      load_planes<DIG>(L.planes + plane_at<DIG>(blk), x);
      const u32x2_t ss = *reinterpret_cast<const u32x2_t*>(L.planes + plane_sum_at<DIG>(blk));
      const int v = (digits_sum<DIG>(w, x, 0) << 1) + ((key >> 8) & 1u ? (int)ss.x : 0);
      to_rows((float)v * (scale_at((key & 31u) << 3, table) * __uint_as_float(ss.y)), key, n);
    };
    listed(X.escape, min(count, 64u));
    if (__builtin_expect(count > 64u, 0)) {  // (a loop instead: 0.1 us of every launch)
      asm volatile("" : "+s"(nb), "+s"(tail_w));  // (as below)
      listed(*reinterpret_cast<const u32x4_t*>(rec + list_at(nb, tail_w) + min(64u + lane, slots - 1u) * 16u), count - 64u);
    }
  } else {
    // More than there was room for: the tile's meta dwords step by step, the next one's on their way, and of the escapes they show one to a
    // lane; those are read 64 at a time.  A launch of 5.6 us takes 10.5 with a tile of twenty (every block of one row after the other, a load
    // to wait for each 64: 30; four steps' dwords together, each with loops of its own: 8.3, and 3 KB more of each of these kernels, which is
    // up to 1 % of a decoded token).
    asm volatile("" : "+s"(nb), "+s"(tail_w), "+v"(lane));  // (what is made of them is made here, and not ahead of the launch's tiles)
    const uint32_t steps = tile_steps(nb), units = tile_units(nb), head = tile_head_bytes(tail_w);
    auto masks = [&](uint32_t s) {
      const uint32_t* piece = reinterpret_cast<const uint32_t*>(rec + step_offset(s, units, head, lane) + 512u);
      return u32x2_t{piece[1], piece[3]};
    };
    u32x2_t next = masks(0);
    uint32_t step = 0, mask = 0, key = 0, n = 0;  // (key: of the lanes without one any block that is there)
#pragma unroll 1
    for (;;) {
      const uint64_t left = __builtin_amdgcn_ballot_w64(mask != 0u);
      if (left != 0u && n < 64u) {
        const uint32_t of = (uint32_t)__builtin_ctzll(left), m = (uint32_t)__builtin_amdgcn_readlane((int)mask, of);
        key = lane == n ? walk_key(step - 1u, of, (uint32_t)__builtin_ctz(m)) : key;
        mask = lane == of ? m & (m - 1u) : mask;
        ++n;
      } else if (left == 0u && step < steps) {
        mask = step * kStepUnits + (lane >> 3) < units ? walk_mask(next.x, next.y) : 0u;
        ++step;
        next = masks(step);  // (past the last: units that are there)
      } else {
        const uint32_t blk = key & 0xFFFFFFFu, r = key >> 28, k = blk & 3u;
        const uint8_t* unit = rec + head + (blk >> 2) * kUnitBytes + (r & 7u) * 16u;
        const u32x2_t d = *reinterpret_cast<const u32x2_t*>(unit + ((r >> 3) * 2u + (k >> 1)) * 128u + (k & 1u) * 8u);
        const u32x2_t sm = *reinterpret_cast<const u32x2_t*>(unit + 512u + (r >> 3) * 8u);
        uint32_t w[3];
        block_octets(d.x, d.y, sm.x << (3u - k), w);
        const BlockEscape e = block_escape(w, (sm.y >> (8u * k)) & 255u);
        w[0] = e.w0;
        int x[3 * DIG];
        load_planes<DIG>(L.planes + plane_at<DIG>(blk), x);
        const u32x2_t ss = *reinterpret_cast<const u32x2_t*>(L.planes + plane_sum_at<DIG>(blk));
        const uint32_t bit = 1u << (4u * (e.at & 7u));  // the coordinate that is 16 below, by itself
        const uint32_t one[3] = {e.at < 8u ? bit : 0u, (e.at >> 3) == 1u ? bit : 0u, (e.at >> 3) == 2u ? bit : 0u};
        const int v = digits_sum<DIG>(w, x, ((int)e.win - 3) * (int)ss.x) - (digits_sum<DIG>(one, x, 0) << 4);
        to_rows((float)(e.negative ? -v : v) * (scale_at(e.slot << 3, table) * __uint_as_float(ss.y)), key, n);
        if (left == 0u) break;
        key = n = 0;
      }
    }
  }
  return fmaf(sum, X.scale, t);
}

// A row's blocks from what its steps left in LDS (sixteen rows a step).
template <uint32_t MAX>
__device__ __forceinline__ float steps_sum(const float* part, uint32_t steps, uint32_t lane) {
  float v[MAX / 4], t = 0.f;
#pragma unroll
  for (uint32_t i = 0; i < MAX / 4; ++i) {
    const uint32_t s = 4u * i + lane_class(lane);
    v[i] = part[sums_read(i, lane_class(lane)) * kTileRows + lane_row(lane)];
    v[i] = s < steps ? v[i] : 0.f;
  }
#pragma unroll
  for (uint32_t i = 0; i < MAX / 4; ++i) t += v[i];
  return classes_sum(t);
}

__device__ __forceinline__ void tile_mat(const GemvArgs& a, uint32_t tile, const uint8_t*& base, void*& y, uint32_t& row0, uint32_t& d_out,
                                         uint32_t& stride, uint32_t& slots) {
  base = a.m[0].base;  // constant indices only: a dynamic one would move the arguments to scratch
  y = a.m[0].y;
  d_out = a.m[0].d_out;
  stride = a.m[0].stride;
  slots = a.m[0].slots;
  uint32_t begin = 0;
#pragma unroll
  for (uint32_t k = 1; k < kMaxGroup; ++k)
    if (k < a.n_mats && tile >= a.m[k].tile_begin) {
      base = a.m[k].base;
      y = a.m[k].y;
      d_out = a.m[k].d_out;
      stride = a.m[k].stride;
      slots = a.m[k].slots;
      begin = a.m[k].tile_begin;
    }
  row0 = (tile - begin) * kTileRows;
}

// y = W x for the rows of up to four matrices that share an activation.
//
// What bounds it: at 10 bytes per block and about 35 vector instructions the weights' way from memory; in a launch of
// a few microseconds the chain launch -> activation -> planes -> product -> store.  So: a team of wavefronts takes a tile of
// sixteen rows, a wavefront a fixed step of it; a tile's loads are all in flight before the
// planes are ready, and each piece's registers are loaded again for the team's next tile as soon as they have been used,
// without a branch, so that every wait is for the oldest load only.  The planes of a unit are read from LDS once for
// the two rows a lane has.  The sums over a team's wavefronts wait in LDS for one barrier per gemv_batch tiles, behind which
// every wavefront finishes one.  The host spreads teams over the CUs first, tiles over teams so that the last, partial round
// meets every CU.
//
// WIDE, rows past 512 blocks, more steps than wavefronts: a workgroup's steps go to its wavefronts in turn (GemvSpread), across the ends of
// tiles.  (As a team with two steps of a tile each, 23 steps were 32, both steps' registers were waited for together and a second tile began
// when both were done: 5120 x 17408 14.4 -> 12.0 us, 4096 x 17408 10.8 -> 8.6, 18000 x 14000 25.7 -> 20.6, rotated 5120 x 17408 21.6 -> 19.7.
// Narrower rows gain nothing from it, or 3 to 7 % where rows of nine to thirteen steps leave a team's workgroup wavefronts without one and
// there are many, and lose up to 7 % elsewhere: 18000 x 4096 8.35 -> 8.95 us, their last wavefronts having steps beside the first tiles' ends.)
//
// GATED: the two matrices are a layer's gate and up, and what is stored is f16(f16(silu(gate)) up) of their rows, both rounded to
// binary16 first (model.rs:831): the bits that the product behind it makes of the two results otherwise, in every one of its workgroups
// (two passes of an exponential and a division for 9728 columns, 2.4 us).  A row's two tiles are neighbouring slots of one workgroup; the
// wavefront of the up tile leaves its scales and extras in LDS in front of the barrier that is there anyway.
template <typename OutT, int SRC, bool WIDE, bool GATED>
__device__ __forceinline__ void tiles_product(const GemvArgs& a) {
  constexpr int DIG = std::is_same<OutT, __half>::value ? 4 : 6;
  static_assert(!(WIDE && GATED), "a pair's tiles are a team's");
  extern __shared__ __align__(16) uint8_t smem[];
  touch_args(a);
  const GemvLds L = gemv_lds<DIG>(smem, gemv_plane_units(a.nb));
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t team = (wave * a.g.inv_team) >> 16, w = wave - team * a.g.team, n_teams = a.g.teams * a.g.grid;
  const uint32_t nb = a.nb, n_steps = tile_steps(nb), units = tile_units(nb), head = tile_head_bytes(a.tail_w);

  struct Record { const uint8_t* rec; const uint8_t* base; uint32_t slots; };
  // A workgroup's slot i of tiles is tile i * grid + its number; with GATED that tile of pairs of slots, the even one in the first matrix.
  const uint32_t n_tiles = GATED ? a.m[1].tile_begin : a.n_tiles;
  auto tile_of = [&](uint32_t slot) { return (GATED ? slot >> 1 : slot) * a.g.grid + blockIdx.x; };
  auto record_of = [&](uint32_t t, uint32_t slot) {
    const uint8_t* base;
    void* y;
    uint32_t row0, d_out, stride, slots;
    if constexpr (GATED) {
      const bool up = slot & 1u;
      base = up ? a.m[1].base : a.m[0].base;
      stride = up ? a.m[1].stride : a.m[0].stride;
      slots = up ? a.m[1].slots : a.m[0].slots;
      row0 = t * kTileRows;
    } else {
      tile_mat(a, t, base, y, row0, d_out, stride, slots);
    }
    return Record{base + kTileTableBytes + (size_t)(row0 / kTileRows) * stride, base, slots};
  };
  // Teams: step w of every tile of the wavefront's is its own (of n_steps and more: none).  WIDE: step `step` of slot `slot`, the sixteenth
  // behind it the next time.  Where a wavefront has no step, or no next one, its loads repeat one: one cache line, and no branch.
  const GemvSpread spread = spread_of(a.g);
  const uint32_t slots = WIDE ? spread.slots - (blockIdx.x < spread.full ? 0u : 1u) : 0u;
  uint32_t off = step_offset(w, units, head, lane);
  uint32_t tile = team < (WIDE ? slots : a.g.teams) ? tile_of(team) : 0xFFFFFFFFu;
  Record cur = record_of(min(tile, n_tiles - 1u), team);
  StepWords W;
  uint32_t table;
  // The tile that this wavefront finishes of those whose rounds begin with r0: the last wavefronts see to the first tiles, since what a tile
  // has besides its steps (tile_extras, 0.8 us for one wavefront) is then not in front of anybody's products where there are
  // wavefronts without any.
  const uint32_t fin = a.g.waves - 1u - wave, batch = WIDE ? spread.batch : gemv_batch(a.g.team);
  const uint32_t my_round = WIDE ? fin : (fin * a.g.inv_teams) >> 16, my_team = WIDE ? 0u : fin - my_round * a.g.teams;
  TileExtras extras;
  uint32_t extras_table;
  // r0: the first of a batch of rounds, or of slots
  auto finished = [&](uint32_t r0) {
    if constexpr (WIDE) return my_round < batch && r0 + fin < slots ? tile_of(r0 + fin) : 0xFFFFFFFFu;
    else return my_round < batch ? tile_of(r0 * a.g.teams + fin) : 0xFFFFFFFFu;
  };
  auto load_finish = [&](uint32_t r0) {
    const uint32_t t = finished(r0);
    const Record r = record_of(min(t, n_tiles - 1u), fin);  // (a batch of rounds has an even number of slots where that matters: gated_teams)
    extras = load_extras(r.rec, nb, a.tail_w, r.slots, t < n_tiles, lane);
    extras_table = scale_table(r.base, lane);
  };
  stage_x<DIG, SRC, WIDE ? 4 : 2>(a.in, nb, a.tail_w, a.g.waves, a.g.passes, L, blockIdx.x == 0, [&]() {
    if constexpr (SRC != kSrcRotated) load_finish(0);  // little, and it has a use while the pieces come
    table = scale_table(cur.base, lane);
    const uint8_t* base = scalar_base(cur.rec);
    load_step(W, base, off & (tile < n_tiles ? 0xFFFFFFFFu : 0u));
  });
  if constexpr (SRC == kSrcRotated) load_finish(0);
  lds_barrier();

  // (In a rotated basis there is no scalar register to keep it in: 2560 x 9728 takes 11.5 us like this, 11.8 with the argument.)
  const uint32_t rounds = WIDE ? slots : SRC == kSrcRotated && !GATED ? (a.n_tiles + n_teams - 1u) / n_teams : a.g.rounds;
  uint32_t slot = 0, step = w;  // (WIDE: every wavefront's first step is one of the first slot)
  for (uint32_t r0 = 0; r0 < rounds; r0 += batch) {
    const uint32_t r1 = min(r0 + batch, rounds), o_tile = finished(r0);
    const float o_scale = extras.scale;
    float o_extra = 0.f;
    if (o_tile < n_tiles) {
      const Record r = record_of(o_tile, fin);
      o_extra = tile_extras<DIG>(extras, r.rec, nb, a.tail_w, r.slots, extras_table, L, lane);
    }
    if constexpr (GATED)
      if ((fin & 1u) && lane_class(lane) == 0u) *reinterpret_cast<float2*>(L.part + gated_at(WIDE) + (fin * kTileRows + lane_row(lane)) * 2u) = make_float2(o_scale, o_extra);
    if (r1 != rounds) load_finish(r1);
    for (uint32_t rd = r0; WIDE ? slot < r1 : rd < r1 && tile < n_tiles; ++rd) {
      uint32_t next_slot = slot, next_step = step;
      if constexpr (WIDE) {
        next_step += kGemvMaxWaves;
        if (next_step >= n_steps) {
          next_step -= n_steps;
          ++next_slot;
        }
      }
      const uint32_t next = WIDE ? (next_slot < slots ? tile_of(next_slot) : 0xFFFFFFFFu) : GATED ? tile_of((rd + 1u) * a.g.teams + team) : tile + n_teams;
      const Record nx = record_of(min(next, n_tiles - 1u), WIDE ? next_slot : (rd + 1u) * a.g.teams + team);
      const uint32_t lanes_table = table, keep = next < n_tiles ? 0xFFFFFFFFu : 0u;
      const uint8_t* base = scalar_base(nx.rec);
      float* const part = L.part + (WIDE ? (slot - r0) * n_steps : sums_at(rd - r0, team, a.g.team, false)) * kTileRows;
      table = scale_table(nx.base, lane);  // in front of the pieces, so that the next round waits for it alone
      if constexpr (WIDE) off = step_offset(next_step, units, head, lane);
      float lo, hi;
      step_product<DIG>(W, L.planes + (min(step, n_steps) * kStepUnits + (lane >> 3)) * XPlanes<DIG>::kDwords, lanes_table, lo, hi,
                        [&](auto piece) __attribute__((always_inline)) { load_piece<decltype(piece)::value>(W, base, off & keep); });
      const float v = rows_sum(lo, hi);
      if (lane_class(lane) == 0u) part[step * kTileRows + lane_row(lane)] = v;
      tile = next;
      slot = next_slot;
      step = next_step;
    }
    // A wavefront per tile of these rounds: everything but the sums themselves is scalar.
    lds_barrier();
    if constexpr (GATED) {
      if (o_tile < n_tiles && !(fin & 1u)) {
        auto sum_of = [&](uint32_t of) {
          const uint32_t round = (of * a.g.inv_teams) >> 16;
          return steps_sum<kGemvMaxWaves>(L.part + sums_at(round, of - round * a.g.teams, a.g.team, false) * kTileRows, n_steps, lane);
        };
        const float2 up_scale = *reinterpret_cast<const float2*>(L.part + gated_at(WIDE) + ((fin + 1u) * kTileRows + lane_row(lane)) * 2u);
        const float gate = fmaf(sum_of(fin), o_scale, o_extra), up = fmaf(sum_of(fin + 1u), up_scale.x, up_scale.y);
        const uint32_t row = o_tile * kTileRows + lane_row(lane);
        if (lane_class(lane) == 0u && row < a.m[0].d_out) store_out<OutT>(a.m[0].y, row, silu_mul(round_half(gate), round_half(up)));
      }
    } else if (o_tile < n_tiles) {
      const uint8_t* o_base;
      void* o_y;
      uint32_t o_row0, o_d_out, o_stride, o_slots;
      tile_mat(a, o_tile, o_base, o_y, o_row0, o_d_out, o_stride, o_slots);
      const float v = steps_sum<kGemvMaxWaves * (WIDE ? kGemvWideSteps : 1u)>(L.part + (WIDE ? fin * n_steps : sums_at(my_round, my_team, a.g.team, false)) * kTileRows, n_steps, lane);
      const uint32_t row = o_row0 + lane_row(lane);
      if (lane_class(lane) == 0u && row < o_d_out) store_out<OutT>(o_y, row, fmaf(v, o_scale, o_extra));
    }
    if (r1 != rounds) lds_barrier();
  }
}

template <typename OutT, int SRC, bool WIDE>
__global__ __launch_bounds__(1024) void gemv_tiles_kernel(GemvArgs a) { tiles_product<OutT, SRC, WIDE, false>(a); }
// gate and up; y of the first matrix takes the result.
template <int SRC>
__global__ __launch_bounds__(1024) void gated_product_kernel(GemvArgs a) { tiles_product<__half, SRC, false, true>(a); }
__host__ inline const void* gated_kernel(bool rotated) {
  return rotated ? reinterpret_cast<const void*>(gated_product_kernel<kSrcRotated>) : reinterpret_cast<const void*>(gated_product_kernel<kSrcAddRmsNorm>);
}

// of a finished activation
template <typename OutT, bool WIDE>
__global__ __launch_bounds__(1024) void finished_product_kernel(GemvArgs a) { tiles_product<OutT, kSrcFinished, WIDE, false>(a); }

template <typename OutT, bool WIDE>
__host__ const void* gemv_kernel_of(int src) {
  switch (src) {
    case kSrcFinished: return reinterpret_cast<const void*>(finished_product_kernel<OutT, WIDE>);
    case kSrcF16: return reinterpret_cast<const void*>(gemv_tiles_kernel<OutT, kSrcF16, WIDE>);
    case kSrcRotated: return reinterpret_cast<const void*>(gemv_tiles_kernel<OutT, kSrcRotated, WIDE>);
    case kSrcSiluMul: return reinterpret_cast<const void*>(gemv_tiles_kernel<OutT, kSrcSiluMul, WIDE>);
    default: return reinterpret_cast<const void*>(gemv_tiles_kernel<OutT, kSrcAddRmsNorm, WIDE>);
  }
}
__host__ inline const void* gemv_kernel(bool f32, int src, bool wide) {
  if (f32) return wide ? gemv_kernel_of<float, true>(src) : gemv_kernel_of<float, false>(src);
  return wide ? gemv_kernel_of<__half, true>(src) : gemv_kernel_of<__half, false>(src);
}
template <class Fn>
__host__ void for_each_gemv_kernel(Fn&& fn) {
  for (int rotated = 0; rotated < 2; ++rotated) fn(gated_kernel(rotated != 0));
  for (int src = kSrcF16; src <= kSrcFinished; ++src)
    for (int v = 0; v < 4; ++v) fn(gemv_kernel(v & 1, src, v & 2));
}

}  // namespace llvq
