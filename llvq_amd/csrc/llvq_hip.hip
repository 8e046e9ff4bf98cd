// C ABI and gfx950 kernels of the fused Leech-lattice dequant-GEMV.
//
// Data in HBM, per matrix: the lattice points of its code stream as tiles of 10 bytes per block, with the row scales and
// tail columns (tiles.h; the stream is unranked once, at upload).  Per runtime: the tables of the unranking.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <type_traits>

#include <algorithm>
#include <cstdio>
#include <cmath>
#include <cstddef>
#include <cstring>
#include <functional>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "../../include/llvq_hip.h"
#include "artifact.hpp"
#include "codebook.hpp"
#include "decode_core.h"
#include "rotation.hpp"

namespace llvq {

// ---- table image --------------------------------------------------------------
// What every workgroup copies into LDS.  The rarely used generic class records
// and the large even-coset tables stay in HBM (they live in L2).
struct TableImage {
  uint64_t starts[kStartsLds];  // first: read twice per block, its offset then needs no add of its own
  FastClass fast[kFastLds];
  double rcp[32];
  double step[(24 - kTailSlots) * 25 * 2];  // rows m >= kTailSlots: the walk's last slots are looked up
  uint8_t pdep4[256];
  uint32_t tail_meta[kTailMetaSlots];
  uint16_t lut[2048];        // a 47-bit field only reaches the lower half of the host table
  uint16_t lut2[kLut2Lds];   // the second-level tables that half refers to
  uint32_t golay[4096];
  uint32_t on_lut[kOnLutSlots];
};
static_assert(sizeof(TableImage) % 16 == 0, "table image is copied in 16-byte units");
constexpr size_t kLdsImageBytes = sizeof(TableImage);  // Golay words and the support-arrangement table included
static_assert(kLdsImageBytes % 16 == 0, "LDS part of the table image is copied in 16-byte units");

struct GlobalTables {
  const TableImage* image;
  const uint64_t* starts;  // the padded table of class starts (kStartsPadded)
  const DevClass* cls;
  const uint32_t* off_lut;
  const uint32_t* expand;
  const uint64_t* tail_codes;
  // what a 48-bit index (shell cap 13) can reach and the LDS image leaves out: every fast-path class record,
  // the whole first level of the class-find table and all its second-level tables
  const FastClass* wide_fast;
  const uint16_t* wide_lut;
  const uint16_t* wide_lut2;
};

// kWide: for 48-bit indices the class records, class starts and class-find tables are the full ones in device
// memory (read through L2); the LDS copies cover what a 47-bit index reaches.
template <bool kWide = false>
__device__ __forceinline__ DecodeTables stage_tables(uint8_t* smem, const GlobalTables& g) {
  const uint4* src = reinterpret_cast<const uint4*>(g.image);
  uint4* dst = reinterpret_cast<uint4*>(smem);
  // five loads per lane in flight at a time (one pass for a 1024-lane workgroup): a load and its
  // store per loop iteration would pay the L2 latency once per iteration
  constexpr uint32_t kUnits = (uint32_t)(sizeof(TableImage) / 16), kLast = kUnits - 1u;
  const uint32_t st = blockDim.x;
  for (uint32_t i0 = threadIdx.x; i0 < kUnits; i0 += 5u * st) {
    const uint32_t i1 = i0 + st, i2 = i1 + st, i3 = i2 + st, i4 = i3 + st;
    const uint4 r0 = src[i0], r1 = src[min(i1, kLast)], r2 = src[min(i2, kLast)], r3 = src[min(i3, kLast)], r4 = src[min(i4, kLast)];
    __builtin_amdgcn_sched_barrier(0);  // keep the loads together, ahead of the first store
    dst[i0] = r0;
    if (i1 < kUnits) dst[i1] = r1;
    if (i2 < kUnits) dst[i2] = r2;
    if (i3 < kUnits) dst[i3] = r3;
    if (i4 < kUnits) dst[i4] = r4;
  }
  const TableImage* s = reinterpret_cast<const TableImage*>(smem);
  if constexpr (kWide)
    return DecodeTables{s->golay, g.cls, g.wide_fast, g.starts, g.starts, g.wide_lut, g.wide_lut2, s->rcp, s->on_lut, g.off_lut,
                        g.expand, s->pdep4, s->step - kTailSlots * 25 * 2, s->tail_meta, g.tail_codes};
  return DecodeTables{s->golay, g.cls, s->fast, s->starts, g.starts, s->lut, s->lut2, s->rcp, s->on_lut, g.off_lut,
                      g.expand, s->pdep4, s->step - kTailSlots * 25 * 2, s->tail_meta, g.tail_codes};
}

// 6-byte big-endian record at a 2-byte-aligned offset of a 4-byte-aligned buffer
// (global or LDS): two dword reads, one funnel shift, two byte swaps.
__device__ __forceinline__ uint64_t read_record(const uint8_t* buf, size_t byte) {
  const uint32_t* w = reinterpret_cast<const uint32_t*>(buf + (byte & ~(size_t)3));
  const uint32_t w0 = w[0], w1 = w[1];
  const bool odd = (byte & 2) != 0;
  const uint32_t first = odd ? __builtin_amdgcn_alignbit(w1, w0, 16) : w0;  // bytes 0..3
  const uint32_t second = odd ? (w1 >> 16) : (w1 & 0xFFFFu);                // bytes 4..5
  return ((uint64_t)__builtin_bswap32(first) << 16) | (uint64_t)(__builtin_bswap32(second) >> 16);
}

// Sum over each row of 16 lanes, left in all 16 (four cross-lane moves inside the row).
template <int CTRL>
__device__ __forceinline__ float dpp_move(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float row16_sum(float x) {
  x += dpp_move<0xB1>(x);   // quad_perm [1,0,3,2]: lane ^ 1
  x += dpp_move<0x4E>(x);   // quad_perm [2,3,0,1]: lane ^ 2
  x += dpp_move<0x141>(x);  // row_half_mirror: the other quad of the half row
  x += dpp_move<0x140>(x);  // row_mirror: the other half of the row
  return x;
}

// Sum over the wavefront, the same value in every lane: the four rows' sums are read as scalars.
__device__ __forceinline__ float wave_sum(float v) {
  v = row16_sum(v);
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0)) + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16)) +
         __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32)) + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
}

// The largest or smallest of the wavefront, the same value in every lane.
template <class Op>
__device__ __forceinline__ float wave_best(float v, Op&& op) {
  v = op(v, dpp_move<0xB1>(v));
  v = op(v, dpp_move<0x4E>(v));
  v = op(v, dpp_move<0x141>(v));
  v = op(v, dpp_move<0x140>(v));
  auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = op(__uint_as_float(p[0]), __uint_as_float(p[1]));
  p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return op(__uint_as_float(p[0]), __uint_as_float(p[1]));
}

constexpr uint32_t kDenseBits = 49;  // bits per block at shell cap 13: a 48-bit index and the gain bit

// ---- parity probe: unrank records to points -----------------------------------
template <bool WIDE>
__global__ __launch_bounds__(256) void decode_blocks_kernel(GlobalTables g, const uint8_t* __restrict__ codes,
                                                            size_t nblocks, int8_t* __restrict__ points,
                                                            uint8_t* __restrict__ gains,
                                                            uint8_t* __restrict__ shells) {
  extern __shared__ __align__(16) uint8_t smem[];
  const DecodeTables T = stage_tables<WIDE>(smem, g);
  __syncthreads();
  if constexpr (WIDE) {
    // 49-bit blocks of a dense stream (shell cap 13): block b is the 49 bits from bit 49 b on, read byte by byte
    // (at most seven bytes hold it), so that no byte past the stream's ceil(49 nblocks / 8) is touched
    for (size_t b = (size_t)blockIdx.x * blockDim.x + threadIdx.x; b < nblocks; b += (size_t)gridDim.x * blockDim.x) {
      const uint64_t bit = (uint64_t)b * kDenseBits;
      const uint32_t sh = (uint32_t)(bit & 7u), nbytes = (sh + kDenseBits + 7u) >> 3;
      uint64_t acc = 0;
      for (uint32_t k = 0; k < 7u; ++k) acc = (acc << 8) | (k < nbytes ? codes[(bit >> 3) + k] : 0u);
      const uint64_t rec = (acc >> (56u - sh - kDenseBits)) & ((1ULL << kDenseBits) - 1u);  // index << 1 | gain
      int8_t* out = points + b * kDim;
      const int ci = decode_index(T, rec >> 1, [&](int p, int v) { out[p] = (int8_t)v; });
      if (gains) gains[b] = (uint8_t)(rec & 1);
      if (shells) shells[b] = ci >= 0 ? (uint8_t)T.cls[ci].shell : (ci == -1 ? 0 : 0xFF);
    }
    return;
  }
  for (size_t b = (size_t)blockIdx.x * blockDim.x + threadIdx.x; b < nblocks;
       b += (size_t)gridDim.x * blockDim.x) {
    // the stream's last record is read byte by byte: the two-dword read would touch up to two
    // bytes past a buffer the caller sized to 6 * nblocks
    uint64_t rec;
    if (b + 1 < nblocks) {
      rec = read_record(codes, 6 * b);
    } else {
      rec = 0;
      for (int k = 0; k < 6; ++k) rec = (rec << 8) | codes[6 * b + k];
    }
    int8_t* out = points + b * kDim;
    const int ci = decode_index(T, rec >> 1, [&](int p, int v) { out[p] = (int8_t)v; });
    if (gains) gains[b] = (uint8_t)(rec & 1);
    if (shells) shells[b] = ci >= 0 ? (uint8_t)T.cls[ci].shell : (ci == -1 ? 0 : 0xFF);
  }
}

// ---- what the product kernels share -----------------------------------------------
constexpr int kMaxGroup = 4;

// What a launch may do to produce its activation before the product.
enum : uint32_t {
  kPrologueNone = 0,
  kPrologueSiluMul = 1,    // x[i] = f16(f16(silu(x2[i])) * x[i])           (model.rs:831)
  kPrologueAddRmsNorm = 2  // r = f16(x[i] + x2[i]) (x2 may be null: r = x[i]); resid_out = r;
                           // x[i] = f16(r / sqrt(mean(r^2) + eps) * norm_w[i])  (model.rs:781, :827-829)
};

// Where a launch's activation comes from, and what it may do to produce it before the product.
struct ActivationIn {
  const __half* x;
  const float* x_f32;  // when set, the activation is these f32 values (a rotated activation) and x is unused
  const __half* x2;
  const __half* norm_w;
  __half* resid_out;   // written by workgroup 0 only; must not alias x
  float eps;
  uint32_t prologue;   // kPrologue*
  // the basis of the matrices, when they are stored rotated and the launch rotates its own activation (see rotate_lds)
  const uint32_t* rot_signbits;
  const void* rot_fragments;  // RotTable
  float rot_inv;
  uint32_t rot_m, rot_k;
};

// A workgroup barrier that orders LDS accesses only: loads from memory stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Eight binary16 values at any 2-byte alignment (one 16-byte load).
struct __attribute__((packed, aligned(2))) HalfOctet { uint32_t w[4]; };
__device__ __forceinline__ float half_lo(uint32_t w) { return __half2float(__ushort_as_half((unsigned short)(w & 0xFFFFu))); }
__device__ __forceinline__ float half_hi(uint32_t w) { return __half2float(__ushort_as_half((unsigned short)(w >> 16))); }

// The rotation x' = (S (x) I_m)(I_k (x) H_m / sqrt m) D x of an activation of n = k m values, by a workgroup of 1024
// lanes (llvq-quant/src/rotation.rs:97-105; f32 like the reference's device rotation, llvq-cuda/kernels/llvq_rot.cuh).
//
// Every workgroup of a batch-1 product rotates its own activation (rows up to those of rot_split_pays), and with sixteen wavefronts on a CU an instruction of
// each costs 7 ns: what bounds a rotation is their number.  (With a value per lane and load, lane exchanges through LDS and a
// pass over LDS per level above 512 a 2560 x 9728 product took 19.2 us; with the levels at 48 instructions, sixteen wavefronts'
// operands asked for where ten have any, and every k on the matrix cores 12.6; 11.1 after that, and 5120 x 5120 8.2 where it was 11.5.  Rows as wide as the former are rotated by
// rotate_split_kernel now, which has both times.)  So:
//  * The five lowest levels are two matrix-core steps: what is rotated is binary16, the entries of H are 0 and +-1, so
//    the products are exact and the sums f32, as butterflies would have them.  A wavefront takes 1024 values; a column of
//    its 32 x 32 result is 32 neighbouring ones, requested by two lanes as two octets each (with their signs).
//  * The next five are lane moves between columns, on the sixteen results a lane holds, an instruction to a result and level
//    (lane_level); the values meet LDS once.
//  * The levels above 1024 are passes over LDS, three levels to a pass, the k x k block is products of scalars for k up to 9, else f32
//    matrix-core steps (rotate_rest).
// A lane's parts of both matrices lie together in a table (RotFragments), the k x k block as it is behind it (RotTable).
// Where an octet spans groups (m < 8) the signed values are put into LDS instead and every level is a pass there.
constexpr uint32_t kRotOctetM = 8;    // the narrowest m that takes the octets
constexpr uint32_t kRotTile = 1024;   // values of a wavefront, and how far the levels before LDS reach
typedef _Float16 rot_h8_t __attribute__((ext_vector_type(8)));
typedef float rot_acc_t __attribute__((ext_vector_type(16)));
struct __attribute__((aligned(16))) RotFragments {   // of lane l: (l32, lh) = (l % 32, l / 32)
  float s[kRotKMax / 2];  // (S / sqrt m)[l32][2 i + lh], zero past k
  rot_h8_t h[2];          // H[l32][16 i + 8 lh + e], H the transform inside groups of min(m, 32)
};
static_assert(sizeof(RotFragments) == 96, "six 16-byte loads");
constexpr uint32_t kRotScalarK = 9;  // the largest k whose block is multiplied as scalars: rows of it are padded to that, with zeros
struct RotTable {
  RotFragments lane[64];
  float rows[kRotScalarK][kRotScalarK + 3];  // (S / sqrt m)[g][i]
};
__device__ __forceinline__ float flip_sign(float v, uint32_t bits, int j) {  // bit j of `bits` is the sign of D
  return __uint_as_float(__float_as_uint(v) ^ (((bits >> j) & 1u) << 31));
}
// Two binary16 values and bits 2 j and 2 j + 1 of their octet's signs.
__device__ __forceinline__ uint32_t flip_signs(uint32_t pair, uint32_t bits, int j) {
  return pair ^ (((bits << (15 - 2 * j)) | (bits << (30 - 2 * j))) & 0x80008000u);
}
// Where a lane's octet i of a tile lies.
__device__ __forceinline__ uint32_t rot_octet_at(uint32_t tile, uint32_t i) {
  const uint32_t lane = threadIdx.x & 63u;
  return tile * kRotTile + (lane & 31u) * 32u + i * 16u + (lane >> 5) * 8u;
}
// A level between lanes that are L apart: v + g * the other lane's v with g = -1 in the lower lane, 1 in the upper one, so that the lower
// one has the difference and the upper one the sum: what lane l holds in the end belongs to column l with the bits of all such
// levels turned over.  The compiler makes a move and a multiply-add of it (v_fmac_f32 takes the move as an operand, but is not
// folded): 16 instructions a level as they stand here, and with a product for the sign, as they were, 48 with the waits in between.  (What a
// lane move reads has to be written two instructions before.)
template <int L>
__device__ __forceinline__ void lane_level(rot_acc_t& v, uint32_t lane) {
  const float g = (lane & (uint32_t)L) ? 1.f : -1.f;
  if constexpr (L == 1) {  // behind the matrix cores, whose results the compiler waits for
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = fmaf(__uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v[r]), 0xB1, 0xF, 0xF, true)), g, v[r]);
    return;
  }
  float a[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) a[r] = v[r];
#define LEVEL(r, move) "v_fmac_f32_dpp %" #r ", %" #r ", %16 " move " row_mask:0xf bank_mask:0xf\n\t"
#define LEVELS(move) "s_nop 1\n\t" LEVEL(0, move) LEVEL(1, move) LEVEL(2, move) LEVEL(3, move) LEVEL(4, move) LEVEL(5, move) LEVEL(6, move) LEVEL(7, move) \
  LEVEL(8, move) LEVEL(9, move) LEVEL(10, move) LEVEL(11, move) LEVEL(12, move) LEVEL(13, move) LEVEL(14, move) LEVEL(15, move) "s_nop 1"
#define SIXTEEN "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7]), "+v"(a[8]), "+v"(a[9]), "+v"(a[10]), "+v"(a[11]), \
  "+v"(a[12]), "+v"(a[13]), "+v"(a[14]), "+v"(a[15])
  if constexpr (L == 2) asm(LEVELS("quad_perm:[2,3,0,1]") : SIXTEEN : "v"(g));
  if constexpr (L == 8) asm(LEVELS("row_ror:8") : SIXTEEN : "v"(g));
  if constexpr (L == 4) {  // lane ^ 7, then lane ^ 3
    float t0, t1, t2, t3;
#define MIRROR(t, r) "v_mov_b32_dpp %" #t ", %" #r " row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
#define TURN(r, t) "v_fmac_f32_dpp %" #r ", %" #t ", %20 quad_perm:[3,2,1,0] row_mask:0xf bank_mask:0xf\n\t"
#define FOUR(r0, r1, r2, r3) MIRROR(16, r0) MIRROR(17, r1) MIRROR(18, r2) MIRROR(19, r3) TURN(r0, 16) TURN(r1, 17) TURN(r2, 18) TURN(r3, 19)
    asm("s_nop 1\n\t" FOUR(0, 1, 2, 3) FOUR(4, 5, 6, 7) FOUR(8, 9, 10, 11) FOUR(12, 13, 14, 15) "s_nop 1"
        : SIXTEEN, "=&v"(t0), "=&v"(t1), "=&v"(t2), "=&v"(t3) : "v"(g));
#undef FOUR
#undef TURN
#undef MIRROR
  }
#undef SIXTEEN
#undef LEVELS
#undef LEVEL
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = a[r];
}
// Where value p of a row under rotation is in LDS: at p, or PLACED.  A lane's results are four neighbours in each of several groups of 32 values, a lane's groups 128 bytes from the
// next one's: eight lanes to a bank.  From m = 512 on, fours of a group change places by the group's number (bits 6 to 8 of p), so that sixteen
// lanes have banks of their own; multiples of m, and of 1024, are added as they are.  (Two thirds of the LDS cycles of rotate_kernel were
// conflicts: rotated q, k, v of 4096 columns at 64 rows 15.2 -> 15.0 us.  In the products' launches, all of whose workgroups do it, what it takes to find
// the places is as long: 2560 x 2560 6.57 -> 6.54, 2560 x 320 5.54 -> 5.60.)
template <bool PLACED>
__device__ __forceinline__ uint32_t rot_place(uint32_t p, uint32_t m) { return PLACED && m >= 512u ? p ^ ((p >> 4) & 0x1Cu) : p; }
// Eight values from p (a multiple of eight) on, PLACED.
__device__ __forceinline__ void rot_octet(const float* v, uint32_t p, uint32_t m, float (&out)[8]) {
  const uint32_t at = rot_place<true>(p, m);
  const float4 a = *reinterpret_cast<const float4*>(v + at), b = *reinterpret_cast<const float4*>(v + (at ^ 4u));
  out[0] = a.x; out[1] = a.y; out[2] = a.z; out[3] = a.w;
  out[4] = b.x; out[5] = b.y; out[6] = b.z; out[7] = b.w;
}
// The levels below min(m, 1024) of a tile whose signed octets a lane holds (zeros past n), into LDS.
template <bool PLACED>
__device__ __forceinline__ void rotate_tile_to(float* v, const uint32_t (&x0)[4], const uint32_t (&x1)[4], const rot_h8_t (&h)[2], uint32_t tile,
                                               uint32_t n, uint32_t m, uint32_t k, float inv) {
  const uint32_t lane = threadIdx.x & 63u;
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  rot_acc_t acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(h[0], __builtin_bit_cast(rot_h8_t, u4{x0[0], x0[1], x0[2], x0[3]}), acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(h[1], __builtin_bit_cast(rot_h8_t, u4{x1[0], x1[1], x1[2], x1[3]}), acc, 0, 0, 0);
  // acc[r] is value 8 (r / 4) + 4 lh + r % 4 of column l32
  uint32_t turned = 0;
  if (m >= 64u) {
    lane_level<1>(acc, lane);
    turned = 1u;
  }
  if (m >= 128u) {
    lane_level<2>(acc, lane);
    turned = 3u;
  }
  if (m >= 256u) {
    lane_level<4>(acc, lane);
    turned = 7u;
  }
  if (m >= 512u) {
    lane_level<8>(acc, lane);
    turned = 15u;
  }
  const bool done = k == 1 && m <= kRotTile;  // nothing follows but the factor
  if (m >= 1024u) {
    // Between the two rows of sixteen lanes results change places, eight against eight: a row has one eight of both, and forms its sums
    // (column below 16) and differences (that one and 16).
    const uint32_t row = (lane >> 4) & 1u, at = rot_place<PLACED>(tile * kRotTile + ((lane & 15u) ^ turned) * 32u + row * 16u + (lane >> 5) * 4u, m);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[r]), __float_as_uint(acc[r + 8]), false, false);
      acc[r] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
      acc[r + 8] = __uint_as_float(p[0]) - __uint_as_float(p[1]);
    }
    if (done) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] *= inv;
    }
#pragma unroll
    for (uint32_t q = 0; q < 4u; ++q)  // (such a tile is whole)
      *reinterpret_cast<float4*>(v + (at ^ 8u * (q & 1u)) + 512u * (q >> 1)) = make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
    return;
  }
  if (done) {
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] *= inv;
  }
  const uint32_t at = tile * kRotTile + ((lane & 31u) ^ turned) * 32u + (lane >> 5) * 4u, place = rot_place<PLACED>(at, m);
#pragma unroll
  for (uint32_t q = 0; q < 4u; ++q)
    if (at + 8u * q < n) *reinterpret_cast<float4*>(v + (place ^ 8u * q)) = make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
}
// log2 R levels from 2^lg on, by all lanes: butterflies over R values 2^lg apart.
template <uint32_t R, bool PLACED>
__device__ __forceinline__ void rotate_levels(float* v, uint32_t n, uint32_t m, uint32_t lg, float factor) {
#pragma unroll 1
  for (uint32_t p = threadIdx.x; p < n / R; p += 1024u) {
    float* at = v + rot_place<PLACED>((p >> lg) * (R << lg) + (p & ((1u << lg) - 1u)), m);
    float r[R];
#pragma unroll
    for (uint32_t i = 0; i < R; ++i) r[i] = at[i << lg];
#pragma unroll
    for (uint32_t l = 1; l < R; l <<= 1)
#pragma unroll
      for (uint32_t i = 0; i < R; ++i)
        if (!(i & l)) {
          const float u = r[i], w = r[i | l];
          r[i] = u + w;
          r[i | l] = u - w;
        }
#pragma unroll
    for (uint32_t i = 0; i < R; ++i) at[i << lg] = r[i] * factor;
  }
}

// The k x k block of K x K numbers as products of scalars: a lane takes whole columns, or where there are fewer than lanes the
// wavefronts share the rows of a column, and read it before any of them writes.  K * K multiply-adds a column, where the matrix cores
// multiply 32 x 32: 5120 values, k = 5, 2.3 us of a launch with the latter.
template <uint32_t K, bool PLACED>
__device__ __forceinline__ void rotate_columns(float* v, uint32_t m, const float* rows) {
  typedef const float __attribute__((address_space(4))) scalar_f;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lg = 31u - (uint32_t)__builtin_clz(m);
  const uint32_t parts = m < 1024u ? 1024u >> lg : 1u, part = m < 1024u ? wave >> (lg - 6u) : 0u;  // (m >= 64: a part is whole wavefronts)
  const uint32_t g0 = K * part / parts, g1 = K * (part + 1u) / parts;
#pragma unroll 1
  for (uint32_t j = threadIdx.x & (m - 1u); j < m; j += 1024u) {
    const uint32_t place = rot_place<PLACED>(j, m);
    float c[K];
#pragma unroll
    for (uint32_t i = 0; i < K; ++i) c[i] = v[i * m + place];
    if (parts > 1u) lds_barrier();
#pragma unroll 1
    for (uint32_t g = g0; g < g1; ++g) {
      scalar_f* s = (scalar_f*)(rows + g * (kRotScalarK + 3u));
      float t = s[0] * c[0];
#pragma unroll
      for (uint32_t i = 1; i < K; ++i) t = fmaf(s[i], c[i], t);
      v[g * m + place] = t;
    }
  }
}
// What rotate_rest needs of the k x k block in registers; its loads are to be out in front of the barrier that rotate_rest is behind.
struct RotBlock { float s[kRotKMax / 2]; };
__device__ __forceinline__ bool rot_scalars(uint32_t m, uint32_t k) { return m >= 64u && k <= kRotScalarK; }
__device__ __forceinline__ RotBlock rot_block(const RotTable* table, uint32_t m, uint32_t k) {
  RotBlock b{};
  const uint32_t lane = threadIdx.x & 63u;
  if (!rot_scalars(m, k)) {
#pragma unroll
    for (uint32_t q = 0; q < 4u; ++q) {
      if (8u * q >= k) break;
      const float4 f = *reinterpret_cast<const float4*>(table->lane[lane].s + 4u * q);
      b.s[4 * q] = f.x;
      b.s[4 * q + 1] = f.y;
      b.s[4 * q + 2] = f.z;
      b.s[4 * q + 3] = f.w;
    }
  }
  return b;
}
// What is left once the levels below 1024 are in LDS (every level, `put_levels`, where the octets were not taken): the values
// are final after the caller's next barrier.  Called behind a barrier.
template <bool PLACED>
__device__ __forceinline__ void rotate_rest(float* v, uint32_t n, uint32_t m, uint32_t k, float inv, const RotTable* table, const RotBlock& B, bool put_levels) {
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t l32 = lane & 31u, lh = lane >> 5;
  // three levels to a pass, what is over in the last
  for (uint32_t lg = put_levels ? 0u : 31u - (uint32_t)__builtin_clz(kRotTile); (1u << lg) < m; lg += 3u) {
    const bool last = (8u << lg) >= m;
    const float factor = last && k == 1 ? inv : 1.f;
    if ((m >> lg) >= 8u) rotate_levels<8, PLACED>(v, n, m, lg, factor);
    else if ((m >> lg) == 4u) rotate_levels<4, PLACED>(v, n, m, lg, factor);
    else rotate_levels<2, PLACED>(v, n, m, lg, factor);
    if (!last || k > 1) lds_barrier();
  }
  if (k == 1 && m == 1) {  // (a row of one value)
    if (tid == 0) v[0] *= inv;
  }
  if (k == 1) return;
  if (rot_scalars(m, k)) {
    const float* rows = &table->rows[0][0];
    if (k == 3u) rotate_columns<3, PLACED>(v, m, rows);
    else if (k == 5u) rotate_columns<5, PLACED>(v, m, rows);
    else if (k == 7u) rotate_columns<7, PLACED>(v, m, rows);
    else rotate_columns<9, PLACED>(v, m, rows);
    return;
  }
  // S (k x k, with the factor 1 / sqrt m) . C (k x m): a wavefront takes 32 columns of C at a time as f32 matrix-core
  // steps of depth 2 (S padded with zeros to 32 x 32; lanes past a narrow m repeat its first column); it reads its columns
  // whole before it writes them, and no other wavefront touches them.
#pragma unroll 1
  for (uint32_t tile = wave; tile * 32u < m; tile += 16) {
    // (in each tile anew: what the steps compare and multiply with would otherwise be formed ahead of the loop and spilled)
    asm volatile("" : "+s"(k), "+s"(m));
    const uint32_t steps = (k + 1u) >> 1;  // k is odd: the last one has no row for the upper half
    const uint32_t j = tile * 32u + l32;
    const float *at = v + rot_place<PLACED>(j < m ? j : 0u, m), *col = at + lh * m;
    rot_acc_t acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
    for (uint32_t s0 = 0; s0 < kRotKMax / 2; s0 += 8u) {  // half the steps at a time: the weights in flight leave registers for that
      if (s0 >= steps) break;
      float c[8];
#pragma unroll
      for (uint32_t i = 0; i < 8u; ++i) {
        if (s0 + i >= steps) break;
        c[i] = s0 + i + 1u == steps ? at[(k - 1u) * m] : col[2u * (s0 + i) * m];
      }
#pragma unroll
      for (uint32_t i = 0; i < 8u; ++i) {
        if (s0 + i >= steps) break;
        float x = c[i];
        if (s0 + i + 1u == steps) x = lh ? 0.f : x;
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(B.s[s0 + i], x, acc, 0, 0, 0);
      }
    }
    // acc[r] is row 8 (r / 4) + 4 lh + r % 4 of column j
    if (j < m) {
      float* out = v + rot_place<PLACED>(j, m) + lh * 4u * m;
#pragma unroll
      for (uint32_t r = 0; r < 16; ++r) {
        const uint32_t g = 8u * (r >> 2) + (r & 3u);
        if (g + 4u < k) out[g * m] = acc[r];
        else if (g < k && !lh) out[g * m] = acc[r];
      }
    }
  }
}

template <typename OutT>
__device__ __forceinline__ void store_out(void* y, uint32_t r, float v);
template <>
__device__ __forceinline__ void store_out<float>(void* y, uint32_t r, float v) {
  reinterpret_cast<float*>(y)[r] = v;
}
template <>
__device__ __forceinline__ void store_out<__half>(void* y, uint32_t r, float v) {
  reinterpret_cast<__half*>(y)[r] = __float2half_rn(v);
}

// Loads and stores of values that another workgroup of the SAME launch produces or consumes (gemv_seq.h): device
// scope, so that they meet in memory and not in an XCD's own L2, which the L2 of another XCD is not coherent with.
// They replace the device-scope fences such an exchange would otherwise need — whose acquire side empties the
// XCD's L2 of the decode tables every time.
template <bool kDeviceScope>
__device__ __forceinline__ __half load_half(const __half* p) {
  if constexpr (kDeviceScope)
    return __ushort_as_half(__hip_atomic_load(reinterpret_cast<const unsigned short*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  else
    return *p;
}
template <bool kDeviceScope>
__device__ __forceinline__ void store_half(__half* p, __half v) {
  if constexpr (kDeviceScope)
    __hip_atomic_store(reinterpret_cast<unsigned short*>(p), __half_as_ushort(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else
    *p = v;
}

// ---- incoherence rotation of an activation ----------------------------------------
// One workgroup per activation row.  Where one batched launch takes all the rows they go out as its octets, 16 bytes to a
// column of them each: the launch that would bring them into that form takes 2.6 us at 64 rows of 4096, 5 at 500.
struct RotArgs {
  const __half* x;        // [rows, n]
  void* out;              // [rows, n] f32 or f16
  const uint32_t* signbits;
  const void* fragments;  // RotTable
  uint32_t n, m, k;
  float inv;
  // to the batched kernels' octets (gemm_kernel.h): `rows` of them, `out` takes the columns from `kcols` on
  uint4* xt;
  uint32_t rows, m_pad, n_oct, kcols;
};
struct RotOctets {};  // in place of an output type
// Where a kernel that makes a batch's rows leaves them for a batched product: xt as the octets gemm_kernel.h describes (`rows` of them, zeros
// behind and past the column kcols), tail columns in the rows themselves.
struct Octets {
  uint4* xt;
  uint32_t rows, m_pad, n_oct, kcols;
};
// The row of workgroup b where a workgroup writes a row's octets: eight rows share the lines of those, and workgroups go to the eight XCDs in
// turn, so rows that share lines are eight apart and a line is made in one L2.  (As they come, every line is written in parts by
// eight of them.  Rotated q, k, v of 64 rows 17.26 -> 16.78 us; and where it paid only up to 256 rows to write octets, it does for all:
// 4096 x 4096 at 300 rows 38.6 us by rows and tile_activations_kernel, 36.4 so, 13000 x 12288 at 1024 310 and 303, 2560 x 9728 94 and 89.)
__device__ __forceinline__ uint32_t octet_row(uint32_t b, uint32_t m_pad) { return m_pad & 63u ? b : (b & ~63u) | (b & 7u) << 3 | ((b >> 3) & 7u); }

// the identity rotation: binary16 -> f32
__global__ __launch_bounds__(256) void widen_kernel(const __half* __restrict__ x, float* __restrict__ out, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = __half2float(x[i]);
}

template <typename OutT>
__global__ __launch_bounds__(1024) void rotate_kernel(RotArgs a) {
  extern __shared__ __align__(16) float rot_s[];
  const uint32_t tid = threadIdx.x, n = a.n, m = a.m, k = a.k;
  uint32_t row = blockIdx.x;
  if constexpr (std::is_same<OutT, RotOctets>::value) {
    row = octet_row(row, a.m_pad);
    const uint32_t live = row < a.rows ? a.kcols / 8u : 0u;  // octets from there on are zero
    for (uint32_t o = live + tid; o < a.n_oct; o += 1024) a.xt[(size_t)o * a.m_pad + row] = make_uint4(0, 0, 0, 0);
    if (row >= a.rows) return;
  }
  const __half* x = a.x + (size_t)row * n;
  const RotTable* table = reinterpret_cast<const RotTable*>(a.fragments);
  if (m >= kRotOctetM) {
    const rot_h8_t h[2] = {table->lane[tid & 63u].h[0], table->lane[tid & 63u].h[1]};
    const uint8_t* signs = reinterpret_cast<const uint8_t*>(a.signbits);
#pragma unroll 1
    for (uint32_t tile = tid >> 6; tile * kRotTile < n; tile += 16u) {
      HalfOctet o[2];
      uint32_t sg[2];
#pragma unroll
      for (uint32_t i = 0; i < 2u; ++i) {
        const uint32_t at = rot_octet_at(tile, i), from = at < n ? at : 0u;
        o[i] = *reinterpret_cast<const HalfOctet*>(x + from);
        sg[i] = signs[from >> 3];
      }
#pragma unroll
      for (uint32_t i = 0; i < 2u; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) o[i].w[j] = rot_octet_at(tile, i) < n ? flip_signs(o[i].w[j], sg[i], j) : 0u;
      rotate_tile_to<true>(rot_s, o[0].w, o[1].w, h, tile, n, m, k, a.inv);
    }
  } else {
    for (uint32_t i = tid; i < n; i += 1024) rot_s[i] = flip_sign(__half2float(x[i]), a.signbits[i >> 5] >> (i & 31u), 0);
  }
  const RotBlock block = rot_block(table, m, k);
  __syncthreads();
  rotate_rest<true>(rot_s, n, m, k, a.inv, table, block, m < kRotOctetM);
  __syncthreads();
  constexpr bool kOctets = std::is_same<OutT, RotOctets>::value, kHalf = kOctets || std::is_same<OutT, __half>::value;
  typedef typename std::conditional<kHalf, __half, float>::type out_t;
  out_t* out = reinterpret_cast<out_t*>(a.out) + (size_t)row * n;
  if constexpr (kHalf) {
    if (kOctets || m >= kRotOctetM) {
      for (uint32_t i = tid * 8u; i < n; i += 8192) {
        HalfOctet o;
        float v[8];
        rot_octet(rot_s, i, m, v);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          o.w[j] = (uint32_t)__half_as_ushort(__float2half_rn(v[2 * j])) | (uint32_t)__half_as_ushort(__float2half_rn(v[2 * j + 1])) << 16;
        if (kOctets && i < a.kcols) a.xt[(size_t)(i / 8u) * a.m_pad + row] = make_uint4(o.w[0], o.w[1], o.w[2], o.w[3]);
        else *reinterpret_cast<HalfOctet*>(out + i) = o;
      }
      return;
    }
  }
  if constexpr (!kOctets)
    for (uint32_t i = tid; i < n; i += 1024) out[i] = (out_t)rot_s[rot_place<true>(i, m)];
}

// One row by kRotSplit workgroups, f32.  Both factors of I_k (x) H_m mix a row's values by bits of their own: workgroup p makes the p-th
// m / 32 values of every group (of three and more, by rot_split_pays), all of H's five highest bits at once as the sums of its sign p over the row (every value of it, once), then
// the others, lane by lane, and the k x k block over the groups' values, which it has all of.
// What bounds it is latency: the launch, a row's way from memory, three barriers; 3.4 to 4.2 us whatever the width.  In the product's launch, where
// every workgroup does all of it, wide rows are several turns of what sixteen wavefronts can at once, and a k x k block past 9 is 32 x 32 on the
// matrix cores: a rotated product of 2560 x 9728 takes 11.2 us there, 10.2 so; 5120 x 17408 19.7 and 16.7, 4096 x 20480 16.0 and 14.2, 4096 x 14336 13.0
// and 12.4, 4096 x 11264 (k = 11) 12.9 and 10.7, 4096 x 8704 (k = 17) 10.6 and 10.0, 4096 x 12288 11.6 and 11.5.  Not 4096 x 10240 (k = 5), 10.4 in both, 4096 x 9216 (k = 9), 9.3
// and 9.8, and 2560 x 5632 (k = 11), 8.8 in both.
constexpr uint32_t kRotSplit = 32, kRotSplitTile = 512;  // workgroups; values of a wavefront
__host__ inline bool rot_split_pays(uint32_t n, uint32_t m, uint32_t k) {  // (m, n: what the kernel is written for)
  return n >= (k > kRotScalarK ? 8192u : 10241u) && m >= 512u && m <= 4096u && n <= kRotSplit * 1024u;
}
__host__ inline size_t rot_split_lds(uint32_t n, uint32_t m) { return (size_t)(n / kRotSplitTile) * (m / kRotSplit) * sizeof(float); }
__global__ __launch_bounds__(1024) void rotate_split_kernel(RotArgs a) {
  extern __shared__ __align__(16) float part[];  // [tile][run]
  __shared__ float mixed[1024];
  asm volatile("" ::"s"(a.x), "s"(a.out), "s"(a.signbits), "s"(a.fragments), "s"(a.n), "s"(a.m), "s"(a.k));  // (all asked for at once)
  const uint32_t tid = threadIdx.x, lane = tid & 63u, n = a.n, m = a.m, k = a.k, p = blockIdx.x;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t run = m / kRotSplit, lg = 31u - (uint32_t)__builtin_clz(run), tiles = n / kRotSplitTile;  // run: 16 .. 128
  const uint8_t* signs = reinterpret_cast<const uint8_t*>(a.signbits);
  HalfOctet o[4];
  uint32_t sg[4];
#pragma unroll
  for (uint32_t i = 0; i < 4u; ++i) {  // (n <= 64 tiles; a wavefront without one repeats the first)
    const uint32_t tile = wave + 16u * i, at = (tile < tiles ? tile : 0u) * kRotSplitTile + lane * 8u;
    o[i] = *reinterpret_cast<const HalfOctet*>(a.x + at);
    sg[i] = signs[at >> 3];
  }
  const uint32_t g = tid >> lg, b = tid & (run - 1u);  // the lane's result: value p * run + b of group g, where g < k
  const RotTable* table = reinterpret_cast<const RotTable*>(a.fragments);
  float s[kRotKMax];
#pragma unroll
  for (uint32_t lh = 0; lh < 2u; ++lh)
#pragma unroll
    for (uint32_t q = 0; q < 4u; ++q) {
      const float4 f = *reinterpret_cast<const float4*>(table->lane[lh * 32u + (g & 31u)].s + 4u * q);
      s[8 * q + lh] = f.x;
      s[8 * q + 2 + lh] = f.y;
      s[8 * q + 4 + lh] = f.z;
      s[8 * q + 6 + lh] = f.w;
    }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (uint32_t i = 0; i < 4u; ++i) {
    const uint32_t tile = wave + 16u * i;
    if (tile >= tiles) break;
    const uint32_t at = tile * kRotSplitTile + lane * 8u;
    const uint32_t bits = sg[i] ^ (__builtin_popcount(((at & (m - 1u)) >> lg) & p) & 1u ? 0xFFu : 0u);
    float v[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t w = flip_signs(o[i].w[j], bits, j);
      v[2 * j] = half_lo(w);
      v[2 * j + 1] = half_hi(w);
    }
    // over the lanes that hold other runs' values of the same places: halves of the wavefront, then rows of sixteen lanes, each
    // going on with half of the values
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const auto t = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[j]), __float_as_uint(v[j + 4]), false, false);
      v[j] = __uint_as_float(t[0]) + __uint_as_float(t[1]);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[j]), __float_as_uint(v[j + 2]), false, false);
      float u = __uint_as_float(t[0]) + __uint_as_float(t[1]);
      if (run <= 64u) u += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(u), 0x128, 0xF, 0xF, false));  // row_ror 8, 4, 2
      if (run <= 32u) u += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(u), 0x124, 0xF, 0xF, false));
      if (run <= 16u) u += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(u), 0x122, 0xF, 0xF, false));
      v[j] = u;
    }
    if ((lane & 15u) * 8u < run)
      *reinterpret_cast<float2*>(part + tile * run + (lane & 15u) * 8u + (lane >> 5) * 4u + ((lane >> 4) & 1u) * 2u) = make_float2(v[0], v[1]);
  }
  __syncthreads();
  const uint32_t each = m / kRotSplitTile;  // tiles of a group
  float v = 0.f;
  if (g < k)
    for (uint32_t t = 0; t < each; ++t) v += part[(g * each + t) * run + b];
  // H's other bits: the upper value of a pair has the difference
  auto level = [&](uint32_t l, float other) __attribute__((always_inline)) { v = b & l ? other - v : other + v; };
  auto lane_move = [&](auto ctrl, float u) __attribute__((always_inline)) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(u), decltype(ctrl)::value, 0xF, 0xF, false));
  };
  level(1u, lane_move(std::integral_constant<int, 0xB1>{}, v));
  level(2u, lane_move(std::integral_constant<int, 0x4E>{}, v));
  level(4u, lane_move(std::integral_constant<int, 0x1B>{}, lane_move(std::integral_constant<int, 0x141>{}, v)));  // lane ^ 7, then ^ 3
  level(8u, lane_move(std::integral_constant<int, 0x128>{}, v));
  if (run >= 32u) level(16u, __shfl_xor(v, 16));
  if (run >= 64u) level(32u, __shfl_xor(v, 32));
  if (run >= 128u) {
    mixed[tid] = v;
    __syncthreads();
    level(64u, mixed[tid ^ 64u]);
    __syncthreads();
  }
  mixed[tid] = v;
  __syncthreads();
  // Few terms in f64, many as four sums (0.1 us of a call): a rotated row is 6 to 28 % nearer to its values in 64 bits than one that a workgroup rotates by
  // itself, ten widths from 8704 to 23552 (17408: 7.4e-8 of its norm, 8.9e-8 there); as one f32 chain it was up to 0.9 % further.
  if (k <= kRotScalarK) {
    double t = 0.;
#pragma unroll
    for (uint32_t i = 0; i < kRotScalarK; ++i) {
      if (i >= k) break;
      t = fma((double)s[i], (double)mixed[(i << lg) + b], t);
    }
    v = (float)t;
  } else {
    float t[4] = {};
#pragma unroll
    for (uint32_t q = 0; q < kRotKMax; q += 8u) {
      if (q >= k) break;
      float c[8];
#pragma unroll
      for (uint32_t i = 0; i < 8u; ++i) c[i] = mixed[(min(q + i, k - 1u) << lg) + b];  // (past k: meets zeros)
#pragma unroll
      for (uint32_t i = 0; i < 8u; ++i) t[i & 3u] = fmaf(s[q + i], c[i], t[i & 3u]);
    }
    v = (t[0] + t[1]) + (t[2] + t[3]);
  }
  if (g < k) reinterpret_cast<float*>(a.out)[g * m + p * run + b] = v;
}

}  // namespace llvq

#include "tiles.h"
#include "gemv_seq.h"
#include "gemm_kernel.h"
#include "gemm_share.h"
#include "decoder.h"

// =================================================================================
// C ABI
// =================================================================================
using namespace llvq;

struct llvq_rt {
  int device = 0;
  hipStream_t stream = nullptr;
  uint8_t* blob = nullptr;  // one device allocation holding every table
  uint8_t* static_scratch = nullptr;  // this device's copy of `scratch` (kStaticScratchBytes)
  GlobalTables tables{};
  int cu_count = 0;
  // rotations by (width, seed), shared by every matrix that consumes the same activation
  // (llvq-llm/src/fused.rs:672-674); an upload may add one, none is changed or moved while launches use it
  struct DevRotation {
    uint32_t n = 0, m = 0, k = 0;
    uint64_t seed = 0;
    float inv = 1.f;
    uint32_t* signbits = nullptr;
    void* fragments = nullptr;  // RotTable
    float* scratch = nullptr;   // one rotated activation, f32, where that is not made in the product's launch: a call's launches use it one behind the other on the runtime's stream
  };
  std::vector<DevRotation*> rotations;
  __half* rot_rows = nullptr;     // rotated batch rows, f16 (matrix-core path)
  size_t rot_rows_bytes = 0;
  // workspace of the wide batched kernel: partial sums of its column splits [splits][padded rows][weight rows, whole tiles]
  float* gemm_ws = nullptr;
  size_t gemm_ws_bytes = 0;
  // a batch's activations as column octets [n_oct][m_pad] of 16 bytes
  __half* gemm_xt = nullptr;
  size_t gemm_xt_bytes = 0;
  // Uploads may come from several threads; launches come from one (llvq_hip.h).  Held while an upload uses what follows
  // and `rotations`.
  std::mutex uploads;
  // where an upload's codes, scales and tail land before they become a matrix's tiles (kUploadBytes at most, kept for the next)
  uint8_t* upload_buf = nullptr;
  size_t upload_bytes = 0;
};

struct llvq_mat {
  std::string name;
  uint32_t d_out = 0, d_in = 0, nblocks = 0, tail_w = 0;
  uint32_t record_bits = 48;  // 48: 6-byte records (shell cap 12); 49: the dense stream of shell cap 13
  float g[2] = {0, 0};
  uint32_t slots = 0, stride = 0;  // places in a tile's list of escapes, bytes of a tile
  uint8_t* tiles = nullptr;  // device: scale table and tiles (tiles.h)
  uint64_t device_bytes = 0;
  uint64_t encoded_bytes = 0;
  bool has_rotation = false;
  uint64_t rotation_seed = 0;
  const llvq_rt::DevRotation* rot = nullptr;  // owned by the runtime
};

struct llvq_seq {
  uint8_t* blob = nullptr;  // one device allocation: units | items | runs | counters | status
  SeqArgs args{};
  const void* kernel = nullptr;
  uint32_t grid = 0, n_items = 0;
  size_t lds = 0;
  uint32_t* own_status = nullptr;  // the status word inside `blob` (args.status may point at a word several sequences share)
};

static thread_local std::string g_last_error;

// Workspace of llvq_hip_gemm_static: device memory the library never allocates or frees.  The
// array's name is only a host-side handle; its device address differs per GPU and is asked for
// once per device, with that device current, at llvq_hip_runtime_create.
constexpr size_t kStaticScratchBytes = (size_t)LLVQ_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) uint8_t scratch[kStaticScratchBytes];
constexpr int kMaxDevices = 64;
static uint8_t* g_scratch_ptr[kMaxDevices] = {};

static int fail(int code, const std::string& msg) {
  g_last_error = msg;
  return code;
}
static int hip_fail(hipError_t e, const char* what) {
  return fail(LLVQ_ERR_DEVICE, std::string(what) + ": " + hipGetErrorString(e));
}
#define HIP_TRY(expr)                                  \
  do {                                                 \
    hipError_t e_ = (expr);                            \
    if (e_ != hipSuccess) return hip_fail(e_, #expr);  \
  } while (0)

extern "C" {

const char* llvq_hip_last_error(void) { return g_last_error.c_str(); }
const char* llvq_hip_version(void) { return "llvq-hip 0.1 (gfx950)"; }

uint64_t llvq_hip_codebook_fingerprint(void) { return codebook_fingerprint(); }

int llvq_hip_host_decode(uint64_t idx, int8_t point[24], int* shell) {
  return host_decode(idx, point, shell) ? 1 : 0;
}

int llvq_hip_runtime_create(int device, void* hip_stream, llvq_rt** out) {
  if (!out) return fail(LLVQ_ERR_INVALID_ARGUMENT, "runtime_create: out is null");
  *out = nullptr;
  const Codebook& cb = codebook();
  if (cb.classes.size() != 383 || codebook_fingerprint() != kFingerprint)
    return fail(LLVQ_ERR_CODEBOOK_MISMATCH, "this build's index map does not reproduce the published fingerprint");
  HIP_TRY(hipSetDevice(device));
  auto* rt = new llvq_rt();
  rt->device = device;
  rt->stream = reinterpret_cast<hipStream_t>(hip_stream);
  hipDeviceProp_t prop;
  hipError_t e = hipGetDeviceProperties(&prop, device);
  if (e != hipSuccess) { delete rt; return hip_fail(e, "hipGetDeviceProperties"); }
  rt->cu_count = prop.multiProcessorCount;
  if (device >= 0 && device < kMaxDevices) {
    if (!g_scratch_ptr[device]) {
      void* p = nullptr;
      e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      if (e != hipSuccess) { delete rt; return hip_fail(e, "hipGetSymbolAddress(scratch)"); }
      g_scratch_ptr[device] = reinterpret_cast<uint8_t*>(p);
    }
    rt->static_scratch = g_scratch_ptr[device];
  }
  // one blob: LDS image | generic class records | off-support table | deposit masks | walk-tail codes
  if (cb.on_lut.size() > (size_t)kOnLutSlots) { delete rt; return fail(LLVQ_ERR_UNSUPPORTED, "support-arrangement table outgrew its LDS slot"); }
  const size_t off_starts = sizeof(TableImage);
  static_assert(sizeof(TableImage) % 8 == 0, "the class starts follow the image 8-byte aligned");
  const size_t off_cls = (off_starts + sizeof(cb.starts) + 15) & ~(size_t)15;
  const size_t off_lut = off_cls + sizeof(cb.dev_classes);
  const size_t off_exp = (off_lut + cb.off_lut.size() * 4 + 15) & ~(size_t)15;
  const size_t off_tail = off_exp + sizeof(cb.expand);
  static_assert(sizeof(cb.expand) % 16 == 0, "the walk-tail codes are read as 8-byte units");
  // ... | every fast-path class record | the whole class-find table, both levels (for 48-bit indices)
  const size_t off_wfast = (off_tail + cb.tail_codes.size() * 8 + 15) & ~(size_t)15;
  const size_t off_wlut = off_wfast + sizeof(cb.fast);
  const size_t off_wlut2 = off_wlut + sizeof(cb.lut);
  const size_t total = off_wlut2 + cb.lut2.size() * 2;
  std::vector<uint8_t> host(total, 0);
  auto* img = reinterpret_cast<TableImage*>(host.data());
  std::memcpy(img->golay, cb.golay, sizeof img->golay);
  std::memcpy(img->fast, cb.fast, sizeof img->fast);
  std::memcpy(img->starts, cb.starts, sizeof img->starts);
  std::memcpy(img->lut, cb.lut, sizeof img->lut);
  // a 47-bit index reaches no class past kFastLds - 2 and no second-level table past kLut2Lds
  uint32_t lut2_used = 0;
  for (uint16_t e : img->lut)
    if (!(e & kLutFinal)) lut2_used = std::max<uint32_t>(lut2_used, (uint32_t)e + (uint32_t)kLut2Span);
  if (lut2_used > (uint32_t)kLut2Lds || lut2_used > cb.lut2.size() || cb.starts[kFastLds - 1] < (1ULL << 47)) {
    delete rt;
    return fail(LLVQ_ERR_UNSUPPORTED, "class-find tables outgrew their LDS slots");
  }
  std::memcpy(img->lut2, cb.lut2.data(), (size_t)lut2_used * 2);
  std::memcpy(host.data() + off_starts, cb.starts, sizeof(cb.starts));
  std::memcpy(img->rcp, cb.rcp, sizeof img->rcp);
  std::memcpy(img->step, cb.step + kTailSlots * 25 * 2, sizeof img->step);
  std::memcpy(img->tail_meta, cb.tail_meta, sizeof img->tail_meta);
  std::memcpy(img->pdep4, cb.pdep4, sizeof img->pdep4);
  std::memcpy(img->on_lut, cb.on_lut.data(), cb.on_lut.size() * 4);
  std::memcpy(host.data() + off_cls, cb.dev_classes, sizeof(cb.dev_classes));
  std::memcpy(host.data() + off_lut, cb.off_lut.data(), cb.off_lut.size() * 4);
  std::memcpy(host.data() + off_exp, cb.expand, sizeof(cb.expand));
  std::memcpy(host.data() + off_tail, cb.tail_codes.data(), cb.tail_codes.size() * 8);
  std::memcpy(host.data() + off_wfast, cb.fast, sizeof(cb.fast));
  std::memcpy(host.data() + off_wlut, cb.lut, sizeof(cb.lut));
  std::memcpy(host.data() + off_wlut2, cb.lut2.data(), cb.lut2.size() * 2);
  e = hipMalloc(reinterpret_cast<void**>(&rt->blob), total);
  if (e != hipSuccess) { delete rt; return hip_fail(e, "hipMalloc(tables)"); }
  e = hipMemcpy(rt->blob, host.data(), total, hipMemcpyHostToDevice);
  if (e != hipSuccess) { (void)hipFree(rt->blob); delete rt; return hip_fail(e, "hipMemcpy(tables)"); }
  rt->tables.image = reinterpret_cast<const TableImage*>(rt->blob);
  rt->tables.starts = reinterpret_cast<const uint64_t*>(rt->blob + off_starts);
  rt->tables.cls = reinterpret_cast<const DevClass*>(rt->blob + off_cls);
  rt->tables.off_lut = reinterpret_cast<const uint32_t*>(rt->blob + off_lut);
  rt->tables.expand = reinterpret_cast<const uint32_t*>(rt->blob + off_exp);
  rt->tables.tail_codes = reinterpret_cast<const uint64_t*>(rt->blob + off_tail);
  rt->tables.wide_fast = reinterpret_cast<const FastClass*>(rt->blob + off_wfast);
  rt->tables.wide_lut = reinterpret_cast<const uint16_t*>(rt->blob + off_wlut);
  rt->tables.wide_lut2 = reinterpret_cast<const uint16_t*>(rt->blob + off_wlut2);
  // the activation tile of a wide matrix pushes dynamic LDS past the 64 KB default
  const int max_lds = 160 * 1024;
  for_each_gemv_kernel([&](const void* kernel) { (void)hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, max_lds); });
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(rotate_kernel<float>), hipFuncAttributeMaxDynamicSharedMemorySize, max_lds);
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(rotate_kernel<__half>), hipFuncAttributeMaxDynamicSharedMemorySize, max_lds);
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(rotate_kernel<RotOctets>), hipFuncAttributeMaxDynamicSharedMemorySize, max_lds);
  for (const void* kernel : {reinterpret_cast<const void*>(gemm_tiles_kernel<1, 1, false>), reinterpret_cast<const void*>(gemm_tiles_kernel<1, 1, true>),
                             reinterpret_cast<const void*>(gemm_tiles_kernel<2, 4, false>), reinterpret_cast<const void*>(gemm_tiles_kernel<1, 4, true>),
                             reinterpret_cast<const void*>(gemm_wide_kernel<4, false>), reinterpret_cast<const void*>(gemm_wide_kernel<4, true>),
                             reinterpret_cast<const void*>(gemm_wide_kernel<8, false>), reinterpret_cast<const void*>(gemm_tall_kernel)})
    (void)hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, max_lds);
  *out = rt;
  return LLVQ_OK;
}

void llvq_hip_runtime_destroy(llvq_rt* rt) {
  if (!rt) return;
  (void)hipSetDevice(rt->device);
  (void)hipFree(rt->blob);
  (void)hipFree(rt->gemm_ws);
  (void)hipFree(rt->gemm_xt);
  (void)hipFree(rt->rot_rows);
  (void)hipFree(rt->upload_buf);
  for (auto* r : rt->rotations) {
    (void)hipFree(r->signbits);
    (void)hipFree(r->fragments);
    (void)hipFree(r->scratch);
    delete r;
  }
  delete rt;
}

int llvq_hip_synchronize(llvq_rt* rt) {
  if (!rt) return fail(LLVQ_ERR_INVALID_ARGUMENT, "synchronize: runtime is null");
  HIP_TRY(hipStreamSynchronize(rt->stream));
  return LLVQ_OK;
}

// Whether the digit planes of rows this wide fit LDS beside what else a launch keeps there.
static bool gemv_fits(uint32_t d_in, bool f32_out, bool rotated) {
  return d_in / kDim <= kGemvMaxBlocks && gemv_tiles_lds_bytes(d_in / kDim, d_in, f32_out, rotated) <= 160 * 1024;
}

// The device tables of rotation (n, seed), built once per runtime.  Called with rt->uploads held.
static int runtime_rotation(llvq_rt* rt, uint32_t n, uint64_t seed, const llvq_rt::DevRotation** out) {
  for (auto* r : rt->rotations)
    if (r->n == n && r->seed == seed) { *out = r; return LLVQ_OK; }
  RotationTables t;
  std::string err;
  if (!build_rotation(n, seed, &t, &err)) return fail(LLVQ_ERR_UNSUPPORTED, err);
  if ((size_t)n * sizeof(float) > 160 * 1024 - 64)
    return fail(LLVQ_ERR_UNSUPPORTED, "width " + std::to_string(n) + " does not fit the rotation kernel's LDS");
  auto* r = new llvq_rt::DevRotation();
  r->n = t.n; r->m = t.m; r->k = t.k; r->seed = seed; r->inv = t.inv;
  hipError_t e = hipMalloc(reinterpret_cast<void**>(&r->signbits), t.signbits.size() * 4);
  if (e == hipSuccess) e = hipMemcpy(r->signbits, t.signbits.data(), t.signbits.size() * 4, hipMemcpyHostToDevice);
  std::vector<RotTable> host(1);
  std::memset(static_cast<void*>(host.data()), 0, sizeof(RotTable));
  RotFragments* const frag = host[0].lane;
  const double unit = 1. / std::sqrt((double)t.m);
  auto scaled = [&](uint32_t g, uint32_t i) { return (float)((double)t.small[(size_t)g * t.k + i] * unit); };
  if (t.k <= kRotScalarK)
    for (uint32_t g = 0; g < t.k; ++g)
      for (uint32_t i = 0; i < t.k; ++i) host[0].rows[g][i] = scaled(g, i);
  const uint32_t inside = std::min(t.m, 32u) - 1u;  // the bits of a column that the transform mixes
  for (uint32_t l = 0; l < 64u; ++l) {
    const uint32_t row = l & 31u, lh = l >> 5;
    for (uint32_t i = 0; i < kRotKMax / 2; ++i) {
      const uint32_t c = 2u * i + lh;
      frag[l].s[i] = row < t.k && c < t.k ? scaled(row, c) : 0.f;
    }
    for (uint32_t i = 0; i < 2u; ++i)
      for (uint32_t e8 = 0; e8 < 8u; ++e8) {
        const uint32_t c = 16u * i + 8u * lh + e8;
        const bool same = ((row ^ c) & ~inside) == 0;
        frag[l].h[i][e8] = (_Float16)(!same ? 0.f : __builtin_popcount(row & c & inside) & 1 ? -1.f : 1.f);
      }
  }
  if (e == hipSuccess) e = hipMalloc(&r->fragments, sizeof(RotTable));
  if (e == hipSuccess) e = hipMemcpy(r->fragments, host.data(), sizeof(RotTable), hipMemcpyHostToDevice);
  // (f32 results have the larger planes: where those fit, all do)
  if (e == hipSuccess && (!gemv_fits(n, true, true) || rot_split_pays(t.n, t.m, t.k))) e = hipMalloc(reinterpret_cast<void**>(&r->scratch), (size_t)n * sizeof(float));
  if (e != hipSuccess) {
    (void)hipFree(r->signbits);
    (void)hipFree(r->fragments);
    delete r;
    return hip_fail(e, "rotation tables");
  }
  rt->rotations.push_back(r);
  *out = r;
  return LLVQ_OK;
}

// Grows a device buffer of the runtime to `need` bytes (contents are not kept).
static hipError_t grow_device(uint8_t** buf, size_t* have, size_t need) {
  if (need <= *have) return hipSuccess;
  (void)hipFree(*buf);
  *buf = nullptr;
  *have = 0;
  const hipError_t e = hipMalloc(reinterpret_cast<void**>(buf), need);
  if (e == hipSuccess) *have = need;
  return e;
}

// Code stream, scales and tail -> the matrix's tiles (tiles.h), through the runtime's staging buffer, kUploadBytes of them
// at a time.  Blocks until done: the host arrays may go, and the staging buffer is free for the next one.  Called with
// rt->uploads held: another upload's copies between this one's and its kernels would end up in this matrix.
constexpr size_t kUploadBytes = 32u << 20;
static hipError_t upload_tiles(llvq_rt* rt, llvq_mat* m, const double* centroids, const float* rscale, const float* tail, const uint8_t* codes) {
  const uint32_t nb = m->nblocks, slots = m->slots, stride = m->stride, n_tiles = tile_count(m->d_out);
  const size_t row_bits = (size_t)nb * m->record_bits;  // sixteen rows are whole bytes whatever the record width
  const uint32_t rows_per = (uint32_t)std::min<size_t>(m->d_out, std::max<size_t>(kTileRows, kUploadBytes * 8 / (row_bits + 32u * (1u + m->tail_w)) / kTileRows * kTileRows));
  TileTable table{};
  for (uint32_t gain = 0; gain < 2; ++gain)
    for (uint32_t shell = 2; shell <= (uint32_t)kMaxShell; ++shell) table.v[gain * 12u + shell - 2u] = (float)centroids[gain] * (float)(1.0 / std::sqrt(16.0 * shell));
  hipError_t e = hipMalloc(reinterpret_cast<void**>(&m->tiles), kTileTableBytes + (size_t)n_tiles * stride + kUnitBytes + 256);  // a tile without a block is read as if it had one
  if (e != hipSuccess) return e;
  const size_t code_room = ((row_bits * rows_per + 7) / 8 + 16 + 255) & ~(size_t)255;
  const size_t scale_room = ((size_t)rows_per * 4 + 255) & ~(size_t)255, tail_room = (size_t)rows_per * m->tail_w * 4;
  if ((e = grow_device(&rt->upload_buf, &rt->upload_bytes, code_room + scale_room + tail_room)) != hipSuccess) return e;
  uint8_t* d_codes = rt->upload_buf;
  float* d_scale = reinterpret_cast<float*>(d_codes + code_room);
  float* d_tail = reinterpret_cast<float*>(d_codes + code_room + scale_room);
  const uint32_t cus = (uint32_t)(rt->cu_count > 0 ? rt->cu_count : 256);
  for (uint32_t r0 = 0; r0 < m->d_out; r0 += rows_per) {
    const uint32_t rows = std::min(rows_per, m->d_out - r0);
    uint8_t* out = m->tiles + kTileTableBytes + (size_t)(r0 / kTileRows) * stride;
    const size_t bytes = (row_bits * rows + 7) / 8;
    if (bytes && (e = hipMemcpyAsync(d_codes, codes + row_bits * r0 / 8, bytes, hipMemcpyHostToDevice, rt->stream)) != hipSuccess) return e;
    if ((e = hipMemcpyAsync(d_scale, rscale + r0, (size_t)rows * 4, hipMemcpyHostToDevice, rt->stream)) != hipSuccess) return e;
    if (m->tail_w && (e = hipMemcpyAsync(d_tail, tail + (size_t)r0 * m->tail_w, (size_t)rows * m->tail_w * 4, hipMemcpyHostToDevice, rt->stream)) != hipSuccess) return e;
    const uint32_t heads = tile_count(rows) * kTileRows * (1u + 4u * tail_depth(m->tail_w));
    hipLaunchKernelGGL(tile_heads_kernel, dim3((heads + 255u) / 256u), dim3(256), 0, rt->stream, table,
                       r0 ? (float*)nullptr : reinterpret_cast<float*>(m->tiles), d_scale, d_tail, out, rows, nb, m->tail_w, slots);
    if (nb) {
      const uint64_t units = (uint64_t)tile_count(rows) * tile_units(nb);
      const uint32_t grid = (uint32_t)std::min<uint64_t>((units + 7) / 8, 2ull * cus);
      if (m->record_bits == 48) hipLaunchKernelGGL(transcode_kernel<false>, dim3(grid), dim3(512), kLdsImageBytes, rt->stream, rt->tables, d_codes, out, rows, nb, m->tail_w, slots);
      else hipLaunchKernelGGL(transcode_kernel<true>, dim3(grid), dim3(512), kLdsImageBytes, rt->stream, rt->tables, d_codes, out, rows, nb, m->tail_w, slots);
    }
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (slots) {
    hipLaunchKernelGGL(sort_lists_kernel, dim3((n_tiles + 3u) / 4u), dim3(256), 0, rt->stream, m->tiles + kTileTableBytes, n_tiles, stride, slots);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  e = hipStreamSynchronize(rt->stream);
  if (rt->upload_bytes > kUploadBytes + 1024) {  // sixteen rows that exceed it by themselves: not kept
    (void)hipFree(rt->upload_buf);
    rt->upload_buf = nullptr;
    rt->upload_bytes = 0;
  }
  return e;
}

static int upload_impl(llvq_rt* rt, const std::string& name, uint32_t d_out, uint32_t d_in,
                       uint32_t shell_cap, uint32_t n_centroids, const double* centroids,
                       const double* row_scales, const float* tail, const uint8_t* codes,
                       size_t code_bytes, bool has_rotation, uint64_t rotation_seed, llvq_mat** out) {
  if (shell_cap > (uint32_t)kMaxShell)
    return fail(LLVQ_ERR_INCONSISTENT, name + ": shell cap " + std::to_string(shell_cap) +
                                           " exceeds the supported ball (m <= 13)");
  // one gain bit is compiled into the kernels (llvq-llm/src/fused.rs:1168-1177)
  if (n_centroids != 2)
    return fail(LLVQ_ERR_UNSUPPORTED, name + ": " + std::to_string(n_centroids) +
                                          " centroids, but the kernels hard-code 1 gain bit");
  const int ib = index_bits(shell_cap);
  if (ib + 1 != 48 && ib + 1 != (int)kDenseBits)
    return fail(LLVQ_ERR_UNSUPPORTED, name + ": shell cap " + std::to_string(shell_cap) + " packs " +
                                          std::to_string(ib + 1) +
                                          " bits per block; the kernels read 6-byte records (cap 12) and the 49-bit stream of cap 13");
  const uint32_t record_bits = (uint32_t)ib + 1u;
  const uint32_t nblocks = d_in / kDim, tail_w = d_in % kDim;
  const uint64_t total_blocks = (uint64_t)d_out * nblocks;
  if ((unsigned __int128)total_blocks * record_bits > (unsigned __int128)code_bytes * 8)
    return fail(LLVQ_ERR_TRUNCATED, "file ends mid-code stream");
  if (d_out == 0 || d_in == 0) return fail(LLVQ_ERR_INVALID_ARGUMENT, name + ": empty matrix");
  if ((total_blocks && !codes) || !centroids || !row_scales || (tail_w && !tail))
    return fail(LLVQ_ERR_INVALID_ARGUMENT, name + ": a required array is null");
  // Index range (format.rs:389-392).  The bound is N(13) whatever the cap; a
  // 47-bit field cannot exceed it (2^47 < N(13)), so at cap 12 this never fires.
  if (ib < 64 && ((1ULL << ib) - 1) > kN13) {
    // (only the 48-bit field of cap 13 can: block b is the record_bits bits from bit record_bits * b on)
    for (uint64_t b = 0; b < total_blocks; ++b) {
      const uint64_t bit = b * record_bits;
      const uint32_t sh = (uint32_t)(bit & 7u), nbytes = (sh + record_bits + 7u) >> 3;
      uint64_t acc = 0;
      for (uint32_t k = 0; k < 7u; ++k) acc = (acc << 8) | (k < nbytes ? codes[(bit >> 3) + k] : 0u);
      const uint64_t v = (acc >> (56u - sh - record_bits)) & ((1ULL << record_bits) - 1u);
      if ((v >> 1) > kN13)
        return fail(LLVQ_ERR_INDEX_OUT_OF_RANGE,
                    name + ": index " + std::to_string(v >> 1) + " is not a codebook member");
    }
  }

  HIP_TRY(hipSetDevice(rt->device));
  std::lock_guard<std::mutex> one_at_a_time(rt->uploads);
  const llvq_rt::DevRotation* rot = nullptr;
  if (has_rotation) {
    const int rc = runtime_rotation(rt, d_in, rotation_seed, &rot);
    if (rc) return rc;
  }
  auto* m = new llvq_mat();
  m->has_rotation = has_rotation;
  m->rotation_seed = rotation_seed;
  m->rot = rot;
  m->name = name;
  m->d_out = d_out;
  m->d_in = d_in;
  m->nblocks = nblocks;
  m->tail_w = tail_w;
  m->record_bits = record_bits;
  m->slots = list_slots(nblocks, record_bits != 48u);
  m->stride = tile_stride(nblocks, tail_w, m->slots);
  m->g[0] = (float)centroids[0];  // fused.rs:1209
  m->g[1] = (float)centroids[1];
  std::vector<float> rs(d_out);
  for (uint32_t r = 0; r < d_out; ++r) rs[r] = (float)row_scales[r];  // fused.rs:1210
  const size_t code_len = (size_t)((total_blocks * record_bits + 7) / 8);
  const size_t tail_len = (size_t)d_out * tail_w * sizeof(float);
  const hipError_t e = upload_tiles(rt, m, centroids, rs.data(), tail, codes);
  if (e != hipSuccess) {
    (void)hipFree(m->tiles);
    delete m;
    return hip_fail(e, "upload_tiles");
  }
  m->device_bytes = kTileTableBytes + (uint64_t)tile_count(d_out) * m->stride;
  m->encoded_bytes = code_len + (uint64_t)d_out * 8 + tail_len + 16;
  *out = m;
  return LLVQ_OK;
}

int llvq_hip_matrix_upload(llvq_rt* rt, const llvq_matrix_desc* d, llvq_mat** out) {
  if (!rt || !d || !out) return fail(LLVQ_ERR_INVALID_ARGUMENT, "matrix_upload: null argument");
  *out = nullptr;
  return upload_impl(rt, d->name ? d->name : "", d->d_out, d->d_in, d->shell_cap, d->n_centroids,
                     d->centroids, d->row_scales, d->tail, d->codes, d->code_bytes,
                     d->has_rotation != 0, d->rotation_seed, out);
}

int llvq_hip_read_header(const uint8_t* buf, size_t len, size_t* pos, uint32_t* version,
                         uint32_t* n_matrices) {
  if (!buf || !pos || !version || !n_matrices || *pos > len)
    return fail(LLVQ_ERR_INVALID_ARGUMENT, "read_header: bad argument");
  std::string err;
  const int rc = parse_header(buf, len, pos, version, n_matrices, &err);
  return rc ? fail(rc, err) : LLVQ_OK;
}

int llvq_hip_parse_matrix_record(const uint8_t* buf, size_t len, size_t* pos, llvq_record_info* out) {
  if (!buf || !pos || !out || *pos > len) return fail(LLVQ_ERR_INVALID_ARGUMENT, "parse_matrix_record: bad argument");
  RecordView r;
  std::string err;
  size_t p = *pos;
  const int rc = parse_matrix_record(buf, len, &p, &r, &err);
  if (rc) return fail(rc, err);
  std::memset(out, 0, sizeof *out);
  std::strncpy(out->name, r.name.c_str(), sizeof out->name - 1);
  out->d_out = r.d_out;
  out->d_in = r.d_in;
  out->shell_cap = r.shell_cap;
  out->n_centroids = r.n_centroids;
  out->rotation_seed = r.rotation_seed;
  out->has_rotation = r.has_rotation ? 1 : 0;
  out->centroids_off = r.centroids_off;
  out->row_scales_off = r.row_scales_off;
  out->tail_off = r.tail_off;
  out->codes_off = r.codes_off;
  out->code_bytes = r.code_bytes;
  *pos = p;
  return LLVQ_OK;
}

int llvq_hip_parse_raw_tensor(const uint8_t* buf, size_t len, size_t* pos, uint32_t version, llvq_raw_info* out) {
  if (!buf || !pos || !out || *pos > len) return fail(LLVQ_ERR_INVALID_ARGUMENT, "parse_raw_tensor: bad argument");
  RawTensorView t;
  std::string err;
  size_t p = *pos;
  const int rc = parse_raw_tensor(buf, len, &p, version, &t, &err);
  if (rc) return fail(rc, err);
  std::memset(out, 0, sizeof *out);
  std::strncpy(out->name, t.name.c_str(), sizeof out->name - 1);
  out->rank = (uint32_t)t.dims.size();
  for (size_t i = 0; i < t.dims.size() && i < 8; ++i) out->dims[i] = t.dims[i];
  out->tag = t.tag;
  out->bits = t.bits;
  out->group = t.group;
  out->count = t.count;
  out->data_off = t.data_off;
  out->data_len = t.data_len;
  out->scales_off = t.scales_off;
  out->biases_off = t.biases_off;
  *pos = p;
  return LLVQ_OK;
}

int llvq_hip_parse_blob(const uint8_t* buf, size_t len, size_t* pos, llvq_blob_info* out) {
  if (!buf || !pos || !out || *pos > len) return fail(LLVQ_ERR_INVALID_ARGUMENT, "parse_blob: bad argument");
  BlobView b;
  std::string err;
  size_t p = *pos;
  const int rc = parse_blob(buf, len, &p, &b, &err);
  if (rc) return fail(rc, err);
  std::memset(out, 0, sizeof *out);
  std::strncpy(out->name, b.name.c_str(), sizeof out->name - 1);
  out->data_off = b.data_off;
  out->data_len = b.data_len;
  *pos = p;
  return LLVQ_OK;
}

int llvq_hip_matrix_from_record(llvq_rt* rt, const uint8_t* buf, size_t len, size_t* pos,
                                llvq_mat** out) {
  if (!rt || !buf || !pos || !out || *pos > len)
    return fail(LLVQ_ERR_INVALID_ARGUMENT, "matrix_from_record: bad argument");
  *out = nullptr;
  RecordView r;
  std::string err;
  size_t p = *pos;
  int rc = parse_matrix_record(buf, len, &p, &r, &err);
  if (rc) return fail(rc, err);
  rc = upload_impl(rt, r.name, r.d_out, r.d_in, r.shell_cap, r.n_centroids, r.centroids.data(),
                   r.row_scales.data(), r.tail.data(), r.codes, r.code_bytes, r.has_rotation, r.rotation_seed, out);
  if (rc == LLVQ_OK) *pos = p;
  return rc;
}

void llvq_hip_matrix_free(llvq_rt* rt, llvq_mat* m) {
  if (!m) return;
  if (rt) (void)hipSetDevice(rt->device);
  (void)hipFree(m->tiles);
  delete m;
}

int llvq_hip_matrix_info(const llvq_mat* m, uint32_t* d_out, uint32_t* d_in, uint32_t* nblocks,
                         uint32_t* tail_w, uint64_t* device_bytes) {
  if (!m) return fail(LLVQ_ERR_INVALID_ARGUMENT, "matrix_info: matrix is null");
  if (d_out) *d_out = m->d_out;
  if (d_in) *d_in = m->d_in;
  if (nblocks) *nblocks = m->nblocks;
  if (tail_w) *tail_w = m->tail_w;
  if (device_bytes) *device_bytes = m->device_bytes;
  return LLVQ_OK;
}

const char* llvq_hip_matrix_name(const llvq_mat* m) { return m ? m->name.c_str() : ""; }

struct Prologue {
  uint32_t kind = kPrologueNone;
  const void* x2 = nullptr;
  const void* norm_w = nullptr;
  void* resid_out = nullptr;
  float eps = 0.f;
};

// One launch of gemv_tiles_kernel over n <= kMaxGroup matrices of equal d_in and basis; `gated`: of gated_product_kernel over two, whose
// one result goes to y[0].
static int launch_group(llvq_rt* rt, const llvq_mat* const* mats, int n, const void* x, void* const* y,
                        int y_dtype, const Prologue* pro = nullptr, const float* x_f32 = nullptr,
                        const llvq_rt::DevRotation* rot = nullptr, bool gated = false) {
  const llvq_mat* m0 = mats[0];
  if (y_dtype != LLVQ_F32 && y_dtype != LLVQ_F16) return fail(LLVQ_ERR_INVALID_ARGUMENT, "gemv: unknown output dtype");
  const bool f32 = y_dtype == LLVQ_F32, rotated = rot != nullptr;
  if (!gemv_fits(m0->d_in, f32, rot != nullptr))
    return fail(LLVQ_ERR_UNSUPPORTED, m0->name + ": d_in " + std::to_string(m0->d_in) + " does not fit the LDS activation tile");
  GemvArgs a{};
  a.in.x = reinterpret_cast<const __half*>(x);
  a.in.x_f32 = x_f32;
  if (pro) {
    a.in.prologue = pro->kind;
    a.in.x2 = reinterpret_cast<const __half*>(pro->x2);
    a.in.norm_w = reinterpret_cast<const __half*>(pro->norm_w);
    a.in.resid_out = reinterpret_cast<__half*>(pro->resid_out);
    a.in.eps = pro->eps;
  }
  if (rot) {
    a.in.rot_signbits = rot->signbits;
    a.in.rot_fragments = rot->fragments;
    a.in.rot_inv = rot->inv;
    a.in.rot_m = rot->m;
    a.in.rot_k = rot->k;
  }
  a.nb = m0->nblocks;
  a.tail_w = m0->tail_w;
  a.n_mats = (uint32_t)n;
  for (int i = 0; i < n; ++i) {
    a.m[i] = TileMat{mats[i]->tiles, gated ? y[0] : y[i], mats[i]->d_out, a.n_tiles, mats[i]->stride, mats[i]->slots};
    a.n_tiles += tile_count(mats[i]->d_out);
  }
  // (The in-launch rotation and the wide rows are written for a full workgroup, whatever of it has a tile.)
  a.g = gemv_grid(a.nb, gated ? a.m[1].tile_begin : a.n_tiles, (uint32_t)(rt->cu_count > 0 ? rt->cu_count : 256), gated, rotated || gemv_wide(a.nb),
                  a.in.prologue == kPrologueAddRmsNorm);
  if (gemv_wide(a.nb)) spread_into(a.g, gemv_spread(a.nb, a.n_tiles, a.g.grid));
  const int src = x_f32 ? kSrcFinished : rotated ? kSrcRotated : a.in.prologue == kPrologueSiluMul ? kSrcSiluMul : a.in.prologue == kPrologueAddRmsNorm ? kSrcAddRmsNorm : kSrcF16;
  void* params[] = {&a};
  HIP_TRY(hipLaunchKernel(gated ? gated_kernel(rotated) : gemv_kernel(f32, src, gemv_wide(a.nb)), dim3(a.g.grid),
                          dim3(a.g.waves * 64u), params, gemv_tiles_lds_bytes(a.nb, m0->d_in, f32, rot != nullptr, gated), rt->stream));
  return LLVQ_OK;
}

// Enqueues x' = Q x for `rows` activation rows of width rot->n.
static RotArgs rot_args(const llvq_rt::DevRotation* rot, const void* x_f16, void* out) {
  RotArgs a{};
  a.x = reinterpret_cast<const __half*>(x_f16);
  a.out = out;
  a.signbits = rot->signbits;
  a.fragments = rot->fragments;
  a.n = rot->n;
  a.m = rot->m;
  a.k = rot->k;
  a.inv = rot->inv;
  return a;
}
static int launch_rotate(llvq_rt* rt, const llvq_rt::DevRotation* rot, const void* x_f16, uint32_t rows, void* out,
                         bool out_f16) {
  const RotArgs a = rot_args(rot, x_f16, out);
  const size_t lds = (size_t)rot->n * sizeof(float);
  if (out_f16) hipLaunchKernelGGL(rotate_kernel<__half>, dim3(rows), dim3(1024), lds, rt->stream, a);
  else hipLaunchKernelGGL(rotate_kernel<float>, dim3(rows), dim3(1024), lds, rt->stream, a);
  HIP_TRY(hipGetLastError());
  return LLVQ_OK;
}

// One row, to f32 (with and without a launch of its own a call has the same bits in either form, llvq_hip_rotate).
static int launch_rotate_row(llvq_rt* rt, const llvq_rt::DevRotation* rot, const void* x_f16, float* out) {
  if (!rot_split_pays(rot->n, rot->m, rot->k)) return launch_rotate(rt, rot, x_f16, 1, out, false);
  const RotArgs a = rot_args(rot, x_f16, out);
  hipLaunchKernelGGL(rotate_split_kernel, dim3(kRotSplit), dim3(1024), rot_split_lds(a.n, a.m), rt->stream, a);
  HIP_TRY(hipGetLastError());
  return LLVQ_OK;
}

static bool same_basis(const llvq_mat* a, const llvq_mat* b) {
  return a->has_rotation == b->has_rotation && (!a->has_rotation || a->rotation_seed == b->rotation_seed);
}

// One activation through projections that share it: consecutive matrices in the
// same basis go out as one launch (at most kMaxGroup).  A launch in a rotated basis
// rotates the activation itself (`pro`, when given, derives it first); rows too wide
// for that, or wide enough that it pays (rot_split_pays), get it rotated once, into the
// rotation's scratch, by a kernel of its own (the former never together with `pro`: the
// caller stages the activation first then).
static int forward_group(llvq_rt* rt, const llvq_mat* const* mats, int n, const void* x, void* const* y, int y_dtype,
                         const Prologue* pro = nullptr) {
  int i = 0;
  while (i < n) {
    int j = i + 1;
    while (j < n && j - i < kMaxGroup && same_basis(mats[i], mats[j])) ++j;
    const float* xr = nullptr;
    if (mats[i]->has_rotation && gemv_fits(mats[i]->d_in, y_dtype == LLVQ_F32, true) && (pro || !rot_split_pays(mats[i]->rot->n, mats[i]->rot->m, mats[i]->rot->k))) {
      const int rc = launch_group(rt, mats + i, j - i, x, y + i, y_dtype, pro, nullptr, mats[i]->rot);
      if (rc) return rc;
      i = j;
      continue;
    }
    if (pro && mats[i]->has_rotation) return fail(LLVQ_ERR_UNSUPPORTED, mats[i]->name + ": prologue with a rotation outside the launch");
    if (mats[i]->has_rotation) {
      // the scratch may still hold this very rotation if the previous run used it; rotating again is cheap and always right
      const int rc = launch_rotate_row(rt, mats[i]->rot, x, mats[i]->rot->scratch);
      if (rc) return rc;
      xr = mats[i]->rot->scratch;
    }
    const int rc = launch_group(rt, mats + i, j - i, x, y + i, y_dtype, pro, xr);
    if (rc) return rc;
    i = j;
  }
  return LLVQ_OK;
}

// Whether a layer's gate and up are one launch that leaves silu(gate) up: 37.8, 44.9 and 63.8 us a layer and token of a decode of four layers at the widths of
// 4B, 8B and 14B models, 38.7, 45.9 and 65.0 as two results that down_proj's launch takes.  In a rotated basis, where down_proj's activation is then as wide as
// rotate_split_kernel wants it and binary16: 50.3, 56.6 and 71.9 us, 53.1, 58.6 and 76.7 with both as parts of down_proj's launch.
// (Rows of up to 8192 columns, a decoder's widest, have as many steps as there are wavefronts at the most, and the sums of pairs fit LDS.)
static bool gated_fits(const llvq_mat* gate, const llvq_mat* up) {
  return same_basis(gate, up) && gate->nblocks && (!gate->has_rotation || gemv_fits(gate->d_in, false, true));
}

static int launch_gemv(llvq_rt* rt, const llvq_mat* m, const void* x, void* y, int y_dtype) {
  return forward_group(rt, &m, 1, x, &y, y_dtype);
}

int llvq_hip_gemv(llvq_rt* rt, const llvq_mat* m, const void* x, void* y, int y_dtype) {
  if (!rt || !m || !x || !y) return fail(LLVQ_ERR_INVALID_ARGUMENT, "gemv: null argument");
  HIP_TRY(hipSetDevice(rt->device));
  return launch_gemv(rt, m, x, y, y_dtype);
}

int llvq_hip_rotate(llvq_rt* rt, const llvq_mat* m, const void* x_f16_dev, float* xr_f32_dev) {
  if (!rt || !m || !x_f16_dev || !xr_f32_dev) return fail(LLVQ_ERR_INVALID_ARGUMENT, "rotate: null argument");
  HIP_TRY(hipSetDevice(rt->device));
  if (m->has_rotation) return launch_rotate_row(rt, m->rot, x_f16_dev, xr_f32_dev);
  hipLaunchKernelGGL(widen_kernel, dim3((m->d_in + 255) / 256), dim3(256), 0, rt->stream,
                     reinterpret_cast<const __half*>(x_f16_dev), xr_f32_dev, m->d_in);
  HIP_TRY(hipGetLastError());
  return LLVQ_OK;
}

int llvq_hip_gemv_rotated(llvq_rt* rt, const llvq_mat* m, const float* xr_f32_dev, void* y, int y_dtype) {
  if (!rt || !m || !xr_f32_dev || !y) return fail(LLVQ_ERR_INVALID_ARGUMENT, "gemv_rotated: null argument");
  HIP_TRY(hipSetDevice(rt->device));
  return launch_group(rt, &m, 1, nullptr, &y, y_dtype, nullptr, xr_f32_dev);
}

int llvq_hip_host_rotate(uint32_t n, uint64_t seed, double* v) {
  if (!v) return fail(LLVQ_ERR_INVALID_ARGUMENT, "host_rotate: null vector");
  RotationTables t;
  std::string err;
  if (!build_rotation(n, seed, &t, &err)) return fail(LLVQ_ERR_UNSUPPORTED, err);
  std::vector<double> w(v, v + n);
  host_rotate(t, &w);
  std::memcpy(v, w.data(), (size_t)n * sizeof(double));
  return LLVQ_OK;
}

int llvq_hip_matrix_rotation(const llvq_mat* m, uint32_t* has_rotation, uint64_t* seed) {
  if (!m) return fail(LLVQ_ERR_INVALID_ARGUMENT, "matrix_rotation: matrix is null");
  if (has_rotation) *has_rotation = m->has_rotation ? 1u : 0u;
  if (seed) *seed = m->rotation_seed;
  return LLVQ_OK;
}

int llvq_hip_gemv_group(llvq_rt* rt, const llvq_mat* const* mats, int n, const void* x,
                        void* const* y, int y_dtype) {
  if (!rt || !mats || !x || !y || n < 0) return fail(LLVQ_ERR_INVALID_ARGUMENT, "gemv_group: bad argument");
  for (int i = 0; i < n; ++i) {
    if (!mats[i] || !y[i]) return fail(LLVQ_ERR_INVALID_ARGUMENT, "gemv_group: null matrix or output");
    if (mats[i]->d_in != mats[0]->d_in)
      return fail(LLVQ_ERR_INVALID_ARGUMENT, mats[i]->name + ": projections of one group must share d_in");
  }
  HIP_TRY(hipSetDevice(rt->device));
  return forward_group(rt, mats, n, x, y, y_dtype);
}

// ---- sequences of group products in one launch (gemv_seq.h) -------------------------------
// One item of a sequence as the library's own callers state it: what a launch_group call takes.
struct SeqSpec {
  const llvq_mat* const* mats = nullptr;
  int n = 0;
  const void* x = nullptr;
  void* const* y = nullptr;
  int y_dtype = LLVQ_F16;
  bool after_previous = false;
  Prologue pro{};
};

constexpr uint32_t kSeqSpinLimit = 1u << 20;  // polls of a wait before it gives up (about a second)

static int seq_create(llvq_rt* rt, const SeqSpec* specs, int n, llvq_seq** out) {
  if (n <= 0) return fail(LLVQ_ERR_INVALID_ARGUMENT, "sequence_create: no items");
  bool dependent = false;
  for (int i = 0; i < n; ++i) {
    const SeqSpec& sp = specs[i];
    if (!sp.mats || sp.n <= 0 || !sp.x || !sp.y) return fail(LLVQ_ERR_INVALID_ARGUMENT, "sequence_create: item " + std::to_string(i) + " has a null or empty field");
    if (sp.y_dtype != LLVQ_F32 && sp.y_dtype != LLVQ_F16) return fail(LLVQ_ERR_INVALID_ARGUMENT, "sequence_create: unknown output dtype");
    if (sp.after_previous && i == 0) return fail(LLVQ_ERR_INVALID_ARGUMENT, "sequence_create: the first item has no item before it");
    if (sp.y_dtype != specs[0].y_dtype) return fail(LLVQ_ERR_INVALID_ARGUMENT, "sequence_create: the items of a sequence share one output dtype");
    for (int j = 0; j < sp.n; ++j) {
      const llvq_mat* m = sp.mats[j];
      if (!m || !sp.y[j]) return fail(LLVQ_ERR_INVALID_ARGUMENT, "sequence_create: null matrix or output in item " + std::to_string(i));
      if (m->d_in != sp.mats[0]->d_in) return fail(LLVQ_ERR_INVALID_ARGUMENT, m->name + ": projections of one item must share d_in");
      if (m->has_rotation) return fail(LLVQ_ERR_UNSUPPORTED, m->name + ": a sequence takes natural-basis matrices only");
      if (m->record_bits != specs[0].mats[0]->record_bits) return fail(LLVQ_ERR_UNSUPPORTED, m->name + ": the matrices of a sequence share one shell cap");
    }
    if (sp.mats[0]->nblocks > 1024u) return fail(LLVQ_ERR_UNSUPPORTED, sp.mats[0]->name + ": rows wider than 24 576 columns do not fit a sequence");
    dependent |= sp.after_previous;
  }
  const bool f32 = specs[0].y_dtype == LLVQ_F32;
  bool prologue = false, wide = false;
  uint32_t max_units = 0;
  for (int i = 0; i < n; ++i) {
    prologue |= specs[i].pro.kind != kPrologueNone;
    wide |= gemv_wide(specs[i].mats[0]->nblocks);
    max_units = std::max(max_units, gemv_plane_units(specs[i].mats[0]->nblocks));
  }
  const size_t lds = gemv_seq_lds_bytes(max_units, f32);
  if (lds > 160 * 1024) return fail(LLVQ_ERR_UNSUPPORTED, "sequence_create: the widest rows do not fit the LDS activation tile");
  const uint32_t grid_cap = (uint32_t)(rt->cu_count > 0 ? rt->cu_count : 256);
  std::vector<SeqUnit> units;
  std::vector<SeqItem> items((size_t)n);
  uint64_t bytes = 0, n_tiles = 0;
  for (int i = 0; i < n; ++i)
    for (int j = 0; j < specs[i].n; ++j) {
      const llvq_mat* m = specs[i].mats[j];
      n_tiles += tile_count(m->d_out);
      bytes += (uint64_t)tile_count(m->d_out) * m->stride;
    }
  // Independent items: runs of equal bytes, workgroup b's ending at the tile with which all before it make up (b + 1) / grid
  // of them; a unit is what a workgroup has of a matrix.  Ordered ones are spread over all workgroups as a launch of their
  // own would be, unit after unit: everyone waits for the slowest.
  uint32_t grid = (uint32_t)std::min<uint64_t>(n_tiles, grid_cap);
  const uint32_t task_steps = dependent ? 1u : seq_task_steps(bytes, grid);
  std::vector<uint32_t> runs{0};
  uint64_t done = 0;
  for (int i = 0; i < n; ++i) {
    const SeqSpec& sp = specs[i];
    const llvq_mat* m0 = sp.mats[0];
    const uint32_t nb = m0->nblocks, steps = tile_steps(nb);
    SeqItem& I = items[(size_t)i];
    std::memset(&I, 0, sizeof I);
    I.x = reinterpret_cast<const __half*>(sp.x);
    I.x2 = reinterpret_cast<const __half*>(sp.pro.x2);
    I.norm_w = reinterpret_cast<const __half*>(sp.pro.norm_w);
    I.resid_out = reinterpret_cast<__half*>(sp.pro.resid_out);
    I.eps = sp.pro.eps;
    I.prologue = sp.pro.kind;
    I.nb = nb;
    I.tail_w = m0->tail_w;
    I.first_unit = (uint32_t)units.size();
    I.wait_item = sp.after_previous ? (uint32_t)(i - 1) : kSeqNoWait;
    I.signals = (i + 1 < n && specs[i + 1].after_previous) ? 1u : 0u;
    I.tasks = seq_tasks(steps, task_steps);
    I.inv_tasks = I.tasks > 1u ? (uint32_t)(((1ull << 32) + I.tasks - 1u) / I.tasks) : 0u;
    const size_t ysz = f32 ? 4 : 2;
    for (int j = 0; j < sp.n; ++j) {
      const llvq_mat* m = sp.mats[j];
      const uint32_t tiles = tile_count(m->d_out), stride = m->stride;
      for (uint32_t t0 = 0, count; t0 < tiles; t0 += count) {
        if (dependent) {
          count = (tiles + grid_cap - 1u) / grid_cap;
        } else {
          uint64_t want;  // the end of the run that the tile begins in
          while ((want = bytes * runs.size() / grid) <= done) runs.push_back((uint32_t)units.size());
          count = (uint32_t)((want - done + stride - 1u) / stride);
        }
        count = std::min(count, tiles - t0);
        SeqUnit t{};
        t.rec = m->tiles + kTileTableBytes + (size_t)t0 * stride;
        t.table = reinterpret_cast<const uint32_t*>(m->tiles);
        t.y = reinterpret_cast<uint8_t*>(sp.y[j]) + (size_t)t0 * kTileRows * ysz;
        t.rows = std::min(count * kTileRows, m->d_out - t0 * kTileRows);
        t.item = (uint32_t)i;
        t.stride = stride;
        t.slots = m->slots;
        units.push_back(t);
        done += (uint64_t)count * stride;
      }
    }
  }
  if (units.size() > 0x7FFFFFFFu) return fail(LLVQ_ERR_UNSUPPORTED, "sequence_create: too many units");
  const uint32_t n_units = (uint32_t)units.size();
  if (dependent) grid = std::min(n_units, grid_cap);
  runs.resize((size_t)grid + 1, n_units);
  for (int i = 0; i < n; ++i) {
    const uint32_t t0 = items[(size_t)i].first_unit, t1 = i + 1 < n ? items[(size_t)i + 1].first_unit : n_units;
    items[(size_t)i].expected = std::min(t1 - t0, grid);
  }
  for (int i = 0; i < n; ++i)
    if (items[(size_t)i].wait_item != kSeqNoWait) items[(size_t)i].wait_expected = items[items[(size_t)i].wait_item].expected;
  HIP_TRY(hipSetDevice(rt->device));
  auto* q = new llvq_seq();
  const size_t off_items = units.size() * sizeof(SeqUnit);
  const size_t off_runs = off_items + items.size() * sizeof(SeqItem);
  const size_t off_counters = (off_runs + runs.size() * 4 + 255) & ~(size_t)255;
  const size_t off_status = off_counters + (((size_t)n * 4 + 255) & ~(size_t)255);
  const size_t total = off_status + 256;
  hipError_t e = hipMalloc(reinterpret_cast<void**>(&q->blob), total);
  if (e == hipSuccess) e = hipMemset(q->blob, 0, total);
  if (e == hipSuccess) e = hipMemcpy(q->blob, units.data(), off_items, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(q->blob + off_items, items.data(), items.size() * sizeof(SeqItem), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(q->blob + off_runs, runs.data(), runs.size() * 4, hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    (void)hipFree(q->blob);
    delete q;
    return hip_fail(e, "sequence tables");
  }
  q->args.units = reinterpret_cast<const SeqUnit*>(q->blob);
  q->args.items = reinterpret_cast<const SeqItem*>(q->blob + off_items);
  q->args.runs = dependent ? nullptr : reinterpret_cast<const uint32_t*>(q->blob + off_runs);
  q->args.n_units = n_units;
  q->args.max_units = max_units;
  q->args.counters = reinterpret_cast<uint32_t*>(q->blob + off_counters);
  q->args.status = reinterpret_cast<uint32_t*>(q->blob + off_status);
  q->own_status = q->args.status;
  q->args.run = 0;
  q->args.spin_limit = kSeqSpinLimit;
  q->args.hold_item = kSeqNoWait;
  const int mode = prologue ? (wide ? kSeqPrologueWide : kSeqPrologue)
                            : dependent ? (wide ? kSeqPrologueWide : kSeqOrdered) : (wide ? kSeqIndependentWide : kSeqIndependent);
  q->kernel = f32 ? seq_kernel_of<float>(mode) : seq_kernel_of<__half>(mode);
  // the activation planes of a wide row push dynamic LDS past the 64 KB default
  (void)hipFuncSetAttribute(q->kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  q->lds = lds;
  q->grid = grid;
  q->n_items = (uint32_t)n;
  *out = q;
  return LLVQ_OK;
}

static int seq_run(llvq_rt* rt, llvq_seq* q) {
  q->args.run += 1;
  SeqArgs a = q->args;
  void* params[] = {&a};
  // An ordinary launch, also with ordered items: sixteen wavefronts a workgroup and no more workgroups than
  // CUs, so on a device this stream has to itself every workgroup is resident and the waits end.  (A cooperative launch
  // would guarantee it, but costs some 200 us per launch here: 4B decode fell from 237 to 85 tokens/s with it.)  Should
  // another queue hold CUs for longer than the bounded wait, the run gives up and says so; it cannot hang.
  HIP_TRY(hipLaunchKernel(q->kernel, dim3(q->grid), dim3(1024), params, q->lds, rt->stream));
  HIP_TRY(hipGetLastError());
  q->args.hold_item = kSeqNoWait;
  return LLVQ_OK;
}

// After a run that gave up: its counters are short, so the next run starts over from zero.
static int seq_reset(llvq_seq* q) {
  HIP_TRY(hipMemset(q->args.counters, 0, (size_t)q->n_items * 4));
  HIP_TRY(hipMemset(q->args.status, 0, 4));
  q->args.run = 0;
  return LLVQ_OK;
}

int llvq_hip_sequence_create(llvq_rt* rt, const llvq_seq_item* items, int n_items, llvq_seq** out) {
  if (!rt || !items || !out || n_items <= 0) return fail(LLVQ_ERR_INVALID_ARGUMENT, "sequence_create: bad argument");
  *out = nullptr;
  std::vector<SeqSpec> specs((size_t)n_items);
  for (int i = 0; i < n_items; ++i) {
    specs[(size_t)i].mats = items[i].mats;
    specs[(size_t)i].n = items[i].n_mats;
    specs[(size_t)i].x = items[i].x_f16_dev;
    specs[(size_t)i].y = items[i].y_dev;
    specs[(size_t)i].y_dtype = items[i].y_dtype;
    specs[(size_t)i].after_previous = items[i].after_previous != 0;
  }
  return seq_create(rt, specs.data(), n_items, out);
}

int llvq_hip_sequence_run(llvq_rt* rt, llvq_seq* seq) {
  if (!rt || !seq) return fail(LLVQ_ERR_INVALID_ARGUMENT, "sequence_run: null argument");
  HIP_TRY(hipSetDevice(rt->device));
  return seq_run(rt, seq);
}

int llvq_hip_sequence_status(llvq_rt* rt, llvq_seq* seq) {
  if (!rt || !seq) return fail(LLVQ_ERR_INVALID_ARGUMENT, "sequence_status: null argument");
  HIP_TRY(hipSetDevice(rt->device));
  HIP_TRY(hipStreamSynchronize(rt->stream));
  uint32_t st = 0;
  HIP_TRY(hipMemcpy(&st, seq->args.status, sizeof st, hipMemcpyDeviceToHost));
  if (!st) return LLVQ_OK;
  // the counters of a run that gave up are short: start over from zero
  const int rc = seq_reset(seq);
  if (rc) return rc;
  return fail(LLVQ_ERR_DEVICE, "sequence: a workgroup gave up waiting for an item; the run's outputs are incomplete");
}

int llvq_hip_sequence_tune(llvq_seq* seq, uint32_t spin_limit, int hold_item) {
  if (!seq) return fail(LLVQ_ERR_INVALID_ARGUMENT, "sequence_tune: null sequence");
  if (hold_item >= (int)seq->n_items) return fail(LLVQ_ERR_INVALID_ARGUMENT, "sequence_tune: no such item");
  seq->args.spin_limit = spin_limit ? spin_limit : kSeqSpinLimit;
  seq->args.hold_item = hold_item >= 0 ? (uint32_t)hold_item : kSeqNoWait;
  return LLVQ_OK;
}

void llvq_hip_sequence_destroy(llvq_rt* rt, llvq_seq* seq) {
  if (!seq) return;
  if (rt) {
    (void)hipSetDevice(rt->device);
    (void)hipStreamSynchronize(rt->stream);
  }
  (void)hipFree(seq->blob);
  delete seq;
}

// Grows a device buffer of the runtime to `need` bytes (contents are not kept).
static int grow_buffer(void** buf, size_t* have, size_t need) {
  if (need <= *have) return LLVQ_OK;
  (void)hipFree(*buf);  // waits for launches that still use it
  *buf = nullptr;
  *have = 0;
  HIP_TRY(hipMalloc(buf, need));
  *have = need;
  return LLVQ_OK;
}

// Where a batched call's device workspaces come from: the runtime's buffers, grown with
// hipMalloc on first use of a larger shape, or (fixed != null) a region the caller of this
// file's helpers provides, which is carved up and never outgrown.
struct GemmWorkspace {
  uint8_t* fixed = nullptr;
  size_t fixed_bytes = 0, used = 0;
};
static int workspace_take(llvq_rt* rt, GemmWorkspace* w, void** runtime_buf, size_t* runtime_have, size_t need, void** out) {
  if (!w || !w->fixed) {
    const int rc = grow_buffer(runtime_buf, runtime_have, need);
    *out = *runtime_buf;
    return rc;
  }
  const size_t at = (w->used + 255) & ~(size_t)255;
  if (need > w->fixed_bytes || at > w->fixed_bytes - need)
    return fail(LLVQ_ERR_UNSUPPORTED, "gemm_static: this shape needs " + std::to_string(at + need) +
                                          " bytes of workspace, the static one holds " + std::to_string(w->fixed_bytes));
  *out = w->fixed + at;
  w->used = at + need;
  return LLVQ_OK;
}

// Rows of activations one batched launch takes; more go out as further launches.  With both terms of the weights (pair)
// half as many where the rows are so wide that their octets would exceed 32 MiB: up to the widest rows a batch-1 product
// takes, such a launch's octets and partial sums (kGemmWsCap) then fit LLVQ_STATIC_SCRATCH_BYTES.
constexpr uint32_t kGemmMaxM = 1024;
static uint32_t gemm_chunk(uint32_t nb, bool pair) { return pair && (nb + 3u) / 4u * 12u > 2048u ? kGemmMaxM / 2 : kGemmMaxM; }
static_assert((kGemvMaxBlocks + 3) / 4 * 12 * (kGemmMaxM / 2) * 16 <= (32u << 20) && 2048u * kGemmMaxM * 16 <= (32u << 20), "octets of a launch");

// Measured times of one step (48 columns) of the wide kernel in us (85 steps less 8, back to back): 256 weight rows by 256
// activation rows; 384 by 128; 256 by 128, two workgroups sharing a CU, each; one of those alone; and with both terms of the
// weights.
constexpr double kWideStep = 1.21, kTallStep = 1.12, kWideHalfStep = 0.76, kWideHalfStepAlone = 0.80, kWidePairStep = 2.5;

// How a batched launch over these matrices at M rows is cut up, and the workspaces it needs.  pair: with both terms of
// the weights (gemm_same_basis says when).
struct GemmPlan {
  uint32_t small;                // 1: up to 16 rows, 2: up to 64 (gemm_tiles_kernel), 0: gemm_wide_kernel
  uint32_t rf, cf, rows_per_tile;  // the wide kernel's form, and weight rows of a workgroup
  uint32_t n_tiles, m_pad, m_tiles, splits, steps_per_split, n_oct;
  size_t ws_bytes, xt_bytes;
};
// The wide kernel's partial sums are kept below this: more column splits than that allows would cost more in memory
// traffic than they gain in filled CUs.
constexpr size_t kGemmWsCap = 32u << 20;
static GemmPlan gemm_plan(const llvq_rt* rt, const llvq_mat* const* mats, int n, uint32_t M, bool pair) {
  const uint32_t cus = (uint32_t)(rt->cu_count > 0 ? rt->cu_count : 256), nb = mats[0]->nblocks;
  GemmPlan p{};
  p.small = M <= 16u ? 1u : M <= kGemmSmallRows ? 2u : 0u;
  p.splits = 1;
  p.m_tiles = 1;
  p.rows_per_tile = pair ? 16u : p.small * 16u;
  const auto tiles_of = [&](uint32_t rows) {
    uint32_t sum = 0;
    for (int i = 0; i < n; ++i) sum += (mats[i]->d_out + rows - 1u) / rows;
    return sum;
  };
  p.n_oct = (nb + 3u) / 4u * 12u;
  if (p.small) {
    p.n_tiles = tiles_of(p.rows_per_tile);
    p.m_pad = p.small == 1u ? 16u : 64u;
    p.xt_bytes = (size_t)p.n_oct * p.m_pad * 16;
    return p;
  }
  // The form and the column splits by the time they should take: rounds of resident workgroups times steps of a
  // workgroup's share of a CU, and for the splits what the partial sums cost on their way through memory.
  // (Rows of a multiple of 8 values that lie off a boundary are not split: what is reserved for such matrices at their usual
  // place holds the octets of either plan, and needs no partial sums for rows that hardly ever come.)
  const uint32_t steps = (nb + 1u) / 2u, most = pair && mats[0]->d_in % 8 == 0 ? 1u : 16u;
  double best = 1e30;
  const auto weigh = [&](uint32_t rf, uint32_t cf, uint32_t most) {
    const uint32_t rows = 128u * rf, n_tiles = tiles_of(rows), m_tiles = (M + 32u * cf - 1u) / (32u * cf), m_pad = m_tiles * 32u * cf;
    const size_t one = (size_t)m_pad * n_tiles * rows * sizeof(float);
    for (uint32_t sp = 1; sp <= most && (sp == 1u || (steps / sp >= 8u && one * sp <= kGemmWsCap)); ++sp) {
      const uint32_t per = (steps + sp - 1u) / sp, wgs = n_tiles * m_tiles * ((steps + per - 1u) / per), per_cu = (wgs + cus - 1u) / cus;
      const double step = pair ? kWidePairStep : rf == 3u ? kTallStep : cf == 8u ? kWideStep : per_cu == 1u ? kWideHalfStepAlone : kWideHalfStep;
      const double cost = per_cu * step * per + (sp > 1u ? 3.0 + 2.0 * (double)one * sp / 4e6 : 0.0);
      if (cost < best) {
        best = cost;
        p.rf = rf;
        p.cf = cf;
        p.rows_per_tile = rows;
        p.n_tiles = n_tiles;
        p.m_tiles = m_tiles;
        p.m_pad = m_pad;
        p.splits = (steps + per - 1u) / per;
        p.steps_per_split = per;
        p.ws_bytes = p.splits > 1u ? one * p.splits : 0;
      }
    }
  };
  if (!pair) weigh(2u, 8u, most);
  weigh(2u, 4u, most);
  // (384 rows are not split: of 150 000 drawn shapes none would be, and no call needs more workspace for them.)
  if (!pair) weigh(3u, 4u, 1u);
  p.xt_bytes = (size_t)p.n_oct * p.m_pad * 16;
  return p;
}

// Sizes the runtime's batched-path buffers for calls over these matrices (grouped as
// llvq_hip_gemm_group groups them) at up to max_rows activation rows, so that those calls find
// them large enough and allocate nothing.
static int reserve_batched(llvq_rt* rt, const llvq_mat* const* mats, int n, uint32_t max_rows) {
  if (n <= 0 || max_rows < 2) return LLVQ_OK;
  size_t ws = 0, xt = 0, rows = 0;
  for (int i0 = 0; i0 < n;) {
    int i1 = i0 + 1;
    while (i1 < n && i1 - i0 < kGemmMaxGroup && mats[i1]->has_rotation == mats[i0]->has_rotation &&
           (!mats[i0]->has_rotation || mats[i1]->rot == mats[i0]->rot))
      ++i1;
    bool six_byte = true;
    for (int i = i0; i < i1; ++i) six_byte &= mats[i]->record_bits == 48;
    if (mats[i0]->nblocks && six_byte) {  // (cap-13 matrices take the row loop, which has no workspace)
      const bool pair = mats[i0]->d_in % 8 != 0;
      const uint32_t chunk = std::min(max_rows, gemm_chunk(mats[i0]->nblocks, pair));
      // every row count up to the chunk: the splits, and so the partial sums, are not monotone in it
      for (uint32_t M = 16;; M = M < 64u ? M + 48u : M < 128u ? 128u : M + 128u) {
        const GemmPlan p = gemm_plan(rt, mats + i0, i1 - i0, M < chunk ? M : chunk, pair);
        ws = p.ws_bytes > ws ? p.ws_bytes : ws;
        xt = p.xt_bytes > xt ? p.xt_bytes : xt;
        if (M >= chunk) break;
      }
    }
    if (mats[i0]->has_rotation) {
      const size_t r = (size_t)max_rows * mats[i0]->d_in * sizeof(__half);
      rows = r > rows ? r : rows;
    }
    i0 = i1;
  }
  int rc = grow_buffer(reinterpret_cast<void**>(&rt->gemm_ws), &rt->gemm_ws_bytes, ws);
  if (!rc) rc = grow_buffer(reinterpret_cast<void**>(&rt->gemm_xt), &rt->gemm_xt_bytes, xt);
  if (!rc) rc = grow_buffer(reinterpret_cast<void**>(&rt->rot_rows), &rt->rot_rows_bytes, rows);
  return rc;
}

// Whether gemm_tiles_kernel reads a small batch where it is, so that no launch makes octets of it (2.2 us).  A load of sixteen rows' pieces
// then meets as many lines as there are rows, three of which cost nothing and each other one 0.065 us for each unit of a wavefront: direct /
// by octets, in us, 4096 x 4096 at 2, 5, 10 and 16 rows 5.4 / 7.5, 5.4 / 7.5, 6.3 / 7.4, 7.4 / 7.5; 12288 x 4096 10.2 / 12.0, 11.3 / 12.1,
// 14.1 / 12.1, 17.4 / 12.2; 2560 x 9728 7.7 / 10.0, 8.4 / 9.8, 10.5 / 9.9, 13.0 / 10.0; 5120 x 17408 19.6 / 21.7, 22.7 / 21.7.  Rows off 16-byte
// boundaries, where a piece is two lines, gain at 2 rows (4096 x 4097 8.4 / 8.8) and lose from 4 (9.6 / 8.3).
static bool gemm_direct(uint32_t M, uint32_t n_tiles, uint32_t nb, uint32_t cus, bool pair) {
  if (pair || M > 16u) return false;
  const uint32_t units = (n_tiles + cus - 1u) / cus * tile_units(nb);  // of the fullest CU
  return M <= 3u || (M - 3u) * units < 20u * 16u;
}
// Whether one of the results lies over the rows, be it in part.  Such rows are not read where they are: octets are whole before the
// product that stores begins.
static bool stored_over_rows(const void* x, size_t x_bytes, const llvq_mat* const* mats, int n, uint32_t M, void* const* y, int y_dtype) {
  const uintptr_t x0 = reinterpret_cast<uintptr_t>(x);
  for (int i = 0; i < n; ++i) {
    const uintptr_t y0 = reinterpret_cast<uintptr_t>(y[i]);
    if (y0 < x0 + x_bytes && x0 < y0 + (size_t)M * mats[i]->d_out * (y_dtype == LLVQ_F32 ? 4u : 2u)) return true;
  }
  return false;
}
// One launch over n <= kGemmMaxGroup matrices of equal d_in that take the same activations
// (already in the matrices' basis), M <= kGemmMaxM rows.  from: rows that are rotated on the way to the octets, their tail
// columns to x.
// make: launches what makes the rows, as octets (and their tail columns in x).  left: takes the results where they are partial ones, to be
// added up by a launch that is enqueued before the next product's (no results in y then).
static int launch_gemm(llvq_rt* rt, const llvq_mat* const* mats, int n, const void* x, uint32_t M, void* const* y,
                       int y_dtype, bool pair, GemmWorkspace* wsp = nullptr, const void* from = nullptr, const std::function<void(const Octets&)>* make = nullptr,
                       GemmSums* left = nullptr) {
  const llvq_mat* m0 = mats[0];
  const __half* xh = reinterpret_cast<const __half*>(x);
  const GemmPlan p = gemm_plan(rt, mats, n, M, pair);
  void* ws_buf = nullptr;
  void* xt_buf = nullptr;
  const size_t mark = wsp ? wsp->used : 0;  // a launch's carvings are released when it has been enqueued: the stream orders the next
  int rc = LLVQ_OK;
  if (p.ws_bytes) rc = workspace_take(rt, wsp, reinterpret_cast<void**>(&rt->gemm_ws), &rt->gemm_ws_bytes, p.ws_bytes, &ws_buf);
  if (rc) return rc;
  rc = workspace_take(rt, wsp, reinterpret_cast<void**>(&rt->gemm_xt), &rt->gemm_xt_bytes, p.xt_bytes, &xt_buf);
  if (rc) return rc;
  if (wsp) wsp->used = mark;
  GemmArgs a{};
  a.xt = reinterpret_cast<const uint4*>(xt_buf);
  a.x = xh;
  a.ws = reinterpret_cast<float*>(ws_buf);
  a.n_mats = (uint32_t)n;
  for (int i = 0; i < n; ++i) {
    a.mat[i] = GemmMat{mats[i]->tiles, y[i], mats[i]->d_out, a.n_tiles, mats[i]->stride, mats[i]->slots};
    a.n_tiles += (mats[i]->d_out + p.rows_per_tile - 1u) / p.rows_per_tile;
  }
  a.y_f32 = y_dtype == LLVQ_F32 ? 1u : 0u;
  a.ldx = m0->d_in;
  a.tail_w = m0->tail_w;
  a.M = M;
  a.m_pad = p.m_pad;
  a.nb = m0->nblocks;
  a.m_tiles = p.m_tiles;
  a.splits = p.splits;
  a.steps_per_split = p.steps_per_split;
  const bool direct = !from && !make && p.small == 1u && gemm_direct(M, a.n_tiles, a.nb, (uint32_t)(rt->cu_count > 0 ? rt->cu_count : 256), pair) &&
                      !stored_over_rows(x, (size_t)M * m0->d_in * 2u, mats, n, M, y, y_dtype);
  a.xs = direct ? reinterpret_cast<const uint8_t*>(x) : reinterpret_cast<const uint8_t*>(xt_buf);
  a.xs_octet = direct ? 16u : p.m_pad * 16u;
  a.xs_block = 3u * a.xs_octet;
  a.xs_unit = 4u * a.xs_block;
  a.xs_row = direct ? a.ldx * 2u : 16u;
  a.xs_last = direct ? M - 1u : 15u;
  if (from) {
    RotArgs ra = rot_args(m0->rot, from, const_cast<void*>(x));
    ra.xt = reinterpret_cast<uint4*>(xt_buf);
    ra.rows = M;
    ra.m_pad = p.m_pad;
    ra.n_oct = p.n_oct;
    ra.kcols = a.nb * kDim;
    hipLaunchKernelGGL(rotate_kernel<RotOctets>, dim3(p.m_pad), dim3(1024), (size_t)ra.n * sizeof(float), rt->stream, ra);
  } else if (make) {
    (*make)(Octets{reinterpret_cast<uint4*>(xt_buf), M, p.m_pad, p.n_oct, a.nb * kDim});
  } else if (!direct) {
    const uint32_t oct_waves = (p.n_oct + 7u) / 8u * (p.m_pad / 8u);
    hipLaunchKernelGGL(tile_activations_kernel, dim3((oct_waves + 3u) / 4u), dim3(256), 0, rt->stream, xh, (const __half*)nullptr, (__half*)nullptr, M,
                       a.ldx, a.nb * 24u, p.m_pad, p.n_oct, reinterpret_cast<uint4*>(xt_buf));
  }
  const dim3 wide_grid(a.n_tiles * p.m_tiles * p.splits);
  auto product = [&](auto pair) {
    constexpr bool kPair = decltype(pair)::value;
    if (p.small == 1u) hipLaunchKernelGGL((gemm_tiles_kernel<1, 1, kPair>), dim3(a.n_tiles), dim3(1024), (gemm_small_lds<1, 1>()), rt->stream, a);
    else if (p.small) hipLaunchKernelGGL((gemm_tiles_kernel<kPair ? 1 : 2, 4, kPair>), dim3(a.n_tiles), dim3(1024), (gemm_small_lds<kPair ? 1 : 2, 4>()), rt->stream, a);
    else if (p.rf == 2u && p.cf == 4u) hipLaunchKernelGGL((gemm_wide_kernel<4, kPair>), wide_grid, dim3(256), (gemm_wide_lds<2, 4, kPair>()), rt->stream, a);
    else if constexpr (!kPair) {
      if (p.rf == 3u) hipLaunchKernelGGL(gemm_tall_kernel, wide_grid, dim3(256), (gemm_wide_lds<3, 4, false>()), rt->stream, a);
      else hipLaunchKernelGGL((gemm_wide_kernel<8, false>), wide_grid, dim3(256), (gemm_wide_lds<2, 8, false>()), rt->stream, a);
    }
  };
  if (pair) product(std::true_type{});
  else product(std::false_type{});
  if (p.splits > 1u && pair) {
    hipLaunchKernelGGL(gemm_reduce_pair_kernel, dim3(a.n_tiles, (M + kReduceM - 1u) / kReduceM), dim3(kReduceRows), 0, rt->stream, a);
  } else if (p.splits > 1u && left) {
    *left = GemmSums{a.ws, p.splits, p.m_pad, a.n_tiles * p.rows_per_tile, {}};
    for (int i = 0; i < n; ++i) left->first[i] = a.mat[i].tile_begin * p.rows_per_tile;
  } else if (p.splits > 1u) {
    hipLaunchKernelGGL(gemm_sum_kernel, dim3(a.n_tiles, (M + 4u * kSumM - 1u) / (4u * kSumM)), dim3(256), 0, rt->stream, a);
  }
  HIP_TRY(hipGetLastError());
  return LLVQ_OK;
}

// What llvq_hip_gemm_static admits of rows on 16-byte boundaries.  The bound is part of its contract (callers choose their
// fallback by it: what it refused stays refused), so it is the one of the partial-sum layout the entry point was specified
// with (gemm_share.h: a band's K-slices shared out over the workgroups, 64 x 64 sums per piece, and a tiled copy of the
// activations).  The kernels need less, and nothing else uses that formula.
static size_t static_admission_bytes(const llvq_rt* rt, const llvq_mat* m, uint32_t M) {
  const uint32_t grid_cap = (uint32_t)(rt->cu_count > 0 ? rt->cu_count : 256), consumers = M <= 256u ? 4u : 8u;
  const uint32_t bands = (m->d_out + 63u) / 64u, spb = (m->nblocks + 15u) / 16u;
  uint32_t ct_shift = 0;
  while ((64u << ct_shift) < M) ++ct_shift;
  const uint32_t kparts = consumers >> ct_shift;
  const GemmShare share = gemm_share(bands ? bands : 1, spb ? spb : 1, grid_cap);
  const uint32_t band0 = kparts == 1 ? share.shared0 : 0u;
  const size_t sums = (size_t)(bands - (band0 < bands ? band0 : bands)) * share.max_pieces * kparts * M * 64 * sizeof(float);
  return ((sums + 255) & ~(size_t)255) + (size_t)spb * 12 * ((M + 63) / 64 * 64) * 64;
}

// Whether one launch takes M rows that come as octets through these matrices (what gemm_same_basis asks of rows in their own basis).
static bool gemm_takes_octets(const llvq_mat* const* mats, int n, uint32_t M) {
  if (n > kGemmMaxGroup || M < 2u || !mats[0]->nblocks || mats[0]->d_in % 8 != 0 || M > gemm_chunk(mats[0]->nblocks, false)) return false;
  for (int i = 0; i < n; ++i)
    if (mats[i]->has_rotation || mats[i]->record_bits != 48 || mats[i]->d_in != mats[0]->d_in) return false;
  return true;
}

// Matrices [0, n) of one group: same d_in, same basis.  What such a call has always been good to decides its way:
//   * rows of a multiple of 8 values from a 16-byte boundary on: weights rounded to binary16 once (error 2e-4 of the
//     results' norm);
//   * other rows, natural basis: both terms of the weights (1e-7 with f32 results, which is what a row by itself has).
//     A second product costs the matrix cores twice the time (13000 x 5121 at 600 rows 250 to 280 us for 115) and a loop of
//     single rows many times that (27 900 us before there were tiles);
//   * row by row, as batch-1 products: a single row, other rows in a rotated basis (the products above take them as
//     binary16, a row by itself in f32; such widths end at 124), matrices without a whole block, and cap-13 matrices,
//     whose rows keep the bits of the single-row product.
static int gemm_same_basis(llvq_rt* rt, const llvq_mat* const* mats, int n, const void* x, int M, void* const* y, int y_dtype,
                           GemmWorkspace* wsp = nullptr, GemmSums* left = nullptr) {
  const llvq_mat* m0 = mats[0];
  const size_t esz = y_dtype == LLVQ_F32 ? 4 : 2;
  const uint8_t* xb = reinterpret_cast<const uint8_t*>(x);
  bool six_byte = true;
  for (int i = 0; i < n; ++i) six_byte &= mats[i]->record_bits == 48;
  const bool pair = m0->d_in % 8 != 0 || (reinterpret_cast<uintptr_t>(x) & 15) != 0;
  if (M < 2 || m0->nblocks == 0 || !six_byte || (pair && m0->has_rotation)) {
    for (int i = 0; i < n; ++i)
      for (int r = 0; r < M; ++r) {
        const int rc = launch_gemv(rt, mats[i], xb + (size_t)r * m0->d_in * 2, reinterpret_cast<uint8_t*>(y[i]) + (size_t)r * mats[i]->d_out * esz, y_dtype);
        if (rc) return rc;
      }
    return LLVQ_OK;
  }
  const int chunk = std::min(M, (int)gemm_chunk(m0->nblocks, pair));
  if (wsp && wsp->fixed) {
    // a call that does not fit is refused whole, before its first launch
    auto after = [](size_t used, size_t bytes) { return ((used + 255) & ~(size_t)255) + bytes; };
    const size_t base = m0->has_rotation ? after(wsp->used, (size_t)M * m0->d_in * sizeof(__half)) : wsp->used;
    size_t need = base;
    if (!pair)  // (rows that pair takes have no such bound, and fit: gemm_chunk)
      for (int m_lo = 0; m_lo < M; m_lo += 512)
        for (int i = 0; i < n; ++i) need = std::max(need, after(base, static_admission_bytes(rt, mats[i], (uint32_t)std::min(M - m_lo, 512))));
    for (int m_lo = 0; m_lo < M; m_lo += chunk)
      for (int i0 = 0; i0 < n; i0 += kGemmMaxGroup) {
        const GemmPlan p = gemm_plan(rt, mats + i0, std::min(n - i0, kGemmMaxGroup), (uint32_t)std::min(M - m_lo, chunk), pair);
        need = std::max(need, after(p.ws_bytes ? after(base, p.ws_bytes) : base, p.xt_bytes));
      }
    if (need > wsp->fixed_bytes)
      return fail(LLVQ_ERR_UNSUPPORTED, "gemm_static: this shape needs " + std::to_string(need) +
                                            " bytes of workspace, the static one holds " + std::to_string(wsp->fixed_bytes));
  }
  if (m0->has_rotation) {
    // rows are rotated (f32 inside) and narrowed to the binary16 the matrix cores take
    void* rows = nullptr;
    const int rc0 = workspace_take(rt, wsp, reinterpret_cast<void**>(&rt->rot_rows), &rt->rot_rows_bytes,
                                   (size_t)M * m0->d_in * sizeof(__half), &rows);
    if (rc0) return rc0;
    if (n <= kGemmMaxGroup && M <= chunk && m0->rot->m >= kRotOctetM)
      return launch_gemm(rt, mats, n, rows, (uint32_t)M, y, y_dtype, pair, wsp, x, nullptr, left);
    const int rc = launch_rotate(rt, m0->rot, x, (uint32_t)M, rows, true);
    if (rc) return rc;
    xb = reinterpret_cast<const uint8_t*>(rows);
  }
  for (int m_lo = 0; m_lo < M; m_lo += chunk) {
    const uint32_t mc = (uint32_t)std::min(M - m_lo, chunk);
    for (int i0 = 0; i0 < n; i0 += kGemmMaxGroup) {
      const int cnt = n - i0 < kGemmMaxGroup ? n - i0 : kGemmMaxGroup;
      void* ys[kGemmMaxGroup];
      for (int i = 0; i < cnt; ++i) ys[i] = reinterpret_cast<uint8_t*>(y[i0 + i]) + (size_t)m_lo * mats[i0 + i]->d_out * esz;
      const int rc = launch_gemm(rt, mats + i0, cnt, xb + (size_t)m_lo * m0->d_in * 2, mc, ys, y_dtype, pair, wsp, nullptr, nullptr,
                                 cnt == n && (int)mc == M ? left : nullptr);
      if (rc) return rc;
    }
  }
  return LLVQ_OK;
}

int llvq_hip_gemm_group(llvq_rt* rt, const llvq_mat* const* mats, int n, const void* x, int M, void* const* y, int y_dtype) {
  if (!rt || !mats || !y || n < 0 || M < 0) return fail(LLVQ_ERR_INVALID_ARGUMENT, "gemm_group: bad argument");
  if (y_dtype != LLVQ_F32 && y_dtype != LLVQ_F16) return fail(LLVQ_ERR_INVALID_ARGUMENT, "gemm_group: unknown output dtype");
  for (int i = 0; i < n; ++i) {
    if (!mats[i]) return fail(LLVQ_ERR_INVALID_ARGUMENT, "gemm_group: null matrix");
    if (mats[i]->d_in != mats[0]->d_in)
      return fail(LLVQ_ERR_INVALID_ARGUMENT, mats[i]->name + ": projections of one group must share d_in");
  }
  if (M == 0 || n == 0) return LLVQ_OK;  // no rows: nothing is read or written, so the pointers may be null
  if (!x) return fail(LLVQ_ERR_INVALID_ARGUMENT, "gemm_group: null activation");
  for (int i = 0; i < n; ++i)
    if (!y[i]) return fail(LLVQ_ERR_INVALID_ARGUMENT, "gemm_group: null output");
  HIP_TRY(hipSetDevice(rt->device));
  // consecutive matrices that share a basis go into one launch; the activation is rotated once per basis
  for (int i0 = 0; i0 < n;) {
    int i1 = i0 + 1;
    while (i1 < n && mats[i1]->has_rotation == mats[i0]->has_rotation && (!mats[i0]->has_rotation || mats[i1]->rot == mats[i0]->rot)) ++i1;
    const int rc = gemm_same_basis(rt, mats + i0, i1 - i0, x, M, y + i0, y_dtype);
    if (rc) return rc;
    i0 = i1;
  }
  return LLVQ_OK;
}

int llvq_hip_gemm(llvq_rt* rt, const llvq_mat* m, const void* x, int M, void* y, int y_dtype) {
  if (!rt || !m || M < 0) return fail(LLVQ_ERR_INVALID_ARGUMENT, "gemm: bad argument");
  if (M == 0) return LLVQ_OK;  // no rows: nothing is read or written, so the pointers may be null
  if (!x || !y) return fail(LLVQ_ERR_INVALID_ARGUMENT, "gemm: null activation or output");
  return llvq_hip_gemm_group(rt, &m, 1, x, M, &y, y_dtype);
}

int llvq_hip_reserve_batched(llvq_rt* rt, const llvq_mat* const* mats, int n, int max_rows) {
  if (!rt || !mats || n < 0 || max_rows < 0) return fail(LLVQ_ERR_INVALID_ARGUMENT, "reserve_batched: bad argument");
  for (int i = 0; i < n; ++i) {
    if (!mats[i]) return fail(LLVQ_ERR_INVALID_ARGUMENT, "reserve_batched: null matrix");
    if (mats[i]->d_in != mats[0]->d_in)
      return fail(LLVQ_ERR_INVALID_ARGUMENT, mats[i]->name + ": projections of one group must share d_in");
  }
  HIP_TRY(hipSetDevice(rt->device));
  return reserve_batched(rt, mats, n, (uint32_t)max_rows);
}

int llvq_hip_gemm_static(llvq_rt* rt, const llvq_mat* m, const void* x, int M, void* y, int y_dtype) {
  if (!rt || !m || M < 0) return fail(LLVQ_ERR_INVALID_ARGUMENT, "gemm_static: bad argument");
  if (y_dtype != LLVQ_F32 && y_dtype != LLVQ_F16) return fail(LLVQ_ERR_INVALID_ARGUMENT, "gemm_static: unknown output dtype");
  if (M == 0) return LLVQ_OK;
  if (!x || !y) return fail(LLVQ_ERR_INVALID_ARGUMENT, "gemm_static: null activation or output");
  if (!rt->static_scratch) return fail(LLVQ_ERR_UNSUPPORTED, "gemm_static: no static workspace on this device");
  HIP_TRY(hipSetDevice(rt->device));
  GemmWorkspace w;
  w.fixed = rt->static_scratch;
  w.fixed_bytes = kStaticScratchBytes;
  return gemm_same_basis(rt, &m, 1, x, M, &y, y_dtype, &w);
}

int llvq_hip_decode_blocks(llvq_rt* rt, const uint8_t* codes_dev, size_t nblocks, int8_t* points_dev,
                           uint8_t* gains_dev, uint8_t* shells_dev) {
  if (!rt) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decode_blocks: runtime is null");
  if (nblocks == 0) return LLVQ_OK;  // an empty stream is valid and writes nothing
  if (!points_dev || !codes_dev) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decode_blocks: null argument");
  if (reinterpret_cast<uintptr_t>(codes_dev) & 3) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decode_blocks: codes must start on a 4-byte boundary");
  HIP_TRY(hipSetDevice(rt->device));
  size_t grid = (nblocks + 255) / 256;
  const size_t cap = (size_t)(rt->cu_count > 0 ? rt->cu_count : 256) * 2;
  if (grid > cap) grid = cap;
  hipLaunchKernelGGL(decode_blocks_kernel<false>, dim3((uint32_t)grid), dim3(256), kLdsImageBytes, rt->stream,
                     rt->tables, codes_dev, nblocks, points_dev, gains_dev, shells_dev);
  HIP_TRY(hipGetLastError());
  return LLVQ_OK;
}

int llvq_hip_decode_stream(llvq_rt* rt, const uint8_t* codes_dev, size_t nblocks, uint32_t shell_cap, int8_t* points_dev,
                           uint8_t* gains_dev, uint8_t* shells_dev) {
  if (!rt) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decode_stream: runtime is null");
  if (shell_cap > (uint32_t)kMaxShell) return fail(LLVQ_ERR_INCONSISTENT, "decode_stream: shell cap " + std::to_string(shell_cap) + " exceeds the supported ball (m <= 13)");
  const int bits = index_bits(shell_cap) + 1;
  if (bits == 48) return llvq_hip_decode_blocks(rt, codes_dev, nblocks, points_dev, gains_dev, shells_dev);
  if (bits != (int)kDenseBits)
    return fail(LLVQ_ERR_UNSUPPORTED, "decode_stream: shell cap " + std::to_string(shell_cap) + " packs " + std::to_string(bits) +
                                          " bits per block; the kernels read 6-byte records (cap 12) and the 49-bit stream of cap 13");
  if (nblocks == 0) return LLVQ_OK;
  if (!points_dev || !codes_dev) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decode_stream: null argument");
  HIP_TRY(hipSetDevice(rt->device));
  size_t grid = (nblocks + 255) / 256;
  const size_t cap = (size_t)(rt->cu_count > 0 ? rt->cu_count : 256) * 2;
  if (grid > cap) grid = cap;
  hipLaunchKernelGGL(decode_blocks_kernel<true>, dim3((uint32_t)grid), dim3(256), kLdsImageBytes, rt->stream,
                     rt->tables, codes_dev, nblocks, points_dev, gains_dev, shells_dev);
  HIP_TRY(hipGetLastError());
  return LLVQ_OK;
}

}  // extern "C"

// =================================================================================
// Batch-1 decode loop (C ABI)
// =================================================================================
struct llvq_decoder {
  llvq_rt* rt = nullptr;
  uint32_t n_layers = 0, hidden = 0, n_heads = 0, n_kv = 0, head_dim = 0, inter = 0, vocab = 0, max_pos = 0;
  float eps = 1e-6f;
  std::vector<const llvq_mat*> proj;  // [n_layers * 7]: q k v o gate up down
  uint8_t* blob = nullptr;            // every dense tensor and buffer below, one allocation
  __half *ln1 = nullptr, *ln2 = nullptr, *qn = nullptr, *kn = nullptr, *fnorm = nullptr;
  __half *embed = nullptr, *head = nullptr, *cos_t = nullptr, *sin_t = nullptr;
  bool embed_q8 = false, head_q8 = false;  // int8 rows instead of binary16
  QuantRows embed_q{}, head_q{};
  __half *kcache = nullptr, *vcache = nullptr;  // [n_layers][n_kv][max_pos][head_dim]
  __half *h = nullptr, *h_alt = nullptr, *normed = nullptr, *q = nullptr, *k = nullptr, *v = nullptr, *ctx = nullptr, *o = nullptr;
  __half *gate = nullptr, *up = nullptr, *act = nullptr, *down = nullptr;
  float* logits = nullptr;      // [vocab], and the chosen token behind them
  float* host_out = nullptr;    // [vocab + 1] pinned memory: a step's last launch leaves logits and token there (null where there is none to be had: copies to the caller's memory)
  float* best_val = nullptr;
  uint32_t* best_idx = nullptr;
  uint32_t* token = nullptr;    // logits + vocab: the token the next step embeds
  uint32_t* history = nullptr;  // [max_pos] tokens chosen by the head
  float* attn_part = nullptr;   // [n_heads][kAttnMaxSplits][head_dim + 2] partial attention sums
  bool kv_q8 = false;           // int8 KV cache (kvq.rs) instead of binary16
  KvQ8 q8{};                    // layer 0's arrays; a layer's are at + layer * (cache_layer or cache_layer / 64 groups)
  uint32_t* attn_counters = nullptr;  // [n_kv][kDecodeCounter], zero between launches
  uint32_t pos = 0;
  uint32_t head_grid = 0;
  // rows of positions at once (llvq_hip_decoder_prefill): [prefill_rows, width] buffers, one allocation
  uint32_t prefill_rows = 0;
  uint8_t* pblob = nullptr;
  __half *ph = nullptr, *ph_alt = nullptr, *pnormed = nullptr, *pq = nullptr, *pk = nullptr, *pv = nullptr, *pctx = nullptr, *po = nullptr;
  __half *pgate = nullptr, *pup = nullptr, *pact = nullptr, *pdown = nullptr;
  uint32_t* ptokens = nullptr;
  // llvq_hip_decoder_generate_phased: events recorded at the phase boundaries of a step (null otherwise)
  std::vector<hipEvent_t>* marks = nullptr;
  size_t next_mark = 0;
  // A position's projections as sequences (empty: one launch of gemv_tiles_kernel per projection group).
  //   chained: seqs[0] = layer 0's q/k/v, seqs[L + 1] = layer L's o_proj, gate/up, down_proj and layer L + 1's q/k/v,
  //            each item ordered behind the one before it;
  //   single:  seqs[4 L + j] = layer L's q/k/v, o_proj, gate/up, down_proj, one item each.
  // They share one status word.
  std::vector<llvq_seq*> seqs;
  bool seq_chained = false;
  uint32_t* seq_status = nullptr;
  ~llvq_decoder() { (void)hipHostFree(host_out); }
};

namespace {

// A phase boundary of a timed step: the next event of the decoder's list goes onto the stream.
void phase_mark(llvq_decoder* d) {
  if (d->marks && d->next_mark < d->marks->size()) (void)hipEventRecord((*d->marks)[d->next_mark++], d->rt->stream);
}

// The head over dec->normed and the argmax, which overwrites *dec->token (and history[slot] when recording) and leaves what `host` asks for there.
void launch_head(llvq_decoder* d, uint32_t history_slot, bool record, const HostResults& host) {
  hipStream_t st = d->rt->stream;
  if (d->head_q8)
    hipLaunchKernelGGL(lm_head_q8_kernel, dim3(d->head_grid), dim3(kHeadThreads), d->hidden * sizeof(float), st, d->head_q, d->normed,
                       d->vocab, d->hidden, d->logits, d->best_val, d->best_idx);
  else
    hipLaunchKernelGGL(lm_head_kernel, dim3(d->head_grid), dim3(kHeadThreads), d->hidden * sizeof(float), st, d->head, d->normed,
                       d->vocab, d->hidden, d->logits, d->best_val, d->best_idx);
  phase_mark(d);
  const uint32_t copies = host.logits ? (d->vocab + kFinalCopy - 1u) / kFinalCopy : 0u;
  hipLaunchKernelGGL(argmax_final_kernel, dim3(1u + copies), dim3(kFinalThreads), 0, st, d->best_val, d->best_idx, d->head_grid * (kHeadThreads / 64),
                     d->token, record ? d->history : (uint32_t*)nullptr, history_slot, d->logits, d->vocab, host);
  phase_mark(d);
}

// Binds a position's projections as sequences (llvq_decoder::seqs), each item with the activation prologue its
// launch would have.  The residual stream alternates between the decoder's two buffers exactly as decoder_step's
// launches alternate them: layer 0's q/k/v reads h; every later prologue reads one buffer and stores the other.
// A model a sequence cannot take (rotated matrices, rows too wide) leaves seqs empty: one launch per group then.
int decoder_bind_sequences(llvq_decoder* d, bool chained) {
  llvq_rt* rt = d->rt;
  d->seq_chained = chained;
  __half *h = d->h, *h_alt = d->h_alt;
  auto give_up = [&](int rc) {
    for (llvq_seq* q : d->seqs) llvq_hip_sequence_destroy(rt, q);
    d->seqs.clear();
    return rc == LLVQ_ERR_UNSUPPORTED ? (int)LLVQ_OK : rc;
  };
  void* qkv_out[3] = {d->q, d->k, d->v};
  void* o_out[1] = {d->o};
  void* gu_out[2] = {d->gate, d->up};
  void* dn_out[1] = {d->down};
  auto qkv_item = [&](uint32_t L, bool ordered) {
    SeqSpec sp;
    sp.mats = d->proj.data() + (size_t)L * 7;
    sp.n = 3;
    sp.x = h;
    sp.y = qkv_out;
    sp.after_previous = ordered;
    sp.pro.kind = kPrologueAddRmsNorm;
    sp.pro.norm_w = d->ln1 + (size_t)L * d->hidden;
    sp.pro.eps = d->eps;
    if (L) {  // the previous layer's MLP output joins the residual stream here
      sp.pro.x2 = d->down;
      sp.pro.resid_out = h_alt;
      std::swap(h, h_alt);
    }
    return sp;
  };
  auto bind = [&](std::vector<SeqSpec>& items) {
    llvq_seq* q = nullptr;
    const int rc = seq_create(rt, items.data(), (int)items.size(), &q);
    if (rc) return rc;
    q->args.status = d->seq_status;
    d->seqs.push_back(q);
    return (int)LLVQ_OK;
  };
  if (!chained) {
    for (uint32_t L = 0; L < d->n_layers; ++L) {
      const llvq_mat* const* P = d->proj.data() + (size_t)L * 7;
      std::vector<SeqSpec> one(1);
      one[0] = qkv_item(L, false);
      int rc = bind(one);
      if (rc) return give_up(rc);
      SeqSpec o;
      o.mats = P + 3; o.n = 1; o.x = d->ctx; o.y = o_out;
      one[0] = o;
      if ((rc = bind(one))) return give_up(rc);
      SeqSpec gu;
      gu.mats = P + 4; gu.n = 2; gu.x = h; gu.y = gu_out;
      gu.pro.kind = kPrologueAddRmsNorm;
      gu.pro.norm_w = d->ln2 + (size_t)L * d->hidden;
      gu.pro.eps = d->eps;
      gu.pro.x2 = d->o;
      gu.pro.resid_out = h_alt;
      std::swap(h, h_alt);
      one[0] = gu;
      if ((rc = bind(one))) return give_up(rc);
      SeqSpec dn;
      dn.mats = P + 6; dn.n = 1; dn.x = d->up; dn.y = dn_out;
      dn.pro.kind = kPrologueSiluMul;
      dn.pro.x2 = d->gate;
      one[0] = dn;
      if ((rc = bind(one))) return give_up(rc);
    }
    return LLVQ_OK;
  }
  for (uint32_t L = 0; L <= d->n_layers; ++L) {
    std::vector<SeqSpec> items;
    if (L == 0) {
      items.push_back(qkv_item(0, false));
    } else {
      const llvq_mat* const* P = d->proj.data() + (size_t)(L - 1) * 7;
      SeqSpec o;
      o.mats = P + 3; o.n = 1; o.x = d->ctx; o.y = o_out;
      items.push_back(o);
      SeqSpec gu;
      gu.mats = P + 4; gu.n = 2; gu.x = h; gu.y = gu_out; gu.after_previous = true;
      gu.pro.kind = kPrologueAddRmsNorm;
      gu.pro.norm_w = d->ln2 + (size_t)(L - 1) * d->hidden;
      gu.pro.eps = d->eps;
      gu.pro.x2 = d->o;
      gu.pro.resid_out = h_alt;
      std::swap(h, h_alt);
      items.push_back(gu);
      SeqSpec dn;
      dn.mats = P + 6; dn.n = 1; dn.x = d->up; dn.y = dn_out; dn.after_previous = true;
      dn.pro.kind = kPrologueSiluMul;
      dn.pro.x2 = d->gate;
      items.push_back(dn);
      if (L < d->n_layers) items.push_back(qkv_item(L, true));
    }
    const int rc = bind(items);
    if (rc) return give_up(rc);
  }
  return LLVQ_OK;
}

// After the stream has drained: whether a workgroup of any sequence gave up waiting since the last check.
int decoder_check_sequences(llvq_decoder* d) {
  if (d->seqs.empty()) return LLVQ_OK;
  uint32_t st = 0;
  HIP_TRY(hipMemcpy(&st, d->seq_status, sizeof st, hipMemcpyDeviceToHost));
  if (!st) return LLVQ_OK;
  for (llvq_seq* q : d->seqs) {
    const int rc = seq_reset(q);
    if (rc) return rc;
  }
  return fail(LLVQ_ERR_DEVICE, "decoder: a workgroup gave up waiting for a projection of the same launch; the position's results are incomplete");
}

// Enqueues one position: embeds *fed (host memory, read here) or, without it, *dec->token, runs the layers at position dec->pos,
// and (want_logits) the head and the argmax, which overwrites *dec->token.
int decoder_step(llvq_decoder* d, bool want_logits, uint32_t history_slot, bool record, const uint32_t* fed = nullptr, const HostResults& host = {}) {
  llvq_rt* rt = d->rt;
  hipStream_t st = rt->stream;
  if (d->pos >= d->max_pos) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decoder: position " + std::to_string(d->pos) + " is past max_positions");
  // the two residual buffers, by local name: a step that fails part-way leaves the decoder as it found it
  __half *h = d->h, *h_alt = d->h_alt;
  phase_mark(d);
  if (d->embed_q8)
    hipLaunchKernelGGL(embed_q8_kernel, dim3((d->hidden + 255) / 256), dim3(256), 0, st, d->embed_q, fed ? (const uint32_t*)nullptr : d->token,
                       fed ? *fed : 0u, d->vocab, d->hidden, h);
  else
    hipLaunchKernelGGL(embed_kernel, dim3((d->hidden + 255) / 256), dim3(256), 0, st, d->embed, fed ? (const uint32_t*)nullptr : d->token,
                       fed ? *fed : 0u, d->vocab, d->hidden, h);
  phase_mark(d);
  const size_t cache_layer = (size_t)d->n_kv * d->max_pos * d->head_dim;
  const uint32_t T = d->pos + 1;
  // heads of another width than 128: about 64 cached positions per workgroup (one batch of four per position class), at most kAttnMaxSplits ranges
  uint32_t n_splits = (T + 63) / 64;
  if (n_splits > (uint32_t)kAttnMaxSplits) n_splits = kAttnMaxSplits;
  const uint32_t groups_per_kv = d->n_heads / d->n_kv;
  // the queries and the wavefronts' running results
  const size_t attn_lds = ((size_t)groups_per_kv * d->head_dim + (size_t)kAttnWaves * groups_per_kv * (d->head_dim + 2) + 4) * sizeof(float);
  const size_t group_layer = cache_layer / kKvGroup;
  // few partials: the last workgroup of a kv head merges them; many: a chip-wide merge kernel does
  const uint32_t merge_inline = n_splits <= (uint32_t)kAttnInlineSplits ? 1u : 0u;
  // Projections derive their activation in the launch's prologue, and rotate it there where their basis
  // is a rotated one; where rows are too wide for that (gemv_fits) the prologue runs as a kernel of its own.
  auto project = [&](const llvq_mat* const* mats, int n, const __half* x, void* const* outs, const Prologue& pro) -> int {
    // every launch of the group can derive (and, in a rotated basis, rotate) the activation itself
    bool fused = true;
    for (int i = 0; i < n; ++i) fused &= gemv_fits(mats[i]->d_in, false, mats[i]->has_rotation);
    if (fused) return forward_group(rt, mats, n, x, outs, LLVQ_F16, &pro);
    const __half* staged = nullptr;
    if (pro.kind == kPrologueAddRmsNorm) {
      hipLaunchKernelGGL(add_rmsnorm_kernel, dim3(1), dim3(norm_threads(d->hidden)), 0, st, x, reinterpret_cast<const __half*>(pro.x2),
                         reinterpret_cast<const __half*>(pro.norm_w), reinterpret_cast<__half*>(pro.resid_out), d->normed,
                         d->hidden, pro.eps, Octets{}, GemmSums{});
      staged = d->normed;
    } else {
      hipLaunchKernelGGL(silu_mul_kernel, dim3((d->inter / 8 + 256) / 256), dim3(256), 0, st, reinterpret_cast<const __half*>(pro.x2),
                         x, d->act, d->inter);
      staged = d->act;
    }
    return forward_group(rt, mats, n, staged, outs, LLVQ_F16);
  };
  // q/k norm, rope and the cache append of this position ride in the attention launch
  auto attention = [&](uint32_t L) {
    KvQ8 lq8 = d->q8;
    if (d->kv_q8) {
      lq8.kq += L * cache_layer; lq8.vq += L * cache_layer;
      lq8.ks += L * group_layer; lq8.kb += L * group_layer; lq8.vs += L * group_layer; lq8.vb += L * group_layer;
    }
    __half* kc = d->kv_q8 ? nullptr : d->kcache + L * cache_layer;
    __half* vc = d->kv_q8 ? nullptr : d->vcache + L * cache_layer;
    AttnNew nw{};
    nw.q_raw = d->q;
    nw.k_raw = d->k;
    nw.v_raw = d->v;
    nw.qn = d->qn + (size_t)L * d->head_dim;
    nw.kn = d->kn + (size_t)L * d->head_dim;
    nw.cos_t = d->cos_t;
    nw.sin_t = d->sin_t;
    nw.kcache = kc;
    nw.vcache = vc;
    nw.eps = d->eps;
    if (d->head_dim == 128u) {
      const uint32_t n = decode_ranges(T, d->n_kv, (uint32_t)(rt->cu_count > 0 ? rt->cu_count : 256));
      const auto kernel = groups_per_kv <= 4u ? (d->kv_q8 ? attn_decode_mfma_kernel<true, 1> : attn_decode_mfma_kernel<false, 1>)
                                              : (d->kv_q8 ? attn_decode_mfma_kernel<true, 2> : attn_decode_mfma_kernel<false, 2>);
      hipLaunchKernelGGL(kernel, dim3(n, d->n_kv), dim3(kDecodeWaves * 64u), 0, st, nw, kc, vc, lq8, d->ctx,
                         d->attn_part, d->attn_counters, groups_per_kv, (T + n - 1u) / n, T, d->max_pos, n);
      return;
    }
    auto attend = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(n_splits, d->n_kv), dim3(kAttnThreads), attn_lds, st, nw, kc, vc, lq8, d->ctx, d->attn_part,
                         d->attn_counters, groups_per_kv, (T + n_splits - 1) / n_splits, d->head_dim, T, d->max_pos, 1.0f / sqrtf((float)d->head_dim), n_splits,
                         merge_inline);
    };
    if (d->kv_q8) {
      if (groups_per_kv <= 2) attend(attn_decode_kernel<true, 2>);
      else if (groups_per_kv <= 4) attend(attn_decode_kernel<true, 4>);
      else if (groups_per_kv <= 5) attend(attn_decode_kernel<true, 5>);
      else attend(attn_decode_kernel<true, kAttnMaxGroup>);
    } else {
      if (groups_per_kv <= 2) attend(attn_decode_kernel<false, 2>);
      else if (groups_per_kv <= 4) attend(attn_decode_kernel<false, 4>);
      else if (groups_per_kv <= 5) attend(attn_decode_kernel<false, 5>);
      else attend(attn_decode_kernel<false, kAttnMaxGroup>);
    }
    if (!merge_inline)
      hipLaunchKernelGGL(attn_merge_kernel, dim3(d->n_heads), dim3(kMergeParts * 128), 0, st, d->attn_part, d->ctx, d->head_dim, n_splits);
  };
  if (!d->seqs.empty() && d->seq_chained) {
    // the projections between two attention launches are one persistent launch each
    int rc = seq_run(rt, d->seqs[0]);
    if (rc) return rc;
    for (uint32_t L = 0; L < d->n_layers; ++L) {
      attention(L);
      rc = seq_run(rt, d->seqs[(size_t)L + 1]);
      if (rc) return rc;
    }
    h = d->n_layers ? d->h_alt : d->h;  // where the last post-attention residual went (decoder_bind_sequences)
  } else if (!d->seqs.empty()) {
    // one launch per projection group, through the sequence kernel's tile loop
    for (uint32_t L = 0; L < d->n_layers; ++L) {
      int rc = seq_run(rt, d->seqs[(size_t)L * 4]);
      if (rc) return rc;
      attention(L);
      for (int j = 1; j < 4; ++j)
        if ((rc = seq_run(rt, d->seqs[(size_t)L * 4 + j]))) return rc;
    }
    h = d->n_layers ? d->h_alt : d->h;
  } else {
  // The residual stream alternates between two buffers: a projection launch whose
  // prologue adds the previous branch reads one and (workgroup 0) writes the other.
  for (uint32_t L = 0; L < d->n_layers; ++L) {
    const llvq_mat* const* P = d->proj.data() + (size_t)L * 7;
    // the previous layer's MLP output joins the residual stream in the q/k/v launch
    Prologue ln1;
    ln1.kind = kPrologueAddRmsNorm;
    ln1.norm_w = d->ln1 + (size_t)L * d->hidden;
    ln1.eps = d->eps;
    if (L) {
      ln1.x2 = d->down;
      ln1.resid_out = h_alt;
    }
    void* qkv_out[3] = {d->q, d->k, d->v};
    int rc = project(P, 3, h, qkv_out, ln1);
    if (rc) return rc;
    if (L) std::swap(h, h_alt);
    attention(L);
    void* o_out[1] = {d->o};
    rc = forward_group(rt, P + 3, 1, d->ctx, o_out, LLVQ_F16);
    if (rc) return rc;
    Prologue ln2;
    ln2.kind = kPrologueAddRmsNorm;
    ln2.norm_w = d->ln2 + (size_t)L * d->hidden;
    ln2.eps = d->eps;
    ln2.x2 = d->o;
    ln2.resid_out = h_alt;
    void* d_out[1] = {d->down};
    if (gated_fits(P[4], P[5])) {
      void* act_out[1] = {d->act};
      rc = launch_group(rt, P + 4, 2, h, act_out, LLVQ_F16, &ln2, nullptr, P[4]->rot, true);
      if (!rc) rc = forward_group(rt, P + 6, 1, d->act, d_out, LLVQ_F16);
    } else {
      void* gu_out[2] = {d->gate, d->up};
      rc = project(P + 4, 2, h, gu_out, ln2);
      if (rc) return rc;
      Prologue act;
      act.kind = kPrologueSiluMul;
      act.x2 = d->gate;
      rc = project(P + 6, 1, d->up, d_out, act);
    }
    if (rc) return rc;
    std::swap(h, h_alt);
  }
  }
  phase_mark(d);
  if (want_logits) {
    hipLaunchKernelGGL(add_rmsnorm_kernel, dim3(1), dim3(norm_threads(d->hidden)), 0, st, h, d->down, d->fnorm, h, d->normed, d->hidden, d->eps, Octets{}, GemmSums{});
    launch_head(d, history_slot, record, host);
  }
  HIP_TRY(hipGetLastError());
  d->pos += 1;
  return LLVQ_OK;
}
// Where a step's last launch leaves what the caller wants of it: in pinned memory, if there is any.
HostResults host_results(llvq_decoder* d, const float* logits_host, const uint32_t* argmax_host) {
  if (!d->host_out) return {};
  return {logits_host ? d->host_out : nullptr, argmax_host ? reinterpret_cast<uint32_t*>(d->host_out + d->vocab) : nullptr};
}
// The wait for a step's results, and their way to the caller's memory.  A copy straight to that (pageable) memory is staged by the
// runtime, one for each result, and begins when the stream has been waited for.  With pinned memory they are there when the
// step ends (argmax_final_kernel has the times), and while it runs the pages that they go to are touched, which for fresh memory is most of
// what moving them costs.
int decoder_results(llvq_decoder* d, float* logits_host, uint32_t* argmax_host) {
  hipStream_t st = d->rt->stream;
  const size_t bytes = (size_t)d->vocab * sizeof(float);
  if (!d->host_out) {
    if (logits_host) HIP_TRY(hipMemcpyAsync(logits_host, d->logits, bytes, hipMemcpyDeviceToHost, st));
    if (argmax_host) HIP_TRY(hipMemcpyAsync(argmax_host, d->token, sizeof(uint32_t), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    return LLVQ_OK;
  }
  if (logits_host) {
    volatile char* page = reinterpret_cast<volatile char*>(logits_host);
    for (size_t at = 0; at < bytes; at += 4096) page[at] = 0;
    page[bytes - 1] = 0;
  }
  HIP_TRY(hipStreamSynchronize(st));
  if (logits_host) std::memcpy(logits_host, d->host_out, bytes);
  if (argmax_host) std::memcpy(argmax_host, d->host_out + d->vocab, sizeof(uint32_t));
  return LLVQ_OK;
}

// n <= prefill_rows positions at once, starting at dec->pos: tokens from dec->ptokens.
// With want_logits the head runs on the last row and leaves its argmax in *dec->token.
int decoder_prefill_pass(llvq_decoder* d, uint32_t n, bool want_logits, uint32_t history_slot, bool record, const HostResults& host) {
  llvq_rt* rt = d->rt;
  hipStream_t st = rt->stream;
  if (d->pos + n > d->max_pos) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decoder_prefill: positions past max_positions");
  __half *ph = d->ph, *ph_alt = d->ph_alt;  // by local name: a pass that fails part-way leaves the decoder as it found it
  if (d->embed_q8)
    hipLaunchKernelGGL(embed_q8_kernel, dim3((d->hidden + 255) / 256, n), dim3(256), 0, st, d->embed_q, d->ptokens, 0u, d->vocab, d->hidden, ph);
  else
    hipLaunchKernelGGL(embed_kernel, dim3((d->hidden + 255) / 256, n), dim3(256), 0, st, d->embed, d->ptokens, 0u, d->vocab, d->hidden, ph);
  const size_t cache_layer = (size_t)d->n_kv * d->max_pos * d->head_dim, group_layer = cache_layer / kKvGroup;
  const float scale = 1.0f / sqrtf((float)d->head_dim);
  // Rows that `make` launches what makes, through projections that share them: straight to the product's octets where one launch takes them
  // all in their own basis, else to x first.
  // left: where the launch that takes the results adds up what the product leaves in parts (the workspace that those are in is as large as any
  // product of a pass needs it, llvq_hip_decoder_create, and is not touched before the next product).
  const auto product = [&](const llvq_mat* const* mats, int n_mats, const __half* x, void* const* y, const std::function<void(const Octets&)>& make,
                           GemmSums* left = nullptr) {
    if (gemm_takes_octets(mats, n_mats, n)) return launch_gemm(rt, mats, n_mats, x, n, y, LLVQ_F16, false, nullptr, nullptr, &make, left);
    make(Octets{});
    bool one_basis = true;
    for (int i = 1; i < n_mats; ++i) one_basis &= same_basis(mats[0], mats[i]);
    if (left && one_basis) return gemm_same_basis(rt, mats, n_mats, x, (int)n, y, LLVQ_F16, nullptr, left);
    return llvq_hip_gemm_group(rt, mats, n_mats, x, (int)n, y, LLVQ_F16);
  };
  GemmSums down_sums{};  // of the layer before
  for (uint32_t L = 0; L < d->n_layers; ++L) {
    const llvq_mat* const* P = d->proj.data() + (size_t)L * 7;
    const uint32_t grp = d->n_heads / d->n_kv;
    // 32 rows per workgroup on the matrix cores where the head width is the one that kernel is built for, the cache walked
    // by two sets of wavefronts, four of two heads each (more than five heads to a set leave it too few registers for a second)
    const bool on_mfma = d->head_dim == 128 && grp <= (uint32_t)kAttnMaxGroup;
    GemmSums qkv_sums{}, o_sums{};
    // residual + previous MLP branch, then the input norm (the branch of layer 0 is absent)
    void* const qkv[3] = {d->pq, d->pk, d->pv};
    int rc = product(P, 3, d->pnormed, qkv, [&](const Octets& to) {
      hipLaunchKernelGGL(add_rmsnorm_kernel, dim3(to.xt ? to.m_pad : n), dim3(norm_threads(d->hidden)), 0, st, ph, L ? d->pdown : (const __half*)nullptr,
                         d->ln1 + (size_t)L * d->hidden, L ? ph_alt : (__half*)nullptr, d->pnormed, d->hidden, d->eps, to, down_sums);
    }, d->head_dim == 128 ? &qkv_sums : nullptr);
    if (rc) return rc;
    if (L) std::swap(ph, ph_alt);
    KvQ8 lq8 = d->q8;
    if (d->kv_q8) {
      lq8.kq += L * cache_layer; lq8.vq += L * cache_layer;
      lq8.ks += L * group_layer; lq8.kb += L * group_layer; lq8.vs += L * group_layer; lq8.vb += L * group_layer;
    }
    __half* kc = d->kv_q8 ? nullptr : d->kcache + L * cache_layer;
    __half* vc = d->kv_q8 ? nullptr : d->vcache + L * cache_layer;
    AttnNew nw{};
    nw.qn = d->qn + (size_t)L * d->head_dim;
    nw.kn = d->kn + (size_t)L * d->head_dim;
    nw.cos_t = d->cos_t;
    nw.sin_t = d->sin_t;
    nw.kcache = kc;
    nw.vcache = vc;
    nw.eps = d->eps;
    const dim3 hgrid((d->n_heads + 2 * d->n_kv + 3) / 4, n), agrid(d->n_kv, n);
    Octets ctx_to{};
    auto attend = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, agrid, dim3(64), 0, st, d->pq, kc, vc, lq8, d->pctx, d->n_heads, d->n_kv, d->head_dim, d->pos, d->max_pos, scale);
    };
    const uint32_t row_blocks = (n + kAttnTile - 1) / kAttnTile;
    const bool by_two = prompt_heads_by_two(d->n_kv, grp, row_blocks, d->pos + n - 1u, (uint32_t)(rt->cu_count > 0 ? rt->cu_count : 256));
    auto attend_mfma = [&](auto kernel, uint32_t heads, uint32_t sets) {
      hipLaunchKernelGGL(kernel, dim3(d->n_kv * ((grp + heads - 1u) / heads), row_blocks), dim3(heads * sets * 64), 0, st, d->pq, kc, vc, lq8, d->pctx, d->n_heads, d->n_kv, d->pos, n, d->max_pos, scale, ctx_to);
    };
    const auto attention = [&]() {
    if (d->kv_q8) {
      hipLaunchKernelGGL(norm_rope_append_rows_kernel<true>, hgrid, dim3(256), 0, st, d->pq, d->pk, d->pv, nw, lq8, d->n_heads, d->n_kv,
                         d->head_dim, d->pos, d->max_pos, qkv_sums);
      if (on_mfma) {
        if (by_two) attend_mfma(attn_rows_mfma_kernel<true, 2, 4>, 2, 4);
        else if (grp <= 2) attend_mfma(attn_rows_mfma_kernel<true, 2, 2>, 2, 2);
        else if (grp <= 4) attend_mfma(attn_rows_mfma_kernel<true, 4, 2>, 4, 2);
        else if (grp <= 5) attend_mfma(attn_rows_mfma_kernel<true, 5, 2>, 5, 2);
        else attend_mfma(attn_rows_mfma_kernel<true, kAttnMaxGroup, 1>, kAttnMaxGroup, 1);
      } else if (grp <= 2) attend(attn_rows_kernel<true, 2>);
      else if (grp <= 4) attend(attn_rows_kernel<true, 4>);
      else if (grp <= 5) attend(attn_rows_kernel<true, 5>);
      else attend(attn_rows_kernel<true, kAttnMaxGroup>);
    } else {
      hipLaunchKernelGGL(norm_rope_append_rows_kernel<false>, hgrid, dim3(256), 0, st, d->pq, d->pk, d->pv, nw, lq8, d->n_heads, d->n_kv,
                         d->head_dim, d->pos, d->max_pos, qkv_sums);
      if (on_mfma) {
        if (by_two) attend_mfma(attn_rows_mfma_kernel<false, 2, 4>, 2, 4);
        else if (grp <= 2) attend_mfma(attn_rows_mfma_kernel<false, 2, 2>, 2, 2);
        else if (grp <= 4) attend_mfma(attn_rows_mfma_kernel<false, 4, 2>, 4, 2);
        else if (grp <= 5) attend_mfma(attn_rows_mfma_kernel<false, 5, 2>, 5, 2);
        else attend_mfma(attn_rows_mfma_kernel<false, kAttnMaxGroup, 1>, kAttnMaxGroup, 1);
      } else if (grp <= 2) attend(attn_rows_kernel<false, 2>);
      else if (grp <= 4) attend(attn_rows_kernel<false, 4>);
      else if (grp <= 5) attend(attn_rows_kernel<false, 5>);
      else attend(attn_rows_kernel<false, kAttnMaxGroup>);
    }
    };
    void* const o_out[1] = {d->po};
    if (on_mfma) {
      rc = product(P + 3, 1, d->pctx, o_out, [&](const Octets& to) {
        ctx_to = to;
        attention();
      }, &o_sums);
    } else {
      attention();
      rc = llvq_hip_gemm(rt, P[3], d->pctx, (int)n, d->po, LLVQ_F16);
    }
    if (rc) return rc;
    void* const gate_up[2] = {d->pgate, d->pup};
    rc = product(P + 4, 2, d->pnormed, gate_up, [&](const Octets& to) {
      hipLaunchKernelGGL(add_rmsnorm_kernel, dim3(to.xt ? to.m_pad : n), dim3(norm_threads(d->hidden)), 0, st, ph, d->po, d->ln2 + (size_t)L * d->hidden,
                         ph_alt, d->pnormed, d->hidden, d->eps, to, o_sums);
    });
    if (rc) return rc;
    std::swap(ph, ph_alt);
    void* const down[1] = {d->pdown};
    down_sums = GemmSums{};
    rc = product(P + 6, 1, d->pact, down, [&](const Octets& to) {
      if (to.xt) {
        const uint32_t waves = (std::max(to.n_oct, d->inter / 8u) + 7u) / 8u * (to.m_pad / 8u);
        hipLaunchKernelGGL(tile_activations_kernel, dim3((waves + 3u) / 4u), dim3(256), 0, st, d->pup, d->pgate, d->pact, n, d->inter, to.kcols, to.m_pad,
                           to.n_oct, to.xt);
        return;
      }
      const uint32_t na = n * d->inter;
      hipLaunchKernelGGL(silu_mul_kernel, dim3(std::min((na / 8u + 256u) / 256u, 4096u)), dim3(256), 0, st, d->pgate, d->pup, d->pact, na);
    }, &down_sums);
    if (rc) return rc;
  }
  if (want_logits) {
    const size_t last = (size_t)(n - 1) * d->hidden;
    if (down_sums.ws) down_sums.ws += (size_t)(n - 1) * down_sums.ld;
    hipLaunchKernelGGL(add_rmsnorm_kernel, dim3(1), dim3(norm_threads(d->hidden)), 0, st, ph + last, d->pdown + last, d->fnorm, d->h, d->normed,
                       d->hidden, d->eps, Octets{}, down_sums);
    launch_head(d, history_slot, record, host);
  }
  HIP_TRY(hipGetLastError());
  d->pos += n;
  return LLVQ_OK;
}

// The prompt through decoder_prefill_pass, prefill_rows positions at a time; the head runs after the last one.
int decoder_prefill(llvq_decoder* d, const uint32_t* tokens, size_t n, uint32_t history_slot, bool record, const HostResults& host = {}) {
  if (!d->prefill_rows) return fail(LLVQ_ERR_UNSUPPORTED, "decoder_prefill: the decoder was created with prefill_rows = 0");
  for (size_t at = 0; at < n; at += d->prefill_rows) {
    const uint32_t c = (uint32_t)(n - at < d->prefill_rows ? n - at : d->prefill_rows);
    HIP_TRY(hipMemcpyAsync(d->ptokens, tokens + at, c * sizeof(uint32_t), hipMemcpyHostToDevice, d->rt->stream));
    const int rc = decoder_prefill_pass(d, c, at + c == n, history_slot, record, host);
    if (rc) return rc;
  }
  return LLVQ_OK;
}

}  // namespace

extern "C" {

int llvq_hip_decoder_create(llvq_rt* rt, const llvq_decoder_desc* c, llvq_decoder** out) {
  if (!rt || !c || !out) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decoder_create: null argument");
  *out = nullptr;
  if (!c->projections || !c->input_norm || !c->post_norm || !c->q_norm || !c->k_norm || !c->final_norm ||
      (!c->embed && !c->embed_q8.codes))
    return fail(LLVQ_ERR_INVALID_ARGUMENT, "decoder_create: a required tensor is null");
  for (const llvq_quant_rows* qr : {&c->embed_q8, &c->lm_head_q8})
    if (qr->codes) {
      if (!qr->scales || !qr->biases) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decoder_create: an int8 tensor without scales or biases");
      // what the kernels compile in (fused_cuda.rs:418-447): 8 bits, groups of 64, whole 16-byte runs per row
      if (qr->bits != 8 || qr->group != kEmbedGroup || c->hidden % 16)
        return fail(LLVQ_ERR_UNSUPPORTED, "decoder_create: int" + std::to_string(qr->bits) + " g" + std::to_string(qr->group) +
                                              " — the kernels hard-code int8 g64 and hidden % 16 = 0");
    }
  if (c->n_layers == 0 || c->hidden == 0 || c->hidden % 8 || c->hidden > 8192 || c->n_heads == 0 || c->n_kv_heads == 0 ||
      c->n_heads % c->n_kv_heads || c->n_heads / c->n_kv_heads > (uint32_t)kAttnMaxGroup || c->head_dim == 0 || c->head_dim % 8 || c->head_dim > 128 || c->intermediate == 0 ||
      c->vocab == 0 || c->max_positions == 0 || c->max_positions > 8192 ||
      (c->kv_mode != LLVQ_KV_F16 && c->kv_mode != LLVQ_KV_Q8) || (c->kv_mode == LLVQ_KV_Q8 && c->head_dim % 64))
    return fail(LLVQ_ERR_UNSUPPORTED,
                "decoder_create: shape outside what the kernels hold (hidden % 8 = 0 and <= 8192, head_dim % 8 = 0 and <= 128, "
                "heads a multiple of kv heads and at most 8 per kv head, max_positions <= 8192, kv_mode f16 or q8 with head_dim % 64 = 0)");
  if (c->prefill_rows > 4096) return fail(LLVQ_ERR_UNSUPPORTED, "decoder_create: the batched prompt path takes at most 4096 rows per pass");
  const uint32_t qd = c->n_heads * c->head_dim, kvd = c->n_kv_heads * c->head_dim;
  static const char* kSite[7] = {"q_proj", "k_proj", "v_proj", "o_proj", "gate_proj", "up_proj", "down_proj"};
  const uint32_t want_out[7] = {qd, kvd, kvd, c->hidden, c->intermediate, c->intermediate, c->hidden};
  const uint32_t want_in[7] = {c->hidden, c->hidden, c->hidden, qd, c->hidden, c->hidden, c->intermediate};
  for (uint32_t L = 0; L < c->n_layers; ++L)
    for (int j = 0; j < 7; ++j) {
      const llvq_mat* m = c->projections[(size_t)L * 7 + j];
      if (!m) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decoder_create: layer " + std::to_string(L) + " " + kSite[j] + " is null");
      if (m->d_out != want_out[j] || m->d_in != want_in[j])
        return fail(LLVQ_ERR_INCONSISTENT, "decoder_create: layer " + std::to_string(L) + " " + kSite[j] + " is " +
                                               std::to_string(m->d_out) + "x" + std::to_string(m->d_in) + ", the architecture needs " +
                                               std::to_string(want_out[j]) + "x" + std::to_string(want_in[j]));
    }
  HIP_TRY(hipSetDevice(rt->device));
  auto* d = new llvq_decoder();
  d->rt = rt;
  d->n_layers = c->n_layers; d->hidden = c->hidden; d->n_heads = c->n_heads; d->n_kv = c->n_kv_heads;
  d->head_dim = c->head_dim; d->inter = c->intermediate; d->vocab = c->vocab; d->max_pos = c->max_positions;
  d->eps = (float)c->rms_eps;
  d->kv_q8 = c->kv_mode == LLVQ_KV_Q8;
  d->proj.assign(c->projections, c->projections + (size_t)c->n_layers * 7);
  d->head_grid = kHeadGroups * (uint32_t)(rt->cu_count > 0 ? rt->cu_count : 256);
  while (d->head_grid > 1 && (uint64_t)d->head_grid * (kHeadThreads / 64) > c->vocab) d->head_grid >>= 1;

  // RoPE tables exactly as Rotary::new builds them (model.rs:163-179): f32 inverse
  // frequencies from an f64 power, f32 angle = position * inv_freq, sin/cos narrowed to binary16.
  const uint32_t half_d = c->head_dim / 2;
  std::vector<__half> cos_h((size_t)c->max_positions * half_d), sin_h(cos_h.size());
  for (uint32_t i = 0; i < half_d; ++i) {
    const float inv = 1.0f / (float)std::pow(c->rope_theta, (double)(2 * i) / (double)c->head_dim);
    for (uint32_t p = 0; p < c->max_positions; ++p) {
      const float ang = (float)p * inv;
      cos_h[(size_t)p * half_d + i] = __float2half_rn(std::cos(ang));
      sin_h[(size_t)p * half_d + i] = __float2half_rn(std::sin(ang));
    }
  }

  // one allocation, 256-byte aligned pieces
  size_t total = 0;
  auto take = [&](size_t bytes) { const size_t at = total; total += (bytes + 255) & ~(size_t)255; return at; };
  const size_t hb = sizeof(__half);
  const size_t o_ln1 = take((size_t)c->n_layers * c->hidden * hb), o_ln2 = take((size_t)c->n_layers * c->hidden * hb);
  const size_t o_qn = take((size_t)c->n_layers * c->head_dim * hb), o_kn = take((size_t)c->n_layers * c->head_dim * hb);
  const size_t o_fn = take((size_t)c->hidden * hb);
  const size_t vh = (size_t)c->vocab * c->hidden, vg = (size_t)c->vocab * ((c->hidden + kEmbedGroup - 1) / kEmbedGroup);
  const bool eq8 = c->embed_q8.codes != nullptr;
  // the head: its own int8 or binary16 tensor, else tied to the embedding in whichever encoding that is
  const bool hq8 = c->lm_head_q8.codes != nullptr || (!c->lm_head && eq8);
  const bool head_own = c->lm_head_q8.codes != nullptr || c->lm_head != nullptr;
  const size_t o_emb = take(eq8 ? vh : vh * hb), o_emb_s = take(eq8 ? vg * hb : 0), o_emb_b = take(eq8 ? vg * hb : 0);
  const size_t o_head = head_own ? take(hq8 ? vh : vh * hb) : o_emb;
  const size_t o_head_s = head_own ? take(hq8 ? vg * hb : 0) : o_emb_s, o_head_b = head_own ? take(hq8 ? vg * hb : 0) : o_emb_b;
  const size_t o_cos = take(cos_h.size() * hb), o_sin = take(sin_h.size() * hb);
  const size_t cache_vals = (size_t)c->n_layers * c->n_kv_heads * c->max_positions * c->head_dim;
  const bool q8 = c->kv_mode == LLVQ_KV_Q8;
  const size_t o_kc = take(cache_vals * (q8 ? 1 : hb)), o_vc = take(cache_vals * (q8 ? 1 : hb));
  const size_t o_ks = take(q8 ? cache_vals / kKvGroup * hb : 0), o_kb = take(q8 ? cache_vals / kKvGroup * hb : 0);
  const size_t o_vs = take(q8 ? cache_vals / kKvGroup * hb : 0), o_vb = take(q8 ? cache_vals / kKvGroup * hb : 0);
  const size_t o_h = take(c->hidden * hb), o_h2 = take(c->hidden * hb), o_nm = take(c->hidden * hb), o_q = take(qd * hb), o_k = take(kvd * hb), o_v = take(kvd * hb);
  const size_t o_ctx = take(qd * hb), o_o = take(c->hidden * hb), o_g = take(c->intermediate * hb), o_u = take(c->intermediate * hb);
  const size_t o_act = take(c->intermediate * hb), o_dn = take(c->hidden * hb);
  const size_t o_log = take(((size_t)c->vocab + 1) * sizeof(float));  // the chosen token behind the logits
  const size_t n_best = (size_t)d->head_grid * (kHeadThreads / 64);
  const size_t o_bv = take(n_best * sizeof(float)), o_bi = take(n_best * sizeof(uint32_t));
  const size_t o_hist = take((size_t)c->max_positions * sizeof(uint32_t));
  const size_t o_ap = take((size_t)c->n_heads * kAttnMaxSplits * (c->head_dim + 2) * sizeof(float)), o_ac = take((size_t)c->n_kv_heads * kDecodeCounter * sizeof(uint32_t));
  const size_t o_seqst = take(256);
  hipError_t e = hipMalloc(reinterpret_cast<void**>(&d->blob), total);
  if (e != hipSuccess) { delete d; return hip_fail(e, "hipMalloc(decoder)"); }
  auto put = [&](size_t at, const void* src, size_t bytes) { return hipMemcpy(d->blob + at, src, bytes, hipMemcpyHostToDevice); };
  e = hipMemset(d->blob, 0, total);
  if (e == hipSuccess) e = put(o_ln1, c->input_norm, (size_t)c->n_layers * c->hidden * hb);
  if (e == hipSuccess) e = put(o_ln2, c->post_norm, (size_t)c->n_layers * c->hidden * hb);
  if (e == hipSuccess) e = put(o_qn, c->q_norm, (size_t)c->n_layers * c->head_dim * hb);
  if (e == hipSuccess) e = put(o_kn, c->k_norm, (size_t)c->n_layers * c->head_dim * hb);
  if (e == hipSuccess) e = put(o_fn, c->final_norm, (size_t)c->hidden * hb);
  if (e == hipSuccess && !eq8) e = put(o_emb, c->embed, vh * hb);
  if (e == hipSuccess && eq8) e = put(o_emb, c->embed_q8.codes, vh);
  if (e == hipSuccess && eq8) e = put(o_emb_s, c->embed_q8.scales, vg * hb);
  if (e == hipSuccess && eq8) e = put(o_emb_b, c->embed_q8.biases, vg * hb);
  if (e == hipSuccess && head_own && !hq8) e = put(o_head, c->lm_head, vh * hb);
  if (e == hipSuccess && head_own && hq8) e = put(o_head, c->lm_head_q8.codes, vh);
  if (e == hipSuccess && head_own && hq8) e = put(o_head_s, c->lm_head_q8.scales, vg * hb);
  if (e == hipSuccess && head_own && hq8) e = put(o_head_b, c->lm_head_q8.biases, vg * hb);
  if (e == hipSuccess) e = put(o_cos, cos_h.data(), cos_h.size() * hb);
  if (e == hipSuccess) e = put(o_sin, sin_h.data(), sin_h.size() * hb);
  if (e != hipSuccess) { (void)hipFree(d->blob); delete d; return hip_fail(e, "decoder upload"); }
  auto H = [&](size_t at) { return reinterpret_cast<__half*>(d->blob + at); };
  d->ln1 = H(o_ln1); d->ln2 = H(o_ln2); d->qn = H(o_qn); d->kn = H(o_kn); d->fnorm = H(o_fn);
  d->embed = H(o_emb); d->head = H(o_head); d->cos_t = H(o_cos); d->sin_t = H(o_sin);
  d->embed_q8 = eq8;
  d->head_q8 = hq8;
  d->embed_q = QuantRows{d->blob + o_emb, H(o_emb_s), H(o_emb_b)};
  d->head_q = QuantRows{d->blob + o_head, H(o_head_s), H(o_head_b)};
  d->kcache = H(o_kc); d->vcache = H(o_vc);
  if (q8) {
    d->q8.kq = d->blob + o_kc; d->q8.vq = d->blob + o_vc;
    d->q8.ks = H(o_ks); d->q8.kb = H(o_kb); d->q8.vs = H(o_vs); d->q8.vb = H(o_vb);
  }
  d->h = H(o_h); d->h_alt = H(o_h2); d->normed = H(o_nm); d->q = H(o_q); d->k = H(o_k); d->v = H(o_v); d->ctx = H(o_ctx); d->o = H(o_o);
  d->gate = H(o_g); d->up = H(o_u); d->act = H(o_act); d->down = H(o_dn);
  d->logits = reinterpret_cast<float*>(d->blob + o_log);
  d->best_val = reinterpret_cast<float*>(d->blob + o_bv);
  d->best_idx = reinterpret_cast<uint32_t*>(d->blob + o_bi);
  d->token = reinterpret_cast<uint32_t*>(d->logits + c->vocab);
  if (hipHostMalloc(reinterpret_cast<void**>(&d->host_out), ((size_t)c->vocab + 1) * sizeof(float), hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    d->host_out = nullptr;
  }
  d->history = reinterpret_cast<uint32_t*>(d->blob + o_hist);
  d->attn_part = reinterpret_cast<float*>(d->blob + o_ap);
  d->attn_counters = reinterpret_cast<uint32_t*>(d->blob + o_ac);
  d->seq_status = reinterpret_cast<uint32_t*>(d->blob + o_seqst);
  if (c->prefill_rows) {
    // row buffers of the batched prompt path, one allocation
    const size_t R = c->prefill_rows;
    size_t ptotal = 0;
    auto ptake = [&](size_t bytes) { const size_t at = ptotal; ptotal += (bytes + 255) & ~(size_t)255; return at; };
    const size_t p_h = ptake(R * c->hidden * hb), p_h2 = ptake(R * c->hidden * hb), p_nm = ptake(R * c->hidden * hb);
    const size_t p_q = ptake(R * qd * hb), p_k = ptake(R * kvd * hb), p_v = ptake(R * kvd * hb), p_ctx = ptake(R * qd * hb);
    const size_t p_o = ptake(R * c->hidden * hb), p_g = ptake(R * c->intermediate * hb), p_u = ptake(R * c->intermediate * hb);
    const size_t p_act = ptake(R * c->intermediate * hb), p_dn = ptake(R * c->hidden * hb), p_tok = ptake(R * sizeof(uint32_t));
    e = hipMalloc(reinterpret_cast<void**>(&d->pblob), ptotal);
    if (e == hipSuccess) e = hipMemset(d->pblob, 0, ptotal);
    if (e != hipSuccess) { (void)hipFree(d->pblob); (void)hipFree(d->blob); delete d; return hip_fail(e, "hipMalloc(decoder prefill rows)"); }
    auto PH = [&](size_t at) { return reinterpret_cast<__half*>(d->pblob + at); };
    d->prefill_rows = c->prefill_rows;
    d->ph = PH(p_h); d->ph_alt = PH(p_h2); d->pnormed = PH(p_nm); d->pq = PH(p_q); d->pk = PH(p_k); d->pv = PH(p_v); d->pctx = PH(p_ctx);
    d->po = PH(p_o); d->pgate = PH(p_g); d->pup = PH(p_u); d->pact = PH(p_act); d->pdown = PH(p_dn);
    d->ptokens = reinterpret_cast<uint32_t*>(d->pblob + p_tok);
    // the batched products of a pass find their workspaces sized: no allocation (and no implicit
    // device synchronisation) between the launches of a prompt
    for (uint32_t L = 0; L < c->n_layers; ++L) {
      const llvq_mat* const* P = d->proj.data() + (size_t)L * 7;
      int rc = reserve_batched(rt, P, 3, c->prefill_rows);
      if (!rc) rc = reserve_batched(rt, P + 3, 1, c->prefill_rows);
      if (!rc) rc = reserve_batched(rt, P + 4, 2, c->prefill_rows);
      if (!rc) rc = reserve_batched(rt, P + 6, 1, c->prefill_rows);
      if (rc) { (void)hipFree(d->pblob); (void)hipFree(d->blob); delete d; return rc; }
    }
  }
  if (c->launch_mode > LLVQ_LAUNCH_CHAINED) {
    (void)hipFree(d->pblob); (void)hipFree(d->blob); delete d;
    return fail(LLVQ_ERR_INVALID_ARGUMENT, "decoder_create: unknown launch_mode");
  }
  if (c->launch_mode != LLVQ_LAUNCH_PER_GROUP) {
    const int rc = decoder_bind_sequences(d, c->launch_mode == LLVQ_LAUNCH_CHAINED);
    if (rc) { (void)hipFree(d->pblob); (void)hipFree(d->blob); delete d; return rc; }
  }
  *out = d;
  return LLVQ_OK;
}

void llvq_hip_decoder_destroy(llvq_decoder* d) {
  if (!d) return;
  (void)hipSetDevice(d->rt->device);
  (void)hipStreamSynchronize(d->rt->stream);
  for (llvq_seq* q : d->seqs) llvq_hip_sequence_destroy(d->rt, q);
  (void)hipFree(d->pblob);
  (void)hipFree(d->blob);
  delete d;
}

int llvq_hip_decoder_reset(llvq_decoder* d) {
  if (!d) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decoder_reset: null decoder");
  d->pos = 0;  // the cache is overwritten position by position; nothing else carries state
  return LLVQ_OK;
}

int llvq_hip_decoder_position(const llvq_decoder* d) { return d ? (int)d->pos : -1; }

int llvq_hip_decoder_seek(llvq_decoder* d, uint32_t position) {
  if (!d) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decoder_seek: null decoder");
  if (position >= d->max_pos) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decoder_seek: position past max_positions");
  d->pos = position;
  return LLVQ_OK;
}

int llvq_hip_decoder_forward_token(llvq_decoder* d, uint32_t token, float* logits_host, uint32_t* argmax_host) {
  if (!d) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decoder_forward_token: null decoder");
  if (token >= d->vocab) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decoder_forward_token: token " + std::to_string(token) + " is outside the vocabulary");
  HIP_TRY(hipSetDevice(d->rt->device));
  const int rc = decoder_step(d, true, 0, false, &token, host_results(d, logits_host, argmax_host));
  if (rc) return rc;
  {
    const int rc1 = decoder_results(d, logits_host, argmax_host);
    if (rc1) return rc1;
  }
  return decoder_check_sequences(d);
}

static int generate_impl(llvq_decoder* d, const uint32_t* prompt, size_t n_prompt, size_t max_new, uint32_t* out, bool batched,
                         const char* who, double* phase_ms = nullptr) {
  if (!d || (n_prompt && !prompt) || (max_new && !out)) return fail(LLVQ_ERR_INVALID_ARGUMENT, std::string(who) + ": null argument");
  if (max_new == 0) return LLVQ_OK;  // model.rs:1052-1054
  if (n_prompt == 0) return fail(LLVQ_ERR_INVALID_ARGUMENT, std::string(who) + ": empty prompt");
  if (n_prompt + max_new - 1 > d->max_pos)
    return fail(LLVQ_ERR_INVALID_ARGUMENT, std::string(who) + ": " + std::to_string(n_prompt + max_new - 1) + " positions exceed max_positions " + std::to_string(d->max_pos));
  for (size_t i = 0; i < n_prompt; ++i)
    if (prompt[i] >= d->vocab) return fail(LLVQ_ERR_INVALID_ARGUMENT, std::string(who) + ": prompt token outside the vocabulary");
  HIP_TRY(hipSetDevice(d->rt->device));
  d->pos = 0;
  // Phase timing: five events per timed step (start, after the embedding, after the layers, after the
  // head, after the argmax); the step that ends the prompt is the first timed one.
  std::vector<hipEvent_t> marks;
  struct MarksGuard {
    llvq_decoder* d;
    std::vector<hipEvent_t>* m;
    ~MarksGuard() {
      d->marks = nullptr;
      for (hipEvent_t e : *m) (void)hipEventDestroy(e);
    }
  } guard{d, &marks};
  if (phase_ms) {
    marks.resize(5 * max_new);
    for (auto& e : marks) {
      e = nullptr;
      HIP_TRY(hipEventCreate(&e));
    }
  }
  if (batched) {
    const int rc = decoder_prefill(d, prompt, n_prompt, 0, true);
    if (rc) return rc;
  } else {
    for (size_t i = 0; i < n_prompt; ++i) {
      if (phase_ms && i + 1 == n_prompt) { d->marks = &marks; d->next_mark = 0; }
      const int rc = decoder_step(d, i + 1 == n_prompt, 0, true, &prompt[i]);
      if (rc) return rc;
    }
  }
  for (size_t t = 1; t < max_new; ++t) {
    const int rc = decoder_step(d, true, (uint32_t)t, true);
    if (rc) return rc;
  }
  HIP_TRY(hipMemcpyAsync(out, d->history, max_new * sizeof(uint32_t), hipMemcpyDeviceToHost, d->rt->stream));
  HIP_TRY(hipStreamSynchronize(d->rt->stream));
  {
    const int rc = decoder_check_sequences(d);
    if (rc) return rc;
  }
  if (phase_ms) {
    auto between = [&](size_t a, size_t b, double* ms) -> int {
      float f = 0.f;
      HIP_TRY(hipEventElapsedTime(&f, marks[a], marks[b]));
      *ms = (double)f;
      return LLVQ_OK;
    };
    for (size_t t = 0; t < max_new; ++t) {
      double* row = phase_ms + 4 * t;
      row[0] = row[1] = row[2] = row[3] = 0.0;
      int rc = between(5 * t + 2, 5 * t + 3, &row[0]);           // final norm + head of the step that chose token t
      if (!rc) rc = between(5 * t + 3, 5 * t + 4, &row[1]);      // argmax
      if (!rc && t + 1 < max_new) rc = between(5 * (t + 1), 5 * (t + 1) + 1, &row[2]);      // embedding of token t
      if (!rc && t + 1 < max_new) rc = between(5 * (t + 1) + 1, 5 * (t + 1) + 2, &row[3]);  // the layers over it
      if (rc) return rc;
    }
  }
  return LLVQ_OK;
}

int llvq_hip_decoder_generate(llvq_decoder* d, const uint32_t* prompt, size_t n_prompt, size_t max_new, uint32_t* out) {
  return generate_impl(d, prompt, n_prompt, max_new, out, false, "decoder_generate");
}

int llvq_hip_decoder_generate_prefilled(llvq_decoder* d, const uint32_t* prompt, size_t n_prompt, size_t max_new, uint32_t* out) {
  return generate_impl(d, prompt, n_prompt, max_new, out, true, "decoder_generate_prefilled");
}

int llvq_hip_decoder_generate_phased(llvq_decoder* d, const uint32_t* prompt, size_t n_prompt, size_t max_new, uint32_t* out,
                                     double* phase_ms) {
  if (max_new && !phase_ms) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decoder_generate_phased: null phase array");
  return generate_impl(d, prompt, n_prompt, max_new, out, false, "decoder_generate_phased", phase_ms);
}

int llvq_hip_decoder_prefill(llvq_decoder* d, const uint32_t* tokens, size_t n, float* logits_host, uint32_t* argmax_host) {
  if (!d || !tokens || n == 0) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decoder_prefill: null or empty argument");
  if (d->pos + n > d->max_pos) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decoder_prefill: positions past max_positions");
  for (size_t i = 0; i < n; ++i)
    if (tokens[i] >= d->vocab) return fail(LLVQ_ERR_INVALID_ARGUMENT, "decoder_prefill: token outside the vocabulary");
  HIP_TRY(hipSetDevice(d->rt->device));
  const int rc = decoder_prefill(d, tokens, n, 0, false, host_results(d, logits_host, argmax_host));
  if (rc) return rc;
  {
    const int rc1 = decoder_results(d, logits_host, argmax_host);
    if (rc1) return rc1;
  }
  return LLVQ_OK;
}

}  // extern "C"
