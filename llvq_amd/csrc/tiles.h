// The weight layout the products read, the kernel that writes it at upload, and the batch-1 product over it.
//
// A code stream is unranked once, on the device, when its matrix is uploaded: unranking costs about 500 vector
// instructions per block, and a product that repeats it is bound by them at 5 % of what HBM delivers (2.26 ms for the
// 150.7 M blocks of a 4B model, 434 GB/s of codes).  A lattice point's 24 coordinates are all even or all odd and at
// most 13 in magnitude, so v = 2 n + p with one bit p per block and n in [-8, 7]: 12 bytes of nibbles and one byte for
// p, the gain bit and the shell.  Nothing is rounded; what a kernel rebuilds from 13 bytes is the integer point itself.
//
//   matrix: 32 floats (gain centroid / sqrt(16 shell), indexed gain << 4 | shell; shell 0, the origin, gives 0),
//           then one record per 8 rows:
//             8 row scales (f32), tail_w x 8 tail values (f32, column by column), nb blocks of 104 bytes
//   block:  8 rows x 12 bytes of nibbles, then 8 rows x 1 byte (gain << 4 | shell) << 2 | p
//   nibble q of dword j holds column 8 j + {0, 2, 4, 6, 1, 3, 5, 7}[q], two's complement: nibbles q and q + 4 are
//           neighbouring columns in the two halves of the dword, which is what a packed binary16 unpack wants, and a
//           dword is the operand of an 8-wide 4-bit dot product.
//
// Eight rows of eight consecutive blocks are 832 consecutive bytes: one step of a wavefront, each lane one (row, block).
#pragma once

namespace llvq {

constexpr uint32_t kTileRows = 8;
constexpr uint32_t kTileBlockBytes = 104;
constexpr uint32_t kTileTableBytes = 128;

__host__ __device__ inline uint32_t tile_head_bytes(uint32_t tail_w) { return 32u + 32u * tail_w; }
// bytes of one record of eight rows (its blocks start 32-byte aligned)
__host__ __device__ inline uint32_t tile_stride(uint32_t nb, uint32_t tail_w) {
  return tile_head_bytes(tail_w) + ((nb * kTileBlockBytes + 31u) & ~31u);
}
__host__ __device__ inline uint32_t tile_count(uint32_t d_out) { return (d_out + kTileRows - 1u) / kTileRows; }

// ---- upload: code stream -> tiles ---------------------------------------------------------------
// One lane per block; lane % 8 is the row inside a record, so that a wavefront writes whole records.  The lanes of a
// wavefront take both coset programs (about 800 instructions per block, 3 ms for a 4B model's blocks): an upload is
// bound by the copy of the codes over PCIe, twenty times that.
// `rows` rows; codes and tiles are those rows' own.
template <bool WIDE>
__global__ __launch_bounds__(512) void transcode_kernel(GlobalTables g, const uint8_t* __restrict__ codes, uint8_t* __restrict__ tiles,
                                                        uint32_t rows, uint32_t nb, uint32_t tail_w) {
  extern __shared__ __align__(16) uint8_t smem[];
  const DecodeTables T = stage_tables<WIDE>(smem, g);
  __syncthreads();
  const uint32_t stride = tile_stride(nb, tail_w), head = tile_head_bytes(tail_w);
  const uint64_t padded = (uint64_t)tile_count(rows) * kTileRows * nb;
  for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < padded; k += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t r = (uint32_t)(k & 7u);
    const uint64_t tb = k >> 3;
    const uint32_t tile = (uint32_t)tb / nb, b = (uint32_t)tb - tile * nb;  // the host keeps a launch's blocks below 2^32
    const uint32_t row = tile * kTileRows + r;
    uint32_t w0 = 0, w1 = 0, w2 = 0, meta = 0;
    if (row < rows) {
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
      uint32_t par = 0;
      const int ci = decode_index(T, rec >> 1, [&](int p, int v) {
        const uint32_t nib = ((uint32_t)(v >> 1) & 15u) << (4u * (((uint32_t)p & 7u) >> 1) + 16u * ((uint32_t)p & 1u));
        par = (uint32_t)v & 1u;
        if (p < 8) w0 |= nib;
        else if (p < 16) w1 |= nib;
        else w2 |= nib;
      });
      if (ci >= 0) meta = ((((uint32_t)rec & 1u) << 4) | T.cls[ci].shell) << 2 | par;
    }
    uint8_t* out = tiles + (size_t)tile * stride + head + (size_t)b * kTileBlockBytes;
    uint32_t* wout = reinterpret_cast<uint32_t*>(out + r * 12u);
    wout[0] = w0;
    wout[1] = w1;
    wout[2] = w2;
    out[96u + r] = (uint8_t)meta;
  }
}

// Row scales and tail columns into the records' heads (zeros for rows past the last), the matrix's block scales to
// `table_out` where that is given (as an argument: a copy of 128 bytes from the host costs an upload 15 us).
struct TileTable { float v[kTileTableBytes / 4]; };
__global__ __launch_bounds__(256) void tile_heads_kernel(TileTable table, float* table_out, const float* __restrict__ rscale, const float* __restrict__ tail, uint8_t* __restrict__ tiles,
                                                         uint32_t rows, uint32_t nb, uint32_t tail_w) {
  if (table_out && blockIdx.x == 0 && threadIdx.x < kTileTableBytes / 4) table_out[threadIdx.x] = table.v[threadIdx.x];
  const uint32_t per = kTileRows * (1u + tail_w), stride = tile_stride(nb, tail_w);
  const uint32_t total = tile_count(rows) * per;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
    const uint32_t tile = i / per, k = i - tile * per, r = k & 7u, j = k >> 3;  // j = 0: the scale, j > 0: tail column j - 1
    const uint32_t row = tile * kTileRows + r;
    float v = 0.f;
    if (row < rows) v = j ? tail[(size_t)row * tail_w + j - 1u] : rscale[row];
    reinterpret_cast<float*>(tiles + (size_t)tile * stride)[k] = v;
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
// In LDS a block is 3 dwords per digit, the sum of its integers (v = 2 n + p: sum v x = 2 sum n x + p sum x) and the scale.
template <int DIG> struct XPlanes { static constexpr uint32_t kDwords = 3 * DIG + 2; };

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
// only takes part in the exchange.  Writes the block's planes at xb.  About 90 instructions for the quad's 24 values.
template <int DIG>
__device__ __forceinline__ void quantize_octet(const float (&v)[8], uint32_t sub, uint32_t* xb) {
  constexpr int kBits = DIG == 4 ? 14 : 22;
  constexpr uint32_t kMagic = 0x4B400000u;  // 1.5 2^23: adding it leaves the rounded integer in the low mantissa bits
  uint32_t m = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) m = max(m, __float_as_uint(v[j]) & 0x7FFFFFFFu);
  m = quad_max(m);
  // Biased exponent of the block's largest, at least the one below which `scale` would leave the normal range (2^-105 with
  // six digits, 2^-113 with four): smaller blocks are quantised at that scale.
  const uint32_t e = max(m >> 23, (uint32_t)kBits);
  const bool bad = m >= 0x7F800000u;     // inf or NaN: the block's products are NaN
  const float up = bad ? 0.f : __uint_as_float((253u + (uint32_t)kBits - e) << 23);
  const float scale = bad ? __builtin_nanf("") : __uint_as_float((e + 1u - (uint32_t)kBits) << 23);
  uint32_t t[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) t[j] = __float_as_uint(fmaf(bad ? 0.f : v[j], up, __uint_as_float(kMagic)));
  int sum = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) sum += (int)(t[j] - kMagic);
  sum = quad_sum(sum);
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
    xb[3 * DIG] = (uint32_t)sum;
    xb[3 * DIG + 1] = __float_as_uint(scale);
  }
}

// ---- batch-1 product ------------------------------------------------------------------------------
constexpr uint32_t kGemvSteps = 4;      // steps of 8 blocks a wavefront takes of a record, ...
constexpr uint32_t kGemvWideSteps = 8;  // ... and of a record wider than 16 wavefronts' worth of those
constexpr uint32_t kGemvMaxWaves = 16;
constexpr uint32_t kGemvRounds = 8;     // records per team between two sums over the team's wavefronts

// How a record's blocks are split over wavefronts: 2^shift of them, wavefront w taking the steps w, w + 2^shift, ...
// It depends on the row length alone, so a matrix gives the same bits whatever it shares a launch with.  The fewest
// wavefronts, at least four, that leave each at most kGemvSteps steps (16 past 512 blocks, with kGemvWideSteps).
// Every wavefront runs all its steps, on zeros where the row has ended: a branch around a load would make every wait
// behind it a wait for all loads in flight.
__host__ __device__ inline uint32_t gemv_split_shift(uint32_t nb) {
  const uint32_t steps = (nb + 7u) >> 3;
  uint32_t s = 2;
  while (s < 4u && (kGemvSteps << s) < steps) ++s;
  return s;
}
__host__ __device__ inline bool gemv_wide(uint32_t nb) { return nb > 8u * kGemvSteps * kGemvMaxWaves; }
constexpr uint32_t kGemvMaxBlocks = 8u * kGemvWideSteps * kGemvMaxWaves;
// Blocks of the planes in LDS: whole steps, and a step of zeros behind them for the wavefronts whose steps end early.
__host__ __device__ inline uint32_t gemv_plane_blocks(uint32_t nb) { return (((nb + 7u) >> 3) + 1u) * 8u; }

// What a launch's activation is made from.
enum : int { kSrcF16 = 0, kSrcRotated = 1, kSrcSiluMul = 2, kSrcAddRmsNorm = 3 };

struct TileMat {
  const uint8_t* base;  // the matrix (table, then records)
  void* y;
  uint32_t d_out;
  uint32_t tile_begin;  // first record of this matrix in the launch
};
struct GemvArgs {
  ActivationIn in;
  uint32_t nb, tail_w, n_mats, n_tiles;
  uint32_t split_shift;
  TileMat m[kMaxGroup];
};

struct GemvLds {
  float* xtail;      // [32]
  float* red;        // [16]
  uint32_t* planes;  // [plane blocks][XPlanes::kDwords]
  float* part;       // [kGemvRounds][16][8]
  float* tpart;      // the same for the tail columns
  float* scales;     // and the rows' scales
  float* xf;         // [d_in] f32 values of a rotated activation
};
__host__ __device__ inline uint32_t gemv_lds_fixed() { return 128u + 64u; }
__host__ __device__ inline size_t gemv_tiles_lds_bytes(uint32_t nb, uint32_t d_in, bool f32_out, bool rotated) {
  const size_t planes = (size_t)gemv_plane_blocks(nb) * (f32_out ? XPlanes<6>::kDwords : XPlanes<4>::kDwords) * 4;
  return gemv_lds_fixed() + planes + 3 * kGemvRounds * kGemvMaxWaves * 8 * 4 + (rotated ? ((size_t)d_in * 4 + 31) / 16 * 16 : 0);
}
template <int DIG>
__device__ __forceinline__ GemvLds gemv_lds(uint8_t* smem, uint32_t plane_blocks) {
  GemvLds L;
  L.xtail = reinterpret_cast<float*>(smem);
  L.red = L.xtail + 32;
  L.planes = reinterpret_cast<uint32_t*>(L.red + 16);
  L.part = reinterpret_cast<float*>(L.planes + (size_t)plane_blocks * XPlanes<DIG>::kDwords);
  L.tpart = L.part + kGemvRounds * kGemvMaxWaves * 8;
  L.scales = L.tpart + kGemvRounds * kGemvMaxWaves * 8;
  L.xf = L.scales + kGemvRounds * kGemvMaxWaves * 8;
  return L;
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
// `request` is called once, right behind the loads of the activation's operands: the first weights go out there.
// PMAX: how often the workgroup's quads pass over the padded blocks, at most.  store_resid: this workgroup is the one
// that stores the new residual.  Ends without a barrier.
template <int DIG, int SRC, int PMAX, bool kDeviceScope = false, class Request>
__device__ __forceinline__ void stage_x(const ActivationIn& in, uint32_t nb, uint32_t tail_w, const GemvLds& L, bool store_resid, Request&& request) {
  constexpr uint32_t kStr = XPlanes<DIG>::kDwords;
  const uint32_t tid = threadIdx.x, n_thr = blockDim.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t sub = tid & 3u, quad = tid >> 2, quads = n_thr >> 2;
  const uint32_t pad = (nb + 7u) & ~7u, d_in = nb * kDim + tail_w;
  const uint32_t passes = (pad + quads - 1u) / quads;
  if (tid < 32u) L.xtail[tid] = 0.f;
  for (uint32_t i = tid; i < 8u * kStr; i += n_thr) L.planes[pad * kStr + i] = 0u;  // the step of zeros
  if constexpr (SRC == kSrcRotated) {
    // The activation is rotated into LDS and quantised from there (a finished f32 one from where it is).
    // A launch in a rotated basis has 1024 lanes.
    float* xf = L.xf;
    if (in.x_f32) {
      request();
    } else {
      const RotFragments F = reinterpret_cast<const RotFragments*>(in.rot_fragments)[lane];
      const bool norm = in.prologue == kPrologueAddRmsNorm, silu = in.prologue == kPrologueSiluMul;
      auto norm_scale = [&](float ss) {
        ss = wave_sum(ss);
        if (lane == 0) L.red[wave] = ss;
        lds_barrier();
        float total = 0.f;
        for (uint32_t w = 0; w < (n_thr >> 6); ++w) total += L.red[w];
        return 1.0f / sqrtf(total / (float)d_in + in.eps);
      };
      if (in.rot_m >= kRotOctetM) {
        // Every operand of a wavefront's tile is requested before the first is used; one that is not there reads x.
        // (Rows past sixteen tiles: a second turn.  Those have no norm in front: a decoder's hidden size ends at 8192.)
        const __half* second = in.x2 ? in.x2 : in.x;
        const __half* third = norm ? in.norm_w : in.x;
        const uint8_t* signs = reinterpret_cast<const uint8_t*>(in.rot_signbits);
        HalfOctet a[2], b[2], g[2];
        uint32_t sg[2];
        auto load_tile = [&](uint32_t tile) {
#pragma unroll
          for (uint32_t i = 0; i < 2u; ++i) {
            const uint32_t from = rot_octet_at(tile, i) < d_in ? rot_octet_at(tile, i) : 0u;
            a[i] = *reinterpret_cast<const HalfOctet*>(in.x + from);
            b[i] = *reinterpret_cast<const HalfOctet*>(second + from);
            g[i] = *reinterpret_cast<const HalfOctet*>(third + from);
            sg[i] = signs[from >> 3];
          }
        };
        auto pack = [](float lo, float hi) { return (uint32_t)__half_as_ushort(__float2half_rn(lo)) | (uint32_t)__half_as_ushort(__float2half_rn(hi)) << 16; };
        load_tile(wave);
        if constexpr (PMAX <= 2) request();
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
              a[i].w[j] = pack(lo, hi);
              ss = fmaf(lo, lo, fmaf(hi, hi, ss));
            }
            if (in.resid_out && store_resid) *reinterpret_cast<HalfOctet*>(in.resid_out + rot_octet_at(wave, i)) = a[i];
          }
          inv = norm_scale(ss);
        }
#pragma unroll 1
        for (uint32_t tile = wave; tile * kRotTile < d_in; tile += 16u) {
          if (tile != wave) load_tile(tile);
#pragma unroll
          for (uint32_t i = 0; i < 2u; ++i) {
            if (silu) {
#pragma unroll
              for (int j = 0; j < 4; ++j)
                a[i].w[j] = pack(silu_mul(half_lo(b[i].w[j]), half_lo(a[i].w[j])), silu_mul(half_hi(b[i].w[j]), half_hi(a[i].w[j])));
            } else if (norm) {
#pragma unroll
              for (int j = 0; j < 4; ++j)
                a[i].w[j] = pack(half_lo(a[i].w[j]) * inv * half_lo(g[i].w[j]), half_hi(a[i].w[j]) * inv * half_hi(g[i].w[j]));
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) a[i].w[j] = rot_octet_at(tile, i) < d_in ? flip_signs(a[i].w[j], sg[i], j) : 0u;
          }
          rotate_tile_to(xf, a[0].w, a[1].w, F, tile, d_in, in.rot_m, in.rot_k, in.rot_inv);
        }
        if constexpr (PMAX > 2) request();  // (no registers for a wide step beside the operands)
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
      lds_barrier();
      rotate_rest(xf, d_in, in.rot_m, in.rot_k, in.rot_inv, F.s, in.rot_m < kRotOctetM);
      lds_barrier();
    }
#pragma unroll 1
    for (uint32_t p = 0; p < passes; ++p) {
      const uint32_t blk = quad + p * quads;
      if (blk >= pad) break;
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = 0.f;
      if (blk < nb && sub < 3u) {
        const uint32_t at = blk * kDim + sub * 8u;
        if (in.x_f32) {
#pragma unroll
          for (int j = 0; j < 8; ++j) v[j] = in.x_f32[at + j];
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) v[j] = xf[at + j];
        }
      }
      quantize_octet<DIG>(v, sub, L.planes + (size_t)blk * kStr);
    }
    if (tid < tail_w) L.xtail[tid] = in.x_f32 ? in.x_f32[nb * kDim + tid] : xf[nb * kDim + tid];
  } else {
    // One or two passes at a time, every operand requested before the first is used; a lane without columns reads the
    // row's first.  The norm's sum comes between two walks: the first leaves the summed values, as binary16, where the
    // second puts the block's planes (or, when two passes are all, in the registers).
    constexpr int kChunk = PMAX > 2 && DIG == 6 ? 1 : 2;
    const __half* second = SRC == kSrcAddRmsNorm ? (in.x2 ? in.x2 : in.x) : in.x2;
    const uint32_t t_at = min(nb * kDim + tid, d_in - 1u);
    float t0 = __half2float(load_half<kDeviceScope>(in.x + t_at)), t1 = 0.f, tg = 0.f;
    if constexpr (SRC != kSrcF16) t1 = __half2float(load_half<kDeviceScope>(second + t_at));
    if constexpr (SRC == kSrcAddRmsNorm) tg = __half2float(in.norm_w[t_at]);
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
      float v[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float lo = half_lo(a[k][j]), hi = half_hi(a[k][j]);
        if constexpr (SRC == kSrcSiluMul) {
          lo = silu_mul(half_lo(b[k][j]), lo);
          hi = silu_mul(half_hi(b[k][j]), hi);
        } else if constexpr (SRC == kSrcAddRmsNorm) {
          lo = round_half(lo * inv * half_lo(g[k][j]));
          hi = round_half(hi * inv * half_hi(g[k][j]));
        }
        v[2 * j] = ok ? lo : 0.f;
        v[2 * j + 1] = ok ? hi : 0.f;
      }
      quantize_octet<DIG>(v, sub, L.planes + (size_t)blk * kStr);
    };
    load_operands(0);
    request();
    __builtin_amdgcn_sched_barrier(0);
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
              a[k][j] = (uint32_t)__half_as_ushort(__float2half_rn(lo)) | (uint32_t)__half_as_ushort(__float2half_rn(hi)) << 16;
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
              uint32_t* keep = L.planes + (size_t)blk * kStr + sub * 4u;
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
      for (uint32_t w = 0; w < (n_thr >> 6); ++w) total += L.red[w];
      inv = 1.0f / sqrtf(total / (float)d_in + in.eps);
    }
    if constexpr (SRC == kSrcAddRmsNorm && PMAX > kChunk) {
#pragma unroll 1
      for (uint32_t p = 0; p < passes; ++p) {
        const uint32_t blk = block_of(p);
        if (blk >= pad) break;
        const bool ok = blk < nb && sub < 3u;
        const uint32_t* kept = L.planes + (size_t)blk * kStr + sub * 4u;
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

// A lane's share of a step: the nibbles and the byte of one (row, block).
struct StepWords {
  uint32_t w0, w1, w2, meta;  // meta: the dword with the bytes of the lane's row and its three neighbours
};
// step_at: the step's first block; lane_off: block lane / 8 and row lane % 8 behind it (12-byte words), meta_off the dword
// with the row's byte.  live = false (uniform) sends every lane to one place instead, a load nobody uses: one cache line,
// and no branch, which would turn every wait behind it into a wait for all loads.
// A record's last step may reach up to seven blocks past it, into the next record or the allocation's slack: such lanes
// meet zeros in the planes.
struct LaneOffsets {
  uint32_t words, meta;
};
__device__ __forceinline__ LaneOffsets lane_offsets(uint32_t lane) {
  const uint32_t r = lane & 7u, bq = lane >> 3;
  return LaneOffsets{bq * kTileBlockBytes + r * 12u, bq * kTileBlockBytes + 96u + (r & 4u)};
}
constexpr uint32_t kStepBytes = 8u * kTileBlockBytes;
__device__ __forceinline__ StepWords load_step(const uint8_t* blocks, uint32_t step, bool live, const LaneOffsets& at) {
  struct __attribute__((packed, aligned(4))) W3 { uint32_t w[3]; };
  typedef const uint8_t __attribute__((address_space(1))) global_u8;
  const uint32_t keep = live ? 0xFFFFFFFFu : 0u;
  uint64_t bits = reinterpret_cast<uint64_t>(blocks + ((step * kStepBytes) & keep));
  asm("" : "+s"(bits));  // a scalar base the compiler cannot take apart again: the loads add a 32-bit lane offset to it
  const uint8_t* base = (const uint8_t*)reinterpret_cast<global_u8*>(bits);
  const W3 w = *reinterpret_cast<const W3*>(base + (at.words & keep));
  // (the byte comes with its dword: a loop-carried byte would be copied, and so waited for, as soon as it is requested)
  return StepWords{w.w[0], w.w[1], w.w[2], *reinterpret_cast<const uint32_t*>(base + (at.meta & keep))};
}

template <int DIG>
struct XBlock {
  int d[3 * DIG];
  int sum;
  float scale;
};
template <int DIG>
__device__ __forceinline__ XBlock<DIG> load_xblock(const uint32_t* xb) {
  XBlock<DIG> x;
  const uint2* p = reinterpret_cast<const uint2*>(xb);
#pragma unroll
  for (int i = 0; i < 3 * DIG / 2; ++i) {
    const uint2 v = p[i];
    x.d[2 * i] = (int)v.x;
    x.d[2 * i + 1] = (int)v.y;
  }
  const uint2 v = p[3 * DIG / 2];
  x.sum = (int)v.x;
  x.scale = __uint_as_float(v.y);
  return x;
}

// acc + (one block's product): exact integer digit products, one f32 conversion, scaled by the block's weight scale and
// the activation's.  12 or 18 dot products and about 10 more instructions.
// table: the matrix's 32 scales, one per lane (the byte & 0x7C is the lane's place in bytes).
template <int DIG>
__device__ __forceinline__ float step_product(const StepWords& w, const XBlock<DIG>& x, uint32_t table, uint32_t r, float acc) {
  const uint32_t meta = w.meta >> (8u * (r & 3u));
  int d[DIG];
#pragma unroll
  for (int k = 0; k < DIG; ++k) {
    d[k] = __builtin_amdgcn_sdot8((int)w.w0, x.d[3 * k], 0, false);
    d[k] = __builtin_amdgcn_sdot8((int)w.w1, x.d[3 * k + 1], d[k], false);
    d[k] = __builtin_amdgcn_sdot8((int)w.w2, x.d[3 * k + 2], d[k], false);
  }
  int s = d[DIG - 1];
#pragma unroll
  for (int k = DIG - 2; k >= 0; --k) s = (s << 4) + d[k];
  s = (s << 1) + (x.sum & -(int)(meta & 1u));
  const float scale = __int_as_float(__builtin_amdgcn_ds_bpermute((int)(meta & 0x7Cu), (int)table));
  return fmaf((float)s, scale * x.scale, acc);
}

// Sum over the lanes that hold the same row (lane % 8): lanes 8, 16 and 32 apart.
__device__ __forceinline__ float row8_sum(float v) {
  v += dpp_move<0x128>(v);  // row_ror:8
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}

// A record's result from what its team's wavefronts left: row lane % 8 in every lane.  part, tpart: 8 floats to a wavefront.
__device__ __forceinline__ float team_sum(const float* part, const float* tpart, float scale, uint32_t split, uint32_t tail_waves, uint32_t lane) {
  const uint32_t k = lane >> 3;
  float v = k < split ? part[lane] : 0.f;
  if (split > 8u) v += part[64u + lane];
  v = row8_sum(v);
  float t = 0.f;
  if (tail_waves) t = row8_sum(k < tail_waves ? tpart[lane] : 0.f);
  return fmaf(v, scale, t);
}

__device__ __forceinline__ void tile_mat(const GemvArgs& a, uint32_t tile, const uint8_t*& base, void*& y, uint32_t& row0, uint32_t& d_out) {
  base = a.m[0].base;  // constant indices only: a dynamic one would move the arguments to scratch
  y = a.m[0].y;
  d_out = a.m[0].d_out;
  uint32_t begin = 0;
#pragma unroll
  for (uint32_t k = 1; k < kMaxGroup; ++k)
    if (k < a.n_mats && tile >= a.m[k].tile_begin) {
      base = a.m[k].base;
      y = a.m[k].y;
      d_out = a.m[k].d_out;
      begin = a.m[k].tile_begin;
    }
  row0 = (tile - begin) * kTileRows;
}

// What a wavefront loads for a record: its steps, its row's scale and a tail column of it, the matrix's block scales (one
// per lane).
template <uint32_t STEPS>
struct RecordWords {
  StepWords step[STEPS];
  float scale, tail;
  uint32_t table;
};
// live: whether the wavefront has a record at all; its j-th step is w + j split of n_steps.
template <uint32_t STEPS>
__device__ __forceinline__ void load_record(RecordWords<STEPS>& W, const uint8_t* rec, const uint8_t* base, uint32_t head, uint32_t w, uint32_t split,
                                            uint32_t n_steps, bool live, uint32_t tail_off, uint32_t lane, const LaneOffsets& at) {
  W.scale = reinterpret_cast<const float*>(rec)[lane & 7u];
  W.table = reinterpret_cast<const uint32_t*>(base)[lane & 31u];
  W.tail = *reinterpret_cast<const float*>(rec + (live ? tail_off : 0u));
#pragma unroll
  for (uint32_t j = 0; j < STEPS; ++j) W.step[j] = load_step(rec + head, w + j * split, live & (w + j * split < n_steps), at);
}

// y = W x for the rows of up to four matrices that share an activation.
//
// What bounds it: at 13 bytes per block and about 25 vector instructions the weights' way from memory; in a launch of
// a few microseconds the chain launch -> activation -> planes -> product -> store.  So: a team of 2^split_shift
// wavefronts takes a record of eight rows, a wavefront a fixed set of its steps; the loads of a record are all in flight
// before the planes are ready, and each step's registers are loaded again for the team's next record as soon as they have
// been used, without a branch, so that every wait is for the oldest load only.  For binary16 results a wavefront reads
// its planes from LDS once and keeps them in registers.  The sums over a team's wavefronts wait in LDS for one barrier
// per kGemvRounds records.  The host spreads teams over the CUs first (a workgroup has four to sixteen wavefronts),
// records over teams so that the last, partial round meets every CU.
// WIDE: rows past 512 blocks, with twice the steps.  Their planes, and the six digits of f32 results, do not fit the
// registers beside the weights: a step then reads its planes from LDS.
template <typename OutT, int SRC, bool WIDE>
__global__ __launch_bounds__(1024) void gemv_tiles_kernel(GemvArgs a) {
  constexpr int DIG = std::is_same<OutT, __half>::value ? 4 : 6;
  constexpr bool XREG = !WIDE && DIG == 4;
  constexpr uint32_t kSteps = WIDE ? kGemvWideSteps : kGemvSteps;
  constexpr uint32_t kStr = XPlanes<DIG>::kDwords;
  extern __shared__ __align__(16) uint8_t smem[];
  const GemvLds L = gemv_lds<DIG>(smem, gemv_plane_blocks(a.nb));
  const uint32_t tid = threadIdx.x, lane = tid & 63u, r = lane & 7u, bq = lane >> 3;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t split = 1u << a.split_shift, team = wave >> a.split_shift, w = wave & (split - 1u);
  const uint32_t teams = (blockDim.x >> 6) >> a.split_shift, n_teams = teams * gridDim.x;
  const uint32_t nb = a.nb, n_steps = (nb + 7u) >> 3;
  const LaneOffsets at = lane_offsets(lane);
  const uint32_t stride = tile_stride(nb, a.tail_w), head = tile_head_bytes(a.tail_w);

  struct Record { const uint8_t* rec; const uint8_t* base; };
  auto record_of = [&](uint32_t t) {
    const uint8_t* base;
    void* y;
    uint32_t row0, d_out;
    tile_mat(a, t, base, y, row0, d_out);
    return Record{base + kTileTableBytes + (size_t)(row0 / kTileRows) * stride, base};
  };
  const uint32_t tail_c = w * 8u + bq;  // the tail column this lane adds for its row
  const uint32_t tail_off = tail_c < a.tail_w ? 32u + tail_c * 32u + r * 4u : 0u;
  const uint32_t tail_waves = (a.tail_w + 7u) >> 3;

  uint32_t tile = team * gridDim.x + blockIdx.x;
  Record cur = record_of(min(tile, a.n_tiles - 1u));
  RecordWords<kSteps> W;
  stage_x<DIG, SRC, WIDE ? 8 : 2>(a.in, nb, a.tail_w, L, blockIdx.x == 0,
                                  [&]() { load_record(W, cur.rec, cur.base, head, w, split, n_steps, tile < a.n_tiles, tail_off, lane, at); });
  lds_barrier();

  XBlock<DIG> X[XREG ? kSteps : 1];
  if constexpr (XREG) {
#pragma unroll
    for (uint32_t j = 0; j < kSteps; ++j) X[j] = load_xblock<DIG>(L.planes + (min(w + j * split, n_steps) * 8u + bq) * kStr);
  }
  const float xt = tail_c < a.tail_w ? L.xtail[tail_c] : 0.f;
  const uint32_t rounds = (a.n_tiles + n_teams - 1u) / n_teams;
  for (uint32_t rd = 0; rd < rounds; ++rd) {
    const uint32_t next = tile + n_teams;
    const bool more = next < a.n_tiles;
    const Record nx = record_of(min(next, a.n_tiles - 1u));
    const uint32_t table = W.table;
    const float tail = W.tail, scale = W.scale;
    W.scale = reinterpret_cast<const float*>(nx.rec)[r];
    W.table = reinterpret_cast<const uint32_t*>(nx.base)[lane & 31u];  // first again, so that the next round waits for them alone
    W.tail = *reinterpret_cast<const float*>(nx.rec + (more ? tail_off : 0u));
    float acc = 0.f;
    if constexpr (XREG) {
#pragma unroll
      for (uint32_t j = 0; j < kSteps; ++j) {
        acc = step_product<DIG>(W.step[j], X[j], table, r, acc);
        __builtin_amdgcn_sched_barrier(0);  // the step's registers are free again only now: the loads need no others
        W.step[j] = load_step(nx.rec + head, w + j * split, more & (w + j * split < n_steps), at);
        __builtin_amdgcn_sched_barrier(0);  // step by step: the products of several at once would not fit the registers
      }
    } else {
#pragma unroll
      for (uint32_t j = 0; j < kSteps; ++j) {
        const uint32_t step = w + j * split;
        acc = step_product<DIG>(W.step[j], load_xblock<DIG>(L.planes + (min(step, n_steps) * 8u + bq) * kStr), table, r, acc);
        __builtin_amdgcn_sched_barrier(0);
        W.step[j] = load_step(nx.rec + head, step, more & (step < n_steps), at);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    acc = row8_sum(acc);
    const uint32_t slot = ((rd % kGemvRounds) * kGemvMaxWaves + wave) * 8u + lane;
    if (lane < 8u) {
      L.part[slot] = acc;
      L.scales[slot] = scale;
    }
    if (w < tail_waves) {
      const float t = row8_sum(tail_c < a.tail_w ? tail * xt : 0.f);
      if (lane < 8u) L.tpart[slot] = t;
    }
    cur = nx;
    tile = next;
    if ((rd + 1u) % kGemvRounds != 0u && rd + 1u != rounds) continue;
    // A wavefront per record of the last rounds: everything but the sums themselves is scalar.  (A lane per row, adding up
    // to sixteen values one behind the other, took 5300 of the 13700 cycles of a 2560 x 9728 product.)
    lds_barrier();
    const uint32_t r0 = rd / kGemvRounds * kGemvRounds, slots = kGemvMaxWaves >> a.split_shift;  // slots: teams to a round
    for (uint32_t q = wave; q < ((rd + 1u - r0) << (4u - a.split_shift)); q += teams << a.split_shift) {
      const uint32_t o_round = q >> (4u - a.split_shift), o_team = q & (slots - 1u);
      const uint32_t o_tile = (r0 + o_round) * n_teams + o_team * gridDim.x + blockIdx.x;
      if (o_team >= teams || o_tile >= a.n_tiles) continue;
      const uint8_t* o_base;
      void* o_y;
      uint32_t o_row0, o_d_out;
      tile_mat(a, o_tile, o_base, o_y, o_row0, o_d_out);
      const uint32_t at0 = (o_round * kGemvMaxWaves + (o_team << a.split_shift)) * 8u;
      const float v = team_sum(L.part + at0, L.tpart + at0, L.scales[at0 + r], split, tail_waves, lane);
      if (lane < 8u && o_row0 + lane < o_d_out) store_out<OutT>(o_y, o_row0 + lane, v);
    }
    if (rd + 1u != rounds) lds_barrier();
  }
}

template <typename OutT, bool WIDE>
__host__ const void* gemv_kernel_of(int src) {
  switch (src) {
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
  for (int src = kSrcF16; src <= kSrcAddRmsNorm; ++src)
    for (int v = 0; v < 4; ++v) fn(gemv_kernel(v & 1, src, v & 2));
}

}  // namespace llvq
