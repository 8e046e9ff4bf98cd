// The batched product Y[M, d_out] = X[M, d_in] W^T on the matrix cores (M >= 2), over the tiles of tiles.h.  Included by
// llvq_hip.hip after it.  The reference runs a row loop of matrix-vector products (llvq-llm/src/model.rs:521-529).
//
// Weights are multiplied as binary16: v centroid[gain] / sqrt(16 shell) rounded once; sums are f32; row scale and tail
// columns are applied in f32 at the end.  The PAIR variants of the kernels multiply what that rounding took as well and keep
// their sums in f64 (of f32 sums over 32 or 48 columns), for the rows whose results are f32 exact (llvq_hip.hip,
// gemm_same_basis).  Relative error of f32 results in norm, 2561 x 1000 at 65 rows: 2.1e-4 with one term, 1.01e-7 with two,
// 0.97e-7 for rows one by one; 13000 columns: 2.2e-4, 1.37e-7, 1.38e-7.  Two terms alone, summed in f32, left up to 6e-7.  A dword of a block's nibbles is eight consecutive columns of a row, which is
// exactly what a lane hands to a 16-deep (32 x 32) or 32-deep (16 x 16) product step, so a wavefront turns the 12 bytes
// its lanes load into its own fragments: no weights pass through LDS, and the order in which the products walk the
// columns is the order the blocks lie in (the lane groups of a fragment hold the same octet of two or four neighbouring
// blocks).  19 instructions per eight weights.
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
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kGemmMaxGroup = 4;
constexpr uint32_t kGemmSmallRows = 64;     // activation rows up to which the split kernel (gemm_tiles_kernel) runs
constexpr uint32_t kGemmTileRowsSmall = 16; // weight rows of a fragment there

// ---- activations as column octets ----------------------------------------------------------------
// One lane per octet; a wavefront takes eight octets of eight rows: 128 consecutive bytes of a row read, 128 of the copy
// written.  Rows from M on and columns from kcols on are zero.
__global__ __launch_bounds__(256) void tile_activations_kernel(const __half* __restrict__ x, uint32_t M, uint32_t ldx, uint32_t kcols,
                                                               uint32_t m_pad, uint32_t n_oct, uint4* __restrict__ xt) {
  const uint32_t lane = threadIdx.x & 63u, wave = blockIdx.x * 4u + (threadIdx.x >> 6);
  const uint32_t groups_m = m_pad >> 3;
  const uint32_t gc = wave / groups_m, gm = wave - gc * groups_m;
  const uint32_t c = gc * 8u + (lane & 7u), m = gm * 8u + (lane >> 3);
  uint4 v = make_uint4(0, 0, 0, 0);
  if (m < M && c * 8u < kcols) {
    const HalfOctet o = *reinterpret_cast<const HalfOctet*>(x + (size_t)m * ldx + c * 8u);
    v = make_uint4(o.w[0], o.w[1], o.w[2], o.w[3]);
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
// The matrix's table of scales for dequant_octet: a lane keeps entry lane % 32 as the sum of two binary16 numbers (low
// half: the entry rounded, high half: what that left), a power of two taken out first that puts the largest entry into
// [8, 16), so that neither number nor an eighth of it leaves the normal range by more than the precision can spare.
// `unit` is that power of two; it goes back in with the row scales.
__device__ __forceinline__ uint32_t split_table(float entry, float& unit) {
  uint32_t e = __float_as_uint(entry) & 0x7F800000u;
#pragma unroll
  for (int k = 1; k < 32; k <<= 1) e = max(e, (uint32_t)__shfl_xor((int)e, k));
  const int ex = min(max((int)(e >> 23) - 130, -100), 100);  // (a table of zeros or with an infinity in it: any power will do)
  unit = ldexpf(1.f, ex);
  const float v = entry * ldexpf(1.f, -ex);
  const _Float16 hi = (_Float16)v;
  const _Float16 lo = (_Float16)(v - (float)hi);
  return __builtin_bit_cast(uint32_t, half2_t{hi, lo});
}
// What a block's meta byte gives a lane: the two parts of its scale (and an eighth of them), and its parity bit where
// dequant_octet wants it.
struct BlockScale {
  half2_t c, c8;
  uint32_t odd, odd8;
};
__device__ __forceinline__ uint32_t block_meta(uint32_t meta_dword, uint32_t r) { return meta_dword >> (8u * (r & 3u)); }
__device__ __forceinline__ uint32_t scale_parts(uint32_t meta, uint32_t table) {
  return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(meta & 0x7Cu), (int)table);
}
__device__ __forceinline__ BlockScale block_scale(uint32_t meta, uint32_t parts) {
  const half2_t c = __builtin_bit_cast(half2_t, parts);
  const uint32_t p = (uint32_t)((int32_t)(meta << 31) >> 31);
  uint32_t odd = (p & 0x00010001u) ^ 0x64106410u, odd8 = (p & 0x00080008u) ^ 0x64806480u;
  asm("" : "+v"(odd), "+v"(odd8));  // (kept whole: taken apart again, a mask and it would no longer be one operation)
  return BlockScale{c, c * half2_t{(_Float16)0.125f, (_Float16)0.125f}, odd, odd8};
}
// One dword of nibbles -> eight weights.  A binary16 number of the form 1024 + k has k in its low bits: with the nibble's
// top bit flipped (two's complement to offset) and the parity bit below it that is 1024 + 16 + v, or 1024 + 128 + 8 v
// where the nibble lies four bits higher.  v (hi + lo) is rounded once: v lo is small enough for its own rounding to be
// lost in that of the sum.  19 instructions, all of which run beside the matrix cores; the mixed-precision
// multiply-add (two fewer) does not: 4 products and 20 of those took 103 ns of a SIMD, with packed or f32 ones 70.
__device__ __forceinline__ half8_t dequant_octet(uint32_t w, const BlockScale& s) {
  const uint32_t t[4] = {((w << 1) & 0x001E001Eu) ^ s.odd, (w & 0x00F000F0u) ^ s.odd8, ((w >> 7) & 0x001E001Eu) ^ s.odd, ((w >> 8) & 0x00F000F0u) ^ s.odd8};
  half8_t out;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const half2_t bias = (i & 1) ? half2_t{(_Float16)1152.f, (_Float16)1152.f} : half2_t{(_Float16)1040.f, (_Float16)1040.f};
    const half2_t v = __builtin_bit_cast(half2_t, t[i]) - bias;
    const half2_t c = (i & 1) ? s.c8 : s.c;
    const half2_t y = __builtin_elementwise_fma(v, half2_t{c.x, c.x}, v * half2_t{c.y, c.y});
    out[2 * i] = y.x;
    out[2 * i + 1] = y.y;
  }
  return out;
}

// The same with what the rounding took as a second binary16 number each: the two make the weight to 2^-22 of it.  (A nibble
// that lies four bits higher is brought down by the operation that takes the bias off, so both halves are v itself; what is
// left of v hi after the first rounding is exact, and v lo joins it in one more.)  27 instructions.
struct WeightPair {
  half8_t hi, lo;
};
__device__ __forceinline__ WeightPair dequant_octet_pair(uint32_t w, const BlockScale& s) {
  const uint32_t t[4] = {((w << 1) & 0x001E001Eu) ^ s.odd, (w & 0x00F000F0u) ^ s.odd8, ((w >> 7) & 0x001E001Eu) ^ s.odd, ((w >> 8) & 0x00F000F0u) ^ s.odd8};
  const half2_t hi = half2_t{s.c.x, s.c.x}, lo = half2_t{s.c.y, s.c.y};
  WeightPair out;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const half2_t u = __builtin_bit_cast(half2_t, t[i]);
    const half2_t v = (i & 1) ? __builtin_elementwise_fma(u, half2_t{(_Float16)0.125f, (_Float16)0.125f}, half2_t{(_Float16)-144.f, (_Float16)-144.f})
                              : u - half2_t{(_Float16)1040.f, (_Float16)1040.f};
    const half2_t y = __builtin_elementwise_fma(v, hi, v * lo);
    const half2_t r = __builtin_elementwise_fma(v, lo, __builtin_elementwise_fma(v, hi, -y));
    out.hi[2 * i] = y.x;
    out.hi[2 * i + 1] = y.y;
    out.lo[2 * i] = r.x;
    out.lo[2 * i + 1] = r.y;
  }
  return out;
}

struct GemmMat {
  const uint8_t* base;  // the matrix (table, then records)
  void* y;
  uint32_t d_out, tile_begin;  // first row tile of this matrix in the launch
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
};

struct GemmTile {
  const uint8_t* base;
  void* y;
  uint32_t row0, d_out;
};
__device__ __forceinline__ GemmTile gemm_tile_at(const GemmArgs& a, uint32_t tile, uint32_t rows_per_tile) {
  GemmTile t{a.mat[0].base, a.mat[0].y, 0u, a.mat[0].d_out};
  uint32_t begin = 0;
#pragma unroll
  for (uint32_t k = 1; k < (uint32_t)kGemmMaxGroup; ++k)
    if (k < a.n_mats && tile >= a.mat[k].tile_begin) {
      t.base = a.mat[k].base;
      t.y = a.mat[k].y;
      t.d_out = a.mat[k].d_out;
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
// 2560 x 2560 at 5 rows: 35.9 -> 10.4 us; rotated q, k, v of 2560 columns at 64 rows, rotation included: 58.1 -> 21.7 us
// (before: codes unranked in the product, partial sums through memory).
// PAIR: both terms of the weights (dequant_octet_pair), 32 columns to a product sum that starts from zero, those added in
// f64; RG = 1 always, two row groups would not fit the registers.  4097 columns, 1024 rows by 64: 16 -> 14 us (twice the
// workgroups), 5000 by 33: 15 -> 22 us.
template <int RG, int MT, bool PAIR>
__global__ __launch_bounds__(1024) void gemm_tiles_kernel(GemmArgs a) {
  extern __shared__ __align__(16) uint8_t smem[];
  constexpr uint32_t kRows = RG * 16, kCols = MT * 16;
  float* part = reinterpret_cast<float*>(smem);           // [16 wavefronts][RG][MT][64 lanes][4]
  float* tw = part + 16 * RG * MT * 256;                  // [kRows][24] tail weights
  float* scale_s = tw + kRows * 24;
  float* tx = scale_s + kRows;                            // [kCols][24] tail activations
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t nb = a.nb, n_quads = (nb + 3u) >> 2;
  const uint32_t stride = tile_stride(nb, a.tail_w), head = tile_head_bytes(a.tail_w);
  const GemmTile t = gemm_tile_at(a, blockIdx.x, kRows);
  const uint8_t* recs = t.base + kTileTableBytes + (size_t)(t.row0 / kTileRows) * stride;
  const uint32_t last_rec = tile_count(t.d_out) - 1u - t.row0 / kTileRows;  // records past the matrix's last repeat it
  const uint32_t r = lane & 7u, g = lane >> 4, m16 = lane & 15u;
  const float entry = reinterpret_cast<const float*>(t.base)[lane & 31u];
  uint32_t rec_off[RG];
#pragma unroll
  for (int k = 0; k < RG; ++k) rec_off[k] = min((uint32_t)k * 2u + ((lane >> 3) & 1u), last_rec) * stride + head + g * kTileBlockBytes;
  const uint32_t x_off = (g * 3u * a.m_pad + m16) * 16u, x_oct = a.m_pad * 16u;

  StepWords W[RG];
  u32x4_t X[3][MT];
  struct __attribute__((packed, aligned(4))) W3 { uint32_t w[3]; };
  auto load_w = [&](uint32_t q, bool live) {
    const uint32_t keep = live ? 0xFFFFFFFFu : 0u;
    const uint8_t* p = uniform_global(recs + ((q * 4u * kTileBlockBytes) & keep));
#pragma unroll
    for (int k = 0; k < RG; ++k) {
      const W3 w = *reinterpret_cast<const W3*>(p + lane_offset((rec_off[k] + r * 12u) & keep));
      W[k] = StepWords{w.w[0], w.w[1], w.w[2], *reinterpret_cast<const uint32_t*>(p + lane_offset((rec_off[k] + 96u + (r & 4u)) & keep))};
    }
  };
  auto load_x = [&](uint32_t j, uint32_t q, bool live) {
    const uint32_t keep = live ? 0xFFFFFFFFu : 0u;
    const uint8_t* p = uniform_global(reinterpret_cast<const uint8_t*>(a.xt) + ((size_t)(q * 12u + j) * x_oct & (size_t)(int64_t)(int32_t)keep));
    const uint32_t off = lane_offset(x_off & keep);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) X[j][mt] = *reinterpret_cast<const u32x4_t*>(p + off + (uint32_t)mt * 256u);
  };
  // The row scales and the tail's operands, needed at the end: asked for first, put down last.
  const uint32_t op_row = tid % kRows, op_col = tid / kRows;  // column 24: the row's scale
  float op_w = 0.f;
  uint32_t op_x[2] = {};
  {
    const uint8_t* rec = recs + (size_t)min(op_row / kTileRows, last_rec) * stride;
    const uint32_t c = op_col < a.tail_w ? op_col + 1u : 0u;
    op_w = reinterpret_cast<const float*>(rec)[c * 8u + (op_row & 7u)];
    if (a.tail_w) {
#pragma unroll
      for (uint32_t i = 0; i < 2; ++i) {
        const uint32_t k = tid + i * 1024u, m = k / a.tail_w;
        op_x[i] = reinterpret_cast<const uint16_t*>(a.x)[(size_t)min(m, a.M - 1u) * a.ldx + nb * kDim + k - m * a.tail_w];
      }
    }
  }
  uint32_t q = wave;
  load_w(q, q < n_quads);
#pragma unroll
  for (uint32_t j = 0; j < 3; ++j) load_x(j, q, q < n_quads);
  float unit;
  const uint32_t table = split_table(entry, unit);
  typedef double sum4_t __attribute__((ext_vector_type(4)));
  typename std::conditional<PAIR, sum4_t, acc4_t>::type acc[RG][MT];
#pragma unroll
  for (int k = 0; k < RG; ++k)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[k][mt] = 0;
  for (; q < n_quads; q += 16u) {
    const uint32_t qn = q + 16u;
    const bool live = qn < n_quads;
    BlockScale s[RG];
#pragma unroll
    for (int k = 0; k < RG; ++k) {
      const uint32_t meta = block_meta(W[k].meta, r);
      s[k] = block_scale(meta, scale_parts(meta, table));
    }
#pragma unroll
    for (uint32_t j = 0; j < 3; ++j) {
      half8_t w[RG], w2[RG];
#pragma unroll
      for (int k = 0; k < RG; ++k) {
        const uint32_t nibbles = j == 0 ? W[k].w0 : j == 1 ? W[k].w1 : W[k].w2;
        if constexpr (PAIR) {
          const WeightPair p = dequant_octet_pair(nibbles, s[k]);
          w[k] = p.hi;
          w2[k] = p.lo;
        } else {
          w[k] = dequant_octet(nibbles, s[k]);
        }
      }
      // a register is asked for again as soon as its contents are used, and not moved from there
      if (j == 2u) {
        __builtin_amdgcn_sched_barrier(0);
        load_w(qn, live);
        __builtin_amdgcn_sched_barrier(0);
      }
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
  if (op_col < a.tail_w) tw[op_row * 24u + op_col] = op_w;
  else if (op_col == 24u) scale_s[op_row] = op_w * unit;
  if (a.tail_w) {
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {
      const uint32_t k = tid + i * 1024u, m = k / a.tail_w;
      if (m < kCols) tx[m * 24u + k - m * a.tail_w] = __half2float(__ushort_as_half((unsigned short)op_x[i]));
    }
  }
  // of a fragment a lane's row is a weight row (lane % 16) and its four elements activation rows 4 (lane / 16) + e
#pragma unroll
  for (int k = 0; k < RG; ++k)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      *reinterpret_cast<acc4_t*>(part + (((wave * RG + k) * MT + mt) * 64u + lane) * 4u) = __builtin_convertvector(acc[k][mt], acc4_t);
  __syncthreads();
  for (uint32_t o = tid; o < kRows * kCols; o += 1024u) {
    const uint32_t row = o % kRows, m = o / kRows;
    if (m >= a.M || t.row0 + row >= t.d_out) continue;
    const uint32_t l = (row & 15u) + 16u * ((m & 15u) >> 2), e = m & 3u;
    const float* p = part + (((row >> 4) * MT + (m >> 4)) * 64u + l) * 4u + e;
    typedef typename std::conditional<PAIR, double, float>::type sum_t;
    sum_t s = 0;
#pragma unroll
    for (uint32_t k = 0; k < 16; ++k) s += (sum_t)p[k * RG * MT * 256];
    float tl = 0.f;
    for (uint32_t c = 0; c < a.tail_w; ++c) tl = fmaf(tw[row * 24u + c], tx[m * 24u + c], tl);
    store_y(t.y, (size_t)m * t.d_out + t.row0 + row, fmaf((float)s, scale_s[row], tl), a.y_f32);
  }
}
template <int RG, int MT>
__host__ constexpr size_t gemm_small_lds() { return (size_t)(16 * RG * MT * 256 + RG * 16 * 25 + MT * 16 * 24) * 4; }
static_assert(gemm_small_lds<2, 4>() <= 160 * 1024, "partial sums of sixteen wavefronts fit a CU's LDS");

// A lane's sixteen results of one activation row (weight rows row + 8 g + 4 h .. + 3, g < 4) into y + at: where y and its
// rows lie on 16-byte boundaries, and one by one.
struct StoreF32 {
  static __device__ __forceinline__ void store(void* y, size_t at, uint32_t row, uint32_t h, uint32_t, const acc16_t& v) {
    float* out = reinterpret_cast<float*>(y) + at + row + 4u * h;
#pragma unroll
    for (int g = 0; g < 4; ++g) *reinterpret_cast<float4*>(out + g * 8) = make_float4(v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]);
  }
};
struct StoreF16 {
  static __device__ __forceinline__ void store(void* y, size_t at, uint32_t row, uint32_t h, uint32_t, const acc16_t& v) {
    uint32_t p[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) p[i] = __builtin_bit_cast(uint32_t, half2_t{(_Float16)v[2 * i], (_Float16)v[2 * i + 1]});
    _Float16* out = reinterpret_cast<_Float16*>(y) + at + row;
#pragma unroll
    for (int g = 0; g < 4; g += 2) {  // the upper half's group g for the lower half's group g + 1: eight rows in a row each
      const auto a = __builtin_amdgcn_permlane32_swap(p[2 * g], p[2 * g + 2], false, false);
      const auto b = __builtin_amdgcn_permlane32_swap(p[2 * g + 1], p[2 * g + 3], false, false);
      *reinterpret_cast<u32x4_t*>(out + (g + h) * 8u) = u32x4_t{a[0], b[0], a[1], b[1]};
    }
  }
};
template <typename Y>
struct StoreEach {
  static __device__ __forceinline__ void store(void* y, size_t at, uint32_t row, uint32_t h, uint32_t d_out, const acc16_t& v) {
    Y* out = reinterpret_cast<Y*>(y) + at;
#pragma unroll
    for (uint32_t e = 0; e < 16; ++e) {
      const uint32_t r = row + 8u * (e >> 2) + 4u * h + (e & 3u);
      if (r < d_out) out[r] = (Y)v[e];
    }
  }
};

// ---- more activation rows ----------------------------------------------------------------------------
// What bounds it: the chain of a step, in which the matrix cores are busy half the time (51 % for CF = 8, counters in
// profiles/; 38 instructions of unpacking run beside every 2 CF products), and tiles that are no multiple of the CUs (192
// workgroups for gate and up of an 8B layer at 512 rows).  A workgroup of four wavefronts takes 256 weight rows by 32 CF activation rows; a wavefront unpacks 64 rows
// (two fragments) against all of the activation rows (CF fragments).  CF = 8: 256 accumulators and one wavefront on a
// SIMD, half the unpacking and a workgroup on every CU (1.28 us a step, where the products alone take 0.85 on numbers
// like these in a loop of nothing else); CF = 4: half of that, two workgroups on a CU (0.69 us a step each) or one (0.8), for batches and matrices
// that do not fill the other.
// Octets and tiles go from memory to LDS without passing through registers, two to three steps of 48 columns (two
// blocks) ahead.
// PAIR: both terms of the weights against the same activations, 2 CF more products a round; every step's sums go to f64
// ones (512 registers: CF = 4 and one wavefront on a SIMD).  2.4 us a step; 13000 x 5121 at 600 rows 115 -> 250 to 280 us.
// Launches with too few tiles to fill the chip split the columns (`splits`): partial sums go to the workspace and
// gemm_reduce_kernel adds them in order; otherwise the tile is finished here.
// Gate and up of an 8B layer (24576 x 4096) at 512 rows: 158 -> 116 us, 886 TFLOP/s; a plain f16 product of that size
// by the vendor's library runs at 1151 on this card (a loop of nothing but products on random numbers reaches 1650).
constexpr uint32_t kWideRows = 256;
constexpr uint32_t kWideTileBytes = 1024;  // four records, two blocks of each (832 bytes) and what the lanes behind them bring
constexpr uint32_t kWideDepth = 4;         // LDS buffers, a step each
template <int CF>
__host__ __device__ constexpr uint32_t gemm_wide_x_bytes() { return 6u * 32u * CF * 16u; }
template <int CF>
__host__ __device__ constexpr uint32_t gemm_wide_buf() { return gemm_wide_x_bytes<CF>() + 8u * kWideTileBytes; }
template <int CF>
__host__ constexpr size_t gemm_wide_lds() { return (size_t)kWideDepth * gemm_wide_buf<CF>(); }
static_assert(kWideDepth * gemm_wide_buf<4>() >= (kWideRows + 128u) * kDim * 4u && kWideDepth * gemm_wide_buf<8>() >= (kWideRows + 256u) * kDim * 4u,
              "the tail's operands fit the buffers");

// 16 bytes per lane from base + offset to LDS, lane after lane from `lds` on.  In assembly because the compiler, which
// cannot tell the buffers apart, would have every read of LDS wait for all of these; the counting is done by hand
// (wide_wait), and there are no other loads in flight where it is.  M0, where the place in LDS goes, is an operand: the
// compiler writes it, and knows that it did.
__device__ __forceinline__ void load_to_lds(uint32_t lds, uint32_t offset, const uint8_t* base) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "{m0}"(lds), "v"(offset), "s"(base) : "memory");
}
template <int N>
__device__ __forceinline__ void wide_wait() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }

template <int CF, bool PAIR>
__global__ __launch_bounds__(256, CF == 8 || PAIR ? 1 : 2) void gemm_wide_kernel(GemmArgs a) {
  constexpr uint32_t kCols = 32u * CF, kBuf = gemm_wide_buf<CF>();
  constexpr int kLoadsX = 3 * CF / 4, kLoadsW = 2, kLoads = kLoadsX + kLoadsW;  // of a wavefront in a step
  extern __shared__ __align__(16) uint8_t smem[];     // [kWideDepth] x { [6 octets][kCols] 16 bytes, [8] x 32 rows of tiles }
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t l32 = lane & 31u, h = lane >> 5, r = lane & 7u;
  // tiles of one row group are neighbours in the grid: they read the same weights
  const uint32_t mt = blockIdx.x % a.m_tiles, rest = blockIdx.x / a.m_tiles;
  const uint32_t tile = rest % a.n_tiles, split = rest / a.n_tiles;
  const uint32_t nb = a.nb, stride = tile_stride(nb, a.tail_w), head = tile_head_bytes(a.tail_w);
  const GemmTile t = gemm_tile_at(a, tile, kWideRows);
  const uint32_t row0 = t.row0 + wave * 64u;            // this wavefront's first row
  const uint32_t n_rec = tile_count(t.d_out);
  const float entry = reinterpret_cast<const float*>(t.base)[lane & 31u];
  const uint32_t n_steps = (nb + 1u) >> 1;
  const uint32_t s0 = split * a.steps_per_split, s1 = min(s0 + a.steps_per_split, n_steps);
  const uint8_t* rec0 = uniform_global(t.base + kTileTableBytes + (size_t)(t.row0 / kTileRows) * stride);
  // records past the matrix's last repeat it: their rows are not stored
  auto record = [&](uint32_t row) __attribute__((always_inline)) { return (min(row / kTileRows, n_rec - 1u) - t.row0 / kTileRows) * stride; };
  // a load of tiles takes four records, 13 lanes each; a load of octets 64 activation rows of one
  uint32_t w_off[kLoadsW], x_off[kLoadsX];
  const uint32_t w_rec = min(lane, 51u) / 13u, w_piece = min(lane, 51u) - w_rec * 13u;
#pragma unroll
  for (uint32_t k = 0; k < (uint32_t)kLoadsW; ++k) w_off[k] = record(t.row0 + (wave * (uint32_t)kLoadsW + k) * 32u + w_rec * 8u) + head + w_piece * 16u;
#pragma unroll
  for (uint32_t i = 0; i < (uint32_t)kLoadsX; ++i) {
    const uint32_t k = i * 4u + wave, o = k / (kCols / 64u), m = k % (kCols / 64u) * 64u + lane;
    x_off[i] = (o * a.m_pad + mt * kCols + m) * 16u;
  }
  const uint32_t x_step = 6u * a.m_pad * 16u, smem_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  const uint8_t* xt = reinterpret_cast<const uint8_t*>(a.xt);
  auto load = [&](uint32_t s, uint32_t buffer) __attribute__((always_inline)) {
    s = min(s, s1 - 1u);  // (steps past the last are loaded too, so that the count of loads in flight is always the same)
    const uint32_t at = smem_at + buffer;
    const uint8_t* xs = uniform_global(xt + (size_t)s * x_step);
    const uint8_t* ws = uniform_global(rec0 + (size_t)s * (2u * kTileBlockBytes));
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)kLoadsX; ++i) load_to_lds(at + (i * 4u + wave) * 1024u, x_off[i], xs);
#pragma unroll
    for (uint32_t k = 0; k < (uint32_t)kLoadsW; ++k) load_to_lds(at + gemm_wide_x_bytes<CF>() + (wave * (uint32_t)kLoadsW + k) * kWideTileBytes, w_off[k], ws);
  };
  acc16_t acc[2][CF];
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int c = 0; c < CF; ++c)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[k][c][e] = 0.f;
  double sum[PAIR ? 2 : 1][PAIR ? CF : 1][16];  // of the steps, with PAIR
  if constexpr (PAIR) {
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int c = 0; c < CF; ++c)
#pragma unroll
        for (int e = 0; e < 16; ++e) sum[k][c][e] = 0.;
  }
  float unit;
  const uint32_t table = split_table(entry, unit);
  // One step: three rounds of eight products, in whose shadow the weights of the round after are unpacked and its
  // activations read.  Behind the first round every wavefront waits for its loads of the next step and then for the
  // others; the step before has been read by then, and its buffer is filled again.  In the second the next step's tiles
  // are read, in the third unpacked.
  struct W3 { uint32_t w[3]; };
  typedef __attribute__((address_space(3))) uint32_t lds_u32;
  half8_t w[2], w2[2], x[CF];
  W3 W[2], Wn[2];
  uint32_t meta[2], parts[2];
  BlockScale sc[2];
  auto unpack = [&](uint32_t j) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if constexpr (PAIR) {
        const WeightPair p = dequant_octet_pair(W[k].w[j], sc[k]);
        w[k] = p.hi;
        w2[k] = p.lo;
      } else {
        w[k] = dequant_octet(W[k].w[j], sc[k]);
      }
    }
  };
  const uint32_t x_at = (h * 3u * kCols + l32) * 16u;
  const uint32_t block_at = gemm_wide_x_bytes<CF>() + wave * 2u * kWideTileBytes + (l32 >> 3) * (2u * kTileBlockBytes) + h * kTileBlockBytes;
  const uint32_t w_at = block_at + r * 12u, meta_at = block_at + 96u + r;
  auto read_x = [&](uint32_t buffer, uint32_t j) __attribute__((always_inline)) {
    const u32x4_t* f = reinterpret_cast<const u32x4_t*>(smem + (buffer + x_at)) + j * kCols;
#pragma unroll
    for (int c = 0; c < CF; ++c) x[c] = __builtin_bit_cast(half8_t, f[(uint32_t)c * 32u]);
  };
  auto read_w = [&](uint32_t buffer) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 2; ++k) meta[k] = smem[(buffer + meta_at) + k * kWideTileBytes];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      // (dword by dword: merged into one read of 12 bytes at 4-byte alignment they took 60 cycles of LDS, not 6)
      const volatile lds_u32* f = (const volatile lds_u32*)(lds_u32*)(smem + (buffer + w_at) + k * (int)kWideTileBytes);
      Wn[k] = W3{{f[0], f[1], f[2]}};
    }
  };
  auto look_up = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 2; ++k) parts[k] = scale_parts(meta[k], table);
  };
  auto scales = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      sc[k] = block_scale(meta[k], parts[k]);
      W[k] = Wn[k];
    }
  };
  auto round = [&](uint32_t buffer, uint32_t next, auto round_j) __attribute__((always_inline)) {
    constexpr uint32_t j = decltype(round_j)::value;
    const half8_t w0[2] = {w[0], w[1]}, w20[2] = {w2[0], w2[1]};
    half8_t x0[CF];
#pragma unroll
    for (int c = 0; c < CF; ++c) x0[c] = x[c];
    if (j < 2u) {
      read_x(buffer, j + 1u);
      unpack(j + 1u);
    } else {
      read_x(next, 0);
      scales();
      unpack(0);
    }
    if constexpr (PAIR) {
#pragma unroll
      for (int c = 0; c < CF; ++c)
#pragma unroll
        for (int k = 0; k < 2; ++k) acc[k][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w20[k], x0[c], acc[k][c], 0, 0, 0);
    }
#pragma unroll
    for (int c = 0; c < CF; ++c)
#pragma unroll
      for (int k = 0; k < 2; ++k) acc[k][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w0[k], x0[c], acc[k][c], 0, 0, 0);
#pragma unroll
    for (int c = 0; c < CF; ++c) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // an LDS read,
#pragma unroll
      for (int i = 0; i < (PAIR ? 4 : 2); ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // a product,
        __builtin_amdgcn_sched_group_barrier(0x002, PAIR ? (CF == 8 ? 2 : 4) : (CF == 8 ? 3 : 5), 0);  // vector instructions
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  load(s0, 0);
  load(s0 + 1u, kBuf);
  load(s0 + 2u, 2u * kBuf);
  wide_wait<2 * kLoads>();
  lds_barrier();
  read_w(0);
  look_up();
  read_x(0, 0);
  scales();
  unpack(0);
  uint32_t buffer = 0, next = kBuf, last = 3u * kBuf, s = s0;
  do {  // (a split has at least one step)
    round(buffer, next, std::integral_constant<uint32_t, 0>{});
    wide_wait<kLoads>();
    lds_barrier();
    load(s + 3u, last);
    read_w(next);
    __builtin_amdgcn_sched_barrier(0);
    round(buffer, next, std::integral_constant<uint32_t, 1>{});
    look_up();
    __builtin_amdgcn_sched_barrier(0);
    round(buffer, next, std::integral_constant<uint32_t, 2>{});
    last = buffer;
    buffer = next;
    next = next + kBuf == kWideDepth * kBuf ? 0u : next + kBuf;
    if constexpr (PAIR) {
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int c = 0; c < CF; ++c)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            sum[k][c][e] += (double)acc[k][c][e];
            acc[k][c][e] = 0.f;
          }
    }
  } while (++s < s1);
  if constexpr (PAIR) {
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int c = 0; c < CF; ++c)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[k][c][e] = (float)sum[k][c][e];
  }
  wide_wait<0>();
  if constexpr (CF == 8) {
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int c = 0; c < CF; ++c) asm volatile("" : "+a"(acc[k][c]));  // one by one from here: all of them would not fit the vector registers
  }
  // A lane's activation row is l32 of a fragment; element e is weight row 8 (e / 4) + 4 h + e % 4 of it.
  // (From the lane's number anew: nothing of this may occupy registers during the loop.)
  const uint32_t lane_e = lane_offset(lane), l32e = lane_e & 31u, he = lane_e >> 5;
  const uint32_t m0 = mt * kCols + l32e;
  if (a.splits > 1u) {
    const uint32_t n_rows = a.n_tiles * kWideRows;
    float* out = a.ws + (size_t)split * a.m_pad * n_rows;
#pragma unroll
    for (int c = 0; c < CF; ++c)
      if (m0 + (uint32_t)c * 32u < a.M) {
#pragma unroll
        for (int k = 0; k < 2; ++k)
          StoreF32::store(out, (size_t)(m0 + (uint32_t)c * 32u) * n_rows, tile * kWideRows + wave * 64u + (uint32_t)k * 32u, he, 0, acc[k][c] * unit);
      }
    return;
  }
  // The tail's operands to LDS, columns of all rows: a lane would wait for each of its loads in turn.
  float* w_tail = reinterpret_cast<float*>(smem);
  float* x_tail = w_tail + kWideRows * kDim;
  if (a.tail_w) {
    __syncthreads();
    for (uint32_t c0 = 0; c0 < a.tail_w; c0 += 8u) {
      float v[8];
      const uint32_t row = tid % kWideRows, m = mt * kCols + tid % kCols;
      // (the columns are shared out where there are two threads to a row)
      const float* rec = reinterpret_cast<const float*>(rec0 + record(t.row0 + row) + 32u) + (row & 7u);
      const __half* tx = a.x + (size_t)min(m, a.M - 1u) * a.ldx + nb * kDim;
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) v[i] = rec[min(c0 + i, a.tail_w - 1u) * 8u];
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i)
        if (tid < kWideRows && c0 + i < a.tail_w) w_tail[(c0 + i) * kWideRows + row] = v[i];
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) v[i] = __half2float(tx[min(c0 + i, a.tail_w - 1u)]);
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i)
        if (tid < kCols && c0 + i < a.tail_w) x_tail[(c0 + i) * kCols + tid] = v[i];
    }
    __syncthreads();
  }
  auto finish = [&](auto to) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const uint32_t row = row0 + (uint32_t)k * 32u;
      float scale[16];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 v = *reinterpret_cast<const float4*>(rec0 + record(row + g * 8u) + he * 16u);
        scale[4 * g] = v.x * unit;
        scale[4 * g + 1] = v.y * unit;
        scale[4 * g + 2] = v.z * unit;
        scale[4 * g + 3] = v.w * unit;
      }
#pragma unroll
      for (int c = 0; c < CF; ++c) {
        // f32 tail columns, two at a time: the halves hold one each.  (One by one on top of the blocks' sum each costs that a
        // rounding: with PAIR they are summed by themselves and meet it last.)
        acc16_t v;
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = PAIR ? 0.f : acc[k][c][e] * scale[e];
        for (uint32_t i = 0; i < a.tail_w; i += 2u) {
          // (Without PAIR they are an even number.  With it a column past the last is zero in both operands: zero times the last
          // one again is not zero where that is infinite.)
          const uint32_t col = PAIR ? min(i + he, a.tail_w - 1u) : i + he;
          const bool there = !PAIR || i + he < a.tail_w;
          const float tw = w_tail[col * kWideRows + wave * 64u + (uint32_t)k * 32u + l32e], tx = x_tail[col * kCols + (uint32_t)c * 32u + l32e];
          v = __builtin_amdgcn_mfma_f32_32x32x2f32(there ? tw : 0.f, there ? tx : 0.f, v, 0, 0, 0);
        }
        if constexpr (PAIR) {
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            float y = fmaf(acc[k][c][e], scale[e], v[e]);
            asm("" : "+v"(y));  // (an f32 value in every store: where they convert one by one it would be one operation, rounded once)
            v[e] = y;
          }
        }
        const uint32_t m = m0 + (uint32_t)c * 32u;
        if (m < a.M) decltype(to)::store(t.y, (size_t)m * t.d_out, row, he, t.d_out, v);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  const bool whole = row0 + 64u <= t.d_out && ((reinterpret_cast<uintptr_t>(t.y) | t.d_out * (a.y_f32 ? 4u : 2u)) & 15u) == 0;
  if (a.y_f32) {
    if (whole) finish(StoreF32{});
    else finish(StoreEach<float>{});
  } else {
    if (whole) finish(StoreF16{});
    else finish(StoreEach<_Float16>{});
  }
}

// The partial sums of the column splits, added in order; row scale and tail columns.  A lane takes one weight row and
// kReduceM activation rows, so that the row's tail is read once for them.
// What bounds it is how many round trips to memory a lane makes: the sums and the tail columns are read four splits and
// eight columns at a time, the activations' tail comes to LDS with the first of them.  (One by one 11.3 us for 500
// rows of 2560 with 8 or 16 tail columns and 14.9 for 6144; so 9.0 and 10.3.)
constexpr uint32_t kReduceM = 8;
constexpr uint32_t kReduceSplits = 4;
struct GemmReduceArgs {
  GemmArgs g;
  uint32_t rows_per_tile, row_chunks;
};
// With PAIR the splits are added in f64 and the tail by itself.
template <bool PAIR>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(GemmReduceArgs ra) {
  typedef typename std::conditional<PAIR, double, float>::type sum_t;
  __shared__ float x_tail[kReduceM][32];
  static_assert(kReduceM * 32u == 256u && kDim <= 32, "a value of the activations' tail per lane");
  const GemmArgs& a = ra.g;
  const uint32_t n_rows = a.n_tiles * ra.rows_per_tile;
  const uint32_t chunk = blockIdx.x % ra.row_chunks, m0 = blockIdx.x / ra.row_chunks * kReduceM;
  const uint32_t mine = chunk * 256u + threadIdx.x, out_row = min(mine, n_rows - 1u);  // lanes past the last row repeat it
  const GemmTile t = gemm_tile_at(a, out_row / ra.rows_per_tile, ra.rows_per_tile);
  const uint32_t my_row = t.row0 + out_row % ra.rows_per_tile, row = min(my_row, t.d_out - 1u);
  const uint32_t stride = tile_stride(a.nb, a.tail_w);
  const uint8_t* rec = t.base + kTileTableBytes + (size_t)(row / kTileRows) * stride;
  const uint32_t r = row & 7u, tail_w = a.tail_w;
  if (tail_w) {
    const uint32_t m = min(m0 + threadIdx.x / 32u, a.M - 1u), c = min(threadIdx.x % 32u, tail_w - 1u);
    x_tail[threadIdx.x / 32u][threadIdx.x % 32u] = __half2float(a.x[(size_t)m * a.ldx + a.nb * kDim + c]);
  }
  const float scale = reinterpret_cast<const float*>(rec)[r];
  sum_t s[kReduceM];
#pragma unroll
  for (uint32_t k = 0; k < kReduceM; ++k) s[k] = 0;
  for (uint32_t p0 = 0; p0 < a.splits; p0 += kReduceSplits) {
    float v[kReduceSplits][kReduceM];
#pragma unroll
    for (uint32_t p = 0; p < kReduceSplits; ++p)
#pragma unroll
      for (uint32_t k = 0; k < kReduceM; ++k)
        v[p][k] = a.ws[((size_t)min(p0 + p, a.splits - 1u) * a.m_pad + min(m0 + k, a.M - 1u)) * n_rows + out_row];
#pragma unroll
    for (uint32_t p = 0; p < kReduceSplits; ++p)
#pragma unroll
      for (uint32_t k = 0; k < kReduceM; ++k) s[k] = p0 + p < a.splits ? s[k] + (sum_t)v[p][k] : s[k];
  }
  float out[kReduceM];
#pragma unroll
  for (uint32_t k = 0; k < kReduceM; ++k) out[k] = PAIR ? 0.f : (float)s[k] * scale;
  if (tail_w) {
    lds_barrier();
    for (uint32_t c0 = 0; c0 < tail_w; c0 += 8u) {
      float tw[8];
#pragma unroll
      for (uint32_t c = 0; c < 8u; ++c) tw[c] = reinterpret_cast<const float*>(rec + 32)[min(c0 + c, tail_w - 1u) * 8u + r];
#pragma unroll
      for (uint32_t c = 0; c < 8u; ++c)
        if (c0 + c < tail_w) {
#pragma unroll
          for (uint32_t k = 0; k < kReduceM; ++k) out[k] = fmaf(tw[c], x_tail[k][c0 + c], out[k]);
        }
    }
  }
  if (mine < n_rows && my_row < t.d_out) {
#pragma unroll
    for (uint32_t k = 0; k < kReduceM; ++k)
      if (m0 + k < a.M) store_y(t.y, (size_t)(m0 + k) * t.d_out + row, PAIR ? fmaf((float)s[k], scale, out[k]) : out[k], a.y_f32);
  }
}

}  // namespace llvq
