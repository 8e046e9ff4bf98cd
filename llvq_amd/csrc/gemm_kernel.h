// The batched product Y[M, d_out] = X[M, d_in] W^T on the matrix cores (M >= 2), over the tiles of tiles.h.  Included by
// llvq_hip.hip after it.  The reference runs a row loop of matrix-vector products (llvq-llm/src/model.rs:521-529).
//
// Weights are multiplied as binary16: v centroid[gain] / sqrt(16 shell) rounded once; sums are f32; row scale and tail
// columns are applied in f32 at the end.  A dword of a block's nibbles is eight consecutive columns of a row, which is
// exactly what a lane hands to a 16-deep (32 x 32) or 32-deep (16 x 16) product step, so a wavefront turns the 12 bytes
// its lanes load into its own fragments: no weights pass through LDS, and the order in which the products walk the
// columns is the order the blocks lie in (the lane groups of a fragment hold the same octet of two or four neighbouring
// blocks).  17 instructions per eight weights.
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
// A block's scale factors for a lane: an unpacked nibble is n in one half of a dword's nibble pairs and 16 n in the other.
struct BlockScale {
  float c, c16, odd;  // 2 s, s / 8, and s if the block's coordinates are odd
};
__device__ __forceinline__ BlockScale block_scale(uint32_t meta_dword, uint32_t r, uint32_t table) {
  const uint32_t meta = meta_dword >> (8u * (r & 3u));
  const float s = __int_as_float(__builtin_amdgcn_ds_bpermute((int)(meta & 0x7Cu), (int)table));
  return BlockScale{2.f * s, 0.125f * s, (meta & 1u) ? s : 0.f};
}
// One dword of nibbles -> eight weights.  1024 + u is a binary16 number whose low bits are u; taking 1032 away leaves
// n = u - 8 exactly (the nibble's top bit is flipped on the way: two's complement to offset), and 16 n likewise; one
// fused multiply-add in f32 per weight, rounded to binary16 once.
// The eight of those are one block of assembly: the compiler does not form them from source, and it does not know what
// an assembly statement does to the registers a matrix instruction reads, so the two wait states that are due between a
// vector write and that read stand at the block's end (and the halves of a register are written four apart).
__device__ __forceinline__ half8_t dequant_octet(uint32_t w, const BlockScale& s) {
  const uint32_t v = w >> 8;
  const uint32_t t[4] = {(w & 0x000F000Fu) ^ 0x64086408u, (w & 0x00F000F0u) ^ 0x64806480u, (v & 0x000F000Fu) ^ 0x64086408u, (v & 0x00F000F0u) ^ 0x64806480u};
  uint32_t n[4], o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const half2_t bias = (i & 1) ? half2_t{(_Float16)1152.f, (_Float16)1152.f} : half2_t{(_Float16)1032.f, (_Float16)1032.f};
    n[i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, t[i]) - bias);
  }
  asm("v_fma_mixlo_f16 %0, %4, %8, %10 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixlo_f16 %1, %5, %9, %10 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixlo_f16 %2, %6, %8, %10 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixlo_f16 %3, %7, %9, %10 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %0, %4, %8, %10 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %1, %5, %9, %10 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %2, %6, %8, %10 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %3, %7, %9, %10 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
      "s_nop 1"
      : "=&v"(o[0]), "=&v"(o[1]), "=&v"(o[2]), "=&v"(o[3])
      : "v"(n[0]), "v"(n[1]), "v"(n[2]), "v"(n[3]), "v"(s.c), "v"(s.c16), "v"(s.odd));
  return __builtin_bit_cast(half8_t, o);
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
template <int RG, int MT>
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
  const uint32_t table = reinterpret_cast<const uint32_t*>(t.base)[lane & 31u];
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
  acc4_t acc[RG][MT];
#pragma unroll
  for (int k = 0; k < RG; ++k)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[k][mt] = acc4_t{0.f, 0.f, 0.f, 0.f};
  for (; q < n_quads; q += 16u) {
    const uint32_t qn = q + 16u;
    const bool live = qn < n_quads;
    BlockScale s[RG];
#pragma unroll
    for (int k = 0; k < RG; ++k) s[k] = block_scale(W[k].meta, r, table);
#pragma unroll
    for (uint32_t j = 0; j < 3; ++j) {
      half8_t w[RG];
#pragma unroll
      for (int k = 0; k < RG; ++k) w[k] = dequant_octet(j == 0 ? W[k].w0 : j == 1 ? W[k].w1 : W[k].w2, s[k]);
      // a register is asked for again as soon as its contents are used, and not moved from there
      if (j == 2u) {
        __builtin_amdgcn_sched_barrier(0);
        load_w(qn, live);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int k = 0; k < RG; ++k)
          acc[k][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, X[j][mt]), w[k], acc[k][mt], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      load_x(j, qn, live);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (op_col < a.tail_w) tw[op_row * 24u + op_col] = op_w;
  else if (op_col == 24u) scale_s[op_row] = op_w;
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
      *reinterpret_cast<acc4_t*>(part + (((wave * RG + k) * MT + mt) * 64u + lane) * 4u) = acc[k][mt];
  __syncthreads();
  for (uint32_t o = tid; o < kRows * kCols; o += 1024u) {
    const uint32_t row = o % kRows, m = o / kRows;
    if (m >= a.M || t.row0 + row >= t.d_out) continue;
    const uint32_t l = (row & 15u) + 16u * ((m & 15u) >> 2), e = m & 3u;
    const float* p = part + (((row >> 4) * MT + (m >> 4)) * 64u + l) * 4u + e;
    float s = 0.f;
#pragma unroll
    for (uint32_t k = 0; k < 16; ++k) s += p[k * RG * MT * 256];
    float tl = 0.f;
    for (uint32_t c = 0; c < a.tail_w; ++c) tl = fmaf(tw[row * 24u + c], tx[m * 24u + c], tl);
    store_y(t.y, (size_t)m * t.d_out + t.row0 + row, fmaf(s, scale_s[row], tl), a.y_f32);
  }
}
template <int RG, int MT>
__host__ constexpr size_t gemm_small_lds() { return (size_t)(16 * RG * MT * 256 + RG * 16 * 25 + MT * 16 * 24) * 4; }
static_assert(gemm_small_lds<2, 4>() <= 160 * 1024, "partial sums of sixteen wavefronts fit a CU's LDS");

// ---- more activation rows ----------------------------------------------------------------------------
// What bounds it: the matrix cores (a 64 x 128 tile of a wavefront is 24 steps of 32 cycles per 48 columns, its two
// weight fragments 120 vector instructions beside them).  A workgroup of four wavefronts takes 64 (4 / WM) weight rows by
// 128 WM activation rows: each wavefront unpacks its own 64 rows (two 32-row fragments, from memory to registers) against
// 128 activation rows (four fragments, from LDS, which the workgroup fills a step of 48 columns ahead from the octets,
// whose order is the fragments' own: a run of 512 bytes each).  128 accumulators and a step's operands fit 256 registers,
// so two workgroups share a CU and one unpacks while the other multiplies.
// Launches with too few tiles to fill the chip split the columns (`splits`): partial sums go to the workspace and
// gemm_reduce_kernel adds them in order; otherwise the tile is finished here.
constexpr uint32_t kWideStepBlocks = 2;  // blocks per step: the halves of a wavefront hold one each
template <int WM>
__host__ __device__ constexpr uint32_t gemm_wide_rows() { return 64u * (4u / WM); }
template <int WM>
__host__ __device__ constexpr uint32_t gemm_wide_cols() { return 128u * WM; }

// Sixteen results of a lane (one weight row, activation rows 8 (e / 4) + e % 4 from m on) into y.
template <typename Y>
__device__ __forceinline__ void store_fragment(Y* y, uint32_t ldy, const acc16_t& v, uint32_t m, uint32_t M) {
#pragma unroll
  for (uint32_t e = 0; e < 16; ++e) {
    const uint32_t me = m + 8u * (e >> 2) + (e & 3u);
    if (me < M) y[(size_t)me * ldy] = (Y)v[e];
  }
}

template <int WM>
__global__ __launch_bounds__(256, 2) void gemm_wide_kernel(GemmArgs a) {
  constexpr uint32_t kCols = gemm_wide_cols<WM>(), kRows = gemm_wide_rows<WM>();
  constexpr uint32_t kPieces = kCols * 6u;            // 16-byte pieces of a step: two blocks of three octets
  constexpr uint32_t kPer = kPieces / 256u;           // of them a lane moves to LDS
  extern __shared__ __align__(16) uint8_t smem[];
  u32x4_t* buf = reinterpret_cast<u32x4_t*>(smem);    // [2][2 blocks][3 octets][kCols]
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t l32 = lane & 31u, h = lane >> 5, r = lane & 7u;
  const uint32_t wm = wave % WM, wr = wave / WM;
  // tiles of one row group are neighbours in the grid: they read the same weights
  const uint32_t mt = blockIdx.x % a.m_tiles, rest = blockIdx.x / a.m_tiles;
  const uint32_t tile = rest % a.n_tiles, split = rest / a.n_tiles;
  const uint32_t nb = a.nb, stride = tile_stride(nb, a.tail_w), head = tile_head_bytes(a.tail_w);
  const GemmTile t = gemm_tile_at(a, tile, kRows);
  const uint32_t row0 = t.row0 + wr * 64u;            // this wavefront's first row
  const uint32_t n_rec = tile_count(t.d_out);
  const uint8_t* recs = t.base + kTileTableBytes;
  const uint32_t table = reinterpret_cast<const uint32_t*>(t.base)[lane & 31u];
  const uint32_t n_steps = (nb + 1u) >> 1;
  const uint32_t s0 = split * a.steps_per_split, s1 = min(s0 + a.steps_per_split, n_steps);
  // records past the matrix's last repeat it: their rows are not stored
  const uint32_t rec0 = min(row0 / kTileRows, n_rec - 1u);
  const uint8_t* wave_rec = recs + (size_t)rec0 * stride;
  uint32_t rec_off[2];
#pragma unroll
  for (uint32_t k = 0; k < 2; ++k) rec_off[k] = (min(row0 / kTileRows + k * 4u + (l32 >> 3), n_rec - 1u) - rec0) * stride;
  const uint32_t in_step = head + h * kTileBlockBytes;
  const uint32_t w_off[2] = {rec_off[0] + in_step + r * 12u, rec_off[1] + in_step + r * 12u};
  const uint32_t meta_off[2] = {rec_off[0] + in_step + 96u + (r & 4u), rec_off[1] + in_step + 96u + (r & 4u)};

  struct __attribute__((packed, aligned(4))) W3 { uint32_t w[3]; };
  StepWords Wa[2], Wb[2];  // of the even and the odd steps
  u32x4_t pre[kPer];
  // piece p of a step: octet p / kCols of the step's six, activation row p % kCols of the tile
  const uint8_t* xt = reinterpret_cast<const uint8_t*>(a.xt + (size_t)mt * kCols);
  uint32_t x_off[kPer];
#pragma unroll
  for (uint32_t i = 0; i < kPer; ++i) x_off[i] = ((tid + i * 256u) / kCols * a.m_pad + (tid + i * 256u) % kCols) * 16u;
  auto load_x = [&](uint32_t s) __attribute__((always_inline)) {
    const uint8_t* xs = uniform_global(xt + (size_t)s * 6u * a.m_pad * 16u);
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) pre[i] = *reinterpret_cast<const u32x4_t*>(xs + lane_offset(x_off[i]));
  };
  auto load_w = [&](StepWords (&W)[2], uint32_t s) __attribute__((always_inline)) {
    const uint8_t* ws = uniform_global(wave_rec + s * (2u * kTileBlockBytes));
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const W3 w = *reinterpret_cast<const W3*>(ws + lane_offset(w_off[k]));
      W[k] = StepWords{w.w[0], w.w[1], w.w[2], *reinterpret_cast<const uint32_t*>(ws + lane_offset(meta_off[k]))};
    }
  };
  acc16_t acc[2][4];
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[k][c][e] = 0.f;
  // One step: the octets fetched during the one before go to LDS, those of the next are fetched, and so are the weights
  // two steps on once this step's are unpacked.
  auto step = [&](StepWords (&W)[2], uint32_t s, u32x4_t* b) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) b[tid + i * 256u] = pre[i];
    lds_barrier();  // (the other buffer was last read before the previous barrier)
    __builtin_amdgcn_sched_barrier(0);
    load_x(min(s + 1u, s1 - 1u));
    __builtin_amdgcn_sched_barrier(0);
    BlockScale sc[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) sc[k] = block_scale(W[k].meta, r, table);
    const u32x4_t* bx = b + h * 3u * kCols + wm * 128u + l32;
    half8_t w[2];
#pragma unroll
    for (uint32_t j = 0; j < 3; ++j) {
      half8_t x[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) x[c] = __builtin_bit_cast(half8_t, bx[j * kCols + (uint32_t)c * 32u]);
#pragma unroll
      for (int k = 0; k < 2; ++k) w[k] = dequant_octet(j == 0 ? W[k].w0 : j == 1 ? W[k].w1 : W[k].w2, sc[k]);
      if (j == 2u) {
        __builtin_amdgcn_sched_barrier(0);
        load_w(W, min(s + 2u, s1 - 1u));
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[k][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[c], w[k], acc[k][c], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  load_x(s0);
  __builtin_amdgcn_sched_barrier(0);
  load_w(Wa, s0);
  load_w(Wb, min(s0 + 1u, s1 - 1u));
  for (uint32_t s = s0;;) {
    step(Wa, s, buf);
    if (++s >= s1) break;
    step(Wb, s, buf + kPieces);
    if (++s >= s1) break;
  }
  // element e of a lane: activation row 8 (e / 4) + 4 h + e % 4 of the fragment, weight row l32 of it
  const uint32_t m0 = mt * kCols + wm * 128u;
  if (a.splits > 1u) {
    const uint32_t n_rows = a.n_tiles * kRows;
    float* out = a.ws + (size_t)split * a.m_pad * n_rows + tile * kRows + wr * 64u + l32;
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int c = 0; c < 4; ++c) store_fragment(out + k * 32, n_rows, acc[k][c], m0 + (uint32_t)c * 32u + 4u * h, a.M);
    return;
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const float* rec = reinterpret_cast<const float*>(wave_rec + rec_off[k]);
    const float scale = rec[r];
    const uint32_t row = row0 + (uint32_t)k * 32u + l32;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      acc16_t v = acc[k][c];
#pragma unroll
      for (int e = 0; e < 16; ++e) v[e] *= scale;
      // f32 tail columns, two at a time: lane half h holds column i + h
      const __half* tx = a.x + (size_t)min(m0 + (uint32_t)c * 32u + l32, a.M - 1u) * a.ldx + nb * kDim;
      for (uint32_t i = 0; i < a.tail_w; i += 2u) {
        const uint32_t col = min(i + h, a.tail_w - 1u);
        const float keep = i + h < a.tail_w ? 1.f : 0.f;
        v = __builtin_amdgcn_mfma_f32_32x32x2f32(__half2float(tx[col]), keep * rec[8u + col * 8u + r], v, 0, 0, 0);
      }
      if (row >= t.d_out) continue;
      const uint32_t m = m0 + (uint32_t)c * 32u + 4u * h;
      if (a.y_f32) store_fragment(reinterpret_cast<float*>(t.y) + row, t.d_out, v, m, a.M);
      else store_fragment(reinterpret_cast<_Float16*>(t.y) + row, t.d_out, v, m, a.M);
    }
  }
}
template <int WM>
__host__ constexpr size_t gemm_wide_lds() { return 2ull * gemm_wide_cols<WM>() * 6 * 16; }

// The partial sums of the column splits, added in order; row scale and tail columns.  A lane takes one weight row and
// kReduceM activation rows, so that the row's tail is read once for them.
constexpr uint32_t kReduceM = 8;
struct GemmReduceArgs {
  GemmArgs g;
  uint32_t rows_per_tile, row_chunks;
};
__global__ __launch_bounds__(256) void gemm_reduce_kernel(GemmReduceArgs ra) {
  const GemmArgs& a = ra.g;
  const uint32_t n_rows = a.n_tiles * ra.rows_per_tile;
  const uint32_t chunk = blockIdx.x % ra.row_chunks, m0 = blockIdx.x / ra.row_chunks * kReduceM;
  const uint32_t out_row = chunk * 256u + threadIdx.x;
  if (out_row >= n_rows) return;
  const GemmTile t = gemm_tile_at(a, out_row / ra.rows_per_tile, ra.rows_per_tile);
  const uint32_t row = t.row0 + out_row % ra.rows_per_tile;
  if (row >= t.d_out) return;
  const uint32_t stride = tile_stride(a.nb, a.tail_w);
  const uint8_t* rec = t.base + kTileTableBytes + (size_t)(row / kTileRows) * stride;
  const uint32_t r = row & 7u;
  float s[kReduceM];
#pragma unroll
  for (uint32_t k = 0; k < kReduceM; ++k) s[k] = 0.f;
  for (uint32_t p = 0; p < a.splits; ++p)
#pragma unroll
    for (uint32_t k = 0; k < kReduceM; ++k) s[k] += a.ws[((size_t)p * a.m_pad + min(m0 + k, a.M - 1u)) * n_rows + out_row];
  const float scale = reinterpret_cast<const float*>(rec)[r];
#pragma unroll
  for (uint32_t k = 0; k < kReduceM; ++k) s[k] *= scale;
  for (uint32_t c = 0; c < a.tail_w; ++c) {
    const float tw = reinterpret_cast<const float*>(rec + 32)[c * 8u + r];
#pragma unroll
    for (uint32_t k = 0; k < kReduceM; ++k) s[k] = fmaf(tw, __half2float(a.x[(size_t)min(m0 + k, a.M - 1u) * a.ldx + a.nb * kDim + c]), s[k]);
  }
#pragma unroll
  for (uint32_t k = 0; k < kReduceM; ++k)
    if (m0 + k < a.M) store_y(t.y, (size_t)(m0 + k) * t.d_out + row, s[k], a.y_f32);
}

}  // namespace llvq
