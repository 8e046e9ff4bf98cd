// Batch-1 greedy decode loop of a Qwen3-architecture model whose seven
// projections per layer are LLVQ matrices: the counterpart of
// Block::forward_cached / Qwen3::hidden_cached / Qwen3::generate
// (llvq-llm/src/model.rs:766-835, :968-982, :1041-1073) at l = 1.
// Included by llvq_hip.hip after the GEMV launcher it drives.
//
// Everything between two projections runs in small hand-written kernels on the
// runtime's stream; the token chosen at one step is read by the next step's
// embedding kernel from device memory, so the host never waits inside a
// generation.  Activations between kernels are binary16 (the run dtype of the
// reference); every kernel computes in f32 and rounds once on output:
//   embed -> h
//   [per layer] add + RMSNorm -> qkv GEMV group -> per-head RMSNorm + RoPE +
//   cache append -> attention over the cache -> o GEMV -> add + RMSNorm ->
//   gate/up GEMV group -> SiLU(gate) * up -> down GEMV
//   add + final RMSNorm -> f16 lm_head GEMV (logits rounded to binary16, as the
//   reference's f16 matmul leaves them) -> argmax, lowest index on ties.
#pragma once

namespace llvq {

// Eight binary16 values per lane of a row's workgroup (rows of up to 8192, a multiple of 8).
__host__ inline uint32_t norm_threads(uint32_t n) { return (n / 8u + 63u) / 64u * 64u; }

// h[row] = embed[token[row]], row = blockIdx.y (token null: the one token `value`)
__global__ __launch_bounds__(256) void embed_kernel(const __half* __restrict__ table, const uint32_t* __restrict__ token, uint32_t value,
                                                    uint32_t vocab, uint32_t hidden, __half* __restrict__ h) {
  const uint32_t t = min(token ? token[blockIdx.y] : value, vocab - 1u);
  h += (size_t)blockIdx.y * hidden;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < hidden; i += gridDim.x * blockDim.x)
    h[i] = table[(size_t)t * hidden + i];
}

// r = f16(h + delta) when delta is given (else h), written to h_out when that is given
// (it may be h itself); normed = f16(r / sqrt(mean(r^2) + eps) * w)
// (candle_nn::RmsNorm: f32 inside, one rounding on the way out).
// One workgroup of norm_threads(n) lanes per row of n values; 16 bytes of an operand per lane: with two bytes, and four
// wavefronts where one has work, 500 rows of 2560 took 5.2 us.
// (A prompt's passes: the launches that brought rows into octets are gone, 500 tokens through twelve 4B layers 3215 -> 3067 us.)
// to: the normed rows go there as octets (a workgroup for each of m_pad rows), and only their tail columns to `normed`.
// sums: delta is what a product left in parts, added up and rounded here.
__global__ __launch_bounds__(1024) void add_rmsnorm_kernel(const __half* h, const __half* __restrict__ delta, const __half* __restrict__ w,
                                                           __half* h_out, __half* __restrict__ normed, uint32_t n, float eps, Octets to, GemmSums sums) {
  __shared__ float red[16];
  const uint32_t at = threadIdx.x * 8u, lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  uint32_t m = blockIdx.x;
  if (to.xt) {
    m = octet_row(m, to.m_pad);
    for (uint32_t o = (m < to.rows ? to.kcols / 8u : 0u) + threadIdx.x; o < to.n_oct; o += blockDim.x) to.xt[(size_t)o * to.m_pad + m] = make_uint4(0, 0, 0, 0);
    if (m >= to.rows) return;
  }
  const size_t row = (size_t)m * n;
  const bool in = at < n;
  const uint32_t from = in ? at : 0u;
  HalfOctet x = *reinterpret_cast<const HalfOctet*>(h + row + from);
  const HalfOctet g = *reinterpret_cast<const HalfOctet*>(w + from);
  if (delta || sums.ws) {  // the residual stream is binary16
    HalfOctet d;
    if (sums.ws) {
      float v[8];
      parts_read(sums, m, sums.first[0] + from, v);
#pragma unroll
      for (int j = 0; j < 4; ++j) d.w[j] = pack_halves(v[2 * j], v[2 * j + 1]);
    } else {
      d = *reinterpret_cast<const HalfOctet*>(delta + row + from);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      x.w[j] = (uint32_t)__half_as_ushort(__float2half_rn(half_lo(x.w[j]) + half_lo(d.w[j]))) |
               (uint32_t)__half_as_ushort(__float2half_rn(half_hi(x.w[j]) + half_hi(d.w[j]))) << 16;
  }
  if (h_out && in) *reinterpret_cast<HalfOctet*>(h_out + row + at) = x;
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) ss = fmaf(half_lo(x.w[j]), half_lo(x.w[j]), fmaf(half_hi(x.w[j]), half_hi(x.w[j]), ss));
  ss = wave_sum(in ? ss : 0.f);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  float total = 0.f;
  for (uint32_t k = 0; k < (blockDim.x >> 6); ++k) total += red[k];  // same order in every lane
  const float inv = 1.0f / sqrtf(total / (float)n + eps);
  if (!in) return;
  HalfOctet o;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    o.w[j] = (uint32_t)__half_as_ushort(__float2half_rn(half_lo(x.w[j]) * inv * half_lo(g.w[j]))) |
             (uint32_t)__half_as_ushort(__float2half_rn(half_hi(x.w[j]) * inv * half_hi(g.w[j]))) << 16;
  if (to.xt && at < to.kcols) to.xt[(size_t)threadIdx.x * to.m_pad + m] = make_uint4(o.w[0], o.w[1], o.w[2], o.w[3]);
  else *reinterpret_cast<HalfOctet*>(normed + row + at) = o;
}

// int8 KV cache (llvq-llm/src/kvq.rs:110-165): asymmetric 8-bit codes per group
// of 64 along head_dim, binary16 scale and bias, chosen from the token alone:
//   s = f16((max - min) / 255), b = f16(min), q = clamp(round((x - b) / (s > 0 ? s : 1)), 0, 255)
// and a reader gets back f16(q s + b).  The reference keeps that reconstructed
// value in its cache; here the codes themselves are stored (1.06 bytes per
// value instead of 2) and the same value is rebuilt on every read.
constexpr uint32_t kKvGroup = 64;
struct KvQ8 {
  uint8_t* kq;    // [n_kv][max_pos][head_dim]
  uint8_t* vq;
  __half* ks;     // [n_kv][max_pos][head_dim / 64] scales
  __half* kb;     //                                biases
  __half* vs;
  __half* vb;
};

// One group of 64 values held one per lane -> code, scale, bias.  (The extremes by lane moves: by __shfl_xor, an LDS instruction each, the twelve
// steps of a group were a microsecond of the decode attention's launch.)
__device__ __forceinline__ uint8_t kv_quantize_group(float x, __half* s_out, __half* b_out) {
  const float mn = wave_best(x, [](float a, float b) { return fminf(a, b); }), mx = wave_best(x, [](float a, float b) { return fmaxf(a, b); });
  const __half sh = __float2half_rn(__fdiv_rn(__fsub_rn(mx, mn), 255.0f));
  const __half bh = __float2half_rn(mn);
  const float s = __half2float(sh), b = __half2float(bh);
  const float safe = s > 0.f ? s : 1.0f;
  const float q = fminf(fmaxf(roundf(__fdiv_rn(__fsub_rn(x, b), safe)), 0.f), 255.f);
  *s_out = sh;
  *b_out = bh;
  return (uint8_t)q;
}

// (q s is exact in f32, 8 bits by 11: the fused operation rounds where the sum alone did.)
__device__ __forceinline__ float kv_dequant(uint32_t q, float s, float b) {
  return __half2float(__float2half_rn(fmaf((float)q, s, b)));
}

// One wavefront: per-head RMSNorm of a q or k head (model.rs:800-808), then RoPE at
// the absolute position in the rotate-half convention (candle_nn::rotary_emb::rope:
// out[i] = x[i] cos - x[i + d/2] sin, out[i + d/2] = x[i] sin + x[i + d/2] cos, with
// the binary16 cos/sin tables of Rotary::new, model.rs:163-179).  Each step rounds to
// binary16 as the reference's tensors do; the results are left, widened, in
// stage[0, head_dim) — an LDS area of this wavefront alone.  head_dim <= 256 (the callers take 128).
__device__ __forceinline__ void wave_lds_sync() {
  // LDS operations of one wavefront execute in order; only the compiler must not move them
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
// The served width, head_dim = 128: a lane's two elements (lane, lane + 64) are a rotation pair, so nothing crosses lanes but
// the sum of squares, and a caller can request the operands of several heads before it finishes the first.
struct HeadOperands { __half x1, x2, w1, w2; };
struct RopeAngle { __half c, s; };
__device__ __forceinline__ HeadOperands head_operands_128(const __half* __restrict__ src, const __half* __restrict__ w, uint32_t a, uint32_t b) {
  return HeadOperands{src[a], src[b], w[a], w[b]};
}
__device__ __forceinline__ float2 norm_rope_128(const HeadOperands& h, const RopeAngle& a, float eps) {
  const float x1 = __half2float(h.x1), x2 = __half2float(h.x2), c = __half2float(a.c), sn = __half2float(a.s);
  const float ss = wave_sum(x1 * x1 + x2 * x2);
  const float inv = 1.0f / sqrtf(ss / 128.0f + eps);
  const float n1 = __half2float(__float2half_rn(x1 * inv * __half2float(h.w1))), n2 = __half2float(__float2half_rn(x2 * inv * __half2float(h.w2)));
  return make_float2(__half2float(__float2half_rn(n1 * c - n2 * sn)), __half2float(__float2half_rn(n1 * sn + n2 * c)));
}
__device__ __forceinline__ void norm_rope_wave(const __half* __restrict__ src, const __half* __restrict__ w,
                                               const __half* __restrict__ cos_t, const __half* __restrict__ sin_t,
                                               uint32_t pos, uint32_t head_dim, float eps, float* stage, uint32_t lane) {
  const uint32_t half_d = head_dim >> 1;
  if (head_dim == 128) {
    const float2 r = norm_rope_128(head_operands_128(src, w, lane, lane + 64u), RopeAngle{cos_t[(size_t)pos * 64 + lane], sin_t[(size_t)pos * 64 + lane]}, eps);
    stage[lane] = r.x;
    stage[lane + 64] = r.y;
    wave_lds_sync();
    return;
  }
  float x[4];  // elements lane, lane + 64, lane + 128, lane + 192
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t i = lane + 64u * j;
    x[j] = i < head_dim ? __half2float(src[i]) : 0.f;
    ss += x[j] * x[j];
  }
  ss = wave_sum(ss);
  const float inv = 1.0f / sqrtf(ss / (float)head_dim + eps);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t i = lane + 64u * j;
    if (i < head_dim) stage[i] = __half2float(__float2half_rn(x[j] * inv * __half2float(w[i])));
  }
  wave_lds_sync();
  float r1[2], r2[2];  // rotated pairs (i, i + d/2) for i = lane, lane + 64
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const uint32_t i = lane + 64u * j;
    r1[j] = r2[j] = 0.f;
    if (i < half_d) {
      const float c = __half2float(cos_t[(size_t)pos * half_d + i]), sn = __half2float(sin_t[(size_t)pos * half_d + i]);
      const float x1 = stage[i], x2 = stage[i + half_d];
      r1[j] = __half2float(__float2half_rn(x1 * c - x2 * sn));
      r2[j] = __half2float(__float2half_rn(x1 * sn + x2 * c));
    }
  }
  wave_lds_sync();
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const uint32_t i = lane + 64u * j;
    if (i < half_d) {
      stage[i] = r1[j];
      stage[i + half_d] = r2[j];
    }
  }
  wave_lds_sync();
}

// What the attention launch is handed about the position being decoded: the raw
// q / k / v rows the projections left, the layer's q and k norm weights and the
// rotary tables.  The launch norms and rotates its own query heads, and the one
// workgroup whose range ends at the new position does the same for k, appends
// k and v to the cache and uses them from LDS.
struct AttnNew {
  const __half* q_raw;  // [n_heads, head_dim]
  const __half* k_raw;  // [n_kv, head_dim]
  const __half* v_raw;  // [n_kv, head_dim]
  const __half* qn;     // [head_dim]
  const __half* kn;     // [head_dim]
  const __half* cos_t;  // [max_pos, head_dim / 2]
  const __half* sin_t;
  __half* kcache;       // this layer's binary16 cache (null with the int8 cache)
  __half* vcache;
  float eps;
};

constexpr int kAttnThreads = 256;
constexpr int kAttnWaves = kAttnThreads / 64;
constexpr uint32_t kAttnClasses = 4 * kAttnWaves;  // position classes of a workgroup, 16 lanes each
constexpr int kAttnRows = 4;                       // positions of a class whose rows are requested together
constexpr int kAttnMaxSplits = 64;  // the cache is cut into at most this many ranges (host picks by length; 128 was measured slower at 8188 positions)
constexpr int kAttnMaxGroup = 8;    // query heads per kv head
constexpr int kAttnInlineSplits = 16;  // up to this many ranges, the workgroup that finishes last merges them itself

// ---- rows of positions at once (prompt processing through the batched product) ----
// One wavefront per (head, row), four to a workgroup: q heads are normed and rotated in place, k heads are
// normed, rotated and appended to the cache at position pos0 + row, v heads are appended.
// Grid (a quarter of n_heads + 2 n_kv, rows).  Same arithmetic as the one-position path.
// sums: heads of 128 come as what the product left in parts, and are added up and rounded here.
template <bool Q8>
__global__ __launch_bounds__(256) void norm_rope_append_rows_kernel(__half* __restrict__ q, const __half* __restrict__ k,
                                                                   const __half* __restrict__ v, AttnNew nw, KvQ8 q8,
                                                                   uint32_t n_heads, uint32_t n_kv, uint32_t head_dim,
                                                                   uint32_t pos0, uint32_t max_pos, GemmSums sums) {
  __shared__ float stages[4][256];
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t head = blockIdx.x * 4u + wave, row = blockIdx.y, lane = threadIdx.x & 63u;
  if (head >= n_heads + 2u * n_kv) return;
  float* stage = stages[wave];
  const uint32_t pos = pos0 + row, kvgroups = head_dim / kKvGroup;
  __half x1{}, x2{};  // of sums: elements lane and lane + 64
  const auto from_sums = [&](const __half* w) {
    const RopeAngle a{nw.cos_t[(size_t)pos * 64 + lane], nw.sin_t[(size_t)pos * 64 + lane]};
    const float2 r = norm_rope_128(HeadOperands{x1, x2, w[lane], w[lane + 64]}, a, nw.eps);
    stage[lane] = r.x;
    stage[lane + 64] = r.y;
    wave_lds_sync();
  };
  if (sums.ws) {
    const uint32_t of = head < n_heads ? head : head < n_heads + n_kv ? head - n_heads : head - n_heads - n_kv;
    const uint32_t first = head < n_heads ? sums.first[0] : head < n_heads + n_kv ? sums.first[1] : sums.first[2];
    const float* from = uniform_global(sums.ws + (size_t)row * sums.ld + first + of * 128u);
    const size_t step = (size_t)sums.m_pad * sums.ld;
    float a = 0.f, b = 0.f;
    for (uint32_t p0 = 0; p0 < sums.splits; p0 += kReduceSplits) {
      float va[kReduceSplits], vb[kReduceSplits];
#pragma unroll
      for (uint32_t p = 0; p < kReduceSplits; ++p) {
        const float* at = from + min(p0 + p, sums.splits - 1u) * step;
        va[p] = at[lane];
        vb[p] = at[lane + 64u];
      }
#pragma unroll
      for (uint32_t p = 0; p < kReduceSplits; ++p) {
        if (p0 + p >= sums.splits) break;
        a += va[p];
        b += vb[p];
      }
    }
    x1 = __float2half_rn(a);
    x2 = __float2half_rn(b);
  }
  if (head < n_heads) {
    __half* qh = q + ((size_t)row * n_heads + head) * head_dim;
    if (sums.ws) from_sums(nw.qn);
    else norm_rope_wave(qh, nw.qn, nw.cos_t, nw.sin_t, pos, head_dim, nw.eps, stage, lane);
    for (uint32_t i = lane; i < head_dim; i += 64) qh[i] = __float2half_rn(stage[i]);
    return;
  }
  const bool is_k = head < n_heads + n_kv;
  const uint32_t kvh = is_k ? head - n_heads : head - n_heads - n_kv;
  const __half* src = (is_k ? k : v) + ((size_t)row * n_kv + kvh) * head_dim;
  if (is_k && sums.ws) from_sums(nw.kn);
  else if (is_k) norm_rope_wave(src, nw.kn, nw.cos_t, nw.sin_t, pos, head_dim, nw.eps, stage, lane);
  else {
    if (sums.ws) {
      stage[lane] = __half2float(x1);
      stage[lane + 64] = __half2float(x2);
    } else {
      for (uint32_t i = lane; i < head_dim; i += 64) stage[i] = __half2float(src[i]);
    }
    wave_lds_sync();
  }
  const size_t crow = (size_t)kvh * max_pos + pos;
  if constexpr (Q8) {
    uint8_t* cq = is_k ? q8.kq : q8.vq;
    __half* cs = is_k ? q8.ks : q8.vs;
    __half* cb = is_k ? q8.kb : q8.vb;
    for (uint32_t g = 0; g < kvgroups; ++g) {
      __half sh, bh;
      const uint8_t code = kv_quantize_group(stage[g * kKvGroup + lane], &sh, &bh);
      cq[crow * head_dim + g * kKvGroup + lane] = code;
      if (lane == 0) {
        cs[crow * kvgroups + g] = sh;
        cb[crow * kvgroups + g] = bh;
      }
    }
  } else {
    __half* dst = (is_k ? nw.kcache : nw.vcache) + crow * head_dim;
    for (uint32_t i = lane; i < head_dim; i += 64) dst[i] = __float2half_rn(stage[i]);
  }
}

// Causal attention of a row of queries over the cache (model.rs:812-822 with the mask of
// :938-960): one wavefront per (kv head, row) serves every query head of the group; the
// query at row r sees positions 0 .. pos0 + r.  Lane (pj, sub) = (lane / 16, lane % 16)
// holds dims [8 sub, 8 sub + 8) of the positions j = pj (mod 4); each of the four position
// classes keeps its own running maximum, sum and weighted V sum (f32), merged at the end.
// head_dim <= 128, a multiple of 8; G >= query heads per kv head sizes the register arrays.  q is already normed and rotated; ctx is rounded once.
template <bool Q8, int G>
__global__ __launch_bounds__(64) void attn_rows_kernel(const __half* __restrict__ q, const __half* __restrict__ kcache,
                                                       const __half* __restrict__ vcache, KvQ8 q8, __half* __restrict__ ctx,
                                                       uint32_t n_heads, uint32_t n_kv, uint32_t head_dim, uint32_t pos0,
                                                       uint32_t max_pos, float scale) {
  const uint32_t kvh = blockIdx.x, row = blockIdx.y, lane = threadIdx.x;
  const uint32_t groups = n_heads / n_kv, T = pos0 + row + 1;
  const uint32_t sub = lane & 15u, pj = lane >> 4, i0 = sub * 8u;
  const bool active = i0 < head_dim;
  const uint32_t kvgroups = head_dim / kKvGroup;
  const size_t base = (size_t)kvh * max_pos;
  float qv[G][8], acc[G][8], m[G], l[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    m[g] = -INFINITY;
    l[g] = 0.f;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      acc[g][t] = 0.f;
      qv[g][t] = ((uint32_t)g < groups && active)
                     ? __half2float(q[((size_t)row * n_heads + kvh * groups + g) * head_dim + i0 + t]) * scale
                     : 0.f;
    }
  }
  // U positions of this lane's class per pass: their rows are requested together, then used in order
  constexpr int U = 4;
  for (uint32_t jb = pj; jb < T; jb += 4 * U) {
    uint4 kraw[U], vraw[U];
    float ks[U], kb[U], vs[U], vb[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t j = jb + 4u * u;
      kraw[u] = vraw[u] = make_uint4(0, 0, 0, 0);
      ks[u] = kb[u] = vs[u] = vb[u] = 0.f;
      if (active && j < T) {
        if constexpr (Q8) {
          const uint2 kc = *reinterpret_cast<const uint2*>(q8.kq + (base + j) * head_dim + i0);
          const uint2 vc = *reinterpret_cast<const uint2*>(q8.vq + (base + j) * head_dim + i0);
          const size_t gi = (base + j) * kvgroups + i0 / kKvGroup;
          kraw[u].x = kc.x; kraw[u].y = kc.y;
          vraw[u].x = vc.x; vraw[u].y = vc.y;
          ks[u] = __half2float(q8.ks[gi]); kb[u] = __half2float(q8.kb[gi]);
          vs[u] = __half2float(q8.vs[gi]); vb[u] = __half2float(q8.vb[gi]);
        } else {
          kraw[u] = *reinterpret_cast<const uint4*>(kcache + (base + j) * head_dim + i0);
          vraw[u] = *reinterpret_cast<const uint4*>(vcache + (base + j) * head_dim + i0);
        }
      }
    }
    // scores of the U positions first (independent exchanges), then the running sums in order
    float sc[U][G], vfs[U][8];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float kf[8];
      if constexpr (Q8) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          kf[t] = kv_dequant((kraw[u].x >> (8 * t)) & 0xFFu, ks[u], kb[u]);
          kf[4 + t] = kv_dequant((kraw[u].y >> (8 * t)) & 0xFFu, ks[u], kb[u]);
          vfs[u][t] = kv_dequant((vraw[u].x >> (8 * t)) & 0xFFu, vs[u], vb[u]);
          vfs[u][4 + t] = kv_dequant((vraw[u].y >> (8 * t)) & 0xFFu, vs[u], vb[u]);
        }
      } else {
        const uint32_t kw[4] = {kraw[u].x, kraw[u].y, kraw[u].z, kraw[u].w}, vw[4] = {vraw[u].x, vraw[u].y, vraw[u].z, vraw[u].w};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          kf[2 * t] = __half2float(__ushort_as_half((unsigned short)(kw[t] & 0xFFFFu)));
          kf[2 * t + 1] = __half2float(__ushort_as_half((unsigned short)(kw[t] >> 16)));
          vfs[u][2 * t] = __half2float(__ushort_as_half((unsigned short)(vw[t] & 0xFFFFu)));
          vfs[u][2 * t + 1] = __half2float(__ushort_as_half((unsigned short)(vw[t] >> 16)));
        }
      }
      if (!active) {
#pragma unroll
        for (int t = 0; t < 8; ++t) kf[t] = vfs[u][t] = 0.f;
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float d = 0.f;
#pragma unroll
        for (int t = 0; t < 8; ++t) d = fmaf(qv[g][t], kf[t], d);
        sc[u][g] = row16_sum(d);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (jb + 4u * u < T) {
#pragma unroll
        for (int g = 0; g < G; ++g)
          if ((uint32_t)g < groups) {
            const float d = sc[u][g];
            const float mn = fmaxf(m[g], d);
            const float c = __expf(m[g] - mn), p = __expf(d - mn);  // c = 0 on the first position (m = -inf)
            l[g] = fmaf(l[g], c, p);
#pragma unroll
            for (int t = 0; t < 8; ++t) acc[g][t] = fmaf(acc[g][t], c, p * vfs[u][t]);
            m[g] = mn;
          }
      }
  }
  // merge the four position classes (a class with no position has m = -inf and weight 0)
#pragma unroll
  for (int off = 16; off <= 32; off <<= 1)
#pragma unroll
    for (int g = 0; g < G; ++g)
      if ((uint32_t)g < groups) {
        const float mo = __shfl_xor(m[g], off, 64), lo = __shfl_xor(l[g], off, 64);
        const float mn = fmaxf(m[g], mo);
        const float c1 = m[g] == -INFINITY ? 0.f : __expf(m[g] - mn), c2 = mo == -INFINITY ? 0.f : __expf(mo - mn);
        l[g] = l[g] * c1 + lo * c2;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          const float ao = __shfl_xor(acc[g][t], off, 64);
          acc[g][t] = acc[g][t] * c1 + ao * c2;
        }
        m[g] = mn;
      }
  if (pj == 0 && active)
#pragma unroll
    for (int g = 0; g < G; ++g)
      if ((uint32_t)g < groups) {
        __half* dst = ctx + ((size_t)row * n_heads + kvh * groups + g) * head_dim + i0;
        const float inv = 1.0f / l[g];
#pragma unroll
        for (int t = 0; t < 8; ++t) dst[t] = __float2half_rn(acc[g][t] * inv);
      }
}

// The same causal attention for 32 rows at a time on the matrix cores (head_dim = 128).
// Workgroup (kv head, block of 32 rows); wavefront w serves query head w of the group and all
// 32 rows.  The cache is walked in tiles of 32 positions, staged in LDS once for all heads:
// K as stored ([position][dim]), V transposed ([dim][position], positions in the order the
// second product wants them).  Per tile and wavefront:
//   S^T = K Q^T      8 x v_mfma_f32_32x32x16_f16; A = K rows from LDS, B = the wavefront's
//                    query rows, held in registers for the whole walk.  Lane (q, h) of the
//                    result holds row q's scores of positions 8a + 4h + b (a, b < 4);
//   online softmax   per row in its two lanes: running maximum and sum in f32, one exchange
//                    between the halves of the wavefront; the causal mask is applied here;
//   O^T += V^T P^T   8 x the same MFMA; B = the probabilities just computed, rounded to
//                    binary16 in the lanes that hold them (no cross-lane movement: the K
//                    index of the product is permuted to match, V^T is stored in that order).
// H sets of wavefronts walk every H-th tile each, and their sums are joined at the end: the walk is a chain (16 tiles for the last rows of a
// 500-row prompt).  A workgroup takes G heads of a kv head's (blockIdx.x: the ceil(heads / G) of each kv head), all of them or two
// (prompt_heads_by_two).  500 rows of 32 heads: 31 us with one set, 22 with two, 17.5 with four and two heads to a workgroup (500 tokens of
// twelve 4B layers 2665 -> 2605 us).
// Scores, maxima, sums and O stay in f32; the context is rounded once.  The next tile's K and
// V rows are requested before the current tile is multiplied.  Positions past the pass's last
// row are read as that row.  Inside a tile a masked position has probability zero and is multiplied
// all the same, so a value that is not finite reaches the rows of its own block of 32 that come
// before it; rows of earlier blocks never meet it.
constexpr int kAttnTile = 32;
constexpr int kAttnKPitch = 128 + 8;   // binary16 elements per K row in LDS
constexpr int kAttnVPitch = 32 + 8;    // per V^T row
template <bool Q8, int G, int H>
__global__ __launch_bounds__(G * H * 64) void attn_rows_mfma_kernel(const __half* __restrict__ q, const __half* __restrict__ kcache,
                                                                const __half* __restrict__ vcache, KvQ8 q8,
                                                                __half* __restrict__ ctx, uint32_t n_heads, uint32_t n_kv,
                                                                uint32_t pos0, uint32_t n_rows, uint32_t max_pos, float scale, Octets to) {
  typedef _Float16 h8 __attribute__((ext_vector_type(8)));
  typedef float f16v __attribute__((ext_vector_type(16)));
  constexpr uint32_t kDimH = 128, kThreads = G * 64;  // threads of a part
  constexpr int CH = (kAttnTile * kDimH / 8 + kThreads - 1) / kThreads;  // 16-byte pieces of a tile per lane
  struct __align__(16) Tile {
    _Float16 k[kAttnTile * kAttnKPitch];
    _Float16 v[kDimH * kAttnVPitch];
  };
  __shared__ Tile tiles[H];
  static_assert(sizeof(tiles) >= (H - 1) * G * 64 * 16 * sizeof(float), "the parts meet in the tiles' memory");
  const uint32_t groups = n_heads / n_kv, of_kv = (groups + G - 1u) / G;
  const uint32_t kvh = blockIdx.x / of_kv, head0 = (blockIdx.x - kvh * of_kv) * G, row0 = blockIdx.y * kAttnTile;
  const uint32_t part = H == 1 ? 0u : (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / kThreads));
  const uint32_t tid = threadIdx.x - part * kThreads, lane = tid & 63u, wave = tid >> 6;
  _Float16 *kt = tiles[part].k, *vt = tiles[part].v;
  const uint32_t l32 = lane & 31u, lh = lane >> 5;
  const bool has_head = head0 + wave < groups;
  const uint32_t head = kvh * groups + min(head0 + wave, groups - 1u);
  const uint32_t my_row = min(row0 + l32, n_rows - 1u);      // rows past the pass repeat its last row and store nothing
  const uint32_t qpos = pos0 + my_row;
  const uint32_t last_pos = pos0 + n_rows - 1u;              // last cached position
  const uint32_t t_end = pos0 + min(row0 + kAttnTile - 1u, n_rows - 1u);
  const uint32_t n_tiles = t_end / kAttnTile + 1u;           // a part takes every H-th; one past the last is staged and not multiplied
  const size_t base = (size_t)kvh * max_pos;
  constexpr uint32_t kvgroups = kDimH / kKvGroup;

  // query rows: B fragments of the first product, dims [16 s + 8 h, +8) of row q
  h8 qf[8];
  {
    const __half* qrow = q + ((size_t)my_row * n_heads + head) * kDimH + lh * 8u;
#pragma unroll
    for (int s8 = 0; s8 < 8; ++s8) qf[s8] = *reinterpret_cast<const h8*>(qrow + s8 * 16);
  }
  f16v o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int j = 0; j < 16; ++j) o[dt][j] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  // staging, 16-byte pieces: piece c of K = position c / 16, dims [8 (c % 16), +8) (rows are read and
  // stored whole); piece c of V = position c % 32, dims [8 (c / 32), +8) (the transposing 2-byte stores
  // of a wavefront then fall into different LDS banks)
  uint4 kreg[CH], vreg[CH];
  float ksc[CH], kbi[CH], vsc[CH], vbi[CH];
  auto request = [&](uint32_t tile) {
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const uint32_t c = tid + (uint32_t)u * kThreads;
      if (c < kAttnTile * kDimH / 8) {
        const uint32_t kpos = min(tile * kAttnTile + c / 16u, last_pos), kd0 = (c & 15u) * 8u;
        const uint32_t vpos = min(tile * kAttnTile + (c & 31u), last_pos), vd0 = (c >> 5) * 8u;
        if constexpr (Q8) {
          const uint2 kc = *reinterpret_cast<const uint2*>(q8.kq + (base + kpos) * kDimH + kd0);
          const uint2 vc = *reinterpret_cast<const uint2*>(q8.vq + (base + vpos) * kDimH + vd0);
          const size_t kgi = (base + kpos) * kvgroups + kd0 / kKvGroup, vgi = (base + vpos) * kvgroups + vd0 / kKvGroup;
          kreg[u] = make_uint4(kc.x, kc.y, 0, 0);
          vreg[u] = make_uint4(vc.x, vc.y, 0, 0);
          ksc[u] = __half2float(q8.ks[kgi]); kbi[u] = __half2float(q8.kb[kgi]);
          vsc[u] = __half2float(q8.vs[vgi]); vbi[u] = __half2float(q8.vb[vgi]);
        } else {
          kreg[u] = *reinterpret_cast<const uint4*>(kcache + (base + kpos) * kDimH + kd0);
          vreg[u] = *reinterpret_cast<const uint4*>(vcache + (base + vpos) * kDimH + vd0);
        }
      }
    }
  };
  auto deposit = [&]() {
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const uint32_t c = tid + (uint32_t)u * kThreads;
      if (c < kAttnTile * kDimH / 8) {
        const uint32_t kp = c / 16u, kd0 = (c & 15u) * 8u, p = c & 31u, vd0 = (c >> 5) * 8u;
        h8 kv8, vv8;
        if constexpr (Q8) {
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            kv8[t] = (_Float16)kv_dequant((kreg[u].x >> (8 * t)) & 0xFFu, ksc[u], kbi[u]);
            kv8[4 + t] = (_Float16)kv_dequant((kreg[u].y >> (8 * t)) & 0xFFu, ksc[u], kbi[u]);
            vv8[t] = (_Float16)kv_dequant((vreg[u].x >> (8 * t)) & 0xFFu, vsc[u], vbi[u]);
            vv8[4 + t] = (_Float16)kv_dequant((vreg[u].y >> (8 * t)) & 0xFFu, vsc[u], vbi[u]);
          }
        } else {
          kv8 = __builtin_bit_cast(h8, kreg[u]);
          vv8 = __builtin_bit_cast(h8, vreg[u]);
        }
        *reinterpret_cast<h8*>(kt + kp * kAttnKPitch + kd0) = kv8;
        // position p = 16 hh + 8 a + 4 h + b sits at column 16 hh + 8 h + 4 a + b of its V^T row
        const uint32_t col = (p & 16u) + ((p >> 2) & 1u) * 8u + ((p >> 3) & 1u) * 4u + (p & 3u);
#pragma unroll
        for (int t = 0; t < 8; ++t) vt[(vd0 + t) * kAttnVPitch + col] = vv8[t];
      }
    }
  };

  request(part);
  for (uint32_t tile = part; tile < n_tiles + part; tile += H) {  // as many turns for every part
    __syncthreads();  // the previous tile has been read by every wavefront
    deposit();
    __syncthreads();
    if (tile + H < n_tiles + part) request(tile + H);
    if (H > 1 && tile >= n_tiles) continue;  // past every row of this block: nothing of it may reach their sums, not even times zero
    // S^T = K Q^T
    f16v sacc;
#pragma unroll
    for (int j = 0; j < 16; ++j) sacc[j] = 0.f;
#pragma unroll
    for (int s8 = 0; s8 < 8; ++s8) {
      const h8 kf = *reinterpret_cast<const h8*>(kt + l32 * kAttnKPitch + s8 * 16 + lh * 8u);
      sacc = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[s8], sacc, 0, 0, 0);
    }
    // online softmax of row q over this tile's positions (16 of them in this lane, 16 in lane ^ 32)
    float sc[16], mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const uint32_t pos = tile * kAttnTile + 8u * (j >> 2) + 4u * lh + (j & 3);
      sc[j] = pos <= qpos ? sacc[j] * scale : -INFINITY;
      mx = fmaxf(mx, sc[j]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m_new = fmaxf(m_run, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;  // a row that has seen nothing yet
    const float alpha = __expf(m_run - m_use);              // 0 while m_run = -inf
    float psum = 0.f;
    h8 pf[2];  // the probabilities as the second product's B fragments
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const float pj = __expf(sc[j] - m_use);
      psum += pj;
      pf[j >> 3][j & 7] = (_Float16)pj;
    }
    psum += __shfl_xor(psum, 32, 64);
    l_run = fmaf(l_run, alpha, psum);
    m_run = m_new;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int j = 0; j < 16; ++j) o[dt][j] *= alpha;
    // O^T += V^T P^T: K index e of half hh <-> position 16 hh + 8 (e / 4) + 4 h + e % 4 = this lane's score 8 hh + e
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) {
        const h8 vf = *reinterpret_cast<const h8*>(vt + (dt * 32 + l32) * kAttnVPitch + hh * 16 + lh * 8u);
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pf[hh], o[dt], 0, 0, 0);
      }
    }
  }
  if constexpr (H > 1) {  // the other parts' sums join the first's in order, a quarter of the dims at a time
    float* const meet = reinterpret_cast<float*>(tiles) + wave * 1024u + lane;
    float* const mine = meet + (part ? part - 1u : 0u) * (G * 1024u);
    __syncthreads();
    if (part) {
      mine[0] = m_run;
      mine[64] = l_run;
    }
    __syncthreads();
    float w[H];
    if (!part) {  // (a part that met no tile of these rows: maximum -inf, weight 0; the first has seen position 0)
      float m = m_run;
#pragma unroll
      for (uint32_t k = 1; k < (uint32_t)H; ++k) m = fmaxf(m, meet[(k - 1u) * (G * 1024u)]);
      w[0] = __expf(m_run - m);
      float l = l_run * w[0];
#pragma unroll
      for (uint32_t k = 1; k < (uint32_t)H; ++k) {
        w[k] = __expf(meet[(k - 1u) * (G * 1024u)] - m);
        l = fmaf(meet[(k - 1u) * (G * 1024u) + 64u], w[k], l);
      }
      l_run = l;
    }
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
      __syncthreads();
      if (part) {
#pragma unroll
        for (int j = 0; j < 16; ++j) mine[j * 64] = o[dt][j];
      }
      __syncthreads();
      if (!part) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          float v = o[dt][j] * w[0];
#pragma unroll
          for (uint32_t k = 1; k < (uint32_t)H; ++k) v = fmaf(meet[(k - 1u) * (G * 1024u) + (uint32_t)j * 64u], w[k], v);
          o[dt][j] = v;
        }
      }
    }
    if (part) return;
  }
  // o[dt][j] = O[q = l32][dim 32 dt + 8 (j / 4) + 4 h + j % 4]
  // (to.xt: a lane's four values are half of an octet, and a line of them eight of the wavefront's rows.  What addresses are made of is made
  // here: nothing of it may occupy registers before.)
  uint32_t lane_e = threadIdx.x & 63u;
  asm volatile("" : "+v"(lane_e));
  const uint32_t row_e = row0 + (lane_e & 31u);
  if (has_head && row_e < n_rows) {
    const float inv = 1.0f / l_run;
    const uint32_t in_rows = row_e * n_heads * (kDimH * 2u) + 8u * (lane_e >> 5), in_octets = row_e * 16u + 8u * (lane_e >> 5);
    uint8_t* const rows = reinterpret_cast<uint8_t*>(ctx + (size_t)head * kDimH);
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const __half2 lo = __float22half2_rn(make_float2(o[dt][4 * a] * inv, o[dt][4 * a + 1] * inv));
        const __half2 hi = __float22half2_rn(make_float2(o[dt][4 * a + 2] * inv, o[dt][4 * a + 3] * inv));
        uint2 pk;
        pk.x = *reinterpret_cast<const uint32_t*>(&lo);
        pk.y = *reinterpret_cast<const uint32_t*>(&hi);
        const uint32_t octet = dt * 4u + a, col = head * kDimH + octet * 8u;
        if (to.xt && col < to.kcols) *reinterpret_cast<uint2*>(reinterpret_cast<uint8_t*>(to.xt + (size_t)(col / 8u) * to.m_pad) + in_octets) = pk;
        else *reinterpret_cast<uint2*>(rows + octet * 16u + in_rows) = pk;
      }
  }
  // columns past the blocks are zero (rows past the pass: nobody has a result of theirs)
  if (to.xt && blockIdx.x == 0u && part == 0u && wave == 0u) {
    if (row_e < n_rows)
      for (uint32_t o = to.kcols / 8u + (lane_e >> 5); o < to.n_oct; o += 2u) to.xt[(size_t)o * to.m_pad + row_e] = make_uint4(0, 0, 0, 0);
  }
}

// Whether a prompt's workgroups take two query heads and the cache by four sets of wavefronts, where else they take all of a kv head's by two sets (one
// past five heads).  Every workgroup brings a kv head's tiles to LDS for itself, so this pays where CUs would be idle, and where the walk is long enough for
// four sets.  us a layer, all heads -> by two, binary16 and int8 caches:
//   up to as many workgroups as CUs: 32 heads of 8, 500 rows at 0 95 -> 91, 102 -> 98, at 2000 154 -> 133, 178 -> 156, at 7600 315 -> 251, 388 -> 313; 40 heads
//     of 8, 300 rows at 500 106 -> 96, 116 -> 105, 256 at 7600 352 -> 245, 431 -> 304; 64 of 8, 256 at 500 115 -> 98, 125 -> 105; 16 of 2, 500 at 0 96 -> 85, 102 -> 89;
//   past that with three to five heads: 40 of 8, 340 rows at 0 92 -> 95, 98 -> 100, 500 at 3000 204 -> 224, 242 -> 276, at 7600 363 -> 422, 447 -> 540;
//   with six to eight: 64 of 8, 300 rows at 0 96 -> 98, 102 -> 105, 400 104 -> 105, 112 -> 115, 500 112 -> 109, 120 -> 118, 300 at 500 118 -> 119, 129 -> 132, 500 135 -> 128,
//     149 -> 145, at 3000 247 -> 231, 294 -> 285;
//   up to 128 positions: 32 of 8, 24 rows at 0 47.7 -> 48.5, 52.9 -> 54.1, 64 53.5 -> 53.8, 55.5 -> 57.1; one and two heads 49.6 -> 50.7, 50.5 -> 51.5
//     (130 rows at 0: within half a us of each other).
inline bool prompt_heads_by_two(uint32_t n_kv, uint32_t groups, uint32_t row_blocks, uint32_t last_pos, uint32_t cus) {
  if (last_pos < 128u) return false;
  if (groups <= 2u || n_kv * ((groups + 1u) / 2u) * row_blocks <= cus) return true;
  return groups > 5u && 2u * n_kv * row_blocks <= cus && last_pos >= 448u;
}

// Attention of one query position over the cache (model.rs:812-822), heads of 128: workgroup (range, kv head) takes the positions
// [range * chunk, + chunk) for all query heads that share the kv head, sixteen positions (a tile) to a wavefront at a time.
//
// What bounds it: round trips to memory (operands and the first rows; partials, the counter and the partials again), so that the rest has to be
// short.  On the vector ALUs a tile was 500 instructions at four query heads (each lane eight columns of a row for every head, sixteen-lane
// sums of the scores); here scores are four matrix instructions (16 positions x 16 columns, of which the query heads take the
// first), the weighted sum of V 32 for every four heads, beside about 130 others (280 with an int8 cache).  The first product leaves a head's scores in the lanes that
// the second takes its weights from: column lane % 16 is head lane % (4 SETS), 4 (lane / 16) + i the position.  V lies in a lane by rows, four of them, eight columns each; in
// the second product a position and column of a lane meet the weights of its four neighbours' heads (16 blocks of 4 heads x 4 columns, 8 cycles each), and every
// quarter of the wavefront has the sums of its own positions until the range ends.  Weights, maxima, sums and scores are f32; K, V and the rotated queries are binary16
// values already.  (Weights as two binary16 terms, of sixteen positions in one instruction, take 6.9 and 11.1 us where these take 7.4 and 12.6, but have no bits below 2^-38
// of the largest, up to 18 % of weights of 2^-37, and where the second term is zero an infinite V is NaN.  f32 products with sixteen columns for the heads, of which
// they are a quarter: 7.9 and 12.8.)  Relative error of the context against 64 bits before it is rounded, in the mean over 3 to 8100 positions, four to eight heads
// and both caches: 1.46e-7; on the vector ALUs 1.58e-7.
// Per launch, on the vector ALUs -> now: 513 positions of a 4B layer 8.3 -> 7.4 us, 8100 of a 14B layer with an int8 cache 19.9 (4.6 of them a merge
// launch) -> 12.6.
//
// The workgroup that arrives last at the kv head's counter merges the ranges' partials in their order and rounds the context once;
// partials go to memory and back at device scope (past the XCDs' own L2s), not between fences, which write back and empty an L2.
constexpr uint32_t kDecodeTile = 16;    // positions of a wavefront at a time
constexpr uint32_t kDecodeWaves = 8;
constexpr uint32_t kDecodeMaxGroup = kAttnMaxGroup;
constexpr uint32_t kDecodeFetch = 32;   // ranges whose partials are asked for together
// log2(e) / sqrt(128), to 9e-9 of itself: scores are exponents of two, with one rounding of a score's difference to the maximum where the scaled
// score, the difference and __expf's product with log2(e) are three.
constexpr float kDecodeScale = 0.127517432f;
// Ranges of T positions: a tile to a wavefront, until the kv heads' workgroups fill the CUs.  us a launch by the number of ranges, on 256 CUs (* the rule's):
//   32 heads of 8, binary16       300: 1 7.3, 2 7.7, 3* 7.1, 8 6.6    1000: 4 8.4, 8* 7.1, 16 7.2, 32 8.7    4000: 8 11.2, 16 9.4, 32* 9.4, 64 16.6    8100: 16 12.4, 32* 12.2, 64 17.7
//   40 heads of 8, int8           300: 1 10.6, 2 9.7, 3* 8.7, 8 7.7   1000: 4 11.1, 8* 8.8, 16 8.3, 32 9.4   4000: 8 16.2, 16 12.1, 32* 10.9, 64 21.3   8100: 16 17.0, 32* 13.8, 64 23.7
//   8 heads of 1, binary16        300: 1 8.4, 2 8.8, 3* 8.2, 8 8.0    1000: 4 10.4, 8* 8.7, 16 8.6, 32 10.0  4000: 8 14.0, 16 11.3, 32* 11.2, 64 12.4   8100: 16 14.4, 32 12.6, 64* 13.0
//   64 heads of 32, binary16      300: 1 6.9, 2 7.3, 3* 6.8, 8 7.4    1000: 4 8.6, 8* 7.8, 16 13.0, 32 22.0  4000: 4 16.9, 8* 14.9, 16 18.0
// (One range has nobody to wait for: 130 positions 5.7 us in one and 7.0 in two.)
inline uint32_t decode_ranges(uint32_t T, uint32_t n_kv, uint32_t cus) {
  const uint32_t n = (T + kDecodeTile * kDecodeWaves - 1u) / (kDecodeTile * kDecodeWaves), fill = (cus + n_kv - 1u) / n_kv;
  return std::min(n, std::min(fill, (uint32_t)kAttnMaxSplits));
}
constexpr uint32_t kDecodeCounter = 64;   // counters are lines of their own: 256 workgroups' additions to one line, behind each other, took 1.5 us

// SETS: of up to four query heads each.
template <bool Q8, int SETS>
__global__ __launch_bounds__(kDecodeWaves * 64) void attn_decode_mfma_kernel(AttnNew nw, const __half* __restrict__ kcache, const __half* __restrict__ vcache,
                                                                             KvQ8 q8, __half* __restrict__ ctx, float* part, uint32_t* __restrict__ counters,
                                                                             uint32_t groups, uint32_t chunk, uint32_t T, uint32_t max_pos, uint32_t n_splits) {
  typedef _Float16 h8 __attribute__((ext_vector_type(8)));
  typedef float f4 __attribute__((ext_vector_type(4)));
  constexpr uint32_t D = 128, kvgroups = D / kKvGroup;
  __shared__ __align__(16) __half qh[kDecodeMaxGroup][D + 8];  // the query heads, normed and rotated
  __shared__ __align__(16) __half knew[D], vnew[D];            // the new position's k and v, or their codes
  __shared__ uint32_t knew_s, knew_b, vnew_s, vnew_b;          // scales and biases of those, a group to a half
  __shared__ __align__(16) float wmax[kDecodeMaxGroup][kDecodeWaves], wsum[kDecodeMaxGroup][kDecodeWaves];
  __shared__ __align__(16) float wacc[kDecodeWaves][4 * SETS][D];
  __shared__ uint32_t arrived;
  const uint32_t kvh = blockIdx.y, split = blockIdx.x, tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t j0 = min(T, split * chunk), j1 = min(T, j0 + chunk), nj = j1 - j0;
  const uint32_t pos = T - 1u;  // the position being decoded
  const bool has_new = nj > 0 && j1 == T;
  const uint32_t n16 = lane & 15u, quarter = lane >> 4;
  const size_t rows = (size_t)kvh * max_pos;

  // A tile's rows: K of position lane % 16, columns 8 (quarter + 4 m) + 0 .. 7 of matrix instruction m (int8: 16 (quarter + 4 m) + 0 .. 15 of
  // 2 m and 2 m + 1); V of positions 4 quarter + u, columns 8 (lane % 16) + 0 .. 7.  Unconditional: past the end the position being
  // decoded is read, whose row this launch writes, and not used.
  uint4 kraw[Q8 ? 2 : 4], vraw[4];
  uint32_t ks = 0, kb = 0;
  __half vs[4], vb[4];
  auto request = [&](uint32_t tile) {
    const uint32_t kp = min(j0 + tile * kDecodeTile + n16, pos);
    if constexpr (Q8) {
      const uint8_t* k = q8.kq + (rows + kp) * D + quarter * 16u;
#pragma unroll
      for (int m = 0; m < 2; ++m) kraw[m] = *reinterpret_cast<const uint4*>(k + m * 64);
      ks = *reinterpret_cast<const uint32_t*>(q8.ks + (rows + kp) * kvgroups);
      kb = *reinterpret_cast<const uint32_t*>(q8.kb + (rows + kp) * kvgroups);
    } else {
      const __half* k = kcache + (rows + kp) * D + quarter * 8u;
#pragma unroll
      for (int m = 0; m < 4; ++m) kraw[m] = *reinterpret_cast<const uint4*>(k + m * 32);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t vp = min(j0 + tile * kDecodeTile + quarter * 4u + (uint32_t)u, pos);
      if constexpr (Q8) {
        const uint2 v = *reinterpret_cast<const uint2*>(q8.vq + (rows + vp) * D + n16 * 8u);
        vraw[u] = make_uint4(v.x, v.y, 0, 0);
        vs[u] = q8.vs[(rows + vp) * kvgroups + (n16 >> 3)];
        vb[u] = q8.vb[(rows + vp) * kvgroups + (n16 >> 3)];
      } else {
        vraw[u] = *reinterpret_cast<const uint4*>(vcache + (rows + vp) * D + n16 * 8u);
      }
    }
  };
  // operands of the wavefront's query head and of the new k and v, in front of the rows (a wavefront without a head: the last one's)
  const RopeAngle angle{nw.cos_t[pos * 64u + lane], nw.sin_t[pos * 64u + lane]};
  const HeadOperands qop = head_operands_128(nw.q_raw + (size_t)(kvh * groups + min(wave, groups - 1u)) * D, nw.qn, lane, lane + 64u);
  const HeadOperands kop = head_operands_128(nw.k_raw + (size_t)kvh * D, nw.kn, lane, lane + 64u);
  const __half v1 = nw.v_raw[(size_t)kvh * D + lane], v2 = nw.v_raw[(size_t)kvh * D + lane + 64u];
  request(wave);
  static_assert(kDecodeMaxGroup <= kDecodeWaves && kDecodeMaxGroup <= 8, "a query head to a wavefront, two sets of them");
  if (wave < groups) {
    const float2 r = norm_rope_128(qop, angle, nw.eps);
    qh[wave][lane] = __float2half_rn(r.x);  // (exact)
    qh[wave][lane + 64u] = __float2half_rn(r.y);
  }
  // The range that ends at the new position owns its k and v: they go to the cache for later positions, and to LDS for this one.
  const auto quantized = [&](float x, uint32_t g, uint8_t* codes, __half* s_row, __half* b_row, __half* fresh, uint32_t* fresh_s, uint32_t* fresh_b) {
    __half sh, bh;
    const uint8_t code = kv_quantize_group(x, &sh, &bh);
    codes[(rows + pos) * D + g * kKvGroup + lane] = code;
    reinterpret_cast<uint8_t*>(fresh)[g * kKvGroup + lane] = code;
    if (lane == 0) {
      s_row[(rows + pos) * kvgroups + g] = sh;
      b_row[(rows + pos) * kvgroups + g] = bh;
      reinterpret_cast<__half*>(fresh_s)[g] = sh;
      reinterpret_cast<__half*>(fresh_b)[g] = bh;
    }
  };
  if (has_new && wave == kDecodeWaves - 1u) {
    const float2 r = norm_rope_128(kop, angle, nw.eps);
    if constexpr (Q8) {
      quantized(r.x, 0, q8.kq, q8.ks, q8.kb, knew, &knew_s, &knew_b);
      quantized(r.y, 1, q8.kq, q8.ks, q8.kb, knew, &knew_s, &knew_b);
    } else {
      nw.kcache[(rows + pos) * D + lane] = knew[lane] = __float2half_rn(r.x);
      nw.kcache[(rows + pos) * D + lane + 64u] = knew[lane + 64u] = __float2half_rn(r.y);
    }
  }
  if (has_new && wave == kDecodeWaves - 2u) {
    if constexpr (Q8) {
      quantized(__half2float(v1), 0, q8.vq, q8.vs, q8.vb, vnew, &vnew_s, &vnew_b);
      quantized(__half2float(v2), 1, q8.vq, q8.vs, q8.vb, vnew, &vnew_s, &vnew_b);
    } else {
      nw.vcache[(rows + pos) * D + lane] = vnew[lane] = v1;
      nw.vcache[(rows + pos) * D + lane + 64u] = vnew[lane + 64u] = v2;
    }
  }
  __syncthreads();

  h8 qf[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const uint32_t col = Q8 ? (quarter + 4u * (m >> 1)) * 16u + (m & 1) * 8u : (quarter + 4u * m) * 8u;
    qf[m] = *reinterpret_cast<const h8*>(&qh[min(n16 % (4u * SETS), groups - 1u)][col]);  // (past the heads: the last head again, not used)
  }
  f4 acc[SETS][8];  // [set][t]: column 8 (lane % 16) + t of heads 4 set + i, of the lane's quarter's positions
#pragma unroll
  for (int set = 0; set < SETS; ++set)
#pragma unroll
    for (int t = 0; t < 8; ++t) acc[set][t] = f4{0.f, 0.f, 0.f, 0.f};
  // Of a value that lane has for head lane % (4 SETS), that of head 4 set + lane % 4.
  const auto of_set = [](int set, float v) {
    if constexpr (SETS == 1) return v;
    const int b = __float_as_int(v);  // quads 1 and 3 take what is in those in front of them; 0 and 2 those behind
    return __int_as_float(set == 0 ? __builtin_amdgcn_update_dpp(b, b, 0x114, 0xF, 0xA, false) : __builtin_amdgcn_update_dpp(b, b, 0x104, 0xF, 0x5, false));
  };
  float m_run = -INFINITY, l_run = 0.f;  // the head's maximum so far; the lane's positions' sum of exponentials
  const auto lane_max = [](float v) {    // over the quarters
    auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
    p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1]));
  };
  const auto lane_sum = [](float v) {
    auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(p[0]) + __uint_as_float(p[1]);
    p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(p[0]) + __uint_as_float(p[1]);
  };
  const auto half_of = [](uint32_t w, uint32_t i) { return __half2float(__ushort_as_half((unsigned short)(w >> (16u * i)))); };
#pragma unroll 1
  for (uint32_t tile = wave; tile * kDecodeTile < nj; tile += kDecodeWaves) {
    const uint32_t left = nj - tile * kDecodeTile;  // positions from the tile's first on
    if (left <= kDecodeTile) {                      // the range's last tile
      if (has_new) {                                // ends in the row that this launch appends
        if (n16 == left - 1u) {
#pragma unroll
          for (int m = 0; m < (Q8 ? 2 : 4); ++m)
            kraw[m] = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint8_t*>(knew) + (quarter + 4u * m) * 16u);
          if constexpr (Q8) {
            ks = knew_s;
            kb = knew_b;
          }
        }
      }
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u) {
        const uint32_t at = quarter * 4u + u;
        if (has_new && at == left - 1u) {
          if constexpr (Q8) {
            const uint2 v = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint8_t*>(vnew) + n16 * 8u);
            vraw[u] = make_uint4(v.x, v.y, 0, 0);
            vs[u] = __ushort_as_half((unsigned short)(vnew_s >> (16u * (n16 >> 3))));
            vb[u] = __ushort_as_half((unsigned short)(vnew_b >> (16u * (n16 >> 3))));
          } else {
            vraw[u] = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint8_t*>(vnew) + n16 * 16u);
          }
        }
        // A row past the range is whatever an earlier use of the cache left.  Its weight is zero, and its values have to be
        // as well: 0 x infinity would reach the sums.
        if (at >= left) {
          vraw[u] = make_uint4(0, 0, 0, 0);
          vs[u] = vb[u] = __ushort_as_half(0);
        }
      }
    }
    // scores
    const f4 zero = {0.f, 0.f, 0.f, 0.f};
    f4 quad[4];  // (each from zero: one behind the other they round more, and wait for each other)
    float va[4][8];  // [u][t]: column t of position u
    if constexpr (Q8) {
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const float sc = half_of(ks, m), bi = half_of(kb, m);
        const uint32_t w[4] = {kraw[m].x, kraw[m].y, kraw[m].z, kraw[m].w};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          h8 k;
#pragma unroll
          for (int t = 0; t < 8; ++t) k[t] = (_Float16)fmaf((float)((w[2 * h + (t >> 2)] >> (8 * (t & 3))) & 0xFFu), sc, bi);  // kv_dequant
          quad[2 * m + h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k, qf[2 * m + h], zero, 0, 0, 0);
        }
      }
      float fs[4], fb[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        fs[u] = __half2float(vs[u]);
        fb[u] = __half2float(vb[u]);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int t = 0; t < 8; ++t) va[u][t] = kv_dequant(((t < 4 ? vraw[u].x : vraw[u].y) >> (8 * (t & 3))) & 0xFFu, fs[u], fb[u]);
    } else {
#pragma unroll
      for (int m = 0; m < 4; ++m) quad[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, kraw[m]), qf[m], zero, 0, 0, 0);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t w[4] = {vraw[u].x, vraw[u].y, vraw[u].z, vraw[u].w};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          va[u][2 * t] = half_lo(w[t]);
          va[u][2 * t + 1] = half_hi(w[t]);
        }
      }
    }
    if ((tile + kDecodeWaves) * kDecodeTile < nj) request(tile + kDecodeWaves);
    float s[4], mt = -INFINITY;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
      s[i] = quarter * 4u + i < left ? (quad[0][i] + quad[1][i]) + (quad[2][i] + quad[3][i]) : -INFINITY;
      mt = fmaxf(mt, s[i]);
    }
    const float mn = fmaxf(m_run, lane_max(mt) * kDecodeScale);
    if (__builtin_amdgcn_ballot_w64(mn != m_run) != 0u) {  // (most tiles of a long range raise nobody's maximum)
      const float e0 = __builtin_amdgcn_exp2f(m_run - mn);  // 0 at the first tile (m_run = -inf)
      m_run = mn;
      l_run *= e0;
#pragma unroll
      for (int set = 0; set < SETS; ++set) {
        const int b = __float_as_int(of_set(set, e0));
        const f4 e = {__int_as_float(__builtin_amdgcn_update_dpp(0, b, 0x00, 0xF, 0xF, false)), __int_as_float(__builtin_amdgcn_update_dpp(0, b, 0x55, 0xF, 0xF, false)),
                      __int_as_float(__builtin_amdgcn_update_dpp(0, b, 0xAA, 0xF, 0xF, false)), __int_as_float(__builtin_amdgcn_update_dpp(0, b, 0xFF, 0xF, 0xF, false))};
#pragma unroll
        for (int t = 0; t < 8; ++t) acc[set][t] *= e;
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float p = __builtin_amdgcn_exp2f(fmaf(s[u], kDecodeScale, -mn));
      l_run += p;
#pragma unroll
      for (int set = 0; set < SETS; ++set) {
        const float ps = of_set(set, p);
#pragma unroll
        for (int t = 0; t < 8; ++t) acc[set][t] = __builtin_amdgcn_mfma_f32_4x4x1f32(ps, va[u][t], acc[set][t], 0, 0, 0);
      }
    }
  }
  // The wavefronts' results meet in LDS.  (One without a position: maximum -inf, weight 0.)
  const float l_all = lane_sum(l_run);
  if (n16 < groups && quarter == 0) {
    wmax[n16][wave] = m_run;
    wsum[n16][wave] = l_all;
  }
  // The quarters' sums meet by lane moves: a move across half the wavefront leaves each half two columns of four, one across a quarter each quarter one.
  const auto quarters = [](float a, float b, float c, float d) {
    auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(c), false, false);
    const float lo = __uint_as_float(p[0]) + __uint_as_float(p[1]);
    p = __builtin_amdgcn_permlane32_swap(__float_as_uint(b), __float_as_uint(d), false, false);
    const float hi = __uint_as_float(p[0]) + __uint_as_float(p[1]);
    p = __builtin_amdgcn_permlane16_swap(__float_as_uint(lo), __float_as_uint(hi), false, false);
    return __uint_as_float(p[0]) + __uint_as_float(p[1]);
  };
#pragma unroll
  for (uint32_t g = 0; g < 4u * SETS; ++g) {
    if (g >= groups) break;
    const f4(&a)[8] = acc[g / 4u];
    const uint32_t i = g % 4u;
    const float x = quarters(a[0][i], a[2][i], a[4][i], a[6][i]), y = quarters(a[1][i], a[3][i], a[5][i], a[7][i]);
    *reinterpret_cast<float2*>(&wacc[wave][g][n16 * 8u + quarter * 2u]) = make_float2(x, y);
  }
  __syncthreads();
  // ---- this workgroup's partial: the wavefronts merged in order, two neighbouring columns to a lane ----
  // part: [head][range][column] weighted sums, behind those of every head's [head][range] {maximum, sum of exponentials}
  float* const part_ml = part + (size_t)gridDim.y * groups * kAttnMaxSplits * D;
  auto put = [&](float* at, float a, float b) {  // read by another workgroup of this launch
    __hip_atomic_store(reinterpret_cast<uint64_t*>(at), (uint64_t)__float_as_uint(a) | (uint64_t)__float_as_uint(b) << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  if (wave < groups) {
    float w[kDecodeWaves], M = -INFINITY, L = 0.f, A = 0.f, B = 0.f;
#pragma unroll
    for (uint32_t k = 0; k < kDecodeWaves; ++k) {
      w[k] = wmax[wave][k];
      M = fmaxf(M, w[k]);
    }
#pragma unroll
    for (uint32_t k = 0; k < kDecodeWaves; ++k) {
      w[k] = w[k] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(w[k] - M);
      const float2 a = *reinterpret_cast<const float2*>(&wacc[k][wave][lane * 2u]);
      L = fmaf(wsum[wave][k], w[k], L);
      A = fmaf(a.x, w[k], A);
      B = fmaf(a.y, w[k], B);
    }
    const uint32_t head = kvh * groups + wave;
    if (n_splits == 1u) {
      reinterpret_cast<__half2*>(ctx + (size_t)head * D)[lane] = __floats2half2_rn(A / L, B / L);
    } else {
      put(part + ((size_t)head * n_splits + split) * D + lane * 2u, A, B);
      if (lane == 0) put(part_ml + (head * n_splits + split) * 2u, M, L);  // (-inf for an empty range)
    }
  }
  if (n_splits == 1u) return;
  // Let the last workgroup of this kv head merge: a lane's partials have arrived in memory before it reaches the barrier,
  // and only then is the workgroup counted.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) arrived = __hip_atomic_fetch_add(&counters[kvh * kDecodeCounter], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (arrived != n_splits - 1u) return;
  // A head to a wavefront: its lanes hold the ranges' maxima and sums, and its weights; then two neighbouring columns each.  The first ranges'
  // partials are requested together with those, every load unconditional (past the last range: the last again, not added).  Sums run in range order.
  static_assert(kAttnMaxSplits <= 64, "a range to a lane");
  if (wave < groups) {
    const uint32_t head = kvh * groups + wave;
    auto load2 = [&](const float* at) { return __hip_atomic_load(reinterpret_cast<const uint64_t*>(at), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    const uint64_t pair = load2(part_ml + (head * n_splits + min(lane, n_splits - 1u)) * 2u);
    uint64_t v[kDecodeFetch];
    auto fetch = [&](uint32_t from) {
#pragma unroll
      for (uint32_t u = 0; u < kDecodeFetch; ++u)
        if (from + (u & ~7u) < n_splits) v[u] = load2(part + ((size_t)head * n_splits + min(from + u, n_splits - 1u)) * D + lane * 2u);
    };
    fetch(0);
    const float mx = lane < n_splits ? __uint_as_float((uint32_t)pair) : -INFINITY;
    const float M = wave_best(mx, [](float a, float b) { return fmaxf(a, b); });
    const float w = mx == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mx - M);  // 0 for an empty range too
    const float L = wave_sum(lane < n_splits ? w * __uint_as_float((uint32_t)(pair >> 32)) : 0.f);
    float A = 0.f, B = 0.f;
#pragma unroll 1
    for (uint32_t from = 0;; from += kDecodeFetch) {
#pragma unroll
      for (uint32_t u0 = 0; u0 < kDecodeFetch; u0 += 8u)
        if (from + u0 < n_splits)
#pragma unroll
          for (uint32_t u = u0; u < u0 + 8u; ++u) {
            const float of = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), (int)(from + u)));
            const float a = fmaf(__uint_as_float((uint32_t)v[u]), of, A), b = fmaf(__uint_as_float((uint32_t)(v[u] >> 32)), of, B);
            A = from + u < n_splits ? a : A;  // (0 x infinity, of the last range's repeats, would reach the sums)
            B = from + u < n_splits ? b : B;
          }
      if (from + kDecodeFetch >= n_splits) break;
      fetch(from + kDecodeFetch);
    }
    reinterpret_cast<__half2*>(ctx + (size_t)(kvh * groups + wave) * D + lane * 2u)[0] = __floats2half2_rn(A / L, B / L);
  }
  if (tid == 0) counters[kvh * kDecodeCounter] = 0;  // ready for the next launch
}

// The same for heads of another width than 128, split over the cache: workgroup (kv head, split) takes a contiguous range of positions
// for all query heads that share the kv head, so every K and V row is fetched
// (and, for the int8 cache, rebuilt) once per group.  The range is walked once:
// sixteen position classes (four per wavefront, 16 lanes x 8 dims each) keep a
// running maximum, a sum of exponentials and a weighted V sum per query head,
// with the K and V rows of four positions requested together; a wavefront's
// four classes meet by lane moves, the wavefronts in LDS, and the workgroup
// leaves an unnormalised partial per query head.  The workgroup that arrives
// last at the kv head's counter merges the partials in split order and rounds
// the context once (past 16 ranges attn_merge_kernel does).  At the lengths of a chat (one batch of rows per class) a
// launch is a chain of round trips: operands and rows, partials to memory, the
// counter, partials from memory.  So the first rows are requested in front of the
// work on the new position's heads, and partials are stored and loaded at
// device scope (past the XCDs' own L2s) instead of between fences, which write
// back and empty an L2.  Scores, softmax and sums stay in
// f32.  head_dim <= 128, a multiple of 8; G >= query heads per kv head sizes
// the register arrays.
template <bool Q8, int G>
__global__ __launch_bounds__(kAttnThreads) void attn_decode_kernel(AttnNew nw, const __half* __restrict__ kcache,
                                                                   const __half* __restrict__ vcache, KvQ8 q8,
                                                                   __half* __restrict__ ctx,
                                                                   float* part, uint32_t* __restrict__ counters,
                                                                   uint32_t groups, uint32_t chunk, uint32_t head_dim,
                                                                   uint32_t T, uint32_t max_pos, float scale, uint32_t n_splits,
                                                                   uint32_t merge_inline) {
  extern __shared__ __align__(16) float att_smem[];
  __shared__ uint32_t arrived;
  __shared__ float stage[kAttnWaves][256];  // one head per wavefront while it is normed and rotated
  __shared__ float knew[256], vnew[256];    // the new position's k and v as the cache returns them
  const uint32_t kvh = blockIdx.y, split = blockIdx.x;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t j0 = min(T, split * chunk), j1 = min(T, j0 + chunk), nj = j1 - j0;
  float* qs = att_smem;                         // [groups][head_dim]
  float* cls = qs + groups * head_dim;          // the wavefronts' results
  const __half* K = kcache + (size_t)kvh * max_pos * head_dim;
  const __half* V = vcache + (size_t)kvh * max_pos * head_dim;
  const uint32_t kvgroups = head_dim / kKvGroup;
  const uint8_t* Kq = q8.kq + (size_t)kvh * max_pos * head_dim;
  const uint8_t* Vq = q8.vq + (size_t)kvh * max_pos * head_dim;
  const __half* Ks = q8.ks + (size_t)kvh * max_pos * kvgroups;
  const __half* Kb = q8.kb + (size_t)kvh * max_pos * kvgroups;
  const __half* Vs = q8.vs + (size_t)kvh * max_pos * kvgroups;
  const __half* Vb = q8.vb + (size_t)kvh * max_pos * kvgroups;
  const uint32_t stride = head_dim + 2;  // floats per partial: max, sum, head_dim sums

  const uint32_t pos = T - 1;  // the position being decoded
  const bool has_new = nj > 0 && j1 == T;
  const uint32_t newj = has_new ? pos : 0xFFFFFFFFu;
  // Lane (pj, sub) = (lane / 16, lane % 16) of wavefront w holds dims [8 sub, 8 sub + 8) of the
  // positions of class c = 4 w + pj: jj = c, c + kAttnClasses, ...  U rows of K and of V are requested
  // together.  The loads are unconditional (a lane with no row, or with the row this launch
  // appends, re-reads a valid one and ignores it): a guarded load would be waited for where it
  // is issued, and the first batch is issued here, ahead of the work on the query heads, which
  // then runs beside the cache's latency.
  const uint32_t sub = lane & 15u, pj = lane >> 4, i0 = sub * 8u, c = wave * 4u + pj;
  const bool active = i0 < head_dim;
  const uint32_t i0c = active ? i0 : 0u;
  constexpr int U = kAttnRows;
  uint4 kraw[U], vraw[U];
  float ksc[U], kbi[U], vsc[U], vbi[U];
  auto request = [&](uint32_t jb) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t j = min(j0 + jb + kAttnClasses * u, pos);
      if constexpr (Q8) {
        const uint2 kc = *reinterpret_cast<const uint2*>(Kq + (size_t)j * head_dim + i0c);
        const uint2 vc = *reinterpret_cast<const uint2*>(Vq + (size_t)j * head_dim + i0c);
        const size_t gi = (size_t)j * kvgroups + i0c / kKvGroup;
        kraw[u] = make_uint4(kc.x, kc.y, 0, 0);
        vraw[u] = make_uint4(vc.x, vc.y, 0, 0);
        ksc[u] = __half2float(Ks[gi]); kbi[u] = __half2float(Kb[gi]);
        vsc[u] = __half2float(Vs[gi]); vbi[u] = __half2float(Vb[gi]);
      } else {
        kraw[u] = *reinterpret_cast<const uint4*>(K + (size_t)j * head_dim + i0c);
        vraw[u] = *reinterpret_cast<const uint4*>(V + (size_t)j * head_dim + i0c);
        ksc[u] = kbi[u] = vsc[u] = vbi[u] = 0.f;
      }
    }
  };
  request(c);
  // the query heads of this kv head: norm, rotate, scale
  for (uint32_t g = wave; g < groups; g += kAttnWaves) {
    norm_rope_wave(nw.q_raw + (size_t)(kvh * groups + g) * head_dim, nw.qn, nw.cos_t, nw.sin_t, pos, head_dim, nw.eps,
                   stage[wave], lane);
    for (uint32_t i = lane; i < head_dim; i += 64) qs[g * head_dim + i] = stage[wave][i] * scale;
    wave_lds_sync();  // stage is rewritten by this wavefront's next head
  }
  // The range that ends at the new position owns its k and v: they go to the
  // cache for later positions, and to LDS, in the form the cache gives back,
  // for this one (nothing else reads that cache row during this launch).
  if (has_new && wave == 0) {
    norm_rope_wave(nw.k_raw + (size_t)kvh * head_dim, nw.kn, nw.cos_t, nw.sin_t, pos, head_dim, nw.eps, stage[0], lane);
    const size_t row = (size_t)kvh * max_pos + pos;
    if constexpr (Q8) {
      for (uint32_t g = 0; g < kvgroups; ++g) {
        __half sh, bh;
        const uint8_t code = kv_quantize_group(stage[0][g * kKvGroup + lane], &sh, &bh);
        q8.kq[row * head_dim + g * kKvGroup + lane] = code;
        if (lane == 0) {
          q8.ks[row * kvgroups + g] = sh;
          q8.kb[row * kvgroups + g] = bh;
        }
        knew[g * kKvGroup + lane] = kv_dequant(code, __half2float(sh), __half2float(bh));
      }
    } else {
      for (uint32_t i = lane; i < head_dim; i += 64) {
        nw.kcache[row * head_dim + i] = __float2half_rn(stage[0][i]);
        knew[i] = stage[0][i];
      }
    }
  }
  if (has_new && wave == 1) {
    const size_t row = (size_t)kvh * max_pos + pos;
    if constexpr (Q8) {
      for (uint32_t g = 0; g < kvgroups; ++g) {
        const float x = __half2float(nw.v_raw[(size_t)kvh * head_dim + g * kKvGroup + lane]);
        __half sh, bh;
        const uint8_t code = kv_quantize_group(x, &sh, &bh);
        q8.vq[row * head_dim + g * kKvGroup + lane] = code;
        if (lane == 0) {
          q8.vs[row * kvgroups + g] = sh;
          q8.vb[row * kvgroups + g] = bh;
        }
        vnew[g * kKvGroup + lane] = kv_dequant(code, __half2float(sh), __half2float(bh));
      }
    } else {
      for (uint32_t i = lane; i < head_dim; i += 64) {
        const __half x = nw.v_raw[(size_t)kvh * head_dim + i];
        nw.vcache[row * head_dim + i] = x;
        vnew[i] = __half2float(x);
      }
    }
  }
  __syncthreads();

  // ---- one pass over the range: scores, running maxima and weighted V sums together ----
  // Each position class keeps its own running maximum, sum of exponentials and weighted V sum
  // (f32); the scores of a batch are formed first (independent cross-lane sums), then folded in
  // order, with the next batch's rows already requested.
  float qv[G][8], acc[G][8], m[G], l[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    m[g] = -INFINITY;
    l[g] = 0.f;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      acc[g][t] = 0.f;
      qv[g][t] = ((uint32_t)g < groups && active) ? qs[g * head_dim + i0 + t] : 0.f;
    }
  }
  for (uint32_t jb = c; jb < nj; jb += kAttnClasses * U) {
    float sc[U][G], vfs[U][8];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t jj = jb + kAttnClasses * u;
      // A row past the range is one of the row this launch is about to write: whatever an earlier use of the cache left.
      // Its weight is zero, and its values have to be as well: 0 x infinity would reach the sums.
      if (jj >= nj) {
        vraw[u] = make_uint4(0, 0, 0, 0);
        vsc[u] = vbi[u] = 0.f;
      }
      float kf[8];
      if (j0 + jj == newj) {  // the row appended by this launch: from LDS, as the cache returns it
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          kf[t] = active ? knew[i0 + t] : 0.f;
          vfs[u][t] = active ? vnew[i0 + t] : 0.f;
        }
      } else if constexpr (Q8) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          kf[t] = kv_dequant((kraw[u].x >> (8 * t)) & 0xFFu, ksc[u], kbi[u]);
          kf[4 + t] = kv_dequant((kraw[u].y >> (8 * t)) & 0xFFu, ksc[u], kbi[u]);
          vfs[u][t] = kv_dequant((vraw[u].x >> (8 * t)) & 0xFFu, vsc[u], vbi[u]);
          vfs[u][4 + t] = kv_dequant((vraw[u].y >> (8 * t)) & 0xFFu, vsc[u], vbi[u]);
        }
      } else {
        const uint32_t kw[4] = {kraw[u].x, kraw[u].y, kraw[u].z, kraw[u].w}, vw[4] = {vraw[u].x, vraw[u].y, vraw[u].z, vraw[u].w};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          kf[2 * t] = __half2float(__ushort_as_half((unsigned short)(kw[t] & 0xFFFFu)));
          kf[2 * t + 1] = __half2float(__ushort_as_half((unsigned short)(kw[t] >> 16)));
          vfs[u][2 * t] = __half2float(__ushort_as_half((unsigned short)(vw[t] & 0xFFFFu)));
          vfs[u][2 * t + 1] = __half2float(__ushort_as_half((unsigned short)(vw[t] >> 16)));
        }
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float d = 0.f;
#pragma unroll
        for (int t = 0; t < 8; ++t) d = fmaf(qv[g][t], kf[t], d);
        sc[u][g] = row16_sum(d);
      }
    }
    if (jb + kAttnClasses * U < nj) request(jb + kAttnClasses * U);
    // the batch's maximum first, so that its exponentials do not wait for each other
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float mn = m[g];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        sc[u][g] = jb + kAttnClasses * u < nj ? sc[u][g] : -INFINITY;
        mn = fmaxf(mn, sc[u][g]);
      }
      const float e0 = __expf(m[g] - mn);  // 0 on the first batch (m = -inf)
      float p[U];
      l[g] *= e0;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        p[u] = __expf(sc[u][g] - mn);
        l[g] += p[u];
      }
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        acc[g][t] *= e0;
#pragma unroll
        for (int u = 0; u < U; ++u) acc[g][t] = fmaf(p[u], vfs[u][t], acc[g][t]);
      }
      m[g] = mn;
    }
  }
  // A wavefront's four classes meet by lane moves; every sixteen lanes then hold the sums, and lanes 16 (g mod 4) on put
  // head g's down.  (A class with no position: maximum -inf, weight 0.)
  float* wmax = cls;                                       // [wavefronts][groups] running maximum,
  float* wsum = wmax + kAttnWaves * groups;                // sum of exponentials,
  float* wacc = qs + ((groups * head_dim + 2u * kAttnWaves * groups + 3u) & ~3u);  // [wavefronts][groups][head_dim] weighted V sums
  // (Heads four at a time: a move across half the wavefront leaves each half two heads of both, one across a quarter
  // each quarter its own head of all four.)
  auto swap32 = [](float a, float b, auto op) {
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return op(__uint_as_float(p[0]), __uint_as_float(p[1]));
  };
  auto swap16 = [](float a, float b, auto op) {
    const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return op(__uint_as_float(p[0]), __uint_as_float(p[1]));
  };
  auto add = [](float a, float b) { return a + b; };
  auto larger = [](float a, float b) { return fmaxf(a, b); };
#pragma unroll
  for (int g0 = 0; g0 < G; g0 += 4) {
    float wgt[4], M = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      wgt[k] = 0.f;
      if (g0 + k < G) {
        const int g = g0 + k;
        float mk = swap32(m[g], m[g], larger);
        mk = swap16(mk, mk, larger);
        wgt[k] = m[g] == -INFINITY ? 0.f : __expf(m[g] - mk);
        M = pj == (uint32_t)k ? mk : M;
      }
    }
    auto quarters = [&](auto value) {  // value(k): head k's; the lane's quarter's own, summed over the classes
      const float lo = swap32(value(0), value(2), add), hi = swap32(value(1), value(3), add);
      return swap16(lo, hi, add);
    };
    const float Lsum = quarters([&](int k) { return g0 + k < G ? l[g0 + k < G ? g0 + k : 0] * wgt[k] : 0.f; });
    float s[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) s[t] = quarters([&](int k) { return g0 + k < G ? acc[g0 + k < G ? g0 + k : 0][t] * wgt[k] : 0.f; });
    const uint32_t g = (uint32_t)g0 + pj;
    if (g < groups) {
      if (sub == 0) {
        wmax[wave * groups + g] = M;
        wsum[wave * groups + g] = Lsum;
      }
      if (active) {
        float4* dst = reinterpret_cast<float4*>(wacc + ((size_t)wave * groups + g) * head_dim + i0);
        dst[0] = make_float4(s[0], s[1], s[2], s[3]);
        dst[1] = make_float4(s[4], s[5], s[6], s[7]);
      }
    }
  }
  __syncthreads();
  // ---- this workgroup's partial: the wavefronts merged in order ----
  auto put = [&](float* at, float v) {  // read by another workgroup of this launch, or by attn_merge_kernel
    __hip_atomic_store(at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  for (uint32_t o = tid; o < groups * head_dim; o += kAttnThreads) {
    const uint32_t g = o / head_dim, i = o - g * head_dim;
    float w[kAttnWaves], M = -INFINITY, L = 0.f, A = 0.f;
#pragma unroll
    for (int k = 0; k < kAttnWaves; ++k) {
      w[k] = wmax[k * groups + g];
      M = fmaxf(M, w[k]);
    }
#pragma unroll
    for (int k = 0; k < kAttnWaves; ++k) {
      w[k] = w[k] == -INFINITY ? 0.f : __expf(w[k] - M);
      L = fmaf(wsum[k * groups + g], w[k], L);
      A = fmaf(wacc[((size_t)k * groups + g) * head_dim + i], w[k], A);
    }
    float* dst = part + ((size_t)(kvh * groups + g) * n_splits + split) * stride;
    if (i == 0) {
      put(dst, M);  // -inf for an empty range
      put(dst + 1, L);
    }
    put(dst + 2 + i, A);
  }
  if (!merge_inline) return;  // attn_merge_kernel finishes (long caches: many partials, merged chip-wide)
  // Let the last workgroup of this kv head merge: a lane's partials have arrived in memory before it reaches the barrier,
  // and only then is the workgroup counted.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) arrived = __hip_atomic_fetch_add(&counters[kvh], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (arrived != n_splits - 1) return;
  // Merge (at most kAttnInlineSplits = 16 ranges): sixteen lanes hold the ranges of a head, form its weights and leave
  // them in LDS; a lane then sums two neighbouring elements.  The first elements are requested together with the
  // (max, sum) pairs, every load unconditional (past the end: a valid one again, of weight zero).  Sums run in range order.
  float* wts = att_smem;                            // [groups][16] weights (the staging of this launch is dead)
  float* tot = wts + groups * kAttnInlineSplits;    // [groups] sums of exponentials
  static_assert(kAttnInlineSplits == 16 && kAttnMaxGroup <= kAttnWaves * 4, "a range per lane of a row, a head per row");
  const uint32_t n_pairs = groups * (head_dim >> 1);
  auto load2 = [&](uint32_t at) {
    return __hip_atomic_load(reinterpret_cast<uint64_t*>(part + at), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  const uint32_t hg = wave * 4u + pj;
  const uint64_t pair = load2(((kvh * groups + min(hg, groups - 1u)) * n_splits + min(sub, n_splits - 1u)) * stride);
  uint64_t v[kAttnInlineSplits];
  auto fetch = [&](uint32_t o) {
    o = min(o, n_pairs - 1u);
    const uint32_t g = o / (head_dim >> 1), i = (o - g * (head_dim >> 1)) * 2u;
    const uint32_t at = (kvh * groups + g) * n_splits * stride + 2u + i;
#pragma unroll
    for (int u = 0; u < kAttnInlineSplits; ++u) v[u] = load2(at + min((uint32_t)u, n_splits - 1u) * stride);
  };
  fetch(tid);
  {
    const float mx = sub < n_splits ? __uint_as_float((uint32_t)pair) : -INFINITY;
    float M = mx;
#pragma unroll
    for (int k = 1; k < 16; k <<= 1) M = fmaxf(M, __shfl_xor(M, k));
    const float w = mx == -INFINITY ? 0.f : __expf(mx - M);  // 0 for an empty range too
    float L = w * (sub < n_splits ? __uint_as_float((uint32_t)(pair >> 32)) : 0.f);
    L = row16_sum(L);
    if (hg < groups) {
      wts[hg * kAttnInlineSplits + sub] = w;
      if (sub == 0) tot[hg] = L;
    }
  }
  __syncthreads();
#pragma unroll 1
  for (uint32_t o = tid; o < n_pairs; o += kAttnThreads) {
    const uint32_t g = o / (head_dim >> 1), i = (o - g * (head_dim >> 1)) * 2u;
    float A = 0.f, B = 0.f;
#pragma unroll
    for (int u = 0; u < kAttnInlineSplits; ++u) {
      const float w = wts[g * kAttnInlineSplits + u];
      A = fmaf(__uint_as_float((uint32_t)v[u]), w, A);
      B = fmaf(__uint_as_float((uint32_t)(v[u] >> 32)), w, B);
    }
    const float L = tot[g];
    reinterpret_cast<__half2*>(ctx + (size_t)(kvh * groups + g) * head_dim + i)[0] = __floats2half2_rn(A / L, B / L);
    if (o + kAttnThreads < n_pairs) fetch(o + kAttnThreads);
  }
  if (tid == 0) counters[kvh] = 0;  // ready for the next launch
}

// Merge of the attention partials as a kernel of its own, for more ranges than the last workgroup merges by itself: a workgroup per query head,
// four lanes to an output dimension, each with sixteen ranges.  What bounds it is round trips to memory: all of a lane's values are
// asked for before the first is looked at, the weights are a wavefront's own.  (A lane to a dimension, eight ranges at a time, behind three
// barriers for the weights: 5.7 us for 64 ranges; eight tokens of four 14B layers at 8100 positions 4470 us, 4380 so.)
constexpr uint32_t kMergeParts = 4;  // of the ranges, two wavefronts each
__global__ __launch_bounds__(kMergeParts * 128) void attn_merge_kernel(const float* __restrict__ part, __half* __restrict__ ctx,
                                                                      uint32_t head_dim, uint32_t n_splits) {
  __shared__ float sums[kMergeParts][128];
  static_assert(kAttnMaxSplits <= 64, "a range's maximum and sum to a lane");
  constexpr uint32_t kRanges = kAttnMaxSplits / kMergeParts;
  const uint32_t head = blockIdx.x, tid = threadIdx.x, lane = tid & 63u, i = tid & 127u;
  const uint32_t p = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 7)), stride = head_dim + 2u;
  const float* src = part + (size_t)head * n_splits * stride;
  // Everything is asked for at once (past the last range: the last again, not added).
  const uint32_t mine = min(lane, n_splits - 1u) * stride, col = 2u + min(i, head_dim - 1u);
  const float m = src[mine], l = src[mine + 1u];
  float v[kRanges];
#pragma unroll
  for (uint32_t u = 0; u < kRanges; ++u) v[u] = src[min(p * kRanges + u, n_splits - 1u) * stride + col];
  const float mx = lane < n_splits ? m : -INFINITY;
  float M = mx;
#pragma unroll
  for (int k = 1; k < 64; k <<= 1) M = fmaxf(M, __shfl_xor(M, k));
  const float w = lane < n_splits ? __expf(mx - M) : 0.f;
  const float L = wave_sum(lane < n_splits ? l * w : 0.f);
  float A = 0.f;
#pragma unroll
  for (uint32_t u = 0; u < kRanges; ++u) {
    const float sum = fmaf(v[u], __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), p * kRanges + u)), A);
    A = p * kRanges + u < n_splits ? sum : A;  // (0 x infinity, of the last range's repeats, would reach the sums)
  }
  sums[p][i] = A;
  __syncthreads();
  if (tid >= head_dim) return;
  float t = sums[0][i];
#pragma unroll
  for (uint32_t k = 1; k < kMergeParts; ++k) t += sums[k][i];
  ctx[(size_t)head * head_dim + i] = __float2half_rn(t / L);
}

// act = f16(f16(silu(gate)) * up)   (model.rs:831: gu[0].apply(act).mul(gu[1]))
// Eight values per lane and turn (two bytes at a time 500 rows of 9728 took 6.9 us); what is over eight goes one by one.
__global__ __launch_bounds__(256) void silu_mul_kernel(const __half* __restrict__ gate, const __half* __restrict__ up,
                                                       __half* __restrict__ out, uint32_t n) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n / 8u; i += gridDim.x * blockDim.x) {
    const HalfOctet g = *reinterpret_cast<const HalfOctet*>(gate + i * 8u), u = *reinterpret_cast<const HalfOctet*>(up + i * 8u);
    HalfOctet o;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      o.w[j] = (uint32_t)__half_as_ushort(__float2half_rn(silu_mul(half_lo(g.w[j]), half_lo(u.w[j])))) |
               (uint32_t)__half_as_ushort(__float2half_rn(silu_mul(half_hi(g.w[j]), half_hi(u.w[j])))) << 16;
    *reinterpret_cast<HalfOctet*>(out + i * 8u) = o;
  }
  const uint32_t i = (n & ~7u) + threadIdx.x;
  if (blockIdx.x == 0 && i < n) out[i] = __float2half_rn(silu_mul(__half2float(gate[i]), __half2float(up[i])));
}

// ---- head -------------------------------------------------------------------------------
// Bound by the read of the head.  One row under way in a wavefront, its loads waiting for the sum of the row before, read
// 151936 rows at 5.5 TB/s (2560 columns in binary16, 140 us) and 5.0 TB/s (5120 in int8, 165 us).  Two rows together, the
// next chunk's loads ahead of this chunk's products and non-temporal (each line is read once): 116 us and 132 us, 6.7 and
// 6.3 TB/s.  Three or four rows (122 and 137 us) have more in flight than the memory takes and a longer last turn.
constexpr int kHeadThreads = 256;
constexpr uint32_t kHeadRows = 2;
// Workgroups to a CU: four took 120 us and 131 us, two 140 us and 165 us; with 2000 to 60000 rows, too, no other number was faster.
constexpr uint32_t kHeadGroups = 3;
typedef uint32_t head_u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ head_u32x4 head_load(const void* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const head_u32x4*>(p));
}

// logits = f16(E h) and every wavefront's best (value, row), lowest row on ties.  W: kValues a lane holds of a chunk,
// Piece, load(row, chunk), dot(piece, h, a) in the order of the row.  A wavefront holds kHeadRows rows together; the
// next chunk's loads, also those of the next rows, leave before this chunk's products.  A row past the end repeats the
// wavefront's first and is not stored, a lane past the row's end the last chunk, which it does not add.
template <class W>
__device__ __forceinline__ void head_rows(const W& w, const __half* __restrict__ h, uint32_t vocab, uint32_t hidden,
                                          float* __restrict__ hs, float* __restrict__ logits, float* __restrict__ best_val,
                                          uint32_t* __restrict__ best_idx) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t gw = __builtin_amdgcn_readfirstlane(blockIdx.x * (kHeadThreads / 64) + (threadIdx.x >> 6));
  const uint32_t nw = gridDim.x * (kHeadThreads / 64);
  const uint32_t chunks = hidden / W::kValues, rounds = (chunks + 63u) >> 6;
  typename W::Piece p[kHeadRows];
  const auto request = [&](uint32_t r0, uint32_t c) {  // r0 < vocab
    const uint32_t cl = min(c * 64u + lane, chunks - 1u);
#pragma unroll
    for (uint32_t i = 0; i < kHeadRows; ++i) {
      const uint32_t r = r0 + i * nw;
      p[i] = w.load(r < vocab ? r : r0, cl);
    }
  };
  if (gw < vocab) request(gw, 0);
  for (uint32_t i = threadIdx.x; i < hidden; i += kHeadThreads) hs[i] = __half2float(h[i]);
  __syncthreads();
  float bv = -INFINITY;
  uint32_t bi = 0xFFFFFFFFu;
  for (uint32_t r0 = gw; r0 < vocab; r0 += kHeadRows * nw) {
    float a[kHeadRows] = {};
    for (uint32_t c = 0; c < rounds; ++c) {
      typename W::Piece now[kHeadRows];
#pragma unroll
      for (uint32_t i = 0; i < kHeadRows; ++i) now[i] = p[i];
      const bool more = c + 1u < rounds;
      const uint32_t rn = more ? r0 : r0 + kHeadRows * nw;
      if (rn < vocab) request(rn, more ? c + 1u : 0u);
      const uint32_t cl = c * 64u + lane;
      if (cl < chunks) {
#pragma unroll
        for (uint32_t i = 0; i < kHeadRows; ++i) a[i] = W::dot(now[i], hs + cl * W::kValues, a[i]);
      }
    }
#pragma unroll
    for (uint32_t i = 0; i < kHeadRows; ++i) {
      const uint32_t r = r0 + i * nw;
      const float l = __half2float(__float2half_rn(wave_sum(a[i])));
      if (r >= vocab) break;
      if (lane == 0) logits[r] = l;
      if (l > bv) {  // rows ascend inside a wavefront, so '>' keeps the lowest row of a tie
        bv = l;
        bi = r;
      }
    }
  }
  if (lane == 0) {
    best_val[gw] = bv;
    best_idx[gw] = bi;
  }
}

// Dense binary16 head (Head::project, model.rs:578-587): eight values a lane and load, f32 accumulate.
struct HalfHead {
  static constexpr uint32_t kValues = 8;
  struct Piece {
    head_u32x4 u;
  };
  const __half* E;
  uint32_t hidden;
  __device__ __forceinline__ Piece load(uint32_t r, uint32_t c) const { return {head_load(E + (size_t)r * hidden + c * 8u)}; }
  static __device__ __forceinline__ float dot(const Piece& p, const float* h, float a) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      a = fmaf(half_lo(p.u[j]), h[2 * j], a);
      a = fmaf(half_hi(p.u[j]), h[2 * j + 1], a);
    }
    return a;
  }
};

__global__ __launch_bounds__(kHeadThreads) void lm_head_kernel(const __half* __restrict__ E, const __half* __restrict__ h,
                                                               uint32_t vocab, uint32_t hidden, float* __restrict__ logits,
                                                               float* __restrict__ best_val, uint32_t* __restrict__ best_idx) {
  extern __shared__ __align__(16) float hs[];  // [hidden]
  head_rows(HalfHead{E, hidden}, h, vocab, hidden, hs, logits, best_val, best_idx);
}

// ---- int8 embedding / head (llvq-llm/kernels/emb_q8.cu) --------------------------------
// One byte per weight, binary16 scale and bias per group of 64 along the row
// (llvq-artifact/src/sealed.rs:64-78): weight = f32(s * q) + b.
constexpr uint32_t kEmbedGroup = 64;
struct QuantRows {
  const uint8_t* q;      // [rows, d]
  const __half* scales;  // [rows, ceil(d / 64)]
  const __half* biases;
};

__device__ __forceinline__ float q8_weight(uint32_t q, float s, float b) {
  return __fadd_rn(__fmul_rn(s, (float)q), b);
}

// h = f16(embedding row of *token)   (emb_q8_gather)
__global__ __launch_bounds__(256) void embed_q8_kernel(QuantRows e, const uint32_t* __restrict__ token, uint32_t value, uint32_t vocab,
                                                       uint32_t hidden, __half* __restrict__ h) {
  const uint32_t t = min(token ? token[blockIdx.y] : value, vocab - 1u);
  h += (size_t)blockIdx.y * hidden;
  const uint32_t gpr = (hidden + kEmbedGroup - 1) / kEmbedGroup;
  for (uint32_t c = blockIdx.x * blockDim.x + threadIdx.x; c < hidden; c += gridDim.x * blockDim.x) {
    const size_t g = (size_t)t * gpr + c / kEmbedGroup;
    h[c] = __float2half_rn(q8_weight(e.q[(size_t)t * hidden + c], __half2float(e.scales[g]), __half2float(e.biases[g])));
  }
}

// int8 head (tv_q8_h): 16 codes per lane and load (a 16-byte run never straddles a group of 64).
struct QuantHead {
  static constexpr uint32_t kValues = 16;
  struct Piece {
    head_u32x4 u;
    __half s, b;
  };
  QuantRows e;
  uint32_t hidden, gpr;
  __device__ __forceinline__ Piece load(uint32_t r, uint32_t c) const {
    const size_t g = (size_t)r * gpr + (c >> 2);
    return {head_load(e.q + (size_t)r * hidden + c * 16u), e.scales[g], e.biases[g]};
  }
  static __device__ __forceinline__ float dot(const Piece& p, const float* h, float a) {
    const float s = __half2float(p.s), b = __half2float(p.b);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int t = 0; t < 4; ++t) a = fmaf(q8_weight((p.u[j] >> (8 * t)) & 0xFFu, s, b), h[4 * j + t], a);
    return a;
  }
};

__global__ __launch_bounds__(kHeadThreads) void lm_head_q8_kernel(QuantRows e, const __half* __restrict__ h, uint32_t vocab,
                                                                  uint32_t hidden, float* __restrict__ logits,
                                                                  float* __restrict__ best_val, uint32_t* __restrict__ best_idx) {
  extern __shared__ __align__(16) float hs[];  // [hidden]
  head_rows(QuantHead{e, hidden, (hidden + kEmbedGroup - 1) / kEmbedGroup}, h, vocab, hidden, hs, logits, best_val, best_idx);
}

// token = argmax over the wavefront winners; lowest row on ties.  Where the caller wants the results, workgroup 0 leaves the token in pinned host
// memory as well, and the others, 4096 values each, the logits: a copy enqueued behind the launch is the copy engine's, which waits
// for the launch by a signal.  (Eight tokens of a 4B model with 151936 logits each 11 640 us with that copy, 11 425 so; four 14B layers 4280 and
// 4110.  Stored by the head itself, a row at a time, they would be writes of four bytes.)
// What bounds workgroup 0 is its round trips: its values are asked for together, and meet in lane moves and one pass over LDS.
constexpr int kFinalThreads = 1024;
constexpr uint32_t kFinalCopy = 4u * kFinalThreads;  // logits of a workgroup
constexpr int kFinalRounds = 4;                      // values of a lane that are asked for together
struct HostResults {  // pinned memory, each null where it is not wanted
  float* logits;
  uint32_t* token;
};
__global__ __launch_bounds__(kFinalThreads) void argmax_final_kernel(const float* __restrict__ best_val, const uint32_t* __restrict__ best_idx,
                                                                     uint32_t n, uint32_t* __restrict__ token_out, uint32_t* __restrict__ history,
                                                                     uint32_t slot, const float* __restrict__ logits, uint32_t vocab, HostResults host) {
  if (blockIdx.x) {
    const uint32_t at = (blockIdx.x - 1u) * kFinalCopy + threadIdx.x * 4u;
    if (at + 4u <= vocab) *reinterpret_cast<float4*>(host.logits + at) = *reinterpret_cast<const float4*>(logits + at);
    else
      for (uint32_t i = at; i < vocab; ++i) host.logits[i] = logits[i];
    return;
  }
  __shared__ float sv[kFinalThreads / 64];
  __shared__ uint32_t si[kFinalThreads / 64];
  float bv = -INFINITY;
  uint32_t bi = 0xFFFFFFFFu;
  const auto take = [&](float v, uint32_t id) {
    const bool better = v > bv || (v == bv && id < bi);
    bv = better ? v : bv;
    bi = better ? id : bi;
  };
  const auto wavefront = [&]() {
#pragma unroll
    for (int k = 1; k < 64; k <<= 1) {
      const float v = __shfl_xor(bv, k);
      const uint32_t id = (uint32_t)__shfl_xor((int)bi, k);
      take(v, id);
    }
  };
  for (uint32_t i0 = threadIdx.x; i0 < n; i0 += kFinalRounds * kFinalThreads) {
    float v[kFinalRounds];
    uint32_t id[kFinalRounds];
#pragma unroll
    for (int u = 0; u < kFinalRounds; ++u) {  // (past the last: the last again)
      const uint32_t i = min(i0 + u * kFinalThreads, n - 1u);
      v[u] = best_val[i];
      id[u] = best_idx[i];
    }
#pragma unroll
    for (int u = 0; u < kFinalRounds; ++u) take(v[u], id[u]);
  }
  wavefront();
  if ((threadIdx.x & 63u) == 0) {
    sv[threadIdx.x >> 6] = bv;
    si[threadIdx.x >> 6] = bi;
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;
  bv = sv[threadIdx.x % (kFinalThreads / 64)];
  bi = si[threadIdx.x % (kFinalThreads / 64)];
  wavefront();
  if (threadIdx.x == 0) {
    *token_out = bi;
    if (history) history[slot] = bi;
    if (host.token) *host.token = bi;
  }
}

}  // namespace llvq
