// A sequence of group products in ONE launch.  Included by llvq_hip.hip after tiles.h, whose steps, planes and record
// layout it shares.
//
// The reference issues two launches per projection and notes that launch latency is about half of a decode token
// (llvq-llm/src/fused_cuda.rs:789-795).  Here the records of every item of a list — an item is what one
// llvq_hip_gemv_group call would be — are cut into units of one workgroup's worth and one persistent 1024-lane
// workgroup per CU walks its share of them without stopping at an item's end but to stage the next activation.
//
//   * Independent items: a workgroup takes one contiguous run of units, the runs equal in bytes, so that it meets two or
//     three items of a model's 144 and streams the rest.  What bounds it is HBM: 13.x bytes per block at 4.6 to 5.2 TB/s; the planes of an
//     item sit in registers, a step's registers are loaded again for the next unit as soon as they have been used
//     (16 wavefronts x 4 steps x 832 bytes in flight per CU), and the sums over a team's wavefronts need no barrier: the
//     wavefront that arrives last at a record's counter in LDS adds them up and stores.  A barrier every four units only
//     bounds how far the wavefronts drift apart (eight record slots).
//   * Ordered items (`wait_item`): the units of an item are dealt round-robin; before a workgroup reads an activation
//     that an earlier item stores it waits for that item's counter, which every workgroup bumps when its last rows of
//     it have arrived in memory (outputs and activations are stored and loaded at device scope, past the XCDs' own L2s).
//     The first unit's weights are requested before the wait.  A workgroup only ever waits for items below the one it is
//     working on and takes its units in ascending order, so with every workgroup resident (grid <= CUs, one workgroup per
//     CU, the device otherwise idle) the waits end.  They are bounded all the same: a wait that reaches `spin_limit`
//     polls sets `*status` and the workgroup returns, which makes every wait behind it give up in turn.
//
// Results are those of the per-item launches bit for bit: a record's split over wavefronts and every order of addition
// depend on the row length alone.
#pragma once

namespace llvq {

constexpr uint32_t kSeqNoWait = 0xFFFFFFFFu;
constexpr uint32_t kSeqSlots = 8;    // records per team whose sums may be pending
constexpr uint32_t kSeqDrift = 4;    // units between two barriers: half of kSeqSlots

struct SeqUnit {           // up to 16 >> split_shift consecutive records of one matrix
  const uint8_t* rec;      // the first record
  const uint32_t* table;   // the matrix's scales
  void* y;                 // the first record's first output element
  uint32_t rows;           // rows of the unit
  uint32_t item;
};
static_assert(sizeof(SeqUnit) == 32, "unit descriptors are read with scalar loads");

struct SeqItem {
  const __half* x;        // the activation, or the prologue's first operand
  const __half* x2;
  const __half* norm_w;
  __half* resid_out;      // stored by the workgroup that takes the item's first unit
  float eps;
  uint32_t prologue;      // kPrologue*
  uint32_t nb, tail_w;
  uint32_t first_unit;
  uint32_t wait_item;     // kSeqNoWait, or the item that must be complete before the activation is read
  uint32_t expected;      // workgroups that take part in this item
  uint32_t signals;       // a later item waits for this one
  uint32_t wait_expected; // `expected` of wait_item
  uint32_t pad[3];
};
static_assert(sizeof(SeqItem) == 80, "item records are read with scalar loads");

struct SeqArgs {
  const SeqUnit* units;
  const SeqItem* items;
  const uint32_t* runs;  // [grid + 1] where each workgroup's run of units begins, or null: dealt round-robin
  uint32_t n_units, max_blocks;  // max_blocks: plane blocks of the widest item
  uint32_t* counters;    // per item: workgroups that have finished it, counted on from run to run
  uint32_t* status;      // set to 1 by a workgroup that gave up waiting
  uint32_t run;          // 1, 2, ...: item i is complete in this run at counters[i] == run * expected
  uint32_t spin_limit;
  uint32_t hold_item;    // kSeqNoWait, or an item this run must treat as never complete (tests of the give-up path)
};

// What a sequence may contain, as far as its kernel has to know.
enum : int {
  kSeqIndependent = 0,      // no item waits, no prologue
  kSeqIndependentWide = 1,  // the same with rows past 512 blocks
  kSeqOrdered = 2,          // items may wait
  kSeqPrologue = 3,         // items may wait and derive their activation
  kSeqPrologueWide = 4      // the same with rows past 512 blocks
};

__host__ __device__ inline size_t gemv_seq_lds_bytes(uint32_t max_blocks, bool f32_out) {
  const size_t planes = (size_t)max_blocks * (f32_out ? XPlanes<6>::kDwords : XPlanes<4>::kDwords) * 4;
  return gemv_lds_fixed() + planes + 2 * kSeqSlots * kGemvMaxWaves * 8 * 4 + kSeqSlots * kGemvMaxWaves * 4 + 16;
}

// The tables are the same for every lane and no kernel writes them: read through the constant address space, they come by
// scalar loads.  As vector loads they would retire behind the weights in flight.
template <typename T>
__device__ __forceinline__ T scalar_read(const T* p) {
  static_assert(sizeof(T) % 4 == 0, "read dword by dword");
  typedef const uint32_t __attribute__((address_space(4))) const_u32;
  struct Raw { uint32_t w[sizeof(T) / 4]; } raw;
  const_u32* src = (const_u32*)reinterpret_cast<const uint32_t*>(p);
#pragma unroll
  for (uint32_t i = 0; i < sizeof(T) / 4; ++i) raw.w[i] = src[i];
  return __builtin_bit_cast(T, raw);
}
__device__ __forceinline__ SeqUnit seq_unit_at(const SeqUnit* units, uint32_t i) {
  SeqUnit u = scalar_read(units + i);
  u.rec = uniform_global(u.rec);
  u.table = uniform_global(u.table);
  u.y = uniform_global(u.y);
  return u;
}

template <typename OutT, int MODE>
__global__ __launch_bounds__(1024) void gemv_seq_kernel(SeqArgs s) {
  constexpr int DIG = std::is_same<OutT, __half>::value ? 4 : 6;
  constexpr bool kWide = MODE == kSeqIndependentWide || MODE == kSeqPrologueWide;
  constexpr bool kWaits = MODE >= kSeqOrdered, kPro = MODE >= kSeqPrologue;
  constexpr uint32_t kSteps = kWide ? kGemvWideSteps : kGemvSteps;
  constexpr uint32_t kStr = XPlanes<DIG>::kDwords;
  extern __shared__ __align__(16) uint8_t smem[];
  GemvLds L;
  L.xtail = reinterpret_cast<float*>(smem);
  L.red = L.xtail + 32;
  L.planes = reinterpret_cast<uint32_t*>(L.red + 16);
  L.part = reinterpret_cast<float*>(L.planes + (size_t)s.max_blocks * kStr);
  L.tpart = L.part + kSeqSlots * kGemvMaxWaves * 8;
  L.xf = nullptr;
  uint32_t* arrived = reinterpret_cast<uint32_t*>(L.tpart + kSeqSlots * kGemvMaxWaves * 8);  // [slot][team]
  uint32_t* verdict = arrived + kSeqSlots * kGemvMaxWaves;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, r = lane & 7u, bq = lane >> 3;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  uint32_t u = s.runs ? scalar_read(s.runs + blockIdx.x) : blockIdx.x;
  const uint32_t u_end = s.runs ? scalar_read(s.runs + blockIdx.x + 1u) : s.n_units, u_step = s.runs ? 1u : gridDim.x;

  uint32_t it = kSeqNoWait, it_signals = 0;  // the item whose activation is in LDS
  uint32_t nb = 0, tail_w = 0, shift = 2, split = 4, team = 0, w = 0, stride = 0, head = 0, n_steps = 0;
  const LaneOffsets at = lane_offsets(lane);
  uint32_t tail_c = 0, tail_off = 0, tail_waves = 0;
  RecordWords<kSteps> W;
  uint32_t slot = 0;
  // this wavefront's record of a unit
  auto request = [&](const SeqUnit& q) {
    const bool mine = team * kTileRows < q.rows;
    const uint8_t* rec = q.rec + (mine ? team * stride : 0u);
    load_record(W, rec, reinterpret_cast<const uint8_t*>(q.table), head, w, split, n_steps, mine, tail_off, lane, at);
  };
  // Every store of this workgroup for item `it` has arrived in memory: tell the items that wait for it.  (The rows went
  // out as device-scope stores; no fence, which would flush or empty the XCD's L2.)
  auto signal_item = [&]() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    if (tid == 0) __hip_atomic_fetch_add(s.counters + it, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };

  if (u >= u_end) return;  // the same for every lane of the workgroup
  SeqUnit cur = seq_unit_at(s.units, u);
  bool last = false;
  for (;;) {  // an item (everything that decides a branch outside a wavefront's own steps is the same for every lane)
    if (it != kSeqNoWait) {
      if (kWaits && it_signals) signal_item();
      else lds_barrier();  // the old planes and slots are no longer read
    }
    const SeqItem I = scalar_read(s.items + cur.item);
    nb = I.nb;
    tail_w = I.tail_w;
    shift = gemv_split_shift(nb);
    split = 1u << shift;
    team = wave >> shift;
    w = wave & (split - 1u);
    n_steps = (nb + 7u) >> 3;
    stride = tile_stride(nb, tail_w);
    head = tile_head_bytes(tail_w);
    tail_c = w * 8u + bq;
    tail_off = tail_c < tail_w ? 32u + tail_c * 32u + r * 4u : 0u;
    tail_waves = (tail_w + 7u) >> 3;
    if (tid < kSeqSlots * kGemvMaxWaves) arrived[tid] = 0;
    slot = 0;
    ActivationIn in{};
    in.x = uniform_global(I.x);
    if constexpr (kPro) {
      in.x2 = uniform_global(I.x2);
      in.norm_w = uniform_global(I.norm_w);
      in.resid_out = uniform_global(I.resid_out);
      in.eps = I.eps;
      in.prologue = I.prologue;
    }
    if constexpr (kWaits) {
      if constexpr (!kWide) request(cur);  // the weights do not depend on the item before
      if (I.wait_item != kSeqNoWait) {
        if (tid == 0) {
          const uint32_t target = s.run * I.wait_expected + (I.wait_item == s.hold_item ? 1u : 0u);
          uint32_t ok = 0;
          for (uint32_t spins = 0; spins <= s.spin_limit; ++spins) {
            const uint32_t v = __hip_atomic_load(s.counters + I.wait_item, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((int32_t)(v - target) >= 0) { ok = 1; break; }
            __builtin_amdgcn_s_sleep(1);
          }
          *verdict = ok;
          if (!ok) __hip_atomic_store(s.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        lds_barrier();
        if (*verdict == 0) return;  // gave up: every lane leaves, and so will whoever waits for this workgroup
      }
    }
    auto ask = [&] { if constexpr (!kWaits && !kWide) request(cur); };
    constexpr int kPasses = kWide ? 4 : 2;
    const bool resid = u == I.first_unit;
    if (kPro && I.prologue == kPrologueSiluMul) stage_x<DIG, kSrcSiluMul, kPasses, kWaits>(in, nb, tail_w, L, resid, ask);
    else if (kPro && I.prologue == kPrologueAddRmsNorm) stage_x<DIG, kSrcAddRmsNorm, kPasses, kWaits>(in, nb, tail_w, L, resid, ask);
    else stage_x<DIG, kSrcF16, kPasses, kWaits>(in, nb, tail_w, L, false, ask);
    if constexpr (kWide) request(cur);  // (the registers are the staging's until here)
    lds_barrier();
    it = cur.item;
    it_signals = I.signals;
    for (;;) {  // its units
      const uint32_t un = u + u_step;
      last = un >= u_end;
      const SeqUnit next = seq_unit_at(s.units, last ? u : un);
      if (slot && slot % kSeqDrift == 0) lds_barrier();
      const bool mine = team * kTileRows < cur.rows;  // whether this wavefront has a record of the unit, and of the next
      const bool more = !last & (next.item == it) & (team * kTileRows < next.rows);
      const uint8_t* nrec = next.rec + (more ? team * stride : 0u);
      const uint32_t table = W.table;
      const float row_scale = W.scale, tail = W.tail;
      W.table = next.table[lane & 31u];  // first, so that the next unit waits for them alone
      W.tail = *reinterpret_cast<const float*>(nrec + (more ? tail_off : 0u));
      W.scale = reinterpret_cast<const float*>(nrec)[r];
      float acc = 0.f;
#pragma unroll
      for (uint32_t j = 0; j < kSteps; ++j) {
        const uint32_t step = w + j * split;
        acc = step_product<DIG>(W.step[j], load_xblock<DIG>(L.planes + (min(step, n_steps) * 8u + bq) * kStr), table, r, acc);
        __builtin_amdgcn_sched_barrier(0);
        W.step[j] = load_step(nrec + head, step, more & (step < n_steps), at);
        __builtin_amdgcn_sched_barrier(0);
      }
      acc = row8_sum(acc);
      if (mine) {
        float* p = L.part + ((slot % kSeqSlots) * kGemvMaxWaves + wave) * 8u;
        float* q = L.tpart + ((slot % kSeqSlots) * kGemvMaxWaves + wave) * 8u;
        if (lane < 8u) p[lane] = acc;
        if (w < tail_waves) {
          const float t = row8_sum(tail_c < tail_w ? tail * L.xtail[tail_c] : 0.f);
          if (lane < 8u) q[lane] = t;
        }
        // whoever sees the count complete sees the sums of the wavefronts that counted
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        uint32_t n = 0;
        if (lane == 0) n = __hip_atomic_fetch_add(arrived + (slot % kSeqSlots) * kGemvMaxWaves + team, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        n = (uint32_t)__builtin_amdgcn_readfirstlane((int)n);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        if (((n + 1u) & (split - 1u)) == 0u) {
          p -= w * 8u;
          q -= w * 8u;
          const float v = team_sum(p, q, row_scale, split, tail_waves, lane);
          const uint32_t row = team * kTileRows + r;
          if (lane < 8u && row < cur.rows) {
            if constexpr (kWaits) {  // a later item of this launch may read it from another XCD
              if constexpr (std::is_same<OutT, __half>::value) store_half<true>(reinterpret_cast<__half*>(cur.y) + row, __float2half_rn(v));
              else __hip_atomic_store(reinterpret_cast<float*>(cur.y) + row, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            } else {
              store_out<OutT>(cur.y, row, v);
            }
          }
        }
      }
      ++slot;
      if (last) break;
      cur = next;
      u = un;
      if (cur.item != it) break;
    }
    if (last) break;
  }
  if (kWaits && it_signals) signal_item();
}

template <typename OutT>
__host__ const void* seq_kernel_of(int mode) {
  switch (mode) {
    case kSeqIndependent: return reinterpret_cast<const void*>(gemv_seq_kernel<OutT, kSeqIndependent>);
    case kSeqIndependentWide: return reinterpret_cast<const void*>(gemv_seq_kernel<OutT, kSeqIndependentWide>);
    case kSeqOrdered: return reinterpret_cast<const void*>(gemv_seq_kernel<OutT, kSeqOrdered>);
    case kSeqPrologue: return reinterpret_cast<const void*>(gemv_seq_kernel<OutT, kSeqPrologue>);
    default: return reinterpret_cast<const void*>(gemv_seq_kernel<OutT, kSeqPrologueWide>);
  }
}

}  // namespace llvq
