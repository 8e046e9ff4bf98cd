// A sequence of group products in ONE launch.  Included by llvq_hip.hip after tiles.h, whose steps, planes and record
// layout it shares.
//
// The reference issues two launches per projection and notes that launch latency is about half of a decode token
// (llvq-llm/src/fused_cuda.rs:789-795).  Here the tiles of every item of a list — an item is what one
// llvq_hip_gemv_group call would be — are shared out over one persistent 1024-lane workgroup per CU, which walks its share
// without stopping at an item's end but to stage the next activation.
//
//   * Independent items: a workgroup takes one contiguous run of tiles, the runs equal in bytes, so that it meets two or
//     three items of a model's 144 and streams the rest.  What bounds it is HBM: 10.x bytes per block, 252 matrices
//     of a 4B model 387 -> 265 us, 5.1 -> 5.8 TB/s (13 bytes before, in lines shared between loads).  A wavefront takes
//     up to four steps of a tile at a time (a task; two where a launch is short); a step's registers are loaded again, piece by piece, for its next
//     step, in this task or the one after, as soon as they have been used: sixteen wavefronts x 5 KB in flight per CU.
//     Rows of one task are a wavefront's own; of wider ones the sums of the steps meet in LDS, the
//     wavefront that arrives last at a tile's counter adds them up and stores, and a barrier every kSeqDrift tasks
//     bounds how far the wavefronts drift apart.
//   * Ordered items (`wait_item`): a step is a task, the tiles are dealt out evenly; before a workgroup reads an activation
//     that an earlier item stores it waits for that item's counter, which every workgroup bumps when its last rows of
//     it have arrived in memory (outputs and activations are stored and loaded at device scope, past the XCDs' own L2s).
//     The first tasks' weights are requested before the wait.  A workgroup only ever waits for items below the one it is
//     working on and takes its units in ascending order, so with every workgroup resident (grid <= CUs, one workgroup per
//     CU, the device otherwise idle) the waits end.  They are bounded all the same: a wait that reaches `spin_limit`
//     polls sets `*status` and the workgroup returns, which makes every wait behind it give up in turn.
//
// Results are those of the per-item launches bit for bit: every order of addition depends on the row length alone.
#pragma once

namespace llvq {

constexpr uint32_t kSeqNoWait = 0xFFFFFFFFu;
struct SeqUnit {           // consecutive tiles of one matrix
  const uint8_t* rec;      // the first tile
  const uint32_t* table;   // the matrix's scales
  void* y;                 // the first tile's first output element
  uint32_t rows;           // rows of the unit
  uint32_t item;
  uint32_t stride, slots;  // of the matrix's tiles
  uint32_t pad[2];
};
static_assert(sizeof(SeqUnit) == 48, "unit descriptors are read with scalar loads");

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
  uint32_t tasks;         // tasks of a tile, its steps shared out evenly
  uint32_t inv_tasks;     // 2^32 / tasks, rounded up (tasks > 1)
  uint32_t pad;
};
static_assert(sizeof(SeqItem) == 80, "item records are read with scalar loads");

struct SeqArgs {
  const SeqUnit* units;
  const SeqItem* items;
  const uint32_t* runs;  // [grid + 1] where each workgroup's run of units begins, or null: dealt round-robin
  uint32_t n_units, max_units;  // max_units: plane units of the widest item
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

__host__ __device__ inline size_t gemv_seq_lds_bytes(uint32_t max_units, bool f32_out) {
  const size_t planes = (size_t)max_units * (f32_out ? XPlanes<6>::kDwords : XPlanes<4>::kDwords) * 4;
  return gemv_lds_fixed() + planes + (kSeqPartSteps + 2 * kSeqMaxSlots) * kTileRows * 4 + kSeqMaxSlots * 4 + 16;
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
  extern __shared__ __align__(16) uint8_t smem[];
  GemvLds L;
  L.xtail = reinterpret_cast<float*>(smem);
  L.red = L.xtail + 32;
  L.planes = reinterpret_cast<uint32_t*>(L.red + 16);
  L.part = reinterpret_cast<float*>(L.planes + (size_t)s.max_units * XPlanes<DIG>::kDwords);  // [slot][step][16 rows]
  L.xf = nullptr;
  float* const tpart = L.part + kSeqPartSteps * kTileRows;                                      // [slot][16 rows] what tile_extras gives,
  float* const scales = tpart + kSeqMaxSlots * kTileRows;                                       // and the row scales
  uint32_t* arrived = reinterpret_cast<uint32_t*>(scales + kSeqMaxSlots * kTileRows);           // [slot]
  uint32_t* verdict = arrived + kSeqMaxSlots;
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  uint32_t u = s.runs ? scalar_read(s.runs + blockIdx.x) : blockIdx.x;
  const uint32_t u_end = s.runs ? scalar_read(s.runs + blockIdx.x + 1u) : s.n_units, u_step = s.runs ? 1u : gridDim.x;

  uint32_t it = kSeqNoWait, it_signals = 0;  // the item whose activation is in LDS
  // Every store of this workgroup for item `it` has arrived in memory: tell the items that wait for it.  (The rows went
  // out as device-scope stores; no fence, which would flush or empty the XCD's L2.)
  auto signal_item = [&]() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    if (tid == 0) __hip_atomic_fetch_add(s.counters + it, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };

  if (u >= u_end) return;  // the same for every lane of the workgroup
  SeqUnit first = seq_unit_at(s.units, u);
  if (tid < kSeqMaxSlots) arrived[tid] = 0;
  for (;;) {  // an item (everything that decides a branch outside a wavefront's own tasks is the same for every lane)
    if (it != kSeqNoWait) {
      if (kWaits && it_signals) signal_item();
      else lds_barrier();  // the old planes and slots are no longer read
    }
    const SeqItem I = scalar_read(s.items + first.item);
    const uint32_t nb = I.nb, tail_w = I.tail_w, n_steps = tile_steps(nb), units = tile_units(nb), head = tile_head_bytes(tail_w);
    const uint32_t tasks = I.tasks, long_steps = n_steps / tasks, long_tasks = n_steps - long_steps * tasks, slots = seq_slots(tasks);
    it = first.item;
    it_signals = I.signals;
    // The workgroup's units of the item, and the tasks in them.
    auto unit_tiles = [&](const SeqUnit& q) { return (q.rows + kTileRows - 1u) / kTileRows; };
    uint32_t total = 0, u_next = u;
    SeqUnit after = first;
    do {
      total += unit_tiles(after) * tasks;
      u_next += u_step;
      if (u_next >= u_end) break;
      after = seq_unit_at(s.units, u_next);
    } while (after.item == it);
    // Where this wavefront is in them: round r's tasks are the sixteen from 16 r on, its own another one of them each time
    // (a tile's tasks may differ in length, and their number divide sixteen).
    SeqUnit at = first;
    uint32_t at_u = u, at_task = 0, at_tile = 0;  // the unit, and the item's tasks and tiles in front of it
    struct Task {
      const uint8_t* rec;
      const uint8_t* table;
      uint8_t* y;
      uint32_t rows;         // of the tile that are there
      uint32_t step, end;    // steps [step, end)
      uint32_t part, slot;   // which of the tile's tasks; where its sums meet
      uint32_t list;         // places in the tile's list of escapes
      bool live;
    };
    auto task_of = [&](uint32_t round) {
      const uint32_t g = round * kSeqWaves + ((wave + round) & (kSeqWaves - 1u));
      const bool live = g < total;
      Task t;
      if (live)
        while (g - at_task >= unit_tiles(at) * tasks) {
          at_task += unit_tiles(at) * tasks;
          at_tile += unit_tiles(at);
          at_u += u_step;
          at = seq_unit_at(s.units, at_u);
        }
      const uint32_t k = live ? g - at_task : 0u, tile = tasks == 1u ? k : __umulhi(k, I.inv_tasks);
      t.part = k - tile * tasks;
      t.rec = at.rec + (size_t)tile * at.stride;
      t.list = at.slots;
      t.table = reinterpret_cast<const uint8_t*>(at.table);
      t.y = reinterpret_cast<uint8_t*>(at.y) + (size_t)tile * (kTileRows * sizeof(OutT));
      t.rows = at.rows - tile * kTileRows;
      t.step = t.part * long_steps + min(t.part, long_tasks);
      t.end = t.step + long_steps + (t.part < long_tasks ? 1u : 0u);
      t.slot = (at_tile + tile) % slots;
      t.live = live;
      return t;
    };
    const uint32_t rounds = (total + kSeqWaves - 1u) / kSeqWaves;
    StepWords W;
    uint32_t table;
    TileExtras extras{};
    auto load_head = [&](const Task& t) {  // a tile's first task sees to them
      if (t.live & (t.part == 0u)) extras = load_extras(t.rec, nb, tail_w, t.list, true, lane);
    };
    Task cur = task_of(0);
    auto request = [&]() {
      table = scale_table(cur.table, lane);
      load_head(cur);
      load_step(W, scalar_base(cur.rec), cur.live ? step_offset(cur.step, units, head, lane) : 0u);
    };
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
      request();  // the weights do not depend on the item before
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
    auto ask = [&] { if constexpr (!kWaits) request(); };
    constexpr int kPasses = kWide ? 4 : 2;
    const bool resid = u == I.first_unit;
    if (kPro && I.prologue == kPrologueSiluMul) stage_x<DIG, kSrcSiluMul, kPasses, kWaits>(in, nb, tail_w, kSeqWaves, stage_passes(nb, kSeqWaves), L, resid, ask);
    else if (kPro && I.prologue == kPrologueAddRmsNorm) stage_x<DIG, kSrcAddRmsNorm, kPasses, kWaits>(in, nb, tail_w, kSeqWaves, stage_passes(nb, kSeqWaves), L, resid, ask);
    else stage_x<DIG, kSrcF16, kPasses, kWaits>(in, nb, tail_w, kSeqWaves, stage_passes(nb, kSeqWaves), L, false, ask);
    lds_barrier();

    auto store_rows = [&](const Task& t, float v) {
      const uint32_t row = lane_row(lane);
      if (lane_class(lane) == 0u && row < t.rows) {
        if constexpr (kWaits) {  // a later item of this launch may read it from another XCD
          if constexpr (std::is_same<OutT, __half>::value) store_half<true>(reinterpret_cast<__half*>(t.y) + row, __float2half_rn(v));
          else __hip_atomic_store(reinterpret_cast<float*>(t.y) + row, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
          store_out<OutT>(t.y, row, v);
        }
      }
    };
    for (uint32_t round = 0; round < rounds; ++round) {
      if (tasks > 1u && round && round % kSeqDrift == 0) lds_barrier();
      const Task next = task_of(round + 1u);
      if (!cur.live) {  // (only in the last round)
        cur = next;
        continue;
      }
      const uint32_t lanes_table = table;
      float* const part = L.part + (size_t)(cur.slot * n_steps) * kTileRows;
      const float row_scale = extras.scale;
      float t = 0.f;
      if (cur.part == 0u) t = tile_extras<DIG>(extras, cur.rec, nb, tail_w, cur.list, lanes_table, L, lane);
      load_head(next);
      float even = 0.f, odd = 0.f;  // steps 0 and 1 of a tile that is one task, and 2 and 3
      for (uint32_t step = cur.step; step < cur.end; ++step) {
        const bool last = step + 1u == cur.end;
        if (last) table = scale_table(next.table, lane);  // in front of the pieces, so that the next task waits for it alone
        const uint8_t* base = scalar_base(last ? next.rec : cur.rec);
        const uint32_t off = last && !next.live ? 0u : step_offset(last ? next.step : step + 1u, units, head, lane);
        float lo, hi;
        step_product<DIG>(W, L.planes + (step * kStepUnits + (lane >> 3)) * XPlanes<DIG>::kDwords, lanes_table, lo, hi,
                          [&](auto piece) __attribute__((always_inline)) { load_piece<decltype(piece)::value>(W, base, off); });
        const float v = rows_sum(lo, hi);
        if (tasks == 1u) {
          if (step & 2u) odd += v;
          else even += v;
        } else if (lane_class(lane) == 0u) {
          part[step * kTileRows + lane_row(lane)] = v;
        }
      }
      if (tasks == 1u) {
        store_rows(cur, fmaf(even + odd, row_scale, t));
      } else {
        if (cur.part == 0u && lane_class(lane) == 0u) {
          tpart[cur.slot * kTileRows + lane_row(lane)] = t;
          scales[cur.slot * kTileRows + lane_row(lane)] = row_scale;
        }
        // whoever sees the count complete sees the sums of the wavefronts that counted
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        uint32_t n = 0;
        if (lane == 0) n = __hip_atomic_fetch_add(arrived + cur.slot, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        n = (uint32_t)__builtin_amdgcn_readfirstlane((int)n);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        if (n + 1u == tasks) {
          const float v = steps_sum<kGemvMaxBlocks / kStepBlocks>(part, n_steps, lane);
          store_rows(cur, fmaf(v, scales[cur.slot * kTileRows + lane_row(lane)], tpart[cur.slot * kTileRows + lane_row(lane)]));
          if (lane == 0) __hip_atomic_store(arrived + cur.slot, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
      }
      cur = next;
    }
    if (u_next >= u_end) break;
    u = u_next;
    first = after;
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
