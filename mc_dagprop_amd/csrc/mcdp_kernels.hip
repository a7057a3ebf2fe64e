// gfx950 kernels of the Monte Carlo DAG propagation path.
//
// walk_kernel fuses the two hot loops of Simulator::run (_core.cpp:323-329
// delay sampling, :332-350 max-plus propagation) for a tile of 64 x kSpl
// samples per workgroup: lane l of every wave carries samples
// tile * 64 kSpl + i * 64 + l, i < kSpl.
//   * plan records (event headers; predecessors with their distribution
//     inline) are wave-uniform and arrive through scalar loads, the next one
//     prefetched while the current one is processed; the distribution switch
//     is a scalar branch taken once for the lane's kSpl samples, whose draws
//     then run as independent instruction chains;
//   * the W waves of a workgroup split each step's events (a step is part of
//     one topological level); results stay in registers until a barrier, then
//     go to LDS slots that later steps read;
//   * LDS is slot-major, a slot holding 64 x kSpl doubles with a lane's
//     samples adjacent, so a lane reads or writes a slot with one ds_read_b64
//     or ds_read_b128;
//   * outputs are sample-contiguous rows, so each store instruction of a wave
//     writes a 512-byte run (nontemporal: nothing reads them back).
// The arithmetic of propagation is FP64 add and compare-select only, in the
// reference's order: t = realized[src] + dur; t = (upper < t) ? upper : t;
// if (t >= best) {best = t; cause = src}; realized = (upper < best) ? upper : best.
// std::min is (b < a) ? b : a, so a NaN candidate is never taken (the fast
// paths take v_min_f64 of a candidate that has won already, see capped_at).
//
// Bound by instruction issue: a wave-activity of the network workload takes
// 107 VALU instructions (4.3 cycles each on a SIMD, 2.4 for one- and
// two-operand 32-bit ones) for its two samples.  200 x 100 events, 100,000
// samples: 11.9 ms -> 11.2 with the integer-indexed logarithm, a lane's two
// draws side by side, output rows addressed by scalar base and lane offset and
// the cap as one instruction (63.8 GB of outputs, 5.7 TB/s; a plain fill of that
// size runs at 6.9); 32,768 samples 3.90 -> 3.57.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "mcdp_kernels.hpp"
#include "mcdp_sampler.hpp"

namespace mcdp {

// A lane's kSpl samples of one LDS slot.
template <int kSpl>
__device__ __forceinline__ void lds_load(const double *lds, int slot, int lane, double (&v)[kSpl]) {
    if constexpr (kSpl == 1) {
        v[0] = lds[slot * kLanes + lane];
    } else {
        static_assert(kSpl == 2, "one or two samples per lane");
        const double2 t = reinterpret_cast<const double2 *>(lds)[slot * kLanes + lane];
        v[0] = t.x;
        v[1] = t.y;
    }
}
template <int kSpl>
__device__ __forceinline__ void lds_store(double *lds, int slot, int lane, const double (&v)[kSpl]) {
    if constexpr (kSpl == 1) {
        lds[slot * kLanes + lane] = v[0];
    } else {
        reinterpret_cast<double2 *>(lds)[slot * kLanes + lane] = double2{v[0], v[1]};
    }
}

// Element offset of (row, column 0) in an array with leading dimension ld:
// a 32 x 32 -> 64-bit product (rows and ld are non-negative and < 2^31).
__device__ __forceinline__ uint64_t row_offset(int32_t row, uint32_t ld) { return (uint64_t)(uint32_t)row * ld; }

// Issue priority from the share of its step's records a wave has left: 3 in
// the first quarter down to 0 in the last.  A SIMD issues its oldest waves
// first at equal priority, so with equal work its youngest wave would finish
// every step last while the others wait at the step's barrier.  A wave later
// on its SIMD (waves go to the four SIMDs in turn: rank wave / 4) counts
// itself a further 1/16 of the step behind per rank.  One comparison per event,
// against the record where the next quarter begins.
struct StepPriority {
    int bound, quarter, prio;
    __device__ __forceinline__ void begin(int r0, int r1, int wave) {
        const int total = r1 - r0;
        quarter = (total + 3) >> 2;
        bound = r0 + quarter + (((wave >> 2) * total) >> 4);
        prio = 3;
        __builtin_amdgcn_s_setprio(3);
    }
    __device__ __forceinline__ void event(int r) {
        if (r < bound) return;
        bound += quarter;
        --prio;
        if (prio == 2)
            __builtin_amdgcn_s_setprio(2);
        else if (prio == 1)
            __builtin_amdgcn_s_setprio(1);
        else
            __builtin_amdgcn_s_setprio(0);
    }
};

// A lane's element of an output row: the row's uniform base and the lane's
// 32-bit byte offset, which a store takes as they are.
template <typename T>
__device__ __forceinline__ T *lane_ptr(T *row, uint32_t &byte) {
#if defined(__HIP_DEVICE_COMPILE__)
    // redefined at each use, so that it is extended there: hoisted out of the
    // loop, the 64-bit offset would be added by an instruction of its own
    asm volatile("" : "+v"(byte));
#endif
    return (T *)((char *)row + byte);
}

// min(a, b) of a candidate b that is not NaN or loses anyway: v_min_f64 keeps
// -0 below +0, so it is (a < b) ? a : b except for a = -0 and b = +0, which the
// host keeps away from this path.
__device__ __forceinline__ double capped_at(double a, double b) {
#if defined(__HIP_DEVICE_COMPILE__)
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
#else
    return a < b ? a : b;
#endif
}

// Alias tables staged in LDS after the slots (fast sampled variant), so an
// empirical draw is a ds_read rather than a vector memory load.
template <bool kInjected, int kPaths, int kSpl>
__device__ __forceinline__ AliasRec *lds_alias_of(const WalkParams &p, double *lds) {
    return reinterpret_cast<AliasRec *>(lds + (size_t)p.slots * kLanes * kSpl);
}
template <bool kInjected, int kPaths, int kSpl>
__device__ __forceinline__ void stage_alias(const WalkParams &p, double *lds) {
    if (!kInjected) {
        if (kPaths == kPathsFast) {
            AliasRec *const dst = lds_alias_of<kInjected, kPaths, kSpl>(p, lds);
            const auto src = as_const_space(p.alias);
            for (int i = threadIdx.x; i < p.n_alias; i += blockDim.x) dst[i] = src[i];
        }
        __syncthreads();
    }
}

// One tile of 64 x kSpl samples of one plan: every step, then the orphan
// activities.  Every wave of the workgroup calls it; it ends with all waves
// past the last step's barrier.
// The LDS slots of one (step, wave)'s events.
template <int K>
struct SlotRow {
    int32_t v[K];
};

// kPos: the cause output is cause_pos (the winning entry's position), not cause.
// kShift: the tile is one of the overlapping ones (see kShiftStep).
template <bool kInjected, int kPaths, int K, int kSpl, bool kPos = false, bool kShift = false>
__device__ __forceinline__ void walk_tile(const WalkParams &p, int32_t tile, double *lds, const LogTable &lt) {
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int W = p.waves;
    const uint32_t ld = (uint32_t)p.ld;
    // records that write their duration row (none when no durations output)
    const uint32_t owner_bit = p.durations ? (uint32_t)kInfoOwner : 0u;
    // The plan never changes during a launch: reading it through the constant
    // address space lets wave-uniform record loads become scalar loads.
    const auto step_off = as_const_space(p.step_off);
    const auto recs = as_const_space(p.recs);
    const auto step_slots = as_const_space(reinterpret_cast<const SlotRow<K> *>(p.step_slots));
    const auto dists = as_const_space(p.dists);
    const auto earliest = as_const_space(p.earliest);

    AliasRec *const lds_alias = lds_alias_of<kInjected, kPaths, kSpl>(p, lds);
    auto draw = [&](const Record &r, const uint32_t(&seed)[kSpl], double(&dur)[kSpl]) {
        if (kPaths == kPathsFast)
            draw_durations<kSpl>(r.info, r.a, r.b, (uint32_t)r.i2, seed, lds_alias, dists, lt, dur);
        else
            draw_durations<kSpl>(r.info, r.a, r.b, (uint32_t)r.i2, seed, as_const_space(p.alias), dists, lt, dur);
    };

    // Lanes past the last sample (last tile only) take over sample n - 1:
    // same seed or injected row, so they compute its values bit for bit and
    // their stores rewrite its bytes unchanged.  No store needs a lane mask.
    uint32_t at8[kSpl];  // byte of the lane's sample in the tile's part of a row of doubles
    uint32_t seed[kSpl];
    // (not with spilled sources: a lane would read back what a neighbour tile stores)
    static_assert(!kShift || (!kInjected && kSpl == 2 && kPaths == kPathsFast && !kPos), "shifted: sampled, fast, spl 2");
    const int32_t s0 = tile * (kShift ? kShiftStep : kLanes * kSpl);
    const uint32_t first_bits = tile == 0 ? 0u : 7u, last_bits = tile == p.n_tiles - 1 ? 8u : 0u;
    // stores v as sample i of the lane to the row at `row`; shifted: if the sample is in the row's part of the tile
    auto put = [&](auto v, auto *row, uint32_t &byte, int i) {
        if (kShift) {
            const uint32_t a = (0u - (uint32_t)((uintptr_t)row / sizeof(*row))) & 7u;
            const bool in = i == 0 ? (uint32_t)lane >= (a & first_bits)
                                   : (uint32_t)lane < (uint32_t)(kShiftStep - kLanes) + (a | last_bits);
            if (!in) return;
        }
        __builtin_nontemporal_store(v, lane_ptr(row, byte));
    };
#pragma unroll
    for (int i = 0; i < kSpl; ++i) {
        const int32_t si = s0 + i * kLanes + lane;
        const int32_t s = si < p.n ? si : p.n - 1;
        at8[i] = (uint32_t)(s - s0) * 8u;
        seed[i] = kInjected ? 0u : (uint32_t)p.seeds[s];
    }
    // the tile's columns of every array
    const double *const dur_in = p.dur_in + s0;
    double *const realized = p.realized + s0, *const durations = p.durations + s0;
    int32_t *const cause = p.cause + s0;
    uint8_t *const cause_pos = p.cause_pos + s0;

    for (int t = 0; t < p.n_steps; ++t) {
        const int r0 = step_off[t * W + wave];
        const int r1 = step_off[t * W + wave + 1];
        double res[K][kSpl];
        int j = 0;
        if (r0 < r1) {
            // One stream of records: an event header, then its predecessors
            // in input order.  The stream ends in a padding record, so the
            // one-ahead prefetch never leaves the array.
            auto rec = recs + r0;
            Record cur = *rec;
            StepPriority priority;
            priority.begin(r0, r1, wave);
            double best[kSpl], upper = 0.0;
            int32_t who[kSpl], event = 0;
            int hdr = r0;  // kPos: the current event's header record (entry k is record hdr + 1 + k)
#pragma unroll
            for (int i = 0; i < kSpl; ++i) {
                best[i] = 0.0;
                who[i] = -1;
            }
            for (int r = r0; r < r1; ++r) {
                const Record nxt = *++rec;
                if (cur.info & kInfoHeader) {
                    priority.event(r);
                    upper = cur.b;
                    // one vector copy per event: the caps and the final clamp
                    // select against it without rebuilding it from SGPRs
                    asm volatile("" : "+v"(upper));
                    event = cur.i0;
                    if (kPos) hdr = r;
#pragma unroll
                    for (int i = 0; i < kSpl; ++i) {
                        best[i] = cur.a;
                        who[i] = -1;
                    }
                } else {
                    double dur[kSpl];
                    if (kInjected) {
#pragma unroll
                        for (int i = 0; i < kSpl; ++i) dur[i] = 0.0;
                        if (cur.info & kInfoEdgeValid) {
                            const uint64_t row = row_offset(cur.i2, ld);
#pragma unroll
                            for (int i = 0; i < kSpl; ++i)
                                dur[i] = __builtin_nontemporal_load(lane_ptr(dur_in + row, at8[i]));
                        }
                    } else {
                        // an edge outside the link table is kind kNone with
                        // minimal duration 0.0, and owns no row
                        draw(cur, seed, dur);
                        if (cur.info & owner_bit) {
                            const uint64_t row = row_offset(cur.i2, ld);
#pragma unroll
                            for (int i = 0; i < kSpl; ++i)
                                put(dur[i], durations + row, at8[i], i);
                        }
                    }
                    double rs[kSpl];
                    if (cur.i1 >= 0) {
                        lds_load<kSpl>(lds, cur.i1, lane, rs);
                    } else if (kPaths == kPathsGeneral && cur.i1 == kSrcGlobal) {
                        const uint64_t row = row_offset(cur.i0, ld);
#pragma unroll
                        for (int i = 0; i < kSpl; ++i) rs[i] = *lane_ptr(realized + row, at8[i]);
                    } else {
                        const double e = earliest[cur.i0];
#pragma unroll
                        for (int i = 0; i < kSpl; ++i) rs[i] = e;
                    }
                    // the cause: the source event, or the entry's position
                    const int32_t tag = kPos ? r - hdr - 1 : cur.i0;
#pragma unroll
                    for (int i = 0; i < kSpl; ++i) {
                        const double tt = rs[i] + dur[i];
                        if (kPaths == kPathsFast) {
                            // best <= upper from the start (max_delay >= 0), so
                            // the capped candidate wins where the bare one does;
                            // a NaN wins neither way
                            const bool wins = tt >= best[i];
                            const double capped = capped_at(upper, tt);
                            best[i] = wins ? capped : best[i];
                            who[i] = wins ? tag : who[i];
                        } else {
                            const double capped = (upper < tt) ? upper : tt;
                            if (capped >= best[i]) {
                                best[i] = capped;
                                who[i] = tag;
                            }
                        }
                    }
                }
                if (cur.info & kInfoLast) {  // the event's last predecessor (or a header with none)
                    const uint64_t row = row_offset(event, ld);
#pragma unroll
                    for (int i = 0; i < kSpl; ++i) {
                        const double rr = kPaths != kPathsFast && upper < best[i] ? upper : best[i];
                        put(rr, realized + row, at8[i], i);
                        if (kPos) {
                            uint32_t at = at8[i] >> 3;
                            if (p.cause_pos) put((uint8_t)who[i], cause_pos + row, at, i);
                        } else if (p.cause) {
                            uint32_t at = at8[i] >> 1;
                            put(who[i], cause + row, at, i);
                        }
                        res[j][i] = rr;
                    }
                    ++j;
                }
                cur = nxt;
            }
        }
        // The step's slots in one scalar load, in flight across the barrier.
        const SlotRow<K> srow = step_slots[t * W + wave];
        // Every read of this step is done before any slot is overwritten,
        // and every commit is visible before the next step reads it.
        __syncthreads();
#pragma unroll
        for (int i = 0; i < K; ++i) {
            const int slot = srow.v[i];
            if (i < j && slot >= 0) lds_store<kSpl>(lds, slot, lane, res[i]);
        }
        __syncthreads();
    }

    // Activities no predecessor entry references still get a duration row.
    if (!kInjected && p.durations) {
        const auto orph = as_const_space(p.orph);
        for (int o = wave; o < p.n_orphans; o += W) {
            const Record rec = orph[o];
            double dur[kSpl];
            draw(rec, seed, dur);
            const uint64_t row = row_offset(rec.i2, ld);
#pragma unroll
            for (int i = 0; i < kSpl; ++i) put(dur[i], durations + row, at8[i], i);
        }
    }
}

template <bool kInjected, int kPaths, int K, int kSpl, bool kPos = false, bool kShift = false>
__global__ void __launch_bounds__(kMaxWaves * kLanes) walk_kernel(WalkParams p) {
    extern __shared__ double lds[];
    __shared__ LogTableLds log_lds;
    if (!kInjected) stage_log_table(log_lds);
    stage_alias<kInjected, kPaths, kSpl>(p, lds);  // its barrier also publishes the log table
    for (int32_t tile = blockIdx.x; tile < p.n_tiles; tile += gridDim.x)
        walk_tile<kInjected, kPaths, K, kSpl, kPos, kShift>(p, tile, lds, log_lds.view());
}

// Several plans in one launch: workgroups take (plan, tile) items from a
// queue (largest plans first, as ordered by the host) until it is empty;
// every workgroup leaves through the same check of the queue head.
template <bool kInjected, int kPaths, int K, int kSpl, bool kPos = false>
__global__ void __launch_bounds__(kMaxWaves * kLanes) walk_batch_kernel(WalkBatchParams b) {
    extern __shared__ double lds[];
    __shared__ int32_t next_item;
    __shared__ LogTableLds log_lds;
    stage_log_table(log_lds);  // published by the loop's first barrier
    int32_t staged = -1;
    const auto item_dag = as_const_space(b.item_dag);
    const auto item_tile = as_const_space(b.item_tile);
    const auto params = as_const_space(b.params);
    for (;;) {
        __syncthreads();  // the previous tile is done with LDS and next_item
        if (threadIdx.x == 0) next_item = atomicAdd(b.counter, 1);
        __syncthreads();
        const int32_t item = __builtin_amdgcn_readfirstlane(next_item);
        if (item >= b.n_items) break;
        const int32_t d = item_dag[item];
        const WalkParams p = params[d];
        if (d != staged) {
            stage_alias<kInjected, kPaths, kSpl>(p, lds);
            staged = d;
        }
        walk_tile<kInjected, kPaths, K, kSpl, kPos>(p, item_tile[item], lds, log_lds.view());
    }
}

// One step of the walk for a few samples, spread over the device instead of
// over one workgroup's waves: workgroup (i, g) is one wave evaluating event
// e0 + i of the schedule for lane group g (samples 64 g + lane).  A
// predecessor's realized time comes from its output row, written by the
// launch of an earlier step (or is its earliest time, when stale), so there
// are no slots and no barriers; the stream orders the steps.  Per sample the
// arithmetic is walk_tile's: the same records, draws and operation order.
template <bool kInjected>
__global__ void __launch_bounds__(kLanes) walk_wide_kernel(WalkParams p, int32_t e0) {
    const int32_t si = (int32_t)blockIdx.y * kLanes + (int32_t)threadIdx.x;
    const int32_t s = si < p.n ? si : p.n - 1;
    const uint32_t ld = (uint32_t)p.ld;
    const auto recs = as_const_space(p.recs);
    const auto earliest = as_const_space(p.earliest);
    const LogTable lt = global_log_table();
    const uint32_t seed[1] = {kInjected ? 0u : (uint32_t)p.seeds[s]};
    const int32_t r0 = as_const_space(p.ev_rec)[e0 + (int32_t)blockIdx.x];
    // The header and the first batch of records load together.
    const Record h = recs[r0];
    Record c[kWideBatch];
#pragma unroll
    for (int u = 0; u < kWideBatch; ++u) c[u] = recs[r0 + 1 + u];
    const double upper = h.b;
    double best = h.a;
    int32_t who = -1;
    // Predecessors in batches: the batch's records (scalar loads), then its
    // predecessor times and injected durations (vector loads), all in flight
    // together; then the draws and the max-plus steps in input order.  The
    // record array ends in kWideBatch padding records, so a batch never
    // reads past it.
    for (int32_t q0 = 0; q0 < h.i2; q0 += kWideBatch) {
        double rs[kWideBatch], dur[kWideBatch];
        if (q0 > 0) {
#pragma unroll
            for (int u = 0; u < kWideBatch; ++u) c[u] = recs[r0 + 1 + q0 + u];
        }
#pragma unroll
        for (int u = 0; u < kWideBatch; ++u) {
            rs[u] = 0.0;
            dur[u] = 0.0;
            if (q0 + u < h.i2) {
                rs[u] = c[u].i1 == kSrcStale ? earliest[c[u].i0] : p.realized[row_offset(c[u].i0, ld) + s];
                if (kInjected && (c[u].info & kInfoEdgeValid)) dur[u] = p.dur_in[row_offset(c[u].i2, ld) + s];
            }
        }
#pragma unroll
        for (int u = 0; u < kWideBatch; ++u) {
            if (q0 + u >= h.i2) break;
            if (!kInjected) {
                double d1[1];
                draw_durations<1>(c[u].info, c[u].a, c[u].b, (uint32_t)c[u].i2, seed, as_const_space(p.alias),
                                  as_const_space(p.dists), lt, d1);
                dur[u] = d1[0];
                if (p.durations && (c[u].info & kInfoOwner))
                    __builtin_nontemporal_store(dur[u], p.durations + row_offset(c[u].i2, ld) + s);
            }
            double tt = rs[u] + dur[u];
            tt = (upper < tt) ? upper : tt;
            if (tt >= best) {
                best = tt;
                who = p.cause_pos ? q0 + u : c[u].i0;  // the entry's position, or the source event
            }
        }
    }
    // realized is read by later steps: an ordinary store; cause is not
    const uint64_t row = row_offset(h.i0, ld);
    p.realized[row + s] = (upper < best) ? upper : best;
    if (p.cause_pos)
        __builtin_nontemporal_store((uint8_t)who, p.cause_pos + row + s);
    else if (p.cause)
        __builtin_nontemporal_store(who, p.cause + row + s);
}

// Durations of the activities no predecessor entry references, for the wide
// steps' samples: workgroup (o, g) draws orphan o for lane group g.
__global__ void __launch_bounds__(kLanes) walk_wide_orphans_kernel(WalkParams p) {
    const int32_t si = (int32_t)blockIdx.y * kLanes + (int32_t)threadIdx.x;
    const int32_t s = si < p.n ? si : p.n - 1;
    const Record rec = as_const_space(p.orph)[blockIdx.x];
    const uint32_t seed[1] = {(uint32_t)p.seeds[s]};
    double dur[1];
    draw_durations<1>(rec.info, rec.a, rec.b, (uint32_t)rec.i2, seed, as_const_space(p.alias), as_const_space(p.dists),
                      global_log_table(), dur);
    p.durations[row_offset(rec.i2, (uint32_t)p.ld) + s] = dur[0];
}

// ---- short runs: all draws, then the propagation level by level -------------
//
// A run far smaller than a round of tiles leaves the fused walk waiting: one
// tile walks the whole DAG on one CU, at a wave's own instruction latency.
// Drawn first, the durations are independent of each other and fill the
// device whatever the sample count; the propagation that is left is a few
// instructions per predecessor.  Measured (one launch per step, or a tile,
// before; two launches now), 200 x 100 events: 1 sample 1.34 -> 0.11 ms, 1,000
// 1.09 -> 0.40, 4,001 1.77 -> 1.20; 60 x 250 events, 12,345 samples 4.8 -> 3.3;
// 20 x 10 events, 1 sample 93 -> 17 us.

// Every link's durations.  kLaneLinks: the lanes of a wave are 64 / group
// links x group samples (short runs: the draw is divergent only where the
// links' laws differ, and the records are sorted by law); otherwise a wave
// takes kDrawSpl samples per lane of one link, its record in scalar registers.
// A wave keeps its samples from link to link, so nothing but scalar loads and
// table reads is waited for in its loop: a seed loaded there would wait for
// the stores before it too.
constexpr int kDrawBlock = 256;
constexpr int kDrawSpl = 4;
constexpr int kDrawBlocksPerCu = 6;  // resident at once: four waves a block, one per SIMD (80 VGPRs)

template <bool kLaneLinks>
__global__ void __launch_bounds__(kDrawBlock, kDrawBlocksPerCu) draw_kernel(DrawParams p, int32_t group, int32_t n_chunks,
                                                          int32_t lds_alias_n) {
    extern __shared__ double lds[];
    __shared__ LogTableLds log_lds;
    stage_log_table(log_lds);
    AliasRec *const alias = reinterpret_cast<AliasRec *>(lds);
    for (int i = threadIdx.x; i < lds_alias_n; i += kDrawBlock) alias[i] = p.alias[i];
    __syncthreads();
    const LogTable lt = log_lds.view();
    const int lane = threadIdx.x & (kLanes - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) + (int)blockIdx.x * (kDrawBlock / kLanes);
    const int waves = (int)gridDim.x * (kDrawBlock / kLanes);
    const uint32_t ld = (uint32_t)p.ld;
    const auto dists = as_const_space(p.dists);
    if (kLaneLinks) {
        // lanes past the last link or sample repeat the last one's draw and
        // rewrite its bytes unchanged
        const int32_t per = kLanes / group, sub = lane / group, sl = lane - sub * group;
        const int32_t s = sl < p.n ? sl : p.n - 1;
        const uint32_t seed[1] = {(uint32_t)p.seeds[s]};
        for (int32_t l0 = wave * per; l0 < p.L; l0 += waves * per) {
            const int32_t li = l0 + sub;
            const Record r = p.recs[li < p.L ? li : p.L - 1];
            double dur[1];
            if (lds_alias_n > 0)
                draw_durations<1>(r.info, r.a, r.b, (uint32_t)r.i2, seed, alias, dists, lt, dur);
            else
                draw_durations<1>(r.info, r.a, r.b, (uint32_t)r.i2, seed, as_const_space(p.alias), dists, lt, dur);
            p.durations[row_offset(r.i2, ld) + s] = dur[0];
        }
    } else {
        // waves chunk, chunk + n_chunks, ... share a chunk's links
        const int32_t slices = waves / n_chunks;
        const int32_t slice = wave / n_chunks, chunk = wave - slice * n_chunks;
        if (slice >= slices) return;
        int32_t s[kDrawSpl];
        uint32_t seed[kDrawSpl];
#pragma unroll
        for (int i = 0; i < kDrawSpl; ++i) {
            const int32_t si = chunk * (kLanes * kDrawSpl) + i * kLanes + lane;
            s[i] = si < p.n ? si : p.n - 1;
            seed[i] = (uint32_t)p.seeds[s[i]];
        }
        for (int32_t li = slice; li < p.L; li += slices) {
            const Record r = as_const_space(p.recs)[li];
            double dur[kDrawSpl];
            if (lds_alias_n > 0)
                draw_durations<kDrawSpl>(r.info, r.a, r.b, (uint32_t)r.i2, seed, alias, dists, lt, dur);
            else
                draw_durations<kDrawSpl>(r.info, r.a, r.b, (uint32_t)r.i2, seed, as_const_space(p.alias), dists, lt, dur);
            double *const row = p.durations + row_offset(r.i2, ld);
#pragma unroll
            for (int i = 0; i < kDrawSpl; ++i) __builtin_nontemporal_store(dur[i], row + s[i]);
        }
    }
}

// The propagation: a workgroup carries `kGroup` samples through every level,
// its threads being (item of the level, sample) pairs, the realized times that
// later levels read in LDS slots.  A slot freed by a level's reads is given out
// again from the next level on, so a level needs one barrier, after its
// results are in their slots.  Nothing but the slots depends on an earlier
// level: an item is loaded three steps ahead and its durations two steps
// ahead, over the barriers, in a ring of four stages (the step is written out
// once per position of the ring, so no stage is ever copied).  Bound by a
// level's latency for few samples (0.45 us per level: loads one step ahead took
// 1.0), by the durations' and results' bytes for many (8,192 samples of 200 x
// 100 events: 5.2 GB in 1.47 ms, 3.6 TB/s, against 4.8 for a plain copy).
struct LevelStage {
    LevelQuad q[kLevelQuads];
    double d[kLevelPreds];
    bool valid, last;  // uniform: there is an item; it is in its level's last pass
    bool live;         // this thread's item exists (a level's last pass may not fill the workgroup)
};

template <int kGroup, bool kZeroEdges>
__global__ void __launch_bounds__(kLevelMaxThreads) level_kernel(LevelParams p) {
    extern __shared__ double lds[];
    const int sl = threadIdx.x & (kGroup - 1);
    const int idx = threadIdx.x / kGroup;
    const int stride = blockDim.x / kGroup;
    // Workgroups go to the eight dies in turn: consecutive groups of samples
    // share the cache lines of every row, so each die takes a run of them.
    const int32_t per = ((int32_t)gridDim.x + 7) / 8;
    const int32_t g = ((int32_t)blockIdx.x & 7) * per + ((int32_t)blockIdx.x >> 3);
    const int32_t si = g * kGroup + sl;
    if (g * kGroup >= p.n) return;  // the whole workgroup: g is uniform
    const uint32_t s = (uint32_t)(si < p.n ? si : p.n - 1);
    const uint32_t ld = (uint32_t)p.ld;
    const auto off = as_const_space(p.off);
    for (int i = idx; i < p.n_init; i += stride) lds[p.init[i].slot * kGroup + sl] = p.init[i].value;
    __syncthreads();

    // the next pass to fetch: items [q, q + stride) of the level ending at
    // end.  Every fetch loads, past the last level its last item again, and
    // every item loads a duration for each position, so that the number of
    // loads is fixed and a wait for older ones leaves these in flight.
    int32_t level = 0, q = off[0], end = off[1], end2 = off[2];
    auto fetch = [&](LevelStage &x) {
        x.valid = q < p.E;
        const int32_t qi = q + idx;
        x.live = qi < end;
        const uint32_t byte = (uint32_t)(x.live ? qi : end - 1) * (uint32_t)sizeof(LevelQuad);
#pragma unroll
        for (int k = 0; k < kLevelQuads; ++k)
            x.q[k] = *reinterpret_cast<const LevelQuad *>(reinterpret_cast<const char *>(p.quad + (int64_t)k * p.E) + byte);
        q += stride;
        x.last = q >= end;
        if (x.last) {
            q = end;
            end = end2;
            ++level;
            end2 = off[level + 2 <= p.n_levels ? level + 2 : p.n_levels];
        }
    };
    auto durations = [&](LevelStage &x) {
#pragma unroll
        for (int k = 0; k < kLevelPreds; ++k) {
            const int32_t e = x.q[2].v[k];
            x.d[k] = p.dur[row_offset(kZeroEdges && e < 0 ? 0 : e, ld) + s];
        }
    };
    auto compute = [&](const LevelStage &x) {
        const double upper = __hiloint2double(x.q[0].v[3], x.q[0].v[2]);
        double best = __hiloint2double(x.q[0].v[1], x.q[0].v[0]);
        int32_t who = -1;  // position of the winning predecessor
        const int32_t event = x.q[1].v[0], slot = (int16_t)x.q[1].v[1], count = (uint32_t)x.q[1].v[1] >> 16;
        auto take = [&](double rs, double d, int32_t k) {
            double tt = rs + d;
            tt = (upper < tt) ? upper : tt;
            const bool wins = tt >= best;
            best = wins ? tt : best;
            who = wins ? k : who;
        };
        double rs[kLevelPreds];
#pragma unroll
        for (int k = 0; k < kLevelPreds; ++k) {
            const uint32_t from = (k & 1) ? (uint32_t)x.q[1].v[2 + k / 2] >> 16 : (uint32_t)x.q[1].v[2 + k / 2] & 0xFFFFu;
            rs[k] = lds[from * kGroup + sl];
        }
#pragma unroll
        for (int k = 0; k < kLevelPreds; ++k) take(rs[k], kZeroEdges && x.q[2].v[k] < 0 ? 0.0 : x.d[k], k);
        int32_t src = -1;
        if (count > kLevelPreds) {
            const int32_t first = p.extra_of[event];
            for (int k = kLevelPreds; k < count; ++k) {
                const LevelPred pr = p.extra[first + k - kLevelPreds];
                double d = 0.0;
                if (!kZeroEdges || pr.edge >= 0) d = p.dur[row_offset(pr.edge, ld) + s];
                take(lds[pr.slot * kGroup + sl], d, k);
                if (who == k) src = pr.src;
            }
        }
        const double rr = (upper < best) ? upper : best;
        if (x.live) {
            if (slot >= 0) lds[slot * kGroup + sl] = rr;
            const uint64_t row = row_offset(event, ld) + s;
            p.realized[row] = rr;
            if (p.cause_pos) {
                p.cause_pos[row] = (uint8_t)who;
            } else if (p.cause) {
#pragma unroll
                for (int k = 0; k < kLevelPreds; ++k) src = who == k ? x.q[3].v[k] : src;
                p.cause[row] = src;
            }
        }
    };
    // one step of the ring: a computed, b's durations in flight, c's issued, d fetched
    auto step = [&](LevelStage &a, LevelStage &b, LevelStage &c, LevelStage &d) {
        fetch(d);
        durations(c);
        compute(a);
        if (!b.valid) return false;
        if (a.last) __syncthreads();
        return true;
    };
    LevelStage a, b, c, d;
    fetch(a);
    fetch(b);
    durations(a);
    fetch(c);
    durations(b);
    while (step(a, b, c, d) && step(b, c, d, a) && step(c, d, a, b) && step(d, a, b, c)) {
    }
}

hipError_t launch_draws(const DrawParams &p, int cus, hipStream_t stream) {
    if (p.L <= 0 || p.n <= 0) return hipSuccess;
    const size_t alias_bytes = (size_t)p.n_alias * sizeof(AliasRec);
    const int32_t lds_alias_n = alias_bytes <= kAliasLdsMaxBytes ? p.n_alias : 0;
    const size_t lds = lds_alias_n > 0 ? alias_bytes : 0;
    constexpr int kWavesPerBlock = kDrawBlock / kLanes;
    const int64_t most = (int64_t)cus * kDrawBlocksPerCu;
    if (p.n < kLanes) {
        int32_t group = 1;
        while (group < p.n) group *= 2;
        const int64_t waves = ((int64_t)p.L * group + kLanes - 1) / kLanes;
        const int64_t blocks = std::min<int64_t>((waves + kWavesPerBlock - 1) / kWavesPerBlock, most);
        hipLaunchKernelGGL((draw_kernel<true>), dim3((unsigned)blocks), dim3(kDrawBlock), lds, stream, p, group, 0,
                           lds_alias_n);
    } else {
        const int64_t chunks = ((int64_t)p.n + kLanes * kDrawSpl - 1) / (kLanes * kDrawSpl);
        const int64_t need = (chunks + kWavesPerBlock - 1) / kWavesPerBlock;  // a wave per chunk
        const int64_t all = (chunks * p.L + kWavesPerBlock - 1) / kWavesPerBlock;
        const int64_t blocks = std::max(need, std::min(all, most));
        hipLaunchKernelGGL((draw_kernel<false>), dim3((unsigned)blocks), dim3(kDrawBlock), lds, stream, p, 0,
                           (int32_t)chunks, lds_alias_n);
    }
    return hipGetLastError();
}

template <int kGroup>
hipError_t launch_levels_of(const LevelParams &p, bool zero_edges, int threads, size_t lds, hipStream_t stream) {
    const void *fn = zero_edges ? (const void *)level_kernel<kGroup, true> : (const void *)level_kernel<kGroup, false>;
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    const int32_t groups = (p.n + kGroup - 1) / kGroup;
    LevelParams args = p;
    void *kargs[] = {&args};
    return hipLaunchKernel(fn, dim3((unsigned)((groups + 7) / 8 * 8)), dim3((unsigned)threads), kargs, lds, stream);
}

hipError_t launch_levels(const LevelParams &p, bool zero_edges, int group, int threads, int slots, hipStream_t stream) {
    if (p.n <= 0 || p.n_levels <= 0) return hipSuccess;
    if (threads < kLanes || threads > kLevelMaxThreads || threads % kLanes || threads % group) return hipErrorInvalidValue;
    if (!p.dur) return hipErrorInvalidValue;
    const size_t lds = (size_t)slots * (size_t)group * sizeof(double);
    if (lds > kLevelLdsMaxBytes) return hipErrorInvalidValue;
    switch (group) {
        case 1: return launch_levels_of<1>(p, zero_edges, threads, lds, stream);
        case 2: return launch_levels_of<2>(p, zero_edges, threads, lds, stream);
        case 4: return launch_levels_of<4>(p, zero_edges, threads, lds, stream);
        case 8: return launch_levels_of<8>(p, zero_edges, threads, lds, stream);
        case 16: return launch_levels_of<16>(p, zero_edges, threads, lds, stream);
        case 32: return launch_levels_of<32>(p, zero_edges, threads, lds, stream);
        case 64: return launch_levels_of<64>(p, zero_edges, threads, lds, stream);
        default: return hipErrorInvalidValue;
    }
}

__global__ void reset_counter_kernel(int32_t *counter) { *counter = 0; }

__global__ void philox_debug_kernel(int variant, int64_t n, const uint32_t *__restrict__ ctr,
                                    const uint32_t *__restrict__ key, uint32_t *__restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (variant == 4) {
        const Words4 w = philox4x32_10(ctr[4 * i], ctr[4 * i + 1], ctr[4 * i + 2], ctr[4 * i + 3], key[2 * i],
                                       key[2 * i + 1]);
        out[4 * i] = w.x;
        out[4 * i + 1] = w.y;
        out[4 * i + 2] = w.z;
        out[4 * i + 3] = w.w;
    } else {
        const Words2 w = philox2x32_10(ctr[2 * i], ctr[2 * i + 1], key[i]);
        out[2 * i] = w.x;
        out[2 * i + 1] = w.y;
    }
}

// The samplers' elementary functions on n inputs: 0 log_tab, 1 cos2pi_fast,
// 2 exp_fast.
__global__ void math_debug_kernel(int fn, int64_t n, const double *__restrict__ x, double *__restrict__ out) {
    __shared__ LogTableLds log_lds;
    stage_log_table(log_lds);
    __syncthreads();
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double v = x[i];
    out[i] = fn == 0 ? log_tab(v, log_lds.view()) : fn == 1 ? cos2pi_fast(v) : exp_fast(v);
}

__global__ void __launch_bounds__(256) copy_kernel(double *__restrict__ dst, const double *__restrict__ src,
                                                   int64_t n) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

hipError_t launch_copy(double *dst, const double *src, int64_t n, hipStream_t stream) {
    const int64_t blocks = std::min<int64_t>((n + 255) / 256, 256 * 64);
    if (blocks > 0) hipLaunchKernelGGL(copy_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, dst, src, n);
    return hipGetLastError();
}

template <bool kInjected, int kPaths, int kSpl, bool kPos>
const void *walk_symbol(int k) {
    switch (k) {
        case 4: return (const void *)walk_kernel<kInjected, kPaths, 4, kSpl, kPos>;
        case 8: return (const void *)walk_kernel<kInjected, kPaths, 8, kSpl, kPos>;
        case 12: return kSpl == 1 ? (const void *)walk_kernel<kInjected, kPaths, 12, 1, kPos> : nullptr;
        case 16: return kSpl == 1 ? (const void *)walk_kernel<kInjected, kPaths, 16, 1, kPos> : nullptr;
        default: return nullptr;
    }
}

template <bool kInjected, int kPaths, bool kPos>
const void *walk_symbol(int k, int spl) {
    return spl == 2   ? walk_symbol<kInjected, kPaths, 2, kPos>(k)
           : spl == 1 ? walk_symbol<kInjected, kPaths, 1, kPos>(k)
                      : nullptr;
}

// Winner positions (v.pos) only for sampled walks.
const void *walk_symbol(WalkVariant v) {
    if (v.shift) {
        if (v.injected || v.paths != kPathsFast || v.spl != 2 || v.pos) return nullptr;
        return v.k == 4   ? (const void *)walk_kernel<false, kPathsFast, 4, 2, false, true>
               : v.k == 8 ? (const void *)walk_kernel<false, kPathsFast, 8, 2, false, true>
                          : nullptr;
    }
    if (v.injected)
        return v.pos ? nullptr
               : v.paths == kPathsFast ? walk_symbol<true, kPathsFast, false>(v.k, v.spl)
                                       : walk_symbol<true, kPathsGeneral, false>(v.k, v.spl);
    if (v.pos)
        return v.paths == kPathsFast ? walk_symbol<false, kPathsFast, true>(v.k, v.spl)
                                     : walk_symbol<false, kPathsGeneral, true>(v.k, v.spl);
    return v.paths == kPathsFast ? walk_symbol<false, kPathsFast, false>(v.k, v.spl)
                                 : walk_symbol<false, kPathsGeneral, false>(v.k, v.spl);
}

template <bool kInjected, int kPaths, int kSpl, bool kPos>
const void *walk_batch_symbol(int k) {
    switch (k) {
        case 4: return (const void *)walk_batch_kernel<kInjected, kPaths, 4, kSpl, kPos>;
        case 8: return (const void *)walk_batch_kernel<kInjected, kPaths, 8, kSpl, kPos>;
        case 12: return kSpl == 1 ? (const void *)walk_batch_kernel<kInjected, kPaths, 12, 1, kPos> : nullptr;
        case 16: return kSpl == 1 ? (const void *)walk_batch_kernel<kInjected, kPaths, 16, 1, kPos> : nullptr;
        default: return nullptr;
    }
}

template <bool kPos>
const void *walk_batch_symbol_of(WalkVariant v) {
    if (v.spl == 1)
        return v.paths == kPathsFast ? walk_batch_symbol<false, kPathsFast, 1, kPos>(v.k)
                                     : walk_batch_symbol<false, kPathsGeneral, 1, kPos>(v.k);
    if (v.spl == 2)
        return v.paths == kPathsFast ? walk_batch_symbol<false, kPathsFast, 2, kPos>(v.k)
                                     : walk_batch_symbol<false, kPathsGeneral, 2, kPos>(v.k);
    return nullptr;
}

// Batches run sampled plans (the injected variant has no batch form); v.pos:
// every plan's cause output is cause_pos.
const void *walk_batch_symbol(WalkVariant v) {
    if (v.injected) return nullptr;
    return v.pos ? walk_batch_symbol_of<true>(v) : walk_batch_symbol_of<false>(v);
}

hipError_t walk_batch_occupancy(WalkVariant v, int waves, size_t lds_bytes, int *blocks_per_cu) {
    const void *fn = walk_batch_symbol(v);
    if (!fn) return hipErrorInvalidValue;
    if (lds_bytes > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
        if (e != hipSuccess) return e;
    }
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, fn, waves * kLanes, lds_bytes);
    if (e != hipSuccess) return e;
    hipFuncAttributes attr;
    e = hipFuncGetAttributes(&attr, fn);
    if (e != hipSuccess) return e;
    if (attr.numRegs > 0) {
        const int granules = (attr.numRegs + 7) / 8;
        const int per_simd = std::min(8, 512 / (granules * 8));
        *blocks_per_cu = std::min(*blocks_per_cu, per_simd / ((waves + 3) / 4));
    }
    return hipSuccess;
}

hipError_t launch_walk_batch(const WalkBatchParams &b, WalkVariant v, int waves, int grid, size_t lds_bytes,
                             hipStream_t stream) {
    const void *fn = walk_batch_symbol(v);
    if (!fn) return hipErrorInvalidValue;
    if (lds_bytes > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(reset_counter_kernel, dim3(1), dim3(1), 0, stream, b.counter);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    WalkBatchParams args = b;
    void *kargs[] = {&args};
    return hipLaunchKernel(fn, dim3(grid), dim3(waves * kLanes), kargs, lds_bytes, stream);
}

hipError_t launch_walk(const WalkParams &p, WalkVariant v, int grid, size_t lds_bytes, hipStream_t stream) {
    const void *fn = walk_symbol(v);
    if (!fn) return hipErrorInvalidValue;
    if (lds_bytes > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
        if (e != hipSuccess) return e;
    }
    WalkParams args = p;
    void *kargs[] = {&args};
    return hipLaunchKernel(fn, dim3(grid), dim3(p.waves * kLanes), kargs, lds_bytes, stream);
}

// Workgroups of the walk kernel resident per CU.  The runtime's figure counts
// waves per CU; a workgroup's waves are spread over the CU's 4 SIMDs, ceil(W/4)
// on the fullest one, so a second workgroup fits only if every SIMD has that
// many wave slots left under the kernel's VGPR budget (512 per lane, in
// granules of 8, at most 8 waves per SIMD).
hipError_t walk_occupancy(WalkVariant v, int waves, size_t lds_bytes, int *blocks_per_cu) {
    const void *fn = walk_symbol(v);
    if (!fn) return hipErrorInvalidValue;
    if (lds_bytes > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
        if (e != hipSuccess) return e;
    }
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, fn, waves * kLanes, lds_bytes);
    if (e != hipSuccess) return e;
    hipFuncAttributes attr;
    e = hipFuncGetAttributes(&attr, fn);
    if (e != hipSuccess) return e;
    if (attr.numRegs > 0) {
        const int granules = (attr.numRegs + 7) / 8;
        const int per_simd = std::min(8, 512 / (granules * 8));
        const int per_wg = (waves + 3) / 4;
        *blocks_per_cu = std::min(*blocks_per_cu, per_simd / per_wg);
    }
    return hipSuccess;
}

hipError_t launch_walk_wide(const WalkParams &p, bool injected, int32_t e0, int32_t n_events, int32_t groups,
                            hipStream_t stream) {
    if (n_events <= 0 || groups <= 0) return hipSuccess;
    if (injected)
        hipLaunchKernelGGL(walk_wide_kernel<true>, dim3((unsigned)n_events, (unsigned)groups), dim3(kLanes), 0, stream,
                           p, e0);
    else
        hipLaunchKernelGGL(walk_wide_kernel<false>, dim3((unsigned)n_events, (unsigned)groups), dim3(kLanes), 0, stream,
                           p, e0);
    return hipGetLastError();
}

hipError_t launch_walk_wide_orphans(const WalkParams &p, int32_t groups, hipStream_t stream) {
    if (p.n_orphans <= 0 || groups <= 0 || !p.durations || !p.seeds) return hipSuccess;
    hipLaunchKernelGGL(walk_wide_orphans_kernel, dim3((unsigned)p.n_orphans, (unsigned)groups), dim3(kLanes), 0, stream,
                       p);
    return hipGetLastError();
}

hipError_t launch_philox_debug(int variant, int64_t n, const uint32_t *ctr, const uint32_t *key, uint32_t *out,
                               hipStream_t stream) {
    const int block = 256;
    const int grid = (int)((n + block - 1) / block);
    if (grid > 0) hipLaunchKernelGGL(philox_debug_kernel, dim3(grid), dim3(block), 0, stream, variant, n, ctr, key, out);
    return hipGetLastError();
}

hipError_t launch_math_debug(int fn, int64_t n, const double *x, double *out, hipStream_t stream) {
    const int block = 256;
    const int grid = (int)((n + block - 1) / block);
    if (grid > 0) hipLaunchKernelGGL(math_debug_kernel, dim3(grid), dim3(block), 0, stream, fn, n, x, out);
    return hipGetLastError();
}

}  // namespace mcdp
