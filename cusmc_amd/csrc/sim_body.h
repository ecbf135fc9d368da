// sim_body.h — the run kernel for gfx950 (compiled once per slot count and
// register policy by sim_variant.hip).
//
// Counterpart of cuSMC's simulation_kernel (simulation/simulation.cu:674-901)
// and its device functions (compute_possible_delay :409-541,
// find_minimum_delay :544-671, SyncInSerial :357-407, check_edge_enabled
// :184-266, take_transition :27-181), and of the expression evaluator
// (simulation/expressions.cu).  Same step semantics, different machine
// mapping:
//
//   * cuSMC runs one block per run and one thread per component, with
//     ~8 + log2(MC) __syncthreads per step and thread-0 serial sections.
//     Here a run is a segment of S = 2^k lanes of one wave64 (64/S runs per
//     wave), and each lane owns C = next_pow2(components)/S component slots
//     (blocked: lane l holds components l*C .. l*C+C-1).  Lanes of a segment
//     talk through cross-lane exchanges, ballots and the wave's LDS; no
//     workgroup barrier is ever needed.
//   * Variables and clocks of each run live in LDS as doubles, clocks as
//     reset stamps (a clock's value is the time minus its stamp), so
//     advancing time is free; time accumulates in FP64.  A component is one
//     word in LDS, its location's record class and the base of its private
//     variables.
//   * The race: cuSMC re-samples every component's delay every step
//     (simulation.cu:513-540) and takes the minimum.  Here the same law is
//     sampled with far fewer draws: zero-delay components (branchpoint,
//     urgent, committed, or a clock bound already reached) win first, lowest
//     index first; otherwise the exponential components are one
//     exponential race — minimum delay Exp(sum of rates) and winner chosen in
//     proportion to its rate — and only components under a clock upper bound
//     draw their own uniform delay.  The rate sum and the proportional
//     choice use one fixed pairwise tree over the next power of two of the
//     component count (in-lane levels, then a butterfly over the segment),
//     so the result does not depend on the launch shape and a sequential
//     host implementation reproduces it bit for bit.
//   * Broadcast receivers compute their enabled sets in parallel and fire
//     all at once where their edges commute, else one at a time in component
//     order (SyncInSerial), each lane executing its own component's
//     transition.  The winner's edges are tested side by side, one per lane
//     of the segment.
//   * Beyond a wave's first, runs are handed out by an atomic counter, so a
//     segment that finishes a short run soon starts the next one.
#pragma once

#include <hip/hip_runtime.h>
#include <float.h>
#include <stdint.h>
#include <type_traits>

#include "device_common.h"
#include "kernels.hpp"

namespace {

// ------------------------------------------------------------ run kernel

// A value that is the same on every lane, as a scalar.
__device__ __forceinline__ unsigned long long first_lane(unsigned long long v) {
    return ((unsigned long long)__builtin_amdgcn_readfirstlane((uint32_t)(v >> 32)) << 32) |
           (unsigned long long)__builtin_amdgcn_readfirstlane((uint32_t)v);
}

// The launch's next n chunks, for the whole wave: the first of them.
__device__ __forceinline__ unsigned long long take_chunks(unsigned long long *counter, uint32_t n, int lane) {
    unsigned long long g = 0;
    if (lane == 0) g = atomicAdd(counter, (unsigned long long)n);
    return first_lane(g);
}

// A run's first state; the reads of several variables and of all state words
// are under way together.
template <int C, bool TRACE>
__device__ __forceinline__ void start_state(const SMC_CONSTANT DevModel &m, double *vars, uint32_t *words,
                                            int32_t *locs, int sl, int S) {
    const int n_vars = m.n_vars, n_comp = m.n_comp;
    const auto *init = m.var_init;
    const auto *word = m.comp_word;
    uint32_t w[C];
#pragma unroll
    for (int j = 0; j < C; ++j) w[j] = sl * C + j < n_comp ? word[sl * C + j] : 0u;
    int v = sl;
#pragma clang loop unroll(disable)
    for (; v + 3 * S < n_vars; v += 4 * S) {
        const double a = init[v], b = init[v + S], c = init[v + 2 * S], d = init[v + 3 * S];
        vars[v] = a;
        vars[v + S] = b;
        vars[v + 2 * S] = c;
        vars[v + 3 * S] = d;
    }
#pragma clang loop unroll(disable)
    for (; v < n_vars; v += S) vars[v] = init[v];
    if (sl == 0) vars[n_vars] = 0.0;
#pragma unroll
    for (int j = 0; j < C; ++j) words[64 * j] = w[j];
    if (TRACE) {
#pragma clang loop unroll(disable)
        for (int j = 0; j < C; ++j) locs[64 * j] = sl * C + j < n_comp ? m.comp_init_loc[sl * C + j] : -1;
    }
}

// A wave starts new runs when its idle lanes have cost it this part of its
// time since the last start.  Times at 1/4, 1/8, 1/16 and 1/32: Fischer-32,
// 1e6 runs, 31.7, 30.9, 30.1 and 31.2 ms; SIR-77, 5e4 runs, 2.39, 2.22, 2.18
// and 2.65 ms.
constexpr uint32_t kWaitShare = 16;

// The launch's counter gives some 80 takes a microsecond, whatever their size:
// thousands of waves that come for the next runs every few turns wait longer for
// it than for their runs.  So a wave begins with runs of its own, and where its runs
// so far took fewer than 64 turns on average, one that comes again within this many
// takes as many more at a time, up to sixteen times its need and half its even share
// of what is left, less one for each of its segments unless the last took under eight
// turns.  One step a run, 1e7 runs: 0.38 ms for 1.98 with a take by need, 2e4 runs
// 10.5 us for 40.9; UppaalWeightTest, 25 steps a run, 1e7 runs 5.9 ms for 12.0.  Longer
// runs wait in a wave while others stand idle: race-8, 1e6 runs, 11.8 ms with the length
// looked at and 13.0 without; SIR-60, 1e5 runs, 1.17 ms with the segments' share left
// and 1.30 without (UppaalWeightTest 4.6).  (Runs of several instances differ too much:
// a chunk at a time.)
constexpr uint32_t kShortRuns = 32;
constexpr int kLengthMost = 1 << 20;

// The same pointer, as far as the optimiser knows another one.
template <class T>
__device__ __forceinline__ const SMC_CONSTANT T *opaque(const SMC_CONSTANT T *p) {
    asm volatile("" : "+s"(p));
    return p;
}

// A wave begins with runs of its own, then takes chunks of runs from the
// launch's queue, and hands the runs to its segments; all its segments work on
// one instance, which (its tables, query and outputs) is thereby uniform across
// the wave and lives in scalar registers.  A chunk of another instance waits until this one's runs are
// done.  A workgroup holds blockDim/64 independent waves.  With TAB
// (single-instance launches) the workgroup first copies the model's tables
// into LDS and every wave reads them there: the race and the transitions are
// chains of dependent table reads, and LDS answers them several times sooner
// than the caches.
//
// What bounds it: VALU issue while the chip is full, the latency of the
// step's chain of dependent reads when it is not.  Both ask for few
// instructions per step and for little code: the lanes of a wave are at
// different points of different runs, so whatever one of them needs, all
// wait for, and a step's code has to stay in the 64 KB instruction cache
// (with per-slot copies of the general code in every branch it was 320 KB).
// Fischer-32, 1e6 runs: 76.2 ms in that form, 51.0 ms with record classes
// and rolled cold paths, 44.2 ms with the slot loop free of branches and its
// invariants out of spilled registers, 40.7 ms with the step's rare parts
// behind branches the whole wave takes or leaves, 36.3 ms with the race's sums
// and windows kept out of LDS, 30.3 ms with runs handed out as below, 29.5 ms
// with the windows of a pair read side by side; SIR-350, 2e5 runs: 355, 117,
// 97, 81.8, 76.7 and 74.6 ms, 66.4 ms with the receivers' picks reduced to a
// comparison, 65.3 ms with half records where nothing is tested.  Now the
// three waves of a SIMD issue a VALU instruction in 88 % of its cycles with
// SIR-350; a wave of Fischer-32, 32 runs and two waves per SIMD, issues
// instructions of all kinds in 52 % of its own.
//
// LDS: [tables: lp.table_bytes, TAB only] then per wave [variables of the
// wave's 64/S runs and a constant 0, an odd number of doubles each][state
// words: 4 bytes per slot and lane][TRACE: locations, the same]; lp.wave_lds
// covers the largest of these over the launch's instances.
//
// When a segment's run ends, it waits: for the last of the wave's runs, or
// until the waiting lanes have cost the wave 1/16 of its time.  Runs of equal
// length then start together and take the same parts of a step in the same
// steps; a Fischer run ends when its goal is reached, and waiting for the
// longest of a chunk left half of the lanes idle.
template <int C, bool TRACE, bool TAB>
__device__ __forceinline__ void sim_body(const LaunchParams &lp) {
    extern __shared__ __attribute__((aligned(16))) double lds[];
    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    double *wbase = lds + (TAB ? lp.table_bytes / 8 : 0) + (size_t)wv * (lp.wave_lds / 8);
    const double INF = __builtin_huge_val();
    using Tables = typename std::conditional<TAB, SmcLdsTables, SmcGlobalTables>::type;
    if (TAB) stage_tables(lp.tables, lp.table_bytes, lds);

  const SMC_CONSTANT LaunchParams *args = (const SMC_CONSTANT LaunchParams *)__builtin_amdgcn_kernarg_segment_ptr();
  // chunks the wave has taken and not begun, the first of them without the queue
  // (not where a caller named more waves than are resident: one that starts late
  // kept its runs waiting, Fischer-32, 2e5 runs, 2560 waves of which 2048 are, 7.8 ms for 6.6)
  unsigned long long g = (unsigned long long)(blockIdx.x * (blockDim.x >> 6) + wv) * lp.first, g_end = g + lp.first;
  if (g >= lp.handed) g = g_end = 0;
  // n more, where any are left
  const auto take = [&](uint32_t n, const SMC_CONSTANT LaunchParams *L) {
      const uint64_t total = L->total_chunks, handed = L->handed;
      if (handed >= total || g_end >= total) {
          g = g_end = total;
      } else {
          g = handed + take_chunks(L->counter, n, lane);
          g_end = g + n;
      }
  };
  for (;;) {
    g = first_lane(g);
    g_end = first_lane(g_end);
    const SMC_CONSTANT LaunchParams *launch = opaque(args);
    if (g == g_end) take(1, launch);
    if (g >= launch->total_chunks) break;
    int lo = 0, hi = launch->n_inst - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (launch->inst[mid].chunk_first <= g) lo = mid;
        else hi = mid - 1;
    }
    // What every step needs of the instance stays in registers; what only a
    // run's start or end needs is read again there (through `inst` made
    // opaque, or it would be loaded here and spilled).
    const SMC_CONSTANT InstDesc *inst = (const SMC_CONSTANT InstDesc *)(uintptr_t)launch->inst + lo;
    DevModelT<Tables> m;
    if constexpr (TAB) {
        const SMC_GLOBAL uint8_t *tables = launch->tables;
        const SMC_LDS uint8_t *copy = (const SMC_LDS uint8_t *)(SMC_LDS double *)lds;
        m.hots = in_lds(inst->m.hots, tables, copy);
        m.locs = in_lds(inst->m.locs, tables, copy);
        m.invs = in_lds(inst->m.invs, tables, copy);
        m.edges = in_lds(inst->m.edges, tables, copy);
        m.guards = in_lds(inst->m.guards, tables, copy);
        m.upds = in_lds(inst->m.upds, tables, copy);
        m.consts = in_lds(inst->m.consts, tables, copy);
        m.code = in_lds(inst->m.code, tables, copy);
    } else {
        m.hots = inst->m.hots;
        m.locs = inst->m.locs;
        m.invs = inst->m.invs;
        m.edges = inst->m.edges;
        m.guards = inst->m.guards;
        m.upds = inst->m.upds;
        m.consts = inst->m.consts;
        m.code = inst->m.code;
    }
    m.loc_edge0 = inst->m.loc_edge0;
    m.rec_shift = inst->m.rec_shift;
    m.base_mask = inst->m.base_mask;
    m.tests = inst->m.tests;
    m.one_rate = inst->m.one_rate;
    m.freeze = inst->m.freeze;
    const uint64_t seed = inst->p.seed;
    const double bound = inst->p.bound;
    const bool reach = inst->p.reach != 0;
    const uint32_t max_steps = inst->p.max_steps;
    // the instance's packing: S lanes per run, 64 / S runs per wave
    const int S0 = inst->lanes;
    const int sl = lane & (S0 - 1);
    const int seg_base = lane - sl;
    const uint64_t seg_ones = (S0 == 64) ? ~0ull : ((1ull << S0) - 1ull);
    const uint64_t seg_mask = seg_ones << seg_base;
    const int stride = (inst->m.n_vars + 1) | 1;
    double *vars = wbase + (lane / S0) * stride;
    uint32_t *words_of = (uint32_t *)(wbase + (64 / S0) * stride);
    uint32_t *words = words_of + lane;
    int32_t *locs = (int32_t *)words_of + 64 * C + lane;  // TRACE only
    // since runs were started: turns of the loop, lanes without a run summed
    // over them
    uint32_t turns = kShortRuns, waited = 0;
    int length = 64;  // turns less what as many runs of 64 turns would have taken, from the first refill on
    uint32_t r_next = 0, r_end = 0;  // runs of chunks begun, not started yet

    bool active = false, done = lane / S0 >= launch->segments;
    uint64_t run = 0;
    uint32_t ridx = 0;
    double t = 0.0;
    uint32_t step = 0, trans = 0;  // trans: edges fired by this lane (the winner's count on lane 0)
    int chan = 0, sender = -1;
    bool goal = false;
    bool over = false;    // no event can follow: the run ends at its clock
    bool changed = true;  // state changed since the last blocking tests
    uint32_t xblk = 0;    // blocked slots at the last change of state (tests of several records)
    uint64_t digest = 0;
    LaneQuery q{inst->p.qvar, 0.0, 0.0};

    // The loop's straight path is one step of every run of the wave; the rest
    // is behind wave-uniform conditions.
    for (;;) {
        const int S = scalar_here(S0);
        // ---- loop test (simulation.cu:835-849)
        const bool in_time = t < bound;
        const bool at_goal = reach & goal & in_time & !over;
        const bool end = active & (!in_time | over | at_goal | (step >= max_steps));
        ++turns;
        if (unlikely(any_lane(end | (!active & !done)))) {
            const SMC_CONSTANT InstDesc *I = opaque(inst);
            if (end) {
                // per-run result (simulation.cu:887-893, statistics.cuh:126-163)
                double qmax = q.qmax, qmin = q.qmin;
                uint32_t fired = trans;
#pragma unroll
                for (int k = 0; k < 6; ++k)
                    if ((1 << k) < S) {
                        qmax = fmax(qmax, seg_xchg(qmax, k));
                        qmin = fmin(qmin, seg_xchg(qmin, k));
                        fired += (uint32_t)__shfl_xor((int)fired, 1 << k);
                    }
                const double value = I->p.is_max ? qmax : qmin;
                if (TRACE) {
                    digest = smc_mix(digest, smc_digest_bits(t));
                    for (int v = 0; v < I->m.n_vars; ++v)
                        digest = smc_mix(digest, smc_digest_bits(I->m.var_clock[v] ? t - vars[v] : vars[v]));
                    for (int c = 0; c < I->m.n_comp; ++c) {
                        const int lv = ((int32_t *)words_of)[64 * C + (c % C) * 64 + seg_base + c / C];
                        digest = smc_mix(digest, (uint64_t)(uint32_t)lv);
                    }
                }
                if (sl == 0) {
                    uint8_t flag;
                    if (reach) flag = at_goal ? 1 : 0;
                    else flag = I->p.is_max ? (value > I->p.threshold) : (value < I->p.threshold);
                    I->p.flag[ridx] = flag;
                    I->p.value[ridx] = value;
                    I->p.steps[ridx] = step;
                    I->p.trans[ridx] = fired;
                    if (I->p.time) I->p.time[ridx] = t;
                    if (TRACE && I->p.digest) I->p.digest[ridx] = digest;
                }
                wave_sync();
                active = false;
            }
            // new runs once none is left, or once the waiting lanes have
            // stood still for a share of the wave's time
            const bool want = !active & !done;
            waited += (uint32_t)__popcll(__ballot(want));
            if (!any_lane(active) || kWaitShare * waited > 64 * turns) {
                const uint32_t idle = (uint32_t)__popcll(__ballot(want));
                const bool brief = 8 * turns < idle;
                length = min(max(length + (int)min(turns, 65536u) - (int)idle, -kLengthMost), kLengthMost);
                const uint32_t more = length < 0 && turns < kShortRuns ? min(kShortRuns / max(turns, 1u), 16u) : 1u;
                waited = turns = 0;
                const uint64_t heads = __ballot(want & (sl == 0));
                const int need = __popcll(heads), rank = __popcll(heads & ((1ull << seg_base) - 1));
                const uint32_t chunk = I->chunk_runs, n_runs = (uint32_t)I->p.n_runs;
                const uint64_t c0 = I->chunk_first, c1 = c0 + (n_runs + (uint64_t)chunk - 1) / chunk;
                uint32_t r = 0xFFFFFFFFu;
                for (int given = 0; given < need;) {
                    if (r_next == r_end) {
                        if (g == g_end) {
                            const SMC_CONSTANT LaunchParams *L = opaque(args);
                            uint32_t n = 1;
                            if (L->n_inst == 1) {
                                const uint64_t total = L->total_chunks, at = max((uint64_t)g, L->handed);
                                const uint64_t left = at < total ? total - at : 0;
                                n = ((uint32_t)(need - given) + chunk - 1) / chunk;
                                const uint64_t half = left >> L->share_shift, keep = brief ? 0u : (uint32_t)L->segments;
                                n = max(n, (uint32_t)min((uint64_t)(n * more), half > keep ? half - keep : 0));
                            }
                            take(n, L);
                        }
                        if (g >= c1) break;
                        const uint64_t stop = g_end < c1 ? g_end : c1, r1 = (stop - c0) * chunk;
                        r_next = (uint32_t)((g - c0) * chunk);
                        r_end = r1 < n_runs ? (uint32_t)r1 : n_runs;
                        g = stop;
                    }
                    const int left = (int)(r_end - r_next), n = left < need - given ? left : need - given;
                    if ((rank >= given) & (rank < given + n)) r = r_next + (uint32_t)(rank - given);
                    r_next += (uint32_t)n;
                    given += n;
                }
                if (want) {
                    if (r == 0xFFFFFFFFu) {
                        done = true;
                    } else {
                        ridx = r;
                        const SMC_CONSTANT uint64_t *round = (const SMC_CONSTANT uint64_t *)(uintptr_t)opaque(args)->round;
                        run = I->p.run_begin + (round ? *round : 0) * I->p.n_runs + r;
                        active = true;
                        t = 0.0; step = 0; trans = 0; chan = 0; sender = -1;
                        goal = false; over = false; changed = true;
                        q.qmax = I->p.qinit; q.qmin = I->p.qinit;
                        digest = TRACE ? smc_mix(0, run) : 0;
                        start_state<C, TRACE>(I->m, vars, words, locs, sl, S);
                        wave_sync();
                    }
                }
                if (!any_lane(active)) break;
                continue;  // a new run passes the loop test first
            }
        }
        if (!active) continue;

        if (any_lane(chan > 0)) {
            // pending broadcast receivers (SyncInSerial simulation.cu:357-407)
            if (chan > 0) {
                bool entered = false;
                fire_receivers<C, TRACE, TRACE>(words, locs, Ctx{vars, t, 0}, m, chan, sender, q, entered, seed,
                                                run, step, lane, sl, S, seg_base, seg_mask, trans, digest);
                changed = true;
                chan = 0;
                sender = -1;
                goal = goal || (__ballot(entered) & seg_mask) != 0;
            }
        }

        // ---- race (compute_possible_delay :409-541, find_minimum_delay
        // :544-671), clock advance, the winner's transition.  A goal entered
        // by this iteration's receivers counts only if this step, raced by
        // every component, keeps t < bound (simulation.cu:409-415, 835-849):
        // no absorption exit and no left-out null racers then.
        const bool full = reach & goal;
        if (unlikely(!m.freeze)) {
            // with frozen racers the race itself ends a run that nothing can
            // leave (no event: blocked racers are out, the rest race at rate
            // 0), so the scan is needed only without them
            if (changed && !full && absorbed<C>(words, Ctx{vars, t, 0}, m, seg_mask)) over = true;
            if (over) continue;
        }
        RaceSlots<C> rs;
        race_slots<C>(rs, words, Ctx{vars, t, 0}, m, changed, xblk);
        changed = full;
        // A frozen component (blocked, exponential) only makes null steps
        // until the next transition.  Leaving it out of the race keeps the
        // law of everything else: exponential racers are memoryless (rates
        // constant between transitions), and a uniform racer redrawn at every
        // step has hazard 1/(W - tau), a function of the absolute time alone
        // (W: the end of its window).  It races as in the reference when the
        // step decides the outcome (full).
        if (unlikely(any_lane(full))) {
            if (m.freeze && full) race_frozen<C>(rs, words, Ctx{vars, t, 0}, m);
        }
        double d = 0.0;
        int w = -1;
        const uint64_t zb = __ballot(rs.zero != 0) & seg_mask;
        if (any_lane(zb == 0)) {
            // some run races (the others' result is replaced below)
            double umin = INF;
            int unif_j = -1;
            // Draws: one for the race, and the uniform delays under clock
            // bounds (slots 2i and 2i+1 of a lane share one; lowest slot
            // first on ties).  The lanes of a run make them side by side: a
            // lane without delays left to draw makes the race's, and its
            // words are handed to the others afterwards.
            // A run without exponential racers needs none for the race.
            const double own = lane_total<C>(rs.leaf);
            const uint64_t racers = __ballot(own > 0.0) & seg_mask;
            smc_u32x4 race{};
            uint64_t got = 0;  // lanes of the run that made the race's draw
            {
                uint32_t b = rs.bounded;
#pragma clang loop unroll(disable)
                do {
                    const bool delay = b != 0;
                    const int j = C > 1 && delay ? (__ffs(b) - 1) & ~1 : 0;
                    const uint32_t c = (uint32_t)(sl * C + j);
                    const smc_u32x4 rw = draw_at(seed, run, step,
                                                 delay ? ((uint32_t)SMC_P_UNIFORM << 24) | smc_uniform_draw(c)
                                                       : (uint32_t)SMC_P_RACE << 24);
                    double left[2];
                    if constexpr (C > 2) {
                        slot_windows(left, words, j, Ctx{vars, t, 0}, m);
                    } else {
                        left[0] = rs.left[0];
                        left[1] = rs.left[C - 1];
                    }
                    const double du = left[0] * smc_uniform_u(rw, c);
                    if (((b >> j) & 1u) && du < umin) { umin = du; unif_j = j; }
                    if (C > 1) {
                        const double du1 = left[1] * smc_uniform_u(rw, c + 1);
                        if (((b >> j) & 2u) && du1 < umin) { umin = du1; unif_j = j + 1; }
                    }
                    b &= ~(3u << j);
                    // every draw of the race is the same: keep the last
                    race.v[0] = delay ? race.v[0] : rw.v[0];
                    race.v[1] = delay ? race.v[1] : rw.v[1];
                    race.v[2] = delay ? race.v[2] : rw.v[2];
                    race.v[3] = delay ? race.v[3] : rw.v[3];
                    got |= __ballot(!delay) & seg_mask;
                } while (any_lane(b != 0 || (got == 0 && racers != 0)));
                const int from = got ? lowest_lane(got) : lane;
#pragma unroll
                for (int k = 0; k < 4; ++k) race.v[k] = (uint32_t)__shfl((int)race.v[k], from);
            }
            // the exponential race, if any run has racers (slotted Aloha,
            // every delay under a clock bound, one run a wave: 61.8 ms with
            // it in every step, 42.7 ms without)
            double dexp = INF;
            if (any_lane(racers != 0)) {
                double level[6] = {};
                const double R = race_total(own, level, S);
                const double e = -device_log2(smc_u01(race.v[0], race.v[1])) / R;
                w = race_pick<C>(rs.leaf, level, smc_u01(race.v[2], race.v[3]) * R, S, seg_base, seg_mask);
                dexp = R > 0.0 ? e : INF;
            }
            d = dexp;
            if (any_lane(unif_j >= 0)) {
                double gu = umin;
#pragma unroll
                for (int k = 0; k < 6; ++k) {
                    if ((1 << k) >= S) break;
                    gu = fmin(gu, seg_xchg(gu, k));
                }
                // the lowest lane holding the least delay (any lane of a run
                // without one: gu is infinite and loses)
                const uint64_t at = __ballot(unif_j >= 0 && umin == gu) & seg_mask;
                const int Lu = at ? lowest_lane(at) : seg_base;
                const int wu = (Lu - seg_base) * C + __shfl(unif_j, Lu);
                if (gu < dexp || (gu == dexp && gu < INF && wu < w)) { d = gu; w = wu; }
            }
            // the step that crosses the bound: the left-out null racers'
            // first event after the bound may come first
            const bool cross = m.freeze && !full && zb == 0 && d < INF && !(t + d < bound);
            if (unlikely(any_lane(cross))) {
                if (cross) {
                    const double Rd = frozen_total<C>(words, Ctx{vars, t, 0}, m, S);
                    if (Rd > 0.0) {
                        const smc_u32x4 dw = draw(seed, run, step, SMC_P_DEAD, 0);
                        const double td = bound + (-device_log2(smc_u01(dw.v[0], dw.v[1])) / Rd);
                        if (td < t + d) { d = td - t; w = -1; }
                    }
                }
            }
        }
        if (any_lane(zb != 0)) {
            // a zero delay wins, the lowest component first
            const int Lz = zb ? lowest_lane(zb) : seg_base;
            const int wz = (Lz - seg_base) * C + __shfl(__ffs(rs.zero) - 1, Lz);
            if (zb) { d = 0.0; w = wz; }
        }
        over = !(d < INF);  // no racer: no event
        if (over) continue;
        // clocks advance (find_minimum_delay :632-651)
        t = t + d;
        if (w >= 0) {
            // the winner's transition (check_enabled_edges :268-305,
            // take_transition :27-181) by every lane of its segment: each
            // tests one of the location's edges; the pick and the updates are
            // the same on all of them
            uint32_t *slot = words_of + (w % C) * 64 + seg_base + w / C;
            const uint32_t ww = *slot;
            const Ctx x{vars, t, word_base(ww, m)};
            const uint4 L1 = load_quad(m.locs + word_rec(ww, m), 1);
            const uint32_t first = L1.x;            // edge_first
            const int ne = (int)(L1.y & 0xFFFFu);   // edge_n
            const uint64_t mask = enabled_mask_by_lanes(first, ne, x, m, S, sl, seg_base, seg_ones);
            if (mask) {
                const int i = pick_edge(mask, first, L1.z, L1.w, seed, run, step, (uint32_t)w, x, m);
                const uint4 head = fire_updates(first + i, x, m, q);
                *slot = (head.x << m.rec_shift) | x.base;
                if (TRACE) {
                    int32_t *wloc = (int32_t *)words_of + 64 * C + (w % C) * 64 + seg_base + w / C;
                    const int32_t lw = *wloc;
                    digest = smc_mix(digest, ((uint64_t)step << 40) | ((uint64_t)w << 20) |
                                                 (uint64_t)(m.loc_edge0[lw] + i));
                    wave_sync();  // every lane has read the location
                    *wloc = lw + rec_at(m.edges, first + i)->dst;
                }
                goal |= (head.y & SMC_EF_GOAL) != 0;
                trans += sl == 0 ? 1u : 0u;
                changed = true;
                chan = (int)head.w > 0 ? (int)head.w : 0;
                sender = chan > 0 ? w : -1;
            }
            wave_sync();
        }
        ++step;
    }
  }
}

// Two register policies of the run kernel: unrestricted (99-123 VGPRs and
// four waves per SIMD up to two slots per lane, 118 and four at four, with
// digests 131 and three, 143-156 and three at eight, 193-206 and two at
// sixteen), and at most 168 (three waves per SIMD), which only sixteen slots
// spill to keep (some thirty registers).  At sixteen it depends on the packing:
// SIR-350, 2e4 runs, 7.2 ms with three waves and 9.5 with two, Fischer-32, 2e5
// runs, whose LDS holds two, 6.6 both; the autotuner measures both.
template <int C, bool TRACE, bool TAB>
__global__ __launch_bounds__(64 * SMC_MAX_GROUP_WAVES) void sim_kernel(LaunchParams lp) {
    sim_body<C, TRACE, TAB>(lp);
}

template <int C, bool TRACE, bool TAB>
__global__ __launch_bounds__(64 * SMC_MAX_GROUP_WAVES) __attribute__((amdgpu_waves_per_eu(3))) void sim_kernel_o3(
    LaunchParams lp) {
    sim_body<C, TRACE, TAB>(lp);
}

}  // namespace
