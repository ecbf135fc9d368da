// is_advance.h — the tilted advance kernel of importance sampling on gfx950
// (compiled once per slot count and register policy by is_variant.hip) and
// the bf16 helpers of the MLP kernels.
//
// No counterpart in the reference (cuSMC estimates by plain Monte Carlo,
// statistics.cuh:126-163).  A proposal multiplies the rate of each
// exponential component by 2^theta, with theta per location given by a small
// MLP of the run's state; each run carries log2 of its likelihood ratio in
// FP64, so that hit * 2^log2lr is an unbiased estimate of the probability.
//
// Runs advance in lock step by macro-steps: one launch of is_advance_kernel
// moves every active run to its next transition (the race, clocks and the
// winner's edge exactly as the run kernel does them, with tilted rates), then
// writes the run's features for the MLP, whose forward pass (MFMA GEMMs
// below) produces the tilts of the next macro-step.
//
// Cross-entropy training replays the elite runs once with the tilts that
// generated them and records, per (run, macro-step), the features at the
// macro-step's start and two statistics per location L of the run's
// components: A_L, the number of races won by the component in L, and B_L,
// its base cumulative hazard over the macro-step's races (r ln2 d per race
// for an exponential racer, -ln(1 - d/M) for a uniform racer on the window
// [0, M]).  The log-density of the macro-step under tilts theta is then
//   ln q = sum_L (ln2 theta_L A_L - 2^theta_L B_L) + terms free of theta,
// so every training epoch is a pass of GEMMs over the recorded pairs.
//
// The proposal: an exponential component's rate r becomes r' = r 2^theta;
// a uniform (clock-bounded) component's hazard 1/(M - d) is multiplied by
// a = 2^theta (a delay-window tilt: survival (1 - d/M)^a on the same window,
// drawn as M (1 - (1 - u)^(1/a))).  Likelihood ratio of one race step
// (exponential base rates r_c summing to R, tilted to R'; delays drawn as
// -log2(u)/rate, so the effective rates carry a factor ln 2):
//   log2 LR = -theta_w + (R' - R) d + sum_{uniform c} (1 - a_c) log2(1 - d/M_c)
// where theta_w is present when an exponential or uniform racer won with its
// own draw.  Zero delays are not tilted and contribute nothing.
#pragma once

#include <hip/hip_runtime.h>

#include "device_common.h"
#include "is_kernels.hpp"

namespace {

__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7F800000u) == 0x7F800000u) return (uint16_t)((u >> 16) | ((u & 0xFFFF) ? 0x40 : 0));
    u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// Features of a run: one-hot of each component's location, scaled
// variables, time / bound.  Each entry is written by exactly one lane.
template <int C>
__device__ __forceinline__ void write_features(const IsParams &P, uint16_t *f, const int32_t *locs, const double *vars,
                                               uint32_t *bits, double t, int sl, int S, int n) {
    const int base = P.m.n_locs, n_vars = P.m.n_vars;
    // the locations held as a bitmap, then eight features a lane and store:
    // written by component they were scattered 2-byte stores, three for each
    for (int k = sl; k < P.lpad / 32; k += S) bits[k] = 0;
    wave_sync();
#pragma unroll
    for (int j = 0; j < C; ++j)
        if (sl * C + j < n) {
            const int at = locs[64 * j];
            atomicOr(&bits[at >> 5], 1u << (at & 31));
        }
    wave_sync();
    const auto two = [](uint32_t b) { return ((b & 1u) | ((b & 2u) << 15)) * 0x3F80u; };
    for (int k = sl; k < base / 8; k += S) {
        const uint32_t b = bits[k >> 2] >> (8 * (k & 3));
        ((uint4 *)f)[k] = uint4{two(b), two(b >> 2), two(b >> 4), two(b >> 6)};
    }
    for (int l = (base & ~7) + sl; l < base; l += S) f[l] = (bits[l >> 5] >> (l & 31)) & 1u ? (uint16_t)0x3F80 : (uint16_t)0;
    for (int v = sl; v < n_vars; v += S) {
        const double x = P.m.var_clock[v] ? t - vars[v] : vars[v];
        f[base + v] = f32_to_bf16((float)(x * P.var_scale[v]));
    }
    if (sl == 0) f[base + n_vars] = f32_to_bf16((float)(t / P.bound));
    for (int k = base + n_vars + 1 + sl; k < P.fpad; k += S) f[k] = 0;
}

// Whether a var-probability query is already decided: the segment-wide
// running max (min) has crossed the threshold.  Every lane tracks the
// updates it executed, so the test reduces over the segment.
__device__ __forceinline__ bool settled(const LaneQuery &q, const IsParams &P, int S) {
    double v = P.is_max ? q.qmax : q.qmin;
#pragma unroll
    for (int k = 0; k < 6; ++k)
        if ((1 << k) < S) v = P.is_max ? fmax(v, seg_xchg(v, k)) : fmin(v, seg_xchg(v, k));
    return P.is_max ? v > P.threshold : v < P.threshold;
}

// ------------------------------------------------------------ advance

// Tilt lookups of the workgroup and its waves (all in LDS): the tilt index
// of every location, and 2^theta precomputed once per theta entry — for the
// whole launch when every run shares one theta vector, else per row.
struct TiltLds {
    const int32_t *tix;   // [lpad]
    const double *ex;     // [theta_len]: 2^theta, shared theta only
    double *row_ex;       // the wave's rows: [64/S][theta_cap] 2^theta
    float *row_th;        // [64/S][theta_cap] theta
    double *scr;          // the wave's slot scratch [C][64] (windows of bounded slots)
    uint32_t *words;      // state words [C][64]
    int32_t *locs;        // locations [C][64]
    uint32_t *bits;       // the wave's rows: locations held, [64/S][lpad / 32]
    double *rec;          // recording build: [C][64] rates, [C][64] int32 locations, [C][64] uint32 wins
};

// REC: the build that records macro-step statistics (elite replays); the
// sampling build leaves the recording state out of its registers.  KEEP: the
// bounded slots' windows are kept in LDS; else they are computed at each use.
template <int C, bool REC, bool KEEP, class MT>
__device__ __forceinline__ void is_advance_rows(const IsParams &P, const MT &m, double *wlds, const TiltLds &tl,
                                                int group) {
    const int lane = threadIdx.x & 63;
    const int S = P.lanes;
    const int sl = lane & (S - 1);
    const int seg_base = lane - sl;
    const uint64_t seg_mask = (S == 64) ? ~0ull : (((1ull << S) - 1ull) << seg_base);
    const int row = group * (64 / S) + lane / S;
    if (row >= P.n_rows) return;  // whole segments only
    const uint64_t seg_ones = (S == 64) ? ~0ull : ((1ull << S) - 1ull);
    double *vars = wlds + (size_t)(lane / S) * P.var_stride;
    double *scr = tl.scr + lane;
    uint32_t *words = tl.words + lane;
    int32_t *locs = tl.locs + lane;
    uint32_t *bits = tl.bits + (lane / S) * (P.lpad / 32);
    const IsRows &st = P.st;
    const int n = m.n_comp;
    const double INF = __builtin_huge_val();

    uint8_t stat = st.status[row];
    if (!(stat & IS_ACTIVE)) return;  // its features and tilts are not read

    // load the run
    const uint64_t run = st.run[row];
    double t = st.t[row];
    double log2lr = st.log2lr[row];
    uint32_t step = st.step[row], trans = 0;  // trans: edges fired by this lane in this launch
    int chan = st.chan[row], sender = st.sender[row];
    bool goal = (stat & IS_GOAL) != 0;
    bool mid = (stat & IS_MID) != 0;
    LaneQuery q{P.qvar, st.qmax[row], st.qmin[row]};
    uint64_t digest = st.digest[row];
    for (int v = sl; v < m.n_vars; v += S) vars[v] = st.vars[(size_t)row * m.n_vars + v];
    if (sl == 0) vars[m.n_vars] = 0.0;
    // recording build: per slot the starting location, the base cumulative
    // hazard over the macro-step's races and the wins, in LDS ([slot][lane])
    double *hz = tl.rec + lane;
    int32_t *loc0 = (int32_t *)(tl.rec + 64 * C) + lane;
    uint32_t *wins = (uint32_t *)(tl.rec + 64 * C) + 64 * C + lane;
    // (the reads of all slots under way together: one after another, two
    // dependent reads each, they were most of a short step)
    int at[C];
    uint32_t rec_of[C], base_of[C];
#pragma unroll
    for (int j = 0; j < C; ++j) at[j] = sl * C + j < n ? (int)st.loc[(size_t)row * n + sl * C + j] : -1;
#pragma unroll
    for (int j = 0; j < C; ++j) base_of[j] = sl * C + j < n ? m.comp_word[sl * C + j] & m.base_mask : 0u;
#pragma unroll
    for (int j = 0; j < C; ++j) rec_of[j] = at[j] >= 0 ? m.loc_rec[at[j]] : 0u;
#pragma unroll
    for (int j = 0; j < C; ++j) {
        locs[64 * j] = at[j];
        words[64 * j] = (rec_of[j] << m.rec_shift) | base_of[j];
        if (REC) {
            loc0[64 * j] = at[j];
            hz[64 * j] = 0.0;
            wins[64 * j] = 0;
        }
    }
    wave_sync();
    // this row's tilts: theta and 2^theta by theta column
    const float *theta = nullptr;
    const double *tex = nullptr;
    if (P.theta) {
        if (P.theta_stride == 0) {
            theta = P.theta;
            tex = tl.ex;
        } else {
            float *th = tl.row_th + (size_t)(lane / S) * P.theta_cap;
            double *ex = tl.row_ex + (size_t)(lane / S) * P.theta_cap;
            const float *src = P.theta + (size_t)row * P.theta_stride;
            for (int i = sl; i < P.theta_len; i += S) {
                const float v = src[i];
                th[i] = v;
                ex[i] = smc_exp2((double)v);
            }
            wave_sync();
            theta = th;
            tex = ex;
        }
    }
    const int rec = (REC && P.rec_pos) ? P.rec_pos[row] : -1;
    if (rec >= 0) {
        write_features<C>(P, P.rec_X + (size_t)rec * P.fpad, locs, vars, bits, t, sl, S, n);
        if (sl == 0) P.rec_w[rec] = P.weight[st.job[row]];
    }
    bool hit = false, end = false, fired_any = false;
    bool changed = true;  // state changed since the last blocking tests
    uint32_t xblk = 0;    // blocked slots at the last change of state (tests of several records)
    auto receivers = [&]() {
        bool entered = false;
        if (P.trace)
            fire_receivers<C, true, true>(words, locs, Ctx{vars, t, 0}, m, chan, sender, q, entered, P.seed, run,
                                          step, lane, sl, S, seg_base, seg_mask, trans, digest);
        else
            fire_receivers<C, false, true>(words, locs, Ctx{vars, t, 0}, m, chan, sender, q, entered, P.seed, run,
                                           step, lane, sl, S, seg_base, seg_mask, trans, digest);
        chan = 0;
        sender = -1;
        goal = goal || (__ballot(entered) & seg_mask) != 0;
    };

    for (;;) {
        bool stop = false;
        if (!mid) {
            // loop test (simulation.cu:835-849), with the early stop of a
            // var-probability query once its outcome is settled
            if (!(t < P.bound)) end = true;
            else if (P.reach && goal) { end = true; hit = true; }
            else if (P.early_stop && !P.reach && settled(q, P, S)) { end = true; hit = true; }
            else if (step >= P.max_steps) end = true;
            if (end) break;
            // after a transition the pending broadcast is processed now, so
            // that the features show it; the next launch resumes at the race
            // (mid-iteration)
            stop = fired_any && P.stop_at_transition;
            if (chan > 0) {
                receivers();
                changed = true;
            }
            if (stop) {
                mid = true;
                break;
            }
        }
        mid = false;
        // a goal entered by receivers: this step is raced in full and
        // decides the hit (as in the run kernel)
        const bool full = P.reach && goal;
        if (!m.freeze && changed && !full && absorbed<C>(words, Ctx{vars, t, 0}, m, seg_mask)) {
            end = true;
            break;
        }
        double d = 0.0;
        int w = -1;
        bool exp_won = false;
        RaceSlots<C> rs;
        race_slots<C>(rs, words, Ctx{vars, t, 0}, m, changed, xblk);
        // windows of the bounded slots
        if (KEEP) {
            for (uint32_t b = rs.bounded; b; b &= b - 1) {
                const int j = __ffs(b) - 1;
                scr[64 * j] = slot_window(words, j, Ctx{vars, t, 0}, m);
            }
        }
        const auto window = [&](int j) { return KEEP ? scr[64 * j] : slot_window(words, j, Ctx{vars, t, 0}, m); };
        if (!full) changed = false;
        // frozen components race only in a full race (as in the run kernel)
        if (m.freeze && full) race_frozen<C>(rs, words, Ctx{vars, t, 0}, m);
        // tilted rates
        double leaft[C];
#pragma unroll
        for (int j = 0; j < C; ++j) {
            leaft[j] = rs.leaf[j];
            if (theta && rs.leaf[j] > 0.0) {
                const int ti = tl.tix[locs[64 * j]];
                if (ti >= 0) leaft[j] = rs.leaf[j] * tex[ti];
            }
        }
        const uint64_t zb = __ballot(rs.zero != 0) & seg_mask;
        if (zb) {
            const int Lz = lowest_lane(zb);
            w = (Lz - seg_base) * C + __shfl(__ffs(rs.zero) - 1, Lz);
        } else {
            // uniform delays; a tilted window (hazard times a = 2^theta)
            // draws M (1 - (1 - u)^(1/a))
            double umin = INF;
            int unif_j = -1;
#pragma clang loop unroll(disable)
            for (uint32_t b = rs.bounded; b;) {
                const int j = __ffs(b) - 1;
                const uint32_t c = (uint32_t)(sl * C + j);
                const smc_u32x4 rw = draw(P.seed, run, step, SMC_P_UNIFORM, smc_uniform_draw(c));
                // slot j, then slot j + 1 when it shares the draw
                const int nj = (C > 1 && !(c & 1u) && ((b >> (j + 1)) & 1u)) ? 2 : 1;
#pragma clang loop unroll(disable)
                for (int k = 0; k < nj; ++k) {
                    const int jk = j + k;
                    const double u = smc_uniform_u(rw, c + (uint32_t)k);
                    const double M = window(jk);
                    const int ti = theta ? tl.tix[locs[64 * jk]] : -1;
                    const bool tilted = ti >= 0 && theta[ti] != 0.0f;
                    const double du = tilted ? M * (1.0 - smc_exp2(device_log2(1.0 - u) / tex[ti])) : M * u;
                    if (du < umin) { umin = du; unif_j = jk; }
                    b &= b - 1;
                }
            }
            // tilted race: the run kernel's tree over the tilted rates
            double lvl[6] = {};
            const double Rt = race_total(lane_total<C>(leaft), lvl, S);
            const double R = theta ? tree_total<C>(rs.leaf, S) : Rt;
            double dexp = INF;
            int wexp = 0x7FFFFFFF;
            if (Rt > 0.0) {
                const smc_u32x4 rw = draw(P.seed, run, step, SMC_P_RACE, 0);
                dexp = -device_log2(smc_u01(rw.v[0], rw.v[1])) / Rt;
                wexp = race_pick<C>(leaft, lvl, smc_u01(rw.v[2], rw.v[3]) * Rt, S, seg_base, seg_mask);
            }
            double gu = umin;
            int wu = 0x7FFFFFFF;
            if (__ballot(unif_j >= 0) & seg_mask) {  // some slot of the run drew a delay
#pragma unroll
                for (int k = 0; k < 6; ++k)
                    if ((1 << k) < S) gu = fmin(gu, seg_xchg(gu, k));
                if (gu < INF) {
                    const int Lu = lowest_lane(__ballot(unif_j >= 0 && umin == gu) & seg_mask);
                    wu = (Lu - seg_base) * C + __shfl(unif_j, Lu);
                }
            }
            bool u_won = false;
            if (gu < dexp || (gu == dexp && wu < wexp)) { d = gu; w = wu; u_won = true; }
            else if (dexp < INF) { d = dexp; w = wexp; exp_won = true; }
            else d = INF;  // no racer: no event
            // the step that crosses the bound: the left-out null racers'
            // first event after it (base rates, no tilt)
            if (m.freeze && !full && d < INF && !(t + d < P.bound)) {
                const double Rd = frozen_total<C>(words, Ctx{vars, t, 0}, m, S);
                if (Rd > 0.0) {
                    const smc_u32x4 rw = draw(P.seed, run, step, SMC_P_DEAD, 0);
                    const double td = P.bound + (-device_log2(smc_u01(rw.v[0], rw.v[1])) / Rd);
                    if (td < t + d) { d = td - t; w = -1; exp_won = false; u_won = false; }
                }
            }
            if (theta && d < INF) {
                // log2 LR of this step: -theta_w (the winner's own draw) +
                // (R' - R) d + the tilted uniform racers' (1 - a) log2(1 -
                // d/M), summed on the race tree
                double th_w = 0.0;
                if (exp_won || u_won) {
                    const int ti = tl.tix[tl.locs[(w % C) * 64 + seg_base + w / C]];
                    if (ti >= 0) th_w = (double)theta[ti];
                }
                log2lr = log2lr - th_w + (Rt - R) * d;
                if (__ballot(rs.bounded != 0) & seg_mask) {
                    double ut[C];
#pragma unroll
                    for (int j = 0; j < C; ++j) {
                        ut[j] = 0.0;
                        if ((rs.bounded >> j) & 1u) {
                            const int ti = tl.tix[locs[64 * j]];
                            if (ti >= 0 && theta[ti] != 0.0f)
                                ut[j] = (1.0 - tex[ti]) * device_log2(1.0 - d / window(j));
                        }
                    }
                    log2lr = log2lr + tree_total<C>(ut, S);
                }
            }
            if ((exp_won || u_won) && rec >= 0) {
                if (lane == seg_base + w / C) wins[64 * (w % C)] += 1u;
            }
            if (REC && rec >= 0 && d < INF) {
                // each racer's base cumulative hazard over this step
                const double LN2 = 0.69314718055994530942;
#pragma unroll
                for (int j = 0; j < C; ++j) {
                    if (rs.leaf[j] > 0.0) hz[64 * j] = hz[64 * j] + LN2 * rs.leaf[j] * d;
                    else if ((rs.bounded >> j) & 1u) hz[64 * j] = hz[64 * j] + -LN2 * device_log2(1.0 - d / window(j));
                }
            }
        }
        if (!(d < INF)) { end = true; break; }  // no event: the run ends at its clock
        t = t + d;  // clocks advance
        if (w >= 0) {
            // the winner's transition, by every lane of its segment (as in
            // the run kernel)
            const int at = (w % C) * 64 + seg_base + w / C;
            const uint32_t ww = tl.words[at];
            const Ctx x{vars, t, word_base(ww, m)};
            const uint4 L1 = load_quad(m.locs + word_rec(ww, m), 1);
            const uint32_t first = L1.x;            // edge_first
            const int ne = (int)(L1.y & 0xFFFFu);   // edge_n
            const uint64_t mask = enabled_mask_by_lanes(first, ne, x, m, S, sl, seg_base, seg_ones);
            if (mask) {
                const int i = pick_edge(mask, first, L1.z, L1.w, P.seed, run, step, (uint32_t)w, x, m);
                const uint4 head = fire_updates(first + i, x, m, q);
                tl.words[at] = (head.x << m.rec_shift) | x.base;
                const int32_t lw = tl.locs[at];
                // the network's edge index (digests name it; records are shared)
                if (P.trace)
                    digest = smc_mix(digest, ((uint64_t)step << 40) | ((uint64_t)w << 20) |
                                                 (uint64_t)(m.loc_edge0[lw] + i));
                wave_sync();  // every lane has read the location
                tl.locs[at] = lw + rec_at(m.edges, first + i)->dst;
                goal |= (head.y & SMC_EF_GOAL) != 0;
                if (sl == 0) ++trans;
                changed = true;
                chan = (int)head.w > 0 ? (int)head.w : 0;
                sender = chan > 0 ? w : -1;
                fired_any = true;
            }
            wave_sync();
        }
        ++step;
    }

    // store the run
    const bool still = !end;
    {
        double qmax = q.qmax, qmin = q.qmin;
#pragma unroll
        for (int k = 0; k < 6; ++k)
            if ((1 << k) < S) {
                qmax = fmax(qmax, seg_xchg(qmax, k));
                qmin = fmin(qmin, seg_xchg(qmin, k));
                trans += (uint32_t)__shfl_xor((int)trans, 1 << k);
            }
        q.qmax = qmax; q.qmin = qmin;
    }
    if (end) {
        if (!hit && !P.reach) hit = P.is_max ? (q.qmax > P.threshold) : (q.qmin < P.threshold);
        if (P.trace) {
            digest = smc_mix(digest, smc_digest_bits(t));
            for (int v = 0; v < m.n_vars; ++v)
                digest = smc_mix(digest, smc_digest_bits(m.var_clock[v] ? t - vars[v] : vars[v]));
            for (int c = 0; c < n; ++c)
                digest = smc_mix(digest, (uint64_t)(uint32_t)tl.locs[(c % C) * 64 + seg_base + c / C]);
        }
    }
#pragma unroll
    for (int j = 0; j < C; ++j)
        if (sl * C + j < n) st.loc[(size_t)row * n + sl * C + j] = (uint16_t)locs[64 * j];
    for (int v = sl; v < m.n_vars; v += S) st.vars[(size_t)row * m.n_vars + v] = vars[v];
    if (sl == 0) {
        st.t[row] = t;
        st.log2lr[row] = log2lr;
        st.step[row] = step;
        st.trans[row] += trans;
        st.chan[row] = chan;
        st.sender[row] = sender;
        st.qmax[row] = q.qmax;
        st.qmin[row] = q.qmin;
        st.digest[row] = digest;
        st.status[row] = (uint8_t)((still ? IS_ACTIVE : 0) | (hit ? IS_HIT : 0) | (goal ? IS_GOAL : 0) |
                                   (still && mid ? IS_MID : 0));
    }
    const uint64_t rows_on = __ballot(still && sl == 0);
    if (P.active_count && rows_on && lane == lowest_lane(rows_on))
        atomicAdd(P.active_count + (blockIdx.x % SMC_IS_COUNTS) * SMC_IS_COUNT_STRIDE, (unsigned int)__popcll(rows_on));
    if (P.feat) write_features<C>(P, P.feat + (size_t)row * P.fpad, locs, vars, bits, t, sl, S, n);
    if (rec >= 0) {
        // statistics of the macro-step for the locations its components
        // started in (a component changes location only at the macro-step's
        // end): wins and base cumulative hazard
        float *A = P.rec_A + (size_t)rec * P.lpad;
        float *B = P.rec_B + (size_t)rec * P.lpad;
#pragma clang loop unroll(disable)
        for (int j = 0; j < C; ++j) {
            const int c = sl * C + j;
            if (c < n) {
                for (int l = m.comp_first_loc[c]; l < m.comp_first_loc[c + 1]; ++l) {
                    float a = 0.f, b = 0.f;
                    if (l == loc0[64 * j] && P.tiltable[l]) {
                        a = (float)wins[64 * j];
                        b = (float)hz[64 * j];
                    }
                    A[l] = a;
                    B[l] = b;
                }
            }
        }
        if (sl == 0)
            for (int k = m.n_locs; k < P.lpad; ++k) { A[k] = 0.f; B[k] = 0.f; }
    }
}

// A workgroup holds blockDim/64 waves; each takes groups of 64/S rows
// (blockIdx.x * waves + wave, then strided by the grid).  With TAB the
// workgroup first stages the model's hot tables in LDS (as the run kernel).
// LDS: [tables: TAB only][per wave: variables of its rows].
template <int C, bool TAB, bool REC, bool KEEP>
__device__ __forceinline__ void is_advance_body(const IsParams &P) {
    extern __shared__ __attribute__((aligned(16))) double lds[];
    const int wv = threadIdx.x >> 6, W = blockDim.x >> 6;
    // LDS: [tables: TAB only][tilt index: lpad int32][2^theta: theta_shared
    //      doubles] then per wave [variables][rows' 2^theta][rows' theta]
    //      [windows: C doubles per lane, if any location has an invariant]
    //      [state words, locations: 4 C bytes per lane each][locations held:
    //      lpad bits per row][recording build: 16 C bytes per lane]
    double *shared = lds + (TAB ? P.table_bytes / 8 : 0);
    int32_t *tix = (int32_t *)shared;
    double *ex = shared + P.lpad / 2;
    double *wlds = shared + P.lpad / 2 + P.theta_shared + (size_t)wv * (P.wave_lds / 8);
    const int R = 64 / P.lanes;
    TiltLds tl;
    tl.tix = tix;
    tl.ex = ex;
    tl.row_ex = wlds + (size_t)R * P.var_stride;
    tl.row_th = (float *)(tl.row_ex + (size_t)R * P.theta_cap);
    tl.scr = (double *)(tl.row_th + (size_t)R * P.theta_cap);
    tl.words = (uint32_t *)(tl.scr + (P.windows > 0 ? 64 * C : 0));
    tl.locs = (int32_t *)tl.words + 64 * C;
    tl.bits = (uint32_t *)(tl.locs + 64 * C);
    tl.rec = (double *)(tl.bits + R * (P.lpad / 32));
#pragma unroll 4
    for (int i = threadIdx.x; i < P.lpad; i += blockDim.x) tix[i] = P.tilt_index[i];
    if (P.theta && P.theta_stride == 0)
        for (int i = threadIdx.x; i < P.theta_len; i += blockDim.x) ex[i] = smc_exp2((double)P.theta[i]);
    if (blockIdx.x == 0 && threadIdx.x < SMC_IS_COUNTS && P.next_count)
        P.next_count[threadIdx.x * SMC_IS_COUNT_STRIDE] = 0;
    const int groups = (P.n_rows + R - 1) / R;
    if constexpr (TAB) {
        stage_tables(P.tables, P.table_bytes, lds);  // ends with the workgroup barrier
        const DevModelT<SmcLdsTables> m = lds_model(P.m, P.tables, lds);
        for (int g = blockIdx.x * W + wv; g < groups; g += gridDim.x * W) {
            is_advance_rows<C, REC, KEEP>(P, m, wlds, tl, g);
            wave_sync();
        }
    } else {
        __syncthreads();
        for (int g = blockIdx.x * W + wv; g < groups; g += gridDim.x * W) {
            is_advance_rows<C, REC, KEEP>(P, P.m, wlds, tl, g);
            wave_sync();
        }
    }
}

// What bounds it: the latency of a row's loads and of its step, and of the
// slowest row of a launch (a row may race several times before an edge
// fires).  Registers unrestricted: 171-243 VGPRs, two waves per SIMD.  Held to
// 168 it spills 43-71 of them at eight slots a lane: SIR-100, 5e4 rows, 24.1
// ms for 22.2.
template <int C, bool TAB, bool REC, bool KEEP = true>
__global__ __launch_bounds__(256) void is_advance_kernel(IsParams P) {
    is_advance_body<C, TAB, REC, KEEP>(P);
}

}  // namespace
