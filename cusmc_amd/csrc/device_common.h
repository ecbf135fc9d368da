// device_common.h — device helpers shared by the run kernel and the
// importance-sampling kernel: expression evaluation, edge enabling and
// choice, transitions, segment exchanges.
#pragma once

#include <hip/hip_runtime.h>
#include <float.h>
#include <stdint.h>

#include "devmodel.h"
#include "expr_ops.h"
#include "smc_stream.h"

namespace {

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ int lowest_lane(uint64_t m) { return __ffsll((unsigned long long)m) - 1; }

// A wave-uniform value, opaque to the optimiser from here on.  What is
// computed from it inside a loop (the round keys of a draw, the levels a
// segment has) stays there: hoisted, these invariants take some sixty scalar
// registers that no kernel here has left, and come back as lane reads of
// spilled registers, one vector instruction each.
__device__ __forceinline__ int scalar_here(int v) {
    asm volatile("" : "+s"(v));
    return v;
}
__device__ __forceinline__ uint64_t scalar_here(uint64_t v) {
    asm volatile("" : "+s"(v));
    return v;
}

// Whether any active lane has c: a wave-uniform condition, so what it guards
// is branched around as a whole, and with `unlikely` laid out away from the
// straight path.  A branch on a lane's own condition is taken whenever no
// lane needs the code, and with few waves on a SIMD the taken branches, not
// the instructions, are a step's latency (a step of the race took 336 of
// them).
__device__ __forceinline__ bool any_lane(bool c) { return __ballot(c) != 0; }
#define unlikely(c) __builtin_expect(!!(c), 0)

__device__ __forceinline__ double scalar_here(double v) {
    asm volatile("" : "+s"(v));
    return v;
}

// smc_log2 (the same operations in the same order) with its coefficients in
// scalar registers, where the compiler would move each into vector registers
// beside every multiply-add, and with the quotient's refinement written out:
// numerator and denominator are far from the ranges that the full division
// sequence scales and fixes up, and without those the steps are its own.
__device__ __forceinline__ double device_log2(double x) {
    const uint64_t b = smc_bits(x);
    int e = (int)((b >> 52) & 0x7FF) - 1023;
    double m = smc_from_bits((b & 0x000FFFFFFFFFFFFFull) | 0x3FF0000000000000ull);
    const bool high = m > 1.4142135623730951;
    m = high ? m * 0.5 : m;
    e += high ? 1 : 0;
    const double n = m - 1.0, d = m + 1.0;
    double r = __builtin_amdgcn_rcp(d);
    r = fma(r, fma(-d, r, 1.0), r);
    r = fma(r, fma(-d, r, 1.0), r);
    const double q = n * r;
    const double s = fma(fma(-d, q, n), r, q);
    const double z = s * s;
    double p = scalar_here(1.0 / 23.0);
    p = fma(p, z, scalar_here(1.0 / 21.0));
    p = fma(p, z, scalar_here(1.0 / 19.0));
    p = fma(p, z, scalar_here(1.0 / 17.0));
    p = fma(p, z, scalar_here(1.0 / 15.0));
    p = fma(p, z, scalar_here(1.0 / 13.0));
    p = fma(p, z, scalar_here(1.0 / 11.0));
    p = fma(p, z, scalar_here(1.0 / 9.0));
    p = fma(p, z, scalar_here(1.0 / 7.0));
    p = fma(p, z, scalar_here(1.0 / 5.0));
    p = fma(p, z, scalar_here(1.0 / 3.0));
    p = fma(p, z, 1.0);
    const double ln_m = (2.0 * s) * p;
    return fma(ln_m, scalar_here(1.4426950408889634074), (double)e);
}

// smc_draw with the key schedule computed at the draw (scalar adds beside
// the rounds).
__device__ __forceinline__ smc_u32x4 draw(uint64_t seed, uint64_t run, uint32_t step, uint32_t purpose,
                                          uint32_t comp) {
    return smc_draw(scalar_here(seed), run, step, purpose, comp);
}

// The same addressed by the counter's second word, (purpose << 24) | index.
__device__ __forceinline__ smc_u32x4 draw_at(uint64_t seed, uint64_t run, uint32_t step, uint32_t where) {
    seed = scalar_here(seed);
    const smc_u32x4 ctr = {{step, where, (uint32_t)run, (uint32_t)(run >> 32)}};
    return smc_philox4x32_10(ctr, (uint32_t)seed, (uint32_t)(seed >> 32));
}

// ------------------------------------------------------------ segment exchange
//
// Level k of a butterfly over an aligned segment: each lane receives the
// value held by the sibling block of 2^k lanes.  Levels 0-1 are DPP quad
// permutes (lane xor 1, xor 2), levels 2-3 DPP mirrors within 8 and 16
// lanes, level 4 a swizzle xor 16, level 5 a cross-half permute.  The
// mirrors reach a lane of the sibling block rather than the xor partner,
// which gives the same value whenever every lane of a block holds the same
// value — true at every level of a butterfly reduction.
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double x) {
    int lo = __double2loint(x), hi = __double2hiint(x);
    lo = __builtin_amdgcn_update_dpp(0, lo, CTRL, 0xF, 0xF, false);
    hi = __builtin_amdgcn_update_dpp(0, hi, CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double seg_xchg(double x, int k) {
    switch (k) {
    case 0: return dpp_f64<0xB1>(x);   // quad_perm [1,0,3,2]
    case 1: return dpp_f64<0x4E>(x);   // quad_perm [2,3,0,1]
    case 2: return dpp_f64<0x141>(x);  // row_half_mirror
    case 3: return dpp_f64<0x140>(x);  // row_mirror
    case 4: {
        int lo = __double2loint(x), hi = __double2hiint(x);
        lo = __builtin_amdgcn_ds_swizzle(lo, 0x401F);  // lane xor 16 within 32
        hi = __builtin_amdgcn_ds_swizzle(hi, 0x401F);
        return __hiloint2double(hi, lo);
    }
    default: return __shfl_xor(x, 32);
    }
}

// The lower and the upper half's value at level k of such a reduction, on
// every lane of the two halves: quad permutes, row shifts into one half of
// the banks, and swaps of rows; none goes through LDS.
__device__ __forceinline__ void seg_halves(double x, int k, double &lower, double &upper) {
    const int lo = __double2loint(x), hi = __double2hiint(x);
    switch (k) {
    case 0:
        lower = dpp_f64<0xA0>(x);  // quad_perm [0,0,2,2]
        upper = dpp_f64<0xF5>(x);  // quad_perm [1,1,3,3]
        return;
    case 1:
        lower = dpp_f64<0x44>(x);  // quad_perm [0,1,0,1]
        upper = dpp_f64<0xEE>(x);  // quad_perm [2,3,2,3]
        return;
    case 2:  // row_shr:4 into banks 1 and 3, row_shl:4 into banks 0 and 2
        lower = __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, 0x114, 0xF, 0xA, false),
                                 __builtin_amdgcn_update_dpp(lo, lo, 0x114, 0xF, 0xA, false));
        upper = __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, 0x104, 0xF, 0x5, false),
                                 __builtin_amdgcn_update_dpp(lo, lo, 0x104, 0xF, 0x5, false));
        return;
    case 3:  // row_shr:8 into banks 2 and 3, row_shl:8 into banks 0 and 1
        lower = __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, 0x118, 0xF, 0xC, false),
                                 __builtin_amdgcn_update_dpp(lo, lo, 0x118, 0xF, 0xC, false));
        upper = __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, 0x108, 0xF, 0x3, false),
                                 __builtin_amdgcn_update_dpp(lo, lo, 0x108, 0xF, 0x3, false));
        return;
    case 4: {
        const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
        lower = __hiloint2double((int)h[0], (int)l[0]);
        upper = __hiloint2double((int)h[1], (int)l[1]);
        return;
    }
    default: {
        const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
        lower = __hiloint2double((int)h[0], (int)l[0]);
        upper = __hiloint2double((int)h[1], (int)l[1]);
        return;
    }
    }
}

// Lanes of the upper halves at level k.
__device__ __forceinline__ uint64_t upper_lanes(int k) {
    constexpr uint64_t m[6] = {0xAAAAAAAAAAAAAAAAull, 0xCCCCCCCCCCCCCCCCull, 0xF0F0F0F0F0F0F0F0ull,
                               0xFF00FF00FF00FF00ull, 0xFFFF0000FFFF0000ull, 0xFFFFFFFF00000000ull};
    return m[k];
}


// Pairwise tree sum over the segment, as in the run kernel (in-lane levels,
// then the butterfly); every lane gets the total.
template <int C>
__device__ __forceinline__ double tree_total(const double (&leaf)[C], int S) {
    double tr[2 * C];
#pragma unroll
    for (int j = 0; j < C; ++j) tr[C + j] = leaf[j];
#pragma unroll
    for (int i = C - 1; i >= 1; --i) tr[i] = tr[2 * i] + tr[2 * i + 1];
    double s = (C == 1) ? leaf[0] : tr[1];
#pragma unroll
    for (int k = 0; k < 6; ++k)
        if ((1 << k) < S) s = s + seg_xchg(s, k);
    return s;
}

// ------------------------------------------------------------ table records

// A whole table record in 16-byte (8-byte) vector loads.  Copying a record
// field by field costs one narrow load per field used (seven for a
// location), each one a separate trip to the cache; the empty asm keeps the
// optimiser from narrowing the vector loads back to the fields used.
template <class T>
__device__ __forceinline__ T load_rec(const SMC_GLOBAL T *p) {
    static_assert(sizeof(T) % 8 == 0, "record size");
    T r;
    if constexpr (sizeof(T) % 16 == 0) {
        const SMC_GLOBAL uint4 *q = (const SMC_GLOBAL uint4 *)p;
        uint4 v[sizeof(T) / 16];
#pragma unroll
        for (int i = 0; i < (int)(sizeof(T) / 16); ++i) {
            v[i] = q[i];
            asm("" : "+v"(v[i].x), "+v"(v[i].y), "+v"(v[i].z), "+v"(v[i].w));
        }
        __builtin_memcpy(&r, v, sizeof(T));
    } else {
        const SMC_GLOBAL uint2 *q = (const SMC_GLOBAL uint2 *)p;
        uint2 v[sizeof(T) / 8];
#pragma unroll
        for (int i = 0; i < (int)(sizeof(T) / 8); ++i) {
            v[i] = q[i];
            asm("" : "+v"(v[i].x), "+v"(v[i].y));
        }
        __builtin_memcpy(&r, v, sizeof(T));
    }
    return r;
}

#if defined(__HIP_DEVICE_COMPILE__)
// The same from LDS (16-byte aligned there too); reads of fields there are
// cheap, so nothing is kept from being narrowed or scheduled.
template <class T>
__device__ __forceinline__ T load_rec(const SMC_LDS T *p) {
    static_assert(sizeof(T) % 8 == 0, "record size");
    T r;
    if constexpr (sizeof(T) % 16 == 0) {
        const SMC_LDS uint4 *q = (const SMC_LDS uint4 *)p;
        uint4 v[sizeof(T) / 16];
#pragma unroll
        for (int i = 0; i < (int)(sizeof(T) / 16); ++i) v[i] = q[i];
        __builtin_memcpy(&r, v, sizeof(T));
    } else {
        const SMC_LDS uint2 *q = (const SMC_LDS uint2 *)p;
        uint2 v[sizeof(T) / 8];
#pragma unroll
        for (int i = 0; i < (int)(sizeof(T) / 8); ++i) v[i] = q[i];
        __builtin_memcpy(&r, v, sizeof(T));
    }
    return r;
}
#endif

// 16 bytes of a record, and an edge's guard interval.
template <class T>
__device__ __forceinline__ uint4 load_quad(const SMC_GLOBAL T *p, int i) {
    return load_rec((const SMC_GLOBAL uint4 *)p + i);
}
struct DevRange { double lo, hi; };
__device__ __forceinline__ DevRange load_range(const SMC_GLOBAL DevEdge *p) {
    return load_rec((const SMC_GLOBAL DevRange *)p + 1);
}
#if defined(__HIP_DEVICE_COMPILE__)
template <class T>
__device__ __forceinline__ uint4 load_quad(const SMC_LDS T *p, int i) {
    return load_rec((const SMC_LDS uint4 *)p + i);
}
__device__ __forceinline__ DevRange load_range(const SMC_LDS DevEdge *p) {
    return load_rec((const SMC_LDS DevRange *)p + 1);
}
#endif
// Record i of a table.  In LDS, which holds fewer than 2^24 records, a 24-bit
// product: a full-rate instruction, where the 32-bit multiply of an index is a
// quarter-rate one.  A table in global memory may be longer.
template <class T>
__device__ __forceinline__ const SMC_GLOBAL T *rec_at(const SMC_GLOBAL T *p, uint32_t i) { return p + i; }
#if defined(__HIP_DEVICE_COMPILE__)
template <class T>
__device__ __forceinline__ const SMC_LDS T *rec_at(const SMC_LDS T *p, uint32_t i) {
    return (const SMC_LDS T *)((const SMC_LDS char *)p + __umul24(i, (uint32_t)sizeof(T)));
}
#endif
__device__ __forceinline__ double quad_f64(const uint4 &q) { return __hiloint2double((int)q.y, (int)q.x); }

// Table pointer of the global arena rebased onto its LDS copy.
template <class T>
__device__ __forceinline__ const SMC_LDS T *in_lds(const SMC_GLOBAL T *p, const SMC_GLOBAL uint8_t *base,
                                                   const SMC_LDS uint8_t *copy) {
    return (const SMC_LDS T *)(copy + ((const SMC_GLOBAL uint8_t *)p - base));
}

// Workgroup-wide copy of n 16-byte words into LDS, eight loads in flight
// per thread before their stores (a plain loop waits on every load).
__device__ __forceinline__ void copy_to_lds(const SMC_GLOBAL uint4 *src, SMC_LDS uint4 *dst, uint32_t n) {
    const uint32_t step = blockDim.x;
    for (uint32_t i = threadIdx.x; i < n; i += 8 * step) {
        uint4 v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            v[u] = uint4{0u, 0u, 0u, 0u};
            if (i + u * step < n) v[u] = src[i + u * step];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (i + u * step < n) dst[i + u * step] = v[u];
    }
}

// Copy the arena prefix [0, bytes) into the start of the workgroup's LDS
// (every thread of the workgroup takes part; ends with a barrier).
__device__ __forceinline__ void stage_tables(const SMC_GLOBAL uint8_t *src, uint32_t bytes, double *lds) {
    const SMC_GLOBAL uint4 *s4 = (const SMC_GLOBAL uint4 *)src;
    SMC_LDS uint4 *d4 = (SMC_LDS uint4 *)(SMC_LDS double *)lds;
    copy_to_lds(s4, d4, bytes / 16);
    __syncthreads();
}

// The model with its hot tables read from the staged copy.
__device__ __forceinline__ DevModelT<SmcLdsTables> lds_model(const DevModel &mg, const SMC_GLOBAL uint8_t *base,
                                                             double *lds) {
    const SMC_LDS uint8_t *tab = (const SMC_LDS uint8_t *)(SMC_LDS double *)lds;
    DevModelT<SmcLdsTables> m;
    m.hots = in_lds(mg.hots, base, tab);
    m.locs = in_lds(mg.locs, base, tab);
    m.invs = in_lds(mg.invs, base, tab);
    m.edges = in_lds(mg.edges, base, tab);
    m.guards = in_lds(mg.guards, base, tab);
    m.upds = in_lds(mg.upds, base, tab);
    m.consts = in_lds(mg.consts, base, tab);
    m.code = in_lds(mg.code, base, tab);
    m.var_init = mg.var_init;
    m.comp_word = mg.comp_word;
    m.comp_init_loc = mg.comp_init_loc;
    m.var_clock = mg.var_clock;
    m.comp_first_loc = mg.comp_first_loc;
    m.loc_edge0 = mg.loc_edge0;
    m.loc_rec = mg.loc_rec;
    m.n_comp = mg.n_comp;
    m.n_vars = mg.n_vars;
    m.n_leaves = mg.n_leaves;
    m.n_locs = mg.n_locs;
    m.rec_shift = mg.rec_shift;
    m.base_mask = mg.base_mask;
    m.tests = mg.tests;
    m.one_rate = mg.one_rate;
    m.freeze = mg.freeze;
    return m;
}

// ------------------------------------------------------------ expressions

// What evaluating an expression of one component needs: the run's variables
// and clock time, and where the component's private variables start.
struct Ctx {
    double *vars;
    double now;
    uint32_t base;
};

// Index of a record's variable operand.
__device__ __forceinline__ uint32_t var_at(uint32_t v, uint32_t base) {
    return (v & 0x7FFFu) + (base & (uint32_t)((int32_t)(v << 16) >> 31));
}
__device__ __forceinline__ uint32_t ref_var(uint32_t ref, uint32_t base) {
    return (ref & 0x1FFFFFFFu) + ((ref & SMC_REF_LOCAL) ? base : 0u);
}

// The operators that few models use, out of line: inlined at every
// expression site they would make up most of the kernels' code.
__attribute__((noinline)) __device__ double rare_op(int op, double a, double b, double c) {
    return smc_apply_op(op, a, b, c);
}

__device__ __forceinline__ double apply_op(int op, double a, double b, double c) {
    switch (op) {
    case SMC_E_ADD: return a + b;
    case SMC_E_SUB: return a - b;
    case SMC_E_MUL: return a * b;
    case SMC_E_DIV: return a / b;
    default: return rare_op(op, a, b, c);
    }
}

// Register-bytecode interpreter (expressions.cu:10-119).
template <class PC, class PI>
__device__ __forceinline__ double eval_code(uint32_t ref, const Ctx &x, PC consts, PI code) {
    const uint32_t first = ref & 0xFFFFFFu, count = (ref >> 24) & 0x3Fu;
    double r0 = 0.0, r1 = 0.0, r2 = 0.0, r3 = 0.0;
#pragma clang loop unroll(disable)
    for (uint32_t k = 0; k < count; ++k) {
        const DevInsn in = load_rec(code + first + k);
        double o[3];
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            const uint16_t w = s == 0 ? in.a : s == 1 ? in.b : in.c;
            const uint32_t kind = w >> 14, i = w & 0x3FFFu;
            if (kind == SMC_OPND_REG) o[s] = i == 0 ? r0 : i == 1 ? r1 : i == 2 ? r2 : r3;
            else if (kind == SMC_OPND_CONST) o[s] = consts[i];
            else {
                const double v = x.vars[(i & (SMC_OPND_LOCAL - 1u)) + ((i & SMC_OPND_LOCAL) ? x.base : 0u)];
                o[s] = kind == SMC_OPND_CLOCK ? x.now - v : v;
            }
        }
        const double v = apply_op(in.op, o[0], o[1], o[2]);
        r0 = in.dst == 0 ? v : r0;
        r1 = in.dst == 1 ? v : r1;
        r2 = in.dst == 2 ? v : r2;
        r3 = in.dst == 3 ? v : r3;
    }
    return r0;
}

// Value of an expression reference: constants and variables inline.
template <class M>
__device__ __forceinline__ double eval_ref(uint32_t ref, const Ctx &x, const M &m) {
    const uint32_t kind = ref >> 30;
    if (kind == SMC_REF_CODE) return eval_code(ref, x, m.consts, m.code);
    if (kind == SMC_REF_CONST) return m.consts[ref & 0x3FFFFFFFu];
    const double v = x.vars[ref_var(ref, x.base)];
    return kind == SMC_REF_CLOCK ? x.now - v : v;
}

template <class M>
__device__ __forceinline__ double location_rate(const DevLoc &L, const Ctx &x, const M &m) {
    const double r = L.rate_const ? L.rate_value : eval_ref(L.rate, x, m);
    return r > 0.0 ? r : 0.0;
}

// The value of a reference that is the same for every lane and reads no
// private variable: the instructions are decoded in scalar registers.
template <class M>
__device__ __forceinline__ double eval_uniform(uint32_t ref, const Ctx &x, const M &m) {
    if ((ref >> 30) != SMC_REF_CODE) return eval_ref(ref, x, m);
    const uint32_t first = ref & 0xFFFFFFu, count = (ref >> 24) & 0x3Fu;
    double r0 = 0.0, r1 = 0.0, r2 = 0.0, r3 = 0.0;
#pragma clang loop unroll(disable)
    for (uint32_t k = 0; k < count; ++k) {
        const DevInsn in = load_rec(m.code + first + k);
        uint32_t lo, hi;
        __builtin_memcpy(&lo, &in, 4);
        __builtin_memcpy(&hi, (const char *)&in + 4, 4);
        lo = __builtin_amdgcn_readfirstlane(lo);
        hi = __builtin_amdgcn_readfirstlane(hi);
        auto operand = [&](uint32_t w) {
            const uint32_t kind = w >> 14, i = w & 0x3FFFu;
            if (kind == SMC_OPND_REG) return i == 0 ? r0 : i == 1 ? r1 : i == 2 ? r2 : r3;
            if (kind == SMC_OPND_CONST) return (double)m.consts[i];
            const double v = x.vars[i];
            return kind == SMC_OPND_CLOCK ? x.now - v : v;
        };
        const int op = (int)(lo & 0xFFu);
        const uint32_t dst = (lo >> 8) & 0xFFu;
        const double a = operand(lo >> 16), b = operand(hi & 0xFFFFu);
        double v;
        if (op == SMC_E_ADD) v = a + b;
        else if (op == SMC_E_SUB) v = a - b;
        else if (op == SMC_E_MUL) v = a * b;
        else if (op == SMC_E_DIV) v = a / b;
        else v = rare_op(op, a, b, operand(hi >> 16));
        if (dst == 0) r0 = v;
        else if (dst == 1) r1 = v;
        else if (dst == 2) r2 = v;
        else r3 = v;
    }
    return r0;
}

// Rotate slot arrays by one (slot 1 to the front): a rolled loop over the
// slots then touches slot 0 only, a constant index, so the arrays stay in
// registers.
template <int C, class T>
__device__ __forceinline__ void rotate_slots(T (&a)[C]) {
    const T f = a[0];
#pragma unroll
    for (int k = 0; k < C - 1; ++k) a[k] = a[k + 1];
    a[C - 1] = f;
}

// ------------------------------------------------------------ slots
//
// A lane's component slots are state words in LDS ([slot][lane]: 64 lanes
// touch 64 consecutive words), so that loops over slots stay rolled where
// they are cold and any lane can read any slot.
template <class M>
__device__ __forceinline__ uint32_t word_rec(uint32_t w, const M &m) { return w >> m.rec_shift; }
template <class M>
__device__ __forceinline__ uint32_t word_base(uint32_t w, const M &m) { return w & m.base_mask; }

// ------------------------------------------------------------ edges

__device__ __forceinline__ bool guard_holds(int op, double x, double r) {
    switch (op) {
    case SMC_C_LE: return x <= r;
    case SMC_C_LT: return x < r;
    case SMC_C_GE: return x >= r;
    case SMC_C_GT: return x > r;
    case SMC_C_EQ: return fabs(x - r) <= SMC_TOL;
    default: return false;
    }
}

template <class M>
__device__ __forceinline__ bool guard_true(const DevGuard &G, const Ctx &x, const M &m) {
    double v = x.vars[var_at(G.var, x.base)];
    if (G.flags & SMC_GF_CLOCK) v = x.now - v;
    bool ok = G.lo <= v && v <= G.hi;
    const bool general = !(G.flags & SMC_GF_RANGE);
    if (unlikely(any_lane(general))) {
        if (general) ok = guard_holds(G.op, v, eval_ref(G.rhs, x, m));
    }
    return ok;
}

// A variable named by a byte offset and a factor (8 or 0) of the base.
__device__ __forceinline__ double *var_ptr(const Ctx &x, uint32_t offset, uint32_t flags) {
    return (double *)((char *)x.vars + offset + __umul24(x.base, flags & 0xFFu));
}

// Whether edge record e is enabled: spontaneous (recv_chan == 0) or a
// receive edge on channel recv_chan (check_enabled_edges
// simulation.cu:268-305, SyncInSerial :363-377).  `here`: the lane has an
// edge to test (others read a valid record all the same).
template <class M>
__device__ __forceinline__ bool edge_enabled(bool here, uint32_t e, int recv_chan, const Ctx &x, const M &m) {
    const uint4 head = load_quad(rec_at(m.edges, e), 0), tail = load_quad(rec_at(m.edges, e), 2);
    const DevRange range = load_range(rec_at(m.edges, e));
    const int channel = (int)head.w;
    double v = *var_ptr(x, tail.x & 0xFFFFu, tail.x >> 16);
    v = (tail.x & (SMC_EG_CLOCK << 16)) ? x.now - v : v;
    bool ok = here & !(head.y & SMC_EF_NEVER) & (recv_chan ? channel == -recv_chan : channel >= 0) &
              (((head.y & SMC_EF_NO_GUARD) != 0) | ((range.lo <= v) & (v <= range.hi)));
    const int more = (int)(tail.z & 0xFFFFu);  // guard_n
    if (any_lane(ok && more)) {
#pragma clang loop unroll(disable)
        for (int g = 0; any_lane(ok && g < more); ++g)
            if (ok && g < more) ok = guard_true(load_rec(rec_at(m.guards, tail.y + g)), x, m);
    }
    return ok;
}

// Enabled edges of a location as a bit mask over its edge list, by one lane.
template <class M>
__device__ __forceinline__ uint64_t enabled_mask(uint32_t edge_first, int edge_n, int recv_chan, const Ctx &x,
                                                 const M &m) {
    uint64_t mask = 0;
#pragma clang loop unroll(disable)
    for (int i = 0; i < edge_n; ++i)
        if (edge_enabled(true, edge_first + i, recv_chan, x, m)) mask |= 1ull << i;
    return mask;
}

// The same for spontaneous edges by all S lanes of a segment, each testing
// one edge at a time.
template <class M>
__device__ __forceinline__ uint64_t enabled_mask_by_lanes(uint32_t edge_first, int edge_n, const Ctx &x, const M &m,
                                                          int S, int sl, int seg_base, uint64_t seg_ones) {
    uint64_t mask = 0;
    int i0 = 0;
#pragma clang loop unroll(disable)
    do {
        const bool here = i0 + sl < edge_n;
        const bool ok = edge_enabled(here, edge_first + (here ? i0 + sl : 0), 0, x, m);
        mask |= ((__ballot(ok) >> seg_base) & seg_ones) << (i0 & 63);
        i0 += S;
    } while (any_lane(i0 < edge_n));
    return mask;
}

template <class M>
__device__ __forceinline__ long long edge_weight(uint32_t e, const Ctx &x, const M &m) {
    const uint4 head = load_quad(rec_at(m.edges, e), 0);
    long long w = (long long)head.z;
    const bool general = !(head.y & SMC_EF_WEIGHT_CONST);
    if (unlikely(any_lane(general))) {
        if (general) {
            const int v = smc_to_int(eval_ref(head.z, x, m));
            w = v > 0 ? v : 0;
        }
    }
    return w;
}

// Weighted choice among the edges in mask (two or more) for the uniform u
// (take_transition simulation.cu:43-79 and get_sum_edge_weight :9-24, with
// the weights of the enabled edges): the sum of the weights first, then from
// the highest edge down.
template <class M>
__device__ __forceinline__ int pick_weighted(uint64_t mask, uint32_t edge_first, double u, const Ctx &x, const M &m) {
    long long W = 0, rnd = 0;
    int pick = lowest_lane(mask);
    uint64_t r = mask;
    bool summed = false;
    // one loop for the sum and the scan, so the weights' expressions are
    // expanded once
#pragma clang loop unroll(disable)
    for (;;) {
        if (!r) {
            if (summed) break;
            summed = true;
            rnd = (long long)((double)W * u);
            r = mask;
        }
        const int i = 63 - __clzll((long long)r);
        r &= ~(1ull << i);
        const long long w = edge_weight(edge_first + i, x, m);
        if (!summed) W += w;
        else {
            W -= w;
            if (W <= rnd) { pick = i; break; }
        }
    }
    return pick;
}

// Weighted choice among the enabled edges in mask; the draw is made only
// when there is a choice.  With all of the location's spontaneous edges
// enabled and their weights constant (full, total: DevLoc.pick_*), the sum is
// known and one upward pass over the edges finds the last whose lower
// neighbours' weights do not exceed the draw.
template <class M>
__device__ __forceinline__ int pick_edge(uint64_t mask, uint32_t edge_first, uint32_t full, uint32_t total,
                                         uint64_t seed, uint64_t run, uint32_t step, uint32_t comp, const Ctx &x,
                                         const M &m) {
    int i = lowest_lane(mask);
    const bool choice = (mask & (mask - 1)) != 0;
    if (any_lane(choice)) {
        const smc_u32x4 w = draw(seed, run, step, SMC_P_WINNER, comp);
        const double u = smc_u01(w.v[0], w.v[1]);
        const bool quick = choice & (mask == (uint64_t)full);
        if (any_lane(quick)) {
            const uint32_t rnd = (uint32_t)((double)total * u);
            uint32_t r = quick ? full : 0u;
            uint32_t below = 0;  // (a lane that is done may wrap it)
#pragma clang loop unroll(disable)
            do {
                const int k = r ? __ffs(r) - 1 : 0;
                const uint32_t wk = rec_at(m.edges, edge_first + k)->weight;
                i = (r && below <= rnd) ? k : i;
                below += wk;
                r &= r - 1;
            } while (any_lane(r != 0));
        }
        const bool slow = choice & !quick;
        if (any_lane(slow)) {
            if (slow) i = pick_weighted(mask, edge_first, u, x, m);
        }
    }
    return i;
}

// The same for component c as a broadcast receiver: its uniform is word
// c & 3 of the receivers' shared draw c >> 2.
template <class M>
__device__ __forceinline__ int pick_receiver(uint64_t mask, uint32_t edge_first, uint64_t seed, uint64_t run,
                                             uint32_t step, uint32_t c, const Ctx &x, const M &m) {
    if ((mask & (mask - 1)) == 0) return lowest_lane(mask);
    const smc_u32x4 w = draw(seed, run, step, SMC_P_RECEIVER, smc_receiver_draw(c));
    return pick_weighted(mask, edge_first, smc_receiver_u(w, c), x, m);
}

struct LaneQuery {
    int qvar;
    double qmax, qmin;
};

// One plain update (value, variable and flags as in DevEdge), with query
// variable tracking.
__device__ __forceinline__ void plain_update(double value, uint32_t var_flags, const Ctx &x, LaneQuery &q) {
    const uint32_t flags = var_flags >> 16;
    double *at = var_ptr(x, var_flags & 0xFFFFu, flags);
    double v = value;
    if (flags & SMC_EU_ADD) v = *at + v;
    if (flags & (SMC_EU_ADD | SMC_EU_SET)) {
        if (at == x.vars + q.qvar) {
            q.qmax = v > q.qmax ? v : q.qmax;
            q.qmin = v < q.qmin ? v : q.qmin;
        }
        *at = (flags & SMC_EU_CLOCK) ? x.now - v : v;
    }
}

// The updates of edge record e in order (take_transition
// simulation.cu:88-180).  Any number of lanes may run it for the same
// component at once: they store the same values.  Returns the record's first
// 16 bytes.
template <class M>
__device__ __forceinline__ uint4 fire_updates(uint32_t e, const Ctx &x, const M &m, LaneQuery &q) {
    const uint4 head = load_quad(rec_at(m.edges, e), 0), more = load_quad(rec_at(m.edges, e), 2);
    const uint4 u0 = load_quad(rec_at(m.edges, e), 3), u1 = load_quad(rec_at(m.edges, e), 4);
    plain_update(quad_f64(u0), u0.z, x, q);
    plain_update(quad_f64(u1), u1.z, x, q);
    const int n = (int)(more.z >> 16);  // upd_n
    if (any_lane(n != 0)) {
#pragma clang loop unroll(disable)
        for (int k = 0; any_lane(k < n); ++k) {
            if (k < n) {
                const DevUpd U = load_rec(m.upds + more.w + k);
                const uint32_t at = var_at(U.var, x.base);
                double v = U.value;
                if (U.kind == SMC_U_ADD) v = x.vars[at] + v;
                const bool general = U.kind == SMC_U_EXPR;
                if (any_lane(general)) {
                    if (general) v = eval_ref(U.expr, x, m);
                }
                if ((int)at == q.qvar) {
                    if (v > q.qmax) q.qmax = v;
                    if (v < q.qmin) q.qmin = v;
                }
                x.vars[at] = U.clock ? x.now - v : v;
            }
        }
    }
    return head;
}

// ------------------------------------------------------------ blocking

// The blocking test of a location flagged SMC_LF_GUARDED: every edge has a
// false clock-free conjunct (one pass over its blocking records).  A blocked
// component cannot fire until a transition changes the variables.
// Locations flagged SMC_LF_DEAD are always blocked and are tested by their
// flag.
template <class M>
__device__ __forceinline__ bool location_blocked(uint32_t block_first, const Ctx &x, const M &m) {
    bool e_blk = false;
#pragma clang loop unroll(disable)
    for (uint32_t k = block_first;; ++k) {
        const DevGuard G = load_rec(rec_at(m.guards, k));
        if (!e_blk) e_blk = !guard_true(G, x, m);
        if (G.flags & SMC_GF_END_EDGE) {
            if (!e_blk) return false;
            e_blk = false;
        }
        if (G.flags & SMC_GF_END_LOC) return true;
    }
}

// Delay window of a location's invariants at this time: the least remaining
// time among the clock bounds still ahead; negative when there is none.
template <class M>
__device__ __forceinline__ double window_of(const DevLoc &L, const Ctx &x, const M &m) {
    double M0 = DBL_MAX;
    bool bounded = false;
#pragma clang loop unroll(disable)
    for (int i = 0; i < L.n_inv; ++i) {
        const DevInv iv = load_rec(m.invs + L.inv_first + i);
        const double bound = iv.bound_const ? iv.bound_value : eval_ref(iv.bound, x, m);
        double ttb = bound - (x.now - x.vars[var_at(iv.var, x.base)]);
        if (iv.strict) ttb -= 1e-6;
        if (ttb >= 0.0) { M0 = ttb < M0 ? ttb : M0; bounded = true; }
    }
    return bounded ? M0 : -1.0;
}

// Whether no component of the segment's run can fire again before the time
// bound: each one is blocked, or is in a location whose rate and spontaneous
// guards read no clock and has no enabled spontaneous edge or races at rate 0
// (an exponential location).  Zero-delay and clock-bounded locations with an
// enabled edge can fire.  Nothing but time changes such a state, so the run's
// outcome is decided.  For models without frozen racers: there the race
// itself ends such a run.
template <int C, class M>
__device__ __forceinline__ bool absorbed(const uint32_t *words, Ctx x, const M &m, uint64_t seg_mask) {
    bool can = false;
#pragma clang loop unroll(disable)
    for (int j = 0; j < C; ++j) {
        const uint32_t w = words[64 * j];
        if (can || !(w >> m.rec_shift)) continue;
        const DevLoc L = load_rec(m.locs + word_rec(w, m));
        x.base = word_base(w, m);
        if (L.klass == SMC_K_ZERO) { can = true; continue; }
        if ((L.flags & SMC_LF_DEAD) || ((L.flags & SMC_LF_GUARDED) && location_blocked(L.block_first, x, m))) continue;
        if (!(L.flags & SMC_LF_TIME_FREE)) { can = true; continue; }
        if (enabled_mask(L.edge_first, L.edge_n, 0, x, m) == 0) continue;
        if (L.klass != SMC_K_EXP || location_rate(L, x, m) > 0.0) can = true;
    }
    return (__ballot(can) & seg_mask) == 0;
}

// ------------------------------------------------------------ race

// What each slot does in the coming step.
template <int C>
struct RaceSlots {
    double leaf[C];         // rate in the exponential race, 0 if not in it
    double left[C];         // window of a bounded slot (kept for up to two slots, else see slot_window)
    uint32_t bounded;       // slots with a clock-bounded delay
    uint32_t zero;          // slots that fire at once: zero-delay locations, bounds reached
};

// A record's variable, given the component's state word.
__device__ __forceinline__ double hot_value(const DevHot &h, uint32_t word, const double *vars) {
    return *(const double *)((const char *)vars + ((word & h.base) << 3) + (h.what & 0xFFFFu));
}

// The delay window of slot j, which is bounded.  (One without an end is
// window_of's largest double.)
template <class M>
__device__ __forceinline__ double slot_window(const uint32_t *words, int j, Ctx x, const M &m) {
    const uint32_t w = words[64 * j];
    const DevHot h = load_rec(m.hots + word_rec(w, m));
    double left = h.a - (x.now - hot_value(h, w, x.vars)) - h.b;
    const bool other = (h.what & (SMC_HF_WINDOW << 16)) != 0;
    if (unlikely(any_lane(other))) {
        if (other) {
            x.base = word_base(w, m);
            left = window_of(load_rec(m.locs + word_rec(w, m)), x, m);
        }
    }
    return left;
}

// The delay windows of slots j and j + 1, read side by side: one after the
// other, three dependent LDS reads each, they were a tenth of a Fischer-32
// step.  Meaningless for a slot that is not bounded.
template <class M>
__device__ __forceinline__ void slot_windows(double (&left)[2], const uint32_t *words, int j, Ctx x, const M &m) {
    uint32_t w[2];
    DevHot h[2];
    double v[2];
    bool other = false;
#pragma unroll
    for (int k = 0; k < 2; ++k) w[k] = words[64 * (j + k)];
#pragma unroll
    for (int k = 0; k < 2; ++k) h[k] = load_rec(m.hots + word_rec(w[k], m));
#pragma unroll
    for (int k = 0; k < 2; ++k) v[k] = hot_value(h[k], w[k], x.vars);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        left[k] = h[k].a - (x.now - v[k]) - h[k].b;
        other |= (h[k].what & (SMC_HF_WINDOW << 16)) != 0;
    }
    if (unlikely(any_lane(other))) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            if (h[k].what & (SMC_HF_WINDOW << 16)) {
                x.base = word_base(w[k], m);
                left[k] = window_of(load_rec(m.locs + word_rec(w[k], m)), x, m);
            }
        }
    }
}

// Classify the lane's slots: one straight line over them, each reading its
// class's 32-byte record and its variable.  No branch depends on a lane or a
// slot: the lanes of a wave hold components in every kind of location, so
// branches would run every kind's code for every slot, and they would keep
// the slots' reads, a chain of three each, from overlapping.  What only some
// slots of a step need (the length of a bounded delay, rates that are
// expressions) is left to later passes over those.  About 17 vector
// instructions a slot with tests; with delays, expressions and zero tests in
// line it was 40.  Without tests half of the record is enough: SIR-350, 2e5
// runs, 65.3 ms for 66.4 with all of it.
// TESTS: some location has an invariant or a guard; RATE: 0 all rates are
// constant, 1 one expression of the value `shared`, 2 several (bits expr).
//
// Slot masks collect one bit a slot by shifting: bit 31 of a word (the sign
// of a zero delay's rate), or the lane's bit of a comparison's result as the
// carry of an addition, the last slot first.
__device__ __forceinline__ uint32_t shift_in_sign(uint32_t mask, uint32_t word) {
    return __builtin_amdgcn_alignbit(mask, word, 31);
}
__device__ __forceinline__ uint32_t shift_in(uint32_t mask, bool c) {
    const uint64_t lanes = __ballot(c);
    asm("v_addc_co_u32 %0, vcc, %0, %0, %1" : "+v"(mask) : "s"(lanes) : "vcc");
    return mask;
}

template <int C, bool TESTS, int RATE, class M>
__device__ __forceinline__ void classify(RaceSlots<C> &rs, const uint32_t *words, const Ctx &x, const M &m,
                                         double shared, uint32_t &expr, uint32_t &own) {
    // slots read at a time: registers for their records
    constexpr int G = C > 8 ? 8 : C;
    uint32_t bounded = 0, ahead = 0, zero = 0;
#pragma unroll
    for (int j0 = C - G; j0 >= 0; j0 -= G) {
        uint32_t w[G];
        DevHot h[G];
        double v[G];
#pragma unroll
        for (int j = 0; j < G; ++j) w[j] = words[64 * (j0 + j)];
#pragma unroll
        for (int j = 0; j < G; ++j) {
            if (TESTS) {
                h[j] = load_rec(m.hots + word_rec(w[j], m));
            } else {
                const uint4 half = load_quad(m.hots + word_rec(w[j], m), 0);
                h[j].rate = quad_f64(half);
                h[j].what = half.z;
                h[j].base = half.w;
            }
        }
        if (TESTS) {
#pragma unroll
            for (int j = 0; j < G; ++j) v[j] = hot_value(h[j], w[j], x.vars);
        }
#pragma unroll
        for (int j = G - 1; j >= 0; --j) {
            const uint32_t bit = 1u << (j0 + j), d = h[j].what;
            double rate = h[j].rate;
            zero = shift_in_sign(zero, (uint32_t)__double2hiint(rate));
            if (RATE == 1) rate = (int32_t)h[j].base < 0 ? shared : rate;
            bool in = true;
            if (TESTS) {
                // an invariant x <= a holds the delay to a - x - b while that
                // is not negative (a - x >= b), and at 0 makes it a zero delay
                const double ax = h[j].a - (x.now - v[j]);
                const bool inv = (int32_t)d < 0;
                const bool bnd = inv & (ax >= h[j].b);
                const bool inside = (h[j].a <= v[j]) & (v[j] <= h[j].b);
                in = inv ? !bnd : inside;
                bounded = shift_in(bounded, bnd);
                ahead = shift_in(ahead, ax > h[j].b);
                if (C <= 2) rs.left[j] = ax - h[j].b;
            }
            rs.leaf[j0 + j] = in ? rate : 0.0;
            if (RATE == 2) {
                expr |= (in & ((d & (SMC_HF_EXPR << 16)) != 0)) ? bit : 0u;
                own |= (d & (SMC_HF_EXPR_LOCAL << 16)) ? bit : 0u;
            }
        }
        if (j0) __builtin_amdgcn_sched_barrier(0);
    }
    rs.bounded = bounded;
    rs.zero = zero | (bounded & ~ahead);
}

// The same, with the invariants, blocking tests and rates that take more than
// a record, on models that have them.  xblk keeps the blocking results until
// the next change of state.
template <int C, class M>
__device__ __forceinline__ void race_slots(RaceSlots<C> &rs, const uint32_t *words, Ctx x, const M &m, bool changed,
                                           uint32_t &xblk) {
    const uint32_t tests = m.tests;
    uint32_t expr = 0;     // slots whose rate is still to be evaluated
    uint32_t own = 0;      // ... from private variables
    const bool with_tests = (tests & (SMC_HF_INV | SMC_HF_GUARD)) != 0;
    if (!(tests & SMC_HF_EXPR)) {
        if (with_tests) classify<C, true, 0>(rs, words, x, m, 0.0, expr, own);
        else classify<C, false, 0>(rs, words, x, m, 0.0, expr, own);
    } else if (m.one_rate != SMC_NO_REF) {
        // one rate expression: evaluated once, for every slot
        double shared = eval_uniform(m.one_rate, x, m);
        shared = shared > 0.0 ? shared : 0.0;
        if (with_tests) classify<C, true, 1>(rs, words, x, m, shared, expr, own);
        else classify<C, false, 1>(rs, words, x, m, shared, expr, own);
    } else {
        classify<C, true, 2>(rs, words, x, m, 0.0, expr, own);
    }
    // (up to two slots' windows are kept, so one without an end is set here)
    constexpr uint32_t kWindow = C <= 2 ? SMC_HF_WINDOW : SMC_HF_XINV;
    if (tests & (kWindow | SMC_HF_XBLK)) {
        if (changed) xblk = 0;
        uint32_t out = 0;
#pragma clang loop unroll(disable)
        for (int j = 0; j < C; ++j) {
            const uint32_t w = words[64 * j], bit = 1u << j;
            const uint32_t f = m.hots[word_rec(w, m)].what >> 16;
            if (f & (kWindow | SMC_HF_XBLK)) {
                const DevLoc L = load_rec(m.locs + word_rec(w, m));
                x.base = word_base(w, m);
                if (f & kWindow) {
                    const double left = window_of(L, x, m);
                    if (left >= 0.0) {
                        rs.bounded |= bit;
                        if (left == 0.0) rs.zero |= bit;
                        out |= bit;
                        if (j == 0) rs.left[0] = left;  // (constant indices: the array stays in registers)
                        else if (C == 2) rs.left[C - 1] = left;
                    }
                }
                if ((f & SMC_HF_XBLK) && changed && location_blocked(L.block_first, x, m)) xblk |= bit;
            }
        }
        out |= xblk;
        expr &= ~out;
#pragma unroll
        for (int j = 0; j < C; ++j) rs.leaf[j] = ((out >> j) & 1u) ? 0.0 : rs.leaf[j];
    }
    // Rates that are expressions: each pass evaluates, on every lane at once,
    // the expression of the lane's first pending slot and hands the value to
    // all of its pending slots with the same expression (unless it reads the
    // component's own variables).  Evaluated slot by slot, the interpreter
    // would run up to C times per race; here once per distinct expression a
    // lane holds.
    if ((tests & SMC_HF_EXPR) && m.one_rate == SMC_NO_REF) {
        uint32_t ref[C];
#pragma unroll
        for (int j = 0; j < C; ++j) ref[j] = m.locs[word_rec(words[64 * j], m)].rate;
        while (any_lane(expr != 0)) {
            double v = 0.0;
            uint32_t r = SMC_NO_REF, first = 0;
            if (expr) {
                first = expr & -expr;
                const uint32_t w = words[64 * (__ffs(first) - 1)];
                r = m.locs[word_rec(w, m)].rate;
                x.base = word_base(w, m);
                v = eval_ref(r, x, m);
                v = v > 0.0 ? v : 0.0;
            }
#pragma unroll
            for (int j = 0; j < C; ++j) {
                const uint32_t bit = 1u << j;
                if ((expr & bit) && (first == bit || (ref[j] == r && !(own & bit)))) {
                    rs.leaf[j] = v;
                    expr &= ~bit;
                }
            }
        }
    }
}

// The rate of slot j if its component is frozen: exponential now and unable
// to fire before the next transition (dead, or blocked by the variables).
// Frozen components leave the race; a step raced in full takes them back,
// and the transition that crosses the time bound still competes with their
// first null event after the bound, drawn from their sum (memoryless races).
template <class M>
__device__ __forceinline__ bool frozen_slot(const uint32_t *words, int j, Ctx x, const M &m, double *rate) {
    const uint32_t w = words[64 * j];
    const DevHot h = load_rec(m.hots + word_rec(w, m));
    const uint32_t d = h.what >> 16;
    const double v = hot_value(h, w, x.vars);
    const bool bnd = (d & SMC_HF_INV) && h.a - (x.now - v) >= h.b;
    bool frozen = (d & SMC_HF_DEAD) || ((d & SMC_HF_GUARD) && !(h.a <= v && v <= h.b));
    frozen = frozen && !bnd;
    *rate = h.rate;
    const bool other = (d & (SMC_HF_XINV | SMC_HF_XBLK)) || (frozen && (d & (SMC_HF_DEAD | SMC_HF_EXPR)));
    if (any_lane(other)) {
        if (other) {
            const DevLoc L = load_rec(m.locs + word_rec(w, m));
            x.base = word_base(w, m);
            if (d & (SMC_HF_XINV | SMC_HF_XBLK))
                frozen = !bnd && !((d & SMC_HF_XINV) && window_of(L, x, m) >= 0.0) &&
                         (frozen || ((d & SMC_HF_XBLK) && location_blocked(L.block_first, x, m)));
            if (frozen) *rate = location_rate(L, x, m);
        }
    }
    return frozen;
}

// Their sum on the race tree (every lane of the segment gets it): leaves in
// order, each completed pair added up at once.
template <int C, class M>
__device__ __forceinline__ double frozen_total(const uint32_t *words, const Ctx &x, const M &m, int S) {
    double half[4] = {0.0, 0.0, 0.0, 0.0}, s = 0.0;
#pragma clang loop unroll(disable)
    for (int j = 0; j < C; ++j) {
        double r;
        const bool frozen = frozen_slot(words, j, x, m, &r);
        s = frozen ? r : 0.0;
#pragma unroll
        for (int k = 0; (1 << k) < C; ++k) {
            if (!((j >> k) & 1)) {
                half[k] = s;
                break;
            }
            s = half[k] + s;
        }
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        if ((1 << k) >= S) break;
        s = s + seg_xchg(s, k);
    }
    return s;
}

// Frozen slots back into the race (their leaves are 0).
template <int C, class M>
__device__ __forceinline__ void race_frozen(RaceSlots<C> &rs, const uint32_t *words, const Ctx &x, const M &m) {
#pragma clang loop unroll(disable)
    for (int j = 0; j < C; ++j) {
        double r;
        if (frozen_slot(words, j, x, m, &r)) rs.leaf[0] = r;
        rotate_slots<C>(rs.leaf);
    }
}

// The exponential race over the segment is a fixed pairwise tree over the
// leaves.  Its levels within the lane:
template <int C>
__device__ __forceinline__ double lane_total(const double (&leaf)[C]) {
    double tr[2 * C];
#pragma unroll
    for (int j = 0; j < C; ++j) tr[C + j] = leaf[j];
#pragma unroll
    for (int i = C - 1; i >= 1; --i) tr[i] = tr[2 * i] + tr[2 * i + 1];
    return (C == 1) ? leaf[0] : tr[1];
}

// The levels above, a butterfly, from the lanes' sums s.  `level` keeps each
// level's own partial sum from the sum to the descent (12 registers; in LDS,
// read back and exchanged through it again, the two took 40 instructions and
// several hundred cycles more on a full segment).  Returns the total.
__device__ __forceinline__ double race_total(double s, double (&level)[6], int S) {
    // one way out of the levels, taken once
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        if ((1 << k) >= S) break;
        level[k] = s;
        if (k < 4) {
            s = s + seg_xchg(s, k);
        } else {
            double lower, upper;
            seg_halves(s, k, lower, upper);
            s = lower + upper;
        }
    }
    return s;
}

// The component reached by descending the tree with v in [0, total): left
// while v is below the left sum (or the right one is 0).  Each lane follows
// the path to itself; the one whose path the descent takes at every level
// (`on`) has it.  Every lane of the segment gets the component.
template <int C>
__device__ __forceinline__ int race_pick(const double (&leaf)[C], const double (&level)[6], double v, int S,
                                         int seg_base, uint64_t seg_mask) {
    uint64_t on = seg_mask;
#pragma unroll
    for (int k = 5; k >= 0; --k) {
        if ((1 << k) < S) {
            double left, right;
            seg_halves(level[k], k, left, right);
            const bool upper = __builtin_amdgcn_inverse_ballot_w64(upper_lanes(k));
            on &= __ballot((v < left) | (right == 0.0)) ^ upper_lanes(k);
            v = v - (upper ? left : 0.0);
        }
    }
    // the lane's tree again, from the same leaves (same sums), halved at
    // each level: cur holds the leaves under the current node
    int node = 0;
    if constexpr (C > 1) {
        double cur[C];
#pragma unroll
        for (int j = 0; j < C; ++j) cur[j] = leaf[j];
#pragma unroll
        for (int half = C / 2; half >= 1; half >>= 1) {
            double l[C / 2 > 0 ? C / 2 : 1], r[C / 2 > 0 ? C / 2 : 1];
#pragma unroll
            for (int j = 0; j < half; ++j) { l[j] = cur[j]; r[j] = cur[half + j]; }
#pragma unroll
            for (int w = half; w > 1; w >>= 1)
#pragma unroll
                for (int j = 0; j < w / 2; ++j) { l[j] = l[2 * j] + l[2 * j + 1]; r[j] = r[2 * j] + r[2 * j + 1]; }
            const bool go_left = v < l[0] || r[0] == 0.0;
            if (!go_left) { v = v - l[0]; node += half; }
#pragma unroll
            for (int j = 0; j < half; ++j) cur[j] = go_left ? cur[j] : cur[half + j];
        }
    }
    const int Lw = on ? lowest_lane(on) : seg_base;
    return (Lw - seg_base) * C + __shfl(node, Lw);
}

// ------------------------------------------------------------ receivers

// Word of the receivers' draw that component c uses.
__device__ __forceinline__ uint32_t receiver_word(const smc_u32x4 &w, uint32_t c) {
    const uint32_t a = (c & 1u) ? w.v[1] : w.v[0], b = (c & 1u) ? w.v[3] : w.v[2];
    return (c & 2u) ? b : a;
}

// A lane's additions to the query variable by receivers that fire at once:
// their sum, and the extremes of its prefixes.
struct ReceiverSums {
    double sum = 0.0, hi = -DBL_MAX, lo = DBL_MAX;
    bool any = false;
};

// The updates (additions and constants) of a receiver's edge record e, whose
// third quarter is `tail`, on the lanes where `on`.
template <class M>
__device__ __forceinline__ void receiver_updates(bool on, uint32_t e, const uint4 &tail, const Ctx &x, const M &m,
                                                 LaneQuery &q, ReceiverSums &sum) {
    auto update = [&](double value, double *at, bool add, bool clock) {
        if (add) {
            if (at == x.vars + q.qvar) {
                sum.sum += value;
                sum.hi = fmax(sum.hi, sum.sum);
                sum.lo = fmin(sum.lo, sum.sum);
                sum.any = true;
            }
            atomicAdd(at, value);
        } else {
            if (at == x.vars + q.qvar) {
                q.qmax = fmax(q.qmax, value);
                q.qmin = fmin(q.qmin, value);
            }
            *at = clock ? x.now - value : value;
        }
    };
    const uint4 u0 = load_quad(rec_at(m.edges, e), 3);
    if (any_lane(on && (u0.z >> 16) >= SMC_EU_ADD)) {
        const uint4 u1 = load_quad(rec_at(m.edges, e), 4);
        if (on && (u0.z >> 16) >= SMC_EU_ADD)
            update(quad_f64(u0), var_ptr(x, u0.z & 0xFFFFu, u0.z >> 16), (u0.z & (SMC_EU_ADD << 16)) != 0,
                   (u0.z & (SMC_EU_CLOCK << 16)) != 0);
        if (on && (u1.z >> 16) >= SMC_EU_ADD)
            update(quad_f64(u1), var_ptr(x, u1.z & 0xFFFFu, u1.z >> 16), (u1.z & (SMC_EU_ADD << 16)) != 0,
                   (u1.z & (SMC_EU_CLOCK << 16)) != 0);
        const int n = on ? (int)(tail.z >> 16) : 0;
        if (any_lane(n != 0)) {
            for (int k = 0; k < n; ++k) {
                const DevUpd U = load_rec(m.upds + tail.w + k);
                update(U.value, x.vars + var_at(U.var, x.base), U.kind == SMC_U_ADD, U.clock != 0);
            }
        }
    }
}

// The query variable's extremes over them, in component order.
__device__ __forceinline__ void receiver_query(const ReceiverSums &sum, double v0, LaneQuery &q, int sl, int S) {
    if (q.qvar >= 0 && any_lane(sum.any)) {
        double incl = sum.sum;
        for (int k = 1; k < S; k <<= 1) {
            const double y = __shfl_up(incl, k, S);
            if (sl >= k) incl += y;
        }
        const double at = v0 + (incl - sum.sum);  // value before this lane's additions
        if (sum.any) {
            q.qmax = fmax(q.qmax, at + sum.hi);
            q.qmin = fmin(q.qmin, at + sum.lo);
        }
    }
}

// Their edges into the digest, in component order.
template <int C>
__device__ __forceinline__ void digest_receivers(const int (&fired)[C], bool any, uint64_t &digest, uint32_t step,
                                                 int seg_base, uint64_t seg_mask) {
    for (uint64_t lanes_with = __ballot(any) & seg_mask; lanes_with; lanes_with &= lanes_with - 1) {
        const int L = lowest_lane(lanes_with);
#pragma unroll
        for (int j = 0; j < C; ++j) {
            const int e = __shfl(fired[j], L);
            if (e >= 0)
                digest = smc_mix(digest, ((uint64_t)step << 40) | ((uint64_t)((L - seg_base) * C + j) << 20) |
                                             (uint64_t)e);
        }
    }
}

// Receivers with guards, on several channels, or with three edges or more.
template <int C, bool TRACE, bool LOCS, class M>
__device__ __forceinline__ void fire_receivers_general(uint32_t *words, int32_t *locs, Ctx x, const M &m, int chan,
                                                       int sender, LaneQuery &q, bool &goal, uint64_t seed,
                                                       uint64_t run, uint32_t step, int lane, int sl, int S,
                                                       int seg_base, uint64_t seg_mask, uint32_t &trans,
                                                       uint64_t &digest) {
    // the enabled receive edges of every slot but the sender's: one bit set
    // each, from its location's record where they are all unguarded on one
    // channel
    uint32_t mk[C];
    uint32_t other = 0;
#pragma unroll
    for (int j = 0; j < C; ++j) {
        const uint4 rv = load_quad(m.locs + word_rec(words[64 * j], m), 0);
        const bool me = sl * C + j == sender;
        mk[j] = (((int)rv.x == chan) & !me) ? rv.y : 0u;
        other |= (((int)rv.x == -1) & !me) ? 1u << j : 0u;
    }
    uint64_t slow = 0;
    uint32_t mk_hi[C];  // edges past the 32nd (only where receivers fire one at a time)
#pragma unroll
    for (int j = 0; j < C; ++j) mk_hi[j] = 0;
    if (any_lane(other != 0)) {
        bool serial = false;
#pragma clang loop unroll(disable)
        for (int j = 0; j < C; ++j) {
            if ((other >> j) & 1u) {
                const uint32_t w = words[64 * j];
                const DevLoc L = load_rec(m.locs + word_rec(w, m));
                x.base = word_base(w, m);
                const uint64_t e = enabled_mask(L.edge_first, L.edge_n, chan, x, m);
                if (e && !(L.flags & SMC_LF_RECV_FAST)) serial = true;
                mk[0] = (uint32_t)e;
                mk_hi[0] = (uint32_t)(e >> 32);
            }
            rotate_slots<C>(mk);
            rotate_slots<C>(mk_hi);
        }
        slow = __ballot(serial) & seg_mask;
    }
    if (!slow) {
        int fired[TRACE ? C : 1];  // the network's index of each slot's edge (digests)
        bool any = false;
        ReceiverSums sum;
        const double v0 = q.qvar >= 0 ? x.vars[q.qvar] : 0.0;
        wave_sync();  // read before any receiver's additions
        // Receivers 4g .. 4g+3 share draw g: the lane's slots of one draw are
        // G consecutive slots (C is a power of two), drawn once at the first
        // of them when any of them has a choice to make.
        constexpr int G = C < 4 ? C : 4;
        smc_u32x4 rw = {{0u, 0u, 0u, 0u}};
#pragma unroll
        for (int j = 0; j < C; ++j) {
            const uint32_t c = (uint32_t)(sl * C + j);
            if (j % G == 0) {
                bool choice = false;
#pragma unroll
                for (int k = j; k < j + G; ++k) choice |= (mk[k] & (mk[k] - 1)) != 0;
                if (any_lane(choice)) rw = draw(seed, run, step, SMC_P_RECEIVER, smc_receiver_draw(c));
            }
            if (any_lane(mk[j] != 0)) {
                const uint32_t w = words[64 * j];
                const bool on = mk[j] != 0, choice = (mk[j] & (mk[j] - 1)) != 0;
                const uint4 rv = load_quad(m.locs + word_rec(w, m), 0);
                const uint32_t ef = m.locs[word_rec(w, m)].edge_first;
                int i = on ? __ffs(mk[j]) - 1 : 0;
                if (any_lane(choice)) {
                    // weighted choice; weights are constants
                    const bool two = choice & ((rv.w & SMC_RF_TWO) != 0) & (mk[j] == rv.y);
                    if (two & (receiver_word(rw, c) >= rv.z)) i = 31 - __clz((int)mk[j]);
                    const bool several = choice & !two;
                    if (unlikely(any_lane(several))) {
                        if (several) {
                            const double u = smc_receiver_u(rw, c);
                            int64_t W = 0;
                            for (uint32_t r = mk[j]; r; r &= r - 1) W += rec_at(m.edges, ef + __ffs(r) - 1)->weight;
                            const int64_t rnd = (int64_t)((double)W * u);
                            for (uint32_t r = mk[j]; r;) {
                                const int k = 31 - __clz((int)r);
                                r &= ~(1u << k);
                                W -= rec_at(m.edges, ef + k)->weight;
                                if (W <= rnd) { i = k; break; }
                            }
                        }
                    }
                }
                const uint32_t e = ef + i;
                const uint4 head = load_quad(rec_at(m.edges, e), 0), tail = load_quad(rec_at(m.edges, e), 2);
                const uint32_t base = word_base(w, m);
                any |= on;
                trans += on ? 1u : 0u;
                goal |= on & ((head.y & SMC_EF_GOAL) != 0);
                if (on) words[64 * j] = (head.x << m.rec_shift) | base;
                if (TRACE) fired[j] = on ? m.loc_edge0[on ? locs[64 * j] : 0] + i : -1;
                if (LOCS && on) locs[64 * j] += rec_at(m.edges, e)->dst;
                x.base = base;
                receiver_updates(on, e, tail, x, m, q, sum);
            } else if (TRACE) fired[j] = -1;
        }
        receiver_query(sum, v0, q, sl, S);
        if constexpr (TRACE) digest_receivers<C>(fired, any, digest, step, seg_base, seg_mask);
    } else {
        // one at a time: the lanes holding enabled receivers in lane order,
        // their slots in slot order; each picks with its own stream
        bool any = false;
#pragma unroll
        for (int j = 0; j < C; ++j) any |= (mk[j] | mk_hi[j]) != 0;
        for (uint64_t lanes_with = __ballot(any) & seg_mask; lanes_with; lanes_with &= lanes_with - 1) {
            const int L = lowest_lane(lanes_with);
#pragma clang loop unroll(disable)
            for (int j = 0; j < C; ++j) {
                const uint64_t mask = ((uint64_t)mk_hi[0] << 32) | mk[0];
                if ((__ballot(mask != 0) >> L) & 1ull) {
                    const int c = (L - seg_base) * C + j;
                    int e_fired = -1;  // the network's index of the fired edge (digests)
                    if (lane == L) {
                        const uint32_t w = words[64 * j];
                        const uint32_t first = m.locs[word_rec(w, m)].edge_first;
                        x.base = word_base(w, m);
                        const int i = pick_receiver(mask, first, seed, run, step, (uint32_t)c, x, m);
                        const uint4 head = fire_updates(first + i, x, m, q);
                        if (head.y & SMC_EF_GOAL) goal = true;
                        words[64 * j] = (head.x << m.rec_shift) | x.base;
                        ++trans;
                        if (TRACE) e_fired = m.loc_edge0[locs[64 * j]] + i;
                        if (LOCS) locs[64 * j] += rec_at(m.edges, first + i)->dst;
                    }
                    wave_sync();
                    if (TRACE) {
                        const int e = __shfl(e_fired, L);
                        digest = smc_mix(digest, ((uint64_t)step << 40) | ((uint64_t)c << 20) | (uint64_t)e);
                    }
                }
                rotate_slots<C>(mk);
                rotate_slots<C>(mk_hi);
            }
        }
    }
    wave_sync();
}

// Receivers of the broadcast `chan` sent by component `sender`
// (SyncInSerial simulation.cu:357-407): the enabled receive edges of every
// other component, then one edge fired per component that has any.
//
// Nearly always every receive edge commutes (SMC_LF_RECV_FAST): constant
// weights make each receiver's pick independent of the others' updates, and
// integer additions and private constants give the same variables in any
// order, so all fire at once.  The query variable's running max/min needs
// the values in component order: they are v0 plus the prefix sums of the
// additions, an exclusive scan over the segment (blocked layout: lane order
// then slot order is component order).  Otherwise they fire one at a time in
// component order, the enabled sets computed before any of them fires.
// TRACE mixes the fired edges into the digest in component order; LOCS keeps
// the network's locations beside the state words; `trans` counts this
// lane's.
template <int C, bool TRACE, bool LOCS, class M>
__device__ __forceinline__ void fire_receivers(uint32_t *words, int32_t *locs, Ctx x, const M &m, int chan,
                                               int sender, LaneQuery &q, bool &goal, uint64_t seed, uint64_t run,
                                               uint32_t step, int lane, int sl, int S, int seg_base, uint64_t seg_mask,
                                               uint32_t &trans, uint64_t &digest) {
    uint32_t on = 0, two = 0, low_idle = 0, high_idle = 0, general = 0;
    uint32_t split[C];
    constexpr int G = C < 8 ? C : 8;  // records read at a time
#pragma unroll
    for (int j0 = C - G; j0 >= 0; j0 -= G) {
        uint4 rv[G];  // recv_chan, recv_mask, recv_split, recv_flags
#pragma unroll
        for (int j = 0; j < G; ++j) rv[j] = load_quad(m.locs + word_rec(words[64 * (j0 + j)], m), 0);
#pragma unroll
        for (int j = G - 1; j >= 0; --j) {
            const bool here = (int)rv[j].x == chan;
            on = shift_in(on, here);
            general = shift_in(general, ((int)rv[j].x == -1) | (here & ((rv[j].w & SMC_RF_MORE) != 0)));
            two = shift_in_sign(two, rv[j].w);
            low_idle = shift_in_sign(low_idle, rv[j].w << 2);
            high_idle = shift_in_sign(high_idle, rv[j].w << 3);
            split[j0 + j] = rv[j].z;
        }
    }
    const uint32_t others = sl == sender / C ? ~(1u << (sender % C)) : ~0u;
    on &= others;
    general &= others;
    if (any_lane(general != 0)) {
        fire_receivers_general<C, TRACE, LOCS>(words, locs, x, m, chan, sender, q, goal, seed, run, step, lane, sl, S,
                                               seg_base, seg_mask, trans, digest);
        return;
    }
    // the picks: receivers 4g .. 4g+3 share draw g, made when any of the
    // lane's slots of it has a choice
    const uint32_t choice = on & two;
    uint32_t high = 0;
    constexpr int D = C < 4 ? C : 4;
#pragma unroll
    for (int j0 = C - D; j0 >= 0; j0 -= D) {
        const uint32_t c0 = (uint32_t)(sl * C + j0);
        if (any_lane(((choice >> j0) & ((1u << D) - 1u)) != 0)) {
            const smc_u32x4 rw = draw(seed, run, step, SMC_P_RECEIVER, smc_receiver_draw(c0));
#pragma unroll
            for (int j = D - 1; j >= 0; --j)
                high = shift_in(high, (D == 4 ? rw.v[j] : receiver_word(rw, c0 + j)) >= split[j0 + j]);
        } else {
            high <<= D;
        }
    }
    high &= choice;
    trans += (uint32_t)__popc(on);
    int fired[TRACE ? C : 1];  // the network's index of each slot's edge (digests)
    if (TRACE) {
#pragma unroll
        for (int j = 0; j < C; ++j) {
            const uint32_t mask = load_quad(m.locs + word_rec(words[64 * j], m), 0).y;
            const int i = (high >> j) & 1u ? 31 - __clz((int)mask) : __ffs(mask) - 1;
            fired[j] = (on >> j) & 1u ? m.loc_edge0[locs[64 * j]] + i : -1;
        }
    }
    const double v0 = q.qvar >= 0 ? x.vars[q.qvar] : 0.0;
    wave_sync();  // read before any receiver's additions
    ReceiverSums sum;
#pragma clang loop unroll(disable)
    for (uint32_t act = on & ~((high & high_idle) | (~high & low_idle)); any_lane(act != 0); act &= act - 1) {
        const bool go = act != 0;
        const int j = go ? __ffs(act) - 1 : 0;
        const uint32_t w = words[64 * j];
        const auto L = m.locs + word_rec(w, m);
        const uint32_t mask = load_quad(L, 0).y;
        const int i = (high >> j) & 1u ? 31 - __clz((int)mask) : __ffs(mask) - 1;
        const uint32_t e = go ? L->edge_first + i : 0u;
        const uint4 head = load_quad(rec_at(m.edges, e), 0), tail = load_quad(rec_at(m.edges, e), 2);
        goal |= go & ((head.y & SMC_EF_GOAL) != 0);
        x.base = word_base(w, m);
        if (go) words[64 * j] = (head.x << m.rec_shift) | x.base;
        if (LOCS && go) locs[64 * j] += rec_at(m.edges, e)->dst;
        receiver_updates(go, e, tail, x, m, q, sum);
    }
    receiver_query(sum, v0, q, sl, S);
    if constexpr (TRACE) digest_receivers<C>(fired, on != 0, digest, step, seg_base, seg_mask);
    wave_sync();
}

}  // namespace
