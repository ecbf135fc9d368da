// devmodel.h — device-side model tables of the run kernel (host and device).
//
// cuSMC keeps a level-major NodeInfo table with 40-byte nodes, 152-byte
// GuardInfo records and one device allocation per expression node
// (simulation/state/shared_model_state.cuh:45-217, shared_model_state.cu:
// 15-161).  Here the model is one arena of small fixed-size records indexed
// by 32-bit offsets, and every expression is either an inline constant, an
// inline variable reference or a short run of register bytecode:
//
//   expression reference (uint32):  bits 31..30 kind
//       SMC_REF_CONST  index into consts[]
//       SMC_REF_VAR    variable operand (an integer variable)
//       SMC_REF_CODE   bits 0..23 first instruction, bits 24..29 count
//       SMC_REF_CLOCK  variable operand of a clock
//
//   instruction (8 bytes): op, dst register, up to three operands; an
//   operand (uint16) is a register r0..r3, a variable, a constant or a
//   clock: bits 15..14 kind (0 reg, 1 var, 2 const, 3 clock), bits 13..0
//   index.  The value of an expression is register r0 after its last
//   instruction.
//
// Variables private to one component are named relative to that component's
// first private variable (the `local` bit of a variable operand), so that the
// instances of one template have the same records: the network's locations
// fall into classes of equal records (DevHot + DevLoc; equal edges, guards,
// updates, and destinations of equal class), and a component's state is one
// word: the class of its location and its private variables' base.
//
// Clocks are stored as reset stamps: a run's variable array holds, for a
// clock x, the time s at which x would have been 0, and its value is t - s
// with t the run's clock time.  Time then advances without a store, however
// many clocks the network has; assigning x := v stores s = t - v.
#pragma once

#include <stdint.h>
#include <type_traits>

#define SMC_REF_CONST 0u
#define SMC_REF_VAR 1u
#define SMC_REF_CODE 2u
#define SMC_REF_CLOCK 3u
#define SMC_NO_REF 0xFFFFFFFFu
#define SMC_REF_KIND(r) ((r) >> 30)
#define SMC_REF_MAKE(kind, payload) (((uint32_t)(kind) << 30) | (uint32_t)(payload))
#define SMC_REF_CODE_MAKE(first, count) (((uint32_t)SMC_REF_CODE << 30) | ((uint32_t)(count) << 24) | (uint32_t)(first))

#define SMC_OPND_REG 0u
#define SMC_OPND_VAR 1u
#define SMC_OPND_CONST 2u
#define SMC_OPND_CLOCK 3u
#define SMC_OPND(kind, idx) ((uint16_t)(((kind) << 14) | (idx)))

// A variable operand: index, and whether it counts from the component's base.
#define SMC_VAR_LOCAL 0x8000u                  // in the records' 16-bit fields
#define SMC_OPND_LOCAL 0x2000u                 // in an instruction's operand
#define SMC_REF_LOCAL 0x20000000u              // in an expression reference
#define SMC_MAX_LOCAL_VARS 8192                // networks with fewer variables use local operands

#define SMC_NREGS 4
#define SMC_MAX_CODE_LEN 63
#define SMC_MAX_OPND_INDEX 16383
#define SMC_MAX_EDGES_PER_LOC 64

// Delay classes of a location (simulation.cu:437-540).
enum smc_delay_class {
    SMC_K_ZERO = 0,     // branchpoint, urgent, committed: delay 0
    SMC_K_EXP = 1,      // exponential at the location's rate
    SMC_K_BOUNDED = 2   // uniform up to the nearest clock upper bound, else exponential
};

// Location flags.
enum {
    SMC_LF_TIME_FREE = 1,   // rate and spontaneous guards read no clock: enabling and rate
                            // change only with transitions
    SMC_LF_DEAD = 2,        // no spontaneous edge can ever fire (each has a `!=` conjunct, or
                            // there is none): always blocked
    SMC_LF_GUARDED = 4,     // blocked or not by the variables: every spontaneous edge without
                            // `!=` has a conjunct that reads no clock (DevLoc.block_first)
    SMC_LF_RECV_FAST = 8    // every receive edge commutes (see DevUpd), constant weights
};

// DevLoc.recv_flags (recv_chan > 0).
enum : uint32_t {
    SMC_RF_TWO = 0x80000000u,     // exactly two receive edges
    SMC_RF_MORE = 0x40000000u,    // three or more
    SMC_RF_LOW_IDLE = 0x20000000u,   // the lower one (or the only one) changes nothing
    SMC_RF_HIGH_IDLE = 0x10000000u   // the higher one of two changes nothing
};

// What a race step has to look at in a location (high half of DevHot.what).
enum {
    SMC_HF_WINDOW = 0x80,   // the delay window is not what the record's invariant leaves: XINV, or with INV one
                            // that may have no end (an infinite or very large bound or clock)
    SMC_HF_EXPR = 0x200,    // the rate is an expression (DevLoc.rate)
    SMC_HF_EXPR_LOCAL = 0x400,  // ... which reads private variables
    SMC_HF_XINV = 0x800,    // other invariants: DevInv records
    SMC_HF_XBLK = 0x1000,   // other blocking tests: guard records from block_first
    SMC_HF_DEAD = 0x2000,   // out of the race unless bounded
    SMC_HF_GUARD = 0x4000,  // leaves the race while its variable is outside [a, b]
    SMC_HF_INV = 0x8000     // one invariant with a constant bound: a = bound, b = 1e-6 if strict
};

#define SMC_HB_EXPR 0x80000000u  // DevHot.base: the rate is an expression

struct DevInsn {
    uint8_t op;
    uint8_t dst;
    uint16_t a, b, c;
};

// The part of a location that every race step reads for every component, 32
// bytes: two 16-byte LDS reads.  `rate` is what the component races at if
// nothing else holds (-0, with its sign bit, for a zero-delay location and
// only there; 0 for one that can never fire and for a rate that is not
// positive).  A location with neither
// invariant nor guard tests a constant 0 (kept behind the run's variables)
// against [-inf, inf], so that all take the same steps.
// The first half is all that a model without invariants and blocking tests
// reads.
struct DevHot {
    double rate;
    uint32_t what;          // low half: the variable's byte offset; high half: SMC_HF_*
    uint32_t base;          // mask of the state word's base: all ones if the variable is private, else 0;
                            // SMC_HB_EXPR, a bit that no state word has
    double a, b;
};

// The rest, 64 bytes: receive edges; spontaneous edges; invariants, blocking
// test and rate.
struct DevLoc {
    int32_t recv_chan;      // every receive edge is unguarded, on this channel, among the first 32 edges, and
                            // they commute; 0 none; -1 other
    uint32_t recv_mask;     // the receive edges, as bits of the edge list
    uint32_t recv_split;    // of two: the least draw that picks the higher one
    uint32_t recv_flags;    // SMC_RF_*
    uint32_t edge_first;    // edges [edge_first, edge_first + edge_n)
    uint16_t edge_n;
    uint8_t klass;
    uint8_t flags;          // SMC_LF_*
    uint32_t pick_mask;     // the spontaneous edges, and the sum of their weights, if these
    uint32_t pick_weight;   // are constants below 2^31 in all (else mask 0)
    uint32_t inv_first;     // clock upper-bound invariants
    uint32_t block_first;   // SMC_LF_GUARDED: the blocking test, guard records from here on
    uint32_t rate;          // expression reference
    uint16_t n_inv;
    uint8_t rate_const;
    uint8_t type;
    double rate_value;      // the rate when it is a constant (rate_const)
    uint64_t pad;
};

struct DevInv {             // x <= bound  (strict: x < bound), 16 bytes
    uint16_t var;
    uint8_t strict;
    uint8_t bound_const;    // bound is the constant bound_value
    uint32_t bound;         // expression reference
    double bound_value;
};

// DevEdge.flags
enum {
    SMC_EF_GOAL = 1,          // destination is a goal location
    SMC_EF_NEVER = 2,         // has a `!=` guard: never enabled (simulation.cu:249-251)
    SMC_EF_WEIGHT_CONST = 4,  // weight is the constant itself (0 if negative), else a reference
    SMC_EF_NO_GUARD = 8       // no guard in the record
};
// DevEdge.g_flags, u0_flags, u1_flags: low byte 8 if the variable counts from
// the component's base, else 0
enum { SMC_EG_CLOCK = 0x100, SMC_EU_ADD = 0x100, SMC_EU_SET = 0x200, SMC_EU_CLOCK = 0x400 };

// An edge, 80 bytes: with its first guard against a constant and its first
// two plain updates (add or set a constant), which is all that most edges
// have, so that firing one is a straight line of three dependent reads.
// Variables are byte offsets.
struct DevEdge {
    uint32_t dst_rec;       // record class of the destination
    uint32_t flags;         // SMC_EF_*
    uint32_t weight;
    int32_t channel;
    double lo, hi;          // the guard holds for values in [lo, hi]
    uint16_t g_var, g_flags;
    uint32_t guard_first;   // other guards
    uint16_t guard_n;
    uint16_t upd_n;         // other updates, after u0 and u1
    uint32_t upd_first;
    double u0_value;
    uint16_t u0_var, u0_flags;  // neither ADD nor SET: no update
    int32_t dst;            // destination relative to the source location
    double u1_value;
    uint16_t u1_var, u1_flags;
    uint32_t pad;
};

// DevGuard.flags
enum {
    SMC_GF_CLOCK_FREE = 1,  // neither var nor rhs reads a clock: fixed between transitions
    SMC_GF_CLOCK = 2,       // var is a clock
    SMC_GF_END_EDGE = 4,    // blocking test: last conjunct of its edge
    SMC_GF_END_LOC = 8,     // blocking test: last record of the location
    SMC_GF_RANGE = 16       // constant right side: holds for values in [lo, hi]
};

// A guard-blocked location's blocking test is a run of guard records (from
// DevLoc.block_first): the clock-free conjuncts of each spontaneous edge
// without `!=`, edge after edge.  The location is blocked when every edge
// has a false conjunct among them.

// variables[var] op rhs, 24 bytes.  With a constant right side every
// operator is the test of an interval of doubles (the tolerance of `==`
// included: the interval's ends are the last values that pass it).
struct DevGuard {
    double lo, hi;
    uint16_t var;
    uint8_t op;             // smc_cons_op, never SMC_C_NE
    uint8_t flags;          // SMC_GF_*
    uint32_t rhs;
};

// Update kinds: integer variable plus a constant, a constant, or anything
// else.  A commuting receive edge has only ADD updates of an integer constant
// and SET updates of a variable written by one component only (or by all
// with the same value), so the receivers of one broadcast can fire in any
// order with the same result.
enum { SMC_U_EXPR = 0, SMC_U_ADD = 1, SMC_U_SET = 2 };

struct DevUpd {             // 16 bytes
    uint16_t var;
    uint8_t kind;           // SMC_U_*
    uint8_t clock;          // var is a clock (stored as a reset stamp)
    uint32_t expr;
    double value;           // the added constant (ADD) or the value (SET)
};

// The tables live in device global memory.  Device code sees their pointers
// in the global address space, so reads compile to global loads (their own
// wait counter) rather than flat loads, which the compiler must also order
// against LDS traffic; host code sees plain pointers of the same size.
// Launch records that no kernel writes are read through the constant address
// space (scalar loads).  A run kernel may stage the tables in LDS and read them through a second
// instance of the same record (DevModelT<SmcLdsTables>).
#if defined(__HIP_DEVICE_COMPILE__)
#define SMC_GLOBAL __attribute__((address_space(1)))
#define SMC_LDS __attribute__((address_space(3)))
#define SMC_CONSTANT __attribute__((address_space(4)))
#else
#define SMC_GLOBAL
#define SMC_LDS
#define SMC_CONSTANT
#endif

struct SmcGlobalTables {
    template <class T> using ptr = const SMC_GLOBAL T *;
};
struct SmcLdsTables {
    template <class T> using ptr = const SMC_LDS T *;
};

// Everything the run kernel needs to know about one model; passed by value.
template <class A>
struct DevModelT {
    typename A::template ptr<DevHot> hots;     // [n_recs] record 0: no component
    typename A::template ptr<DevLoc> locs;     // [n_recs]
    typename A::template ptr<DevInv> invs;
    typename A::template ptr<DevEdge> edges;
    typename A::template ptr<DevGuard> guards;
    typename A::template ptr<DevUpd> upds;
    typename A::template ptr<double> consts;
    typename A::template ptr<DevInsn> code;
    const SMC_GLOBAL double *var_init;     // stored form at time 0: initial value, -initial value for a clock
    const SMC_GLOBAL uint32_t *comp_word;      // [n_comp] initial state word (class << rec_shift | base)
    const SMC_GLOBAL int32_t *comp_init_loc;   // [n_comp]
    const SMC_GLOBAL uint8_t *var_clock;   // [n_vars] 1: the variable is a clock
    const SMC_GLOBAL int32_t *comp_first_loc;  // [n_comp + 1] location range of each component
    const SMC_GLOBAL int32_t *loc_edge0;       // [n_locs] the network's index of each location's first edge
                                               // (edge records are shared: digests name network edges)
    const SMC_GLOBAL uint32_t *loc_rec;        // [n_locs] record class of each location
    int32_t n_comp;
    int32_t n_vars;
    int32_t n_leaves;           // next power of two >= n_comp
    int32_t n_locs;
    int32_t rec_shift;          // state word: class << rec_shift | base of the private variables
    uint32_t base_mask;         // (1 << rec_shift) - 1
    uint32_t tests;             // every SMC_HF_* flag some location has
    uint32_t one_rate;          // the one rate expression of the network (reading no private
                                // variable), or SMC_NO_REF
    int32_t freeze;             // no rate reads a clock: blocked components may leave the race
};
using DevModel = DevModelT<SmcGlobalTables>;
