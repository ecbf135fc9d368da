// compile.cpp — lowers an smc_network to the run kernel's tables.
//
// What the reference does at this point (shared_model_state.cu:164-689,
// pn_compile_visitor.cpp) and what is done here instead:
//   * expressions: cuSMC keeps guard right-hand sides as pointer trees and
//     compiles the rest to a Polish-notation array evaluated with a
//     10-double stack in local memory (expressions.cu:97-119).  Here every
//     expression becomes an inline constant, an inline variable or a short
//     three-address program over four registers (Sethi-Ullman order), with
//     identical programs and constants shared across components.
//   * invariants: only conjuncts that can bound a delay are kept — a clock
//     on the left, `<` or `<=` (simulation.cu:464-509); the kernel never
//     reads any other invariant.
//   * guards: only conjuncts on a variable are kept (simulation.cu:209); an
//     edge with a `!=` conjunct can never be enabled (simulation.cu:249-251)
//     and is flagged instead.
//   * locations get a delay class so the kernel does not re-derive it, and
//     what every race step reads of them is laid out apart (DevHot).
//   * comparisons with a constant become interval tests.
//   * locations with equal records share one record class: the instances of
//     a template differ only in their private variables, which are named
//     relative to the component (CSMA/CA with 100 processes: 1,800 locations,
//     28 classes, and tables of a few kilobytes that every kernel can keep in
//     LDS).
#include "compile.hpp"

#include <cstring>
#include <functional>
#include <map>
#include <stdexcept>
#include <algorithm>
#include <cmath>
#include <string>
#include <unordered_map>
#include "expr_ops.h"
#include "network.hpp"

namespace smc {

namespace {

class Lowerer {
public:
    // base: first private variable of each component (-1: none); owner: the
    // component a variable is private to (-1: none).  Without them variables
    // keep their own indices.
    Lowerer(const smc_network &n, ModelImage &img, const std::vector<int> *owner = nullptr,
            const std::vector<int> *base = nullptr)
        : n_(n), img_(img), owner_(owner), base_(base) {}

    // Later references belong to component c.
    void set_component(int c) { comp_ = c; }
    bool local(int v) const { return owner_ && (*owner_)[v] == comp_ && comp_ >= 0; }
    uint32_t index(int v) const { return (uint32_t)(local(v) ? v - (*base_)[comp_] : v); }
    // Variable operand of a record's 16-bit field.
    uint16_t field(int v) const { return (uint16_t)(index(v) | (local(v) ? SMC_VAR_LOCAL : 0u)); }

    uint32_t ref(int e, double dflt) {
        if (e < 0) return SMC_REF_MAKE(SMC_REF_CONST, const_index(dflt));
        const smc_expr_node &x = n_.exprs[e];
        if (x.op == SMC_E_LIT) return SMC_REF_MAKE(SMC_REF_CONST, const_index(x.value));
        if (x.op == SMC_E_RANDOM) return SMC_REF_MAKE(SMC_REF_CONST, const_index(1.0));
        if (x.op == SMC_E_VAR)
            return SMC_REF_MAKE(n_.var_kind[x.var] == SMC_VAR_CLOCK ? SMC_REF_CLOCK : SMC_REF_VAR,
                                index(x.var) | (local(x.var) ? SMC_REF_LOCAL : 0u));
        std::vector<DevInsn> prog;
        int maxreg = 0;
        uint16_t r = emit(e, 0, prog, &maxreg);
        if (r != SMC_OPND(SMC_OPND_REG, 0)) throw std::runtime_error("internal: expression result not in r0");
        if ((int)prog.size() > SMC_MAX_CODE_LEN)
            throw std::runtime_error("limit: expression needs more than 63 instructions");
        std::string key((const char *)prog.data(), prog.size() * sizeof(DevInsn));
        auto it = code_cache_.find(key);
        uint32_t first;
        if (it != code_cache_.end()) first = it->second;
        else {
            first = (uint32_t)img_.code.size();
            if (first + prog.size() >= (1u << 24)) throw std::runtime_error("limit: bytecode larger than 16M instructions");
            img_.code.insert(img_.code.end(), prog.begin(), prog.end());
            code_cache_[key] = first;
        }
        return SMC_REF_CODE_MAKE(first, prog.size());
    }

private:
    const smc_network &n_;
    ModelImage &img_;
    const std::vector<int> *owner_, *base_;
    int comp_ = -1;
    std::unordered_map<uint64_t, uint32_t> const_cache_;
    std::unordered_map<std::string, uint32_t> code_cache_;

    uint32_t const_index(double v) {
        uint64_t b;
        memcpy(&b, &v, 8);
        auto it = const_cache_.find(b);
        if (it != const_cache_.end()) return it->second;
        uint32_t i = (uint32_t)img_.consts.size();
        if (i > SMC_MAX_OPND_INDEX) throw std::runtime_error("limit: more than 16384 distinct constants");
        img_.consts.push_back(v);
        const_cache_[b] = i;
        return i;
    }

    int need(int e) const {
        const smc_expr_node &x = n_.exprs[e];
        if (x.op == SMC_E_LIT || x.op == SMC_E_VAR || x.op == SMC_E_RANDOM) return 0;
        int ar = smc_op_arity(x.op);
        const int kids[3] = {x.a, x.b, x.c};
        int nk[3] = {0, 0, 0};
        for (int i = 0; i < ar; ++i) nk[i] = need(kids[i]);
        // evaluate neediest first; each evaluated non-leaf child holds one register
        int order[3] = {0, 1, 2};
        for (int i = 0; i < ar; ++i)
            for (int j = i + 1; j < ar; ++j)
                if (nk[order[j]] > nk[order[i]]) std::swap(order[i], order[j]);
        int held = 0, peak = 1;
        for (int i = 0; i < ar; ++i) {
            int k = order[i];
            if (nk[k] > 0) { peak = std::max(peak, held + nk[k]); ++held; }
        }
        return std::max(peak, 1);
    }

    uint16_t emit(int e, int base, std::vector<DevInsn> &prog, int *maxreg) {
        const smc_expr_node &x = n_.exprs[e];
        if (x.op == SMC_E_LIT) return SMC_OPND(SMC_OPND_CONST, const_index(x.value));
        if (x.op == SMC_E_RANDOM) return SMC_OPND(SMC_OPND_CONST, const_index(1.0));
        if (x.op == SMC_E_VAR) {
            if (x.var > SMC_MAX_OPND_INDEX) throw std::runtime_error("limit: variable index above 16383 in an expression");
            return SMC_OPND(n_.var_kind[x.var] == SMC_VAR_CLOCK ? SMC_OPND_CLOCK : SMC_OPND_VAR,
                            index(x.var) | (local(x.var) ? SMC_OPND_LOCAL : 0u));
        }
        int ar = smc_op_arity(x.op);
        const int kids[3] = {x.a, x.b, x.c};
        int nk[3] = {0, 0, 0};
        for (int i = 0; i < ar; ++i) nk[i] = need(kids[i]);
        int order[3] = {0, 1, 2};
        for (int i = 0; i < ar; ++i)
            for (int j = i + 1; j < ar; ++j)
                if (nk[order[j]] > nk[order[i]]) std::swap(order[i], order[j]);
        uint16_t opnd[3] = {0, 0, 0};
        int r = base;
        for (int i = 0; i < ar; ++i) {
            int k = order[i];
            opnd[k] = emit(kids[k], r, prog, maxreg);
            if ((opnd[k] >> 14) == SMC_OPND_REG) ++r;
        }
        if (base >= SMC_NREGS) throw std::runtime_error("limit: expression needs more than 4 registers");
        *maxreg = std::max(*maxreg, base);
        DevInsn in{};
        in.op = (uint8_t)x.op;
        in.dst = (uint8_t)base;
        in.a = opnd[0]; in.b = opnd[1]; in.c = opnd[2];
        prog.push_back(in);
        return SMC_OPND(SMC_OPND_REG, (uint32_t)base);
    }
};

// The component each variable is private to (read and written by it alone),
// or -1, and each component's first private variable.
void private_variables(const smc_network &n, std::vector<int> &owner, std::vector<int> &base) {
    constexpr int kNone = -1, kShared = -2;
    owner.assign(n.n_vars, kNone);
    base.assign(n.n_components, 0);
    auto use = [&](int v, int c) { owner[v] = owner[v] == kNone || owner[v] == c ? c : kShared; };
    std::function<void(int, int)> use_expr = [&](int x, int c) {
        if (x < 0) return;
        const smc_expr_node &nd = n.exprs[x];
        if (nd.op == SMC_E_VAR) use(nd.var, c);
        const int kids[3] = {nd.a, nd.b, nd.c};
        for (int k = 0; k < smc_op_arity(nd.op); ++k) use_expr(kids[k], c);
    };
    auto use_constraint = [&](const smc_constraint &C, int c) {
        if (C.uses_variable) use(C.var, c);
        use_expr(C.rhs, c);
    };
    for (int c = 0; c < n.n_components; ++c)
        for (int l = n.comp_first_loc[c]; l < n.comp_first_loc[c + 1]; ++l) {
            const smc_location &L = n.locations[l];
            use_expr(L.rate, c);
            for (int k = 0; k < L.inv_count; ++k) use_constraint(n.constraints[L.inv_first + k], c);
            for (int k = 0; k < L.edge_count; ++k) {
                const smc_edge &E = n.edges[L.edge_first + k];
                use_expr(E.weight, c);
                for (int g = 0; g < E.guard_count; ++g) use_constraint(n.constraints[E.guard_first + g], c);
                for (int u = 0; u < E.upd_count; ++u) {
                    use(n.updates[E.upd_first + u].var, c);
                    use_expr(n.updates[E.upd_first + u].expr, c);
                }
            }
        }
    std::vector<uint8_t> seen(n.n_components, 0);
    for (int v = 0; v < n.n_vars; ++v) {
        if (owner[v] < 0) { owner[v] = -1; continue; }
        if (!seen[owner[v]]) { seen[owner[v]] = 1; base[owner[v]] = v; }
    }
}

// Doubles in the order of their values, as integers.
int64_t order_of(double x) {
    int64_t b;
    memcpy(&b, &x, 8);
    return b < 0 ? (int64_t)0x8000000000000000ull - b : b;
}
double double_of(int64_t o) {
    const int64_t b = o < 0 ? (int64_t)0x8000000000000000ull - o : o;
    double x;
    memcpy(&x, &b, 8);
    return x;
}

// The interval of values x for which `x op r` holds (empty: lo > hi).  For
// `==` the ends are the first and last x with |x - r| <= SMC_TOL in doubles:
// the rounded difference is monotonic in x, so they are found by bisection.
void range_of(int op, double r, double *lo, double *hi) {
    const double INF = HUGE_VAL;
    *lo = INF;
    *hi = -INF;
    if (r != r) return;
    switch (op) {
    case SMC_C_LE: *lo = -INF; *hi = r; return;
    case SMC_C_GE: *lo = r; *hi = INF; return;
    case SMC_C_LT: if (r > -INF) { *lo = -INF; *hi = std::nextafter(r, -INF); } return;
    case SMC_C_GT: if (r < INF) { *lo = std::nextafter(r, INF); *hi = INF; } return;
    case SMC_C_EQ: break;
    default: return;
    }
    if (std::fabs(r) == INF) return;
    auto end = [&](double outside) {
        int64_t in = order_of(r), out = order_of(outside);  // the test holds at `in`, fails at `out`
        // (the two may lie further apart than a signed difference holds)
        const auto apart = [&] { return in > out ? (uint64_t)in - (uint64_t)out : (uint64_t)out - (uint64_t)in; };
        while (apart() > 1) {
            const int64_t mid = in / 2 + out / 2 + (in % 2 + out % 2) / 2;
            if (std::fabs(double_of(mid) - r) <= SMC_TOL) in = mid;
            else out = mid;
        }
        return double_of(in);
    };
    *lo = end(-INF);
    *hi = end(INF);
}

// Index of the run of n records in `out`, stored once per content.
template <class T>
uint32_t intern(std::vector<T> &out, std::unordered_map<std::string, uint32_t> &map, const T *first, size_t n) {
    if (n == 0) return 0;
    std::string key((const char *)first, n * sizeof(T));
    auto it = map.find(key);
    if (it != map.end()) return it->second;
    const uint32_t at = (uint32_t)out.size();
    out.insert(out.end(), first, first + n);
    map.emplace(std::move(key), at);
    return at;
}

// One location before classes are formed.
struct RawEdge {
    DevEdge e{};
    int dst_loc = 0;
    std::vector<DevGuard> guards;
    std::vector<DevUpd> upds;
};
struct RawLoc {
    DevHot hot{};
    DevLoc loc{};
    std::vector<RawEdge> edges;
    std::vector<DevInv> invs;
    std::vector<DevGuard> block;
};

// A record's variable operand as a byte offset and its local factor.
void inline_var(uint16_t v, uint16_t *offset, uint16_t *flags) {
    *offset = (uint16_t)((v & ~SMC_VAR_LOCAL) * 8u);
    *flags = (uint16_t)(*flags | ((v & SMC_VAR_LOCAL) ? 8 : 0));
}

// Move an edge's first constant guard and its leading plain updates (at most
// two) into its record.
void inline_edge(RawEdge &re) {
    DevEdge &e = re.e;
    e.flags |= SMC_EF_NO_GUARD;
    for (size_t k = 0; k < re.guards.size(); ++k) {
        const DevGuard G = re.guards[k];
        if (!(G.flags & SMC_GF_RANGE)) continue;
        e.flags &= ~(uint32_t)SMC_EF_NO_GUARD;
        e.lo = G.lo;
        e.hi = G.hi;
        if (G.flags & SMC_GF_CLOCK) e.g_flags |= SMC_EG_CLOCK;
        inline_var(G.var, &e.g_var, &e.g_flags);
        re.guards.erase(re.guards.begin() + k);
        break;
    }
    size_t u = 0;
    for (; u < 2 && u < re.upds.size() && re.upds[u].kind != SMC_U_EXPR; ++u) {
        const DevUpd &U = re.upds[u];
        uint16_t &var = u ? e.u1_var : e.u0_var, &flags = u ? e.u1_flags : e.u0_flags;
        (u ? e.u1_value : e.u0_value) = U.value;
        flags |= (uint16_t)((U.kind == SMC_U_ADD ? SMC_EU_ADD : SMC_EU_SET) | (U.clock ? SMC_EU_CLOCK : 0));
        inline_var(U.var, &var, &flags);
    }
    re.upds.erase(re.upds.begin(), re.upds.begin() + u);
    e.guard_n = (uint16_t)re.guards.size();
    e.upd_n = (uint16_t)re.upds.size();
}

// Partition of the locations into classes of equal records: first by their
// own content, then, until nothing splits, by the classes their edges lead
// to.  The model fixtures are stable after one to three passes; a chain of equal
// locations separates by one link a pass.  Where 64 passes do not do, the
// locations at the same place of equal components are a class: instances of a
// template still share their records.
std::vector<uint32_t> classes_of(const smc_network &net, const std::vector<RawLoc> &raw, uint32_t *count) {
    const size_t n = raw.size();
    std::vector<uint32_t> cls(n), next(n);
    auto put = [](std::string &k, const auto &v) {
        const uint32_t c = (uint32_t)v.size();
        k.append((const char *)&c, 4);
        if (c) k.append((const char *)v.data(), c * sizeof(v[0]));
    };
    std::unordered_map<std::string, uint32_t> ids;
    for (size_t l = 0; l < n; ++l) {
        std::string k((const char *)&raw[l].hot, sizeof(DevHot));
        k.append((const char *)&raw[l].loc, sizeof(DevLoc));
        put(k, raw[l].invs);
        put(k, raw[l].block);
        for (const RawEdge &e : raw[l].edges) {
            k.append((const char *)&e.e, sizeof(DevEdge));
            put(k, e.guards);
            put(k, e.upds);
        }
        cls[l] = ids.emplace(std::move(k), (uint32_t)ids.size()).first->second;
    }
    *count = (uint32_t)ids.size();
    const std::vector<uint32_t> own = cls;  // by their own content, destinations relative to the location
    for (int pass = 0; pass < 64; ++pass) {
        ids.clear();
        for (size_t l = 0; l < n; ++l) {
            std::string k((const char *)&cls[l], 4);
            for (const RawEdge &e : raw[l].edges) k.append((const char *)&cls[e.dst_loc], 4);
            next[l] = ids.emplace(std::move(k), (uint32_t)ids.size()).first->second;
        }
        cls.swap(next);
        if (ids.size() == *count) return cls;
        *count = (uint32_t)ids.size();
    }
    ids.clear();
    *count = 0;
    for (int c = 0; c < net.n_components; ++c) {
        const int l0 = net.comp_first_loc[c], locs = net.comp_first_loc[c + 1] - l0;
        std::string k((const char *)&own[l0], (size_t)locs * 4);
        const auto at = ids.emplace(std::move(k), *count);  // the component's first class
        if (at.second) *count += (uint32_t)locs;
        for (int l = 0; l < locs; ++l) cls[l0 + l] = at.first->second + (uint32_t)l;
    }
    return cls;
}

// use_locals: private variables named relative to their component.
ModelImage lower(const smc_network &n, bool use_locals) {
    ModelImage img;
    img.n_comp = n.n_components;
    img.n_vars = n.n_vars;
    int leaves = 1;
    while (leaves < n.n_components) leaves <<= 1;
    img.n_leaves = leaves;

    img.var_init.assign(n.var_init, n.var_init + n.n_vars);
    img.var_kind.assign(n.var_kind, n.var_kind + n.n_vars);
    for (int v = 0; v < n.n_vars; ++v) img.var_clock.push_back(n.var_kind[v] == SMC_VAR_CLOCK ? 1 : 0);
    img.comp_init_loc.assign(n.comp_init_loc, n.comp_init_loc + n.n_components);
    img.comp_first_loc.assign(n.comp_first_loc, n.comp_first_loc + n.n_components + 1);

    std::vector<int> owner, base;
    private_variables(n, owner, base);
    if (!use_locals) std::fill(base.begin(), base.end(), 0);
    Lowerer lw(n, img, use_locals ? &owner : nullptr, use_locals ? &base : nullptr);
    // expression identities across components (rates, for tilt groups)
    ModelImage plain;
    Lowerer lw_plain(n, plain);

    std::vector<int8_t> clock_memo(n.n_exprs, -1);
    std::function<bool(int)> reads_clock = [&](int x) -> bool {
        if (x < 0) return false;
        if (clock_memo[x] >= 0) return clock_memo[x] != 0;
        const smc_expr_node &nd = n.exprs[x];
        bool r = nd.op == SMC_E_VAR && n.var_kind[nd.var] == SMC_VAR_CLOCK;
        if (!r && nd.op != SMC_E_LIT && nd.op != SMC_E_VAR)
            r = reads_clock(nd.a) || reads_clock(nd.b) || reads_clock(nd.c);
        clock_memo[x] = r ? 1 : 0;
        return r;
    };
    std::function<bool(int)> reads_local = [&](int x) -> bool {
        if (x < 0) return false;
        const smc_expr_node &nd = n.exprs[x];
        if (nd.op == SMC_E_VAR) return lw.local(nd.var);
        const int kids[3] = {nd.a, nd.b, nd.c};
        for (int k = 0; k < smc_op_arity(nd.op); ++k)
            if (reads_local(kids[k])) return true;
        return false;
    };
    auto literal = [&](int x, double *v) {
        if (x < 0 || n.exprs[x].op != SMC_E_LIT) return false;
        *v = n.exprs[x].value;
        return true;
    };
    auto is_var = [&](int x, int var) { return x >= 0 && n.exprs[x].op == SMC_E_VAR && n.exprs[x].var == var; };

    // Forms of an update: ADD (integer variable += constant), SET (:= a
    // constant).  Subtracting a constant is adding its negative, exactly.
    auto form = [&](const smc_update &U, double *c) -> int {
        const smc_expr_node *x = U.expr >= 0 ? &n.exprs[U.expr] : nullptr;
        if (!x) return SMC_U_EXPR;
        if (n.var_kind[U.var] == SMC_VAR_INT &&
            ((x->op == SMC_E_ADD && is_var(x->a, U.var) && literal(x->b, c)) ||
             (x->op == SMC_E_ADD && literal(x->a, c) && is_var(x->b, U.var)) ||
             (x->op == SMC_E_SUB && is_var(x->a, U.var) && literal(x->b, c) && ((*c = -*c), true))))
            return SMC_U_ADD;
        if (literal(U.expr, c)) return SMC_U_SET;
        return SMC_U_EXPR;
    };
    auto whole = [](double c) { return c == std::floor(c) && std::fabs(c) < 2147483648.0; };
    // Receive edges whose updates commute within one broadcast: additions
    // are of integer constants, and per variable over all receive edges all
    // are ADD, or all SET of one value, or it is written by a single
    // component — then the writes of one broadcast's receivers give the same
    // result in any order.
    struct VarUse { int add = 0, set = 0, other = 0, writer = -1; bool one_value = true; double value = 0.0; };
    std::vector<VarUse> use(n.n_vars);
    for (int c = 0; c < n.n_components; ++c)
        for (int l = n.comp_first_loc[c]; l < n.comp_first_loc[c + 1]; ++l)
            for (int k = 0; k < n.locations[l].edge_count; ++k) {
                const smc_edge &E = n.edges[n.locations[l].edge_first + k];
                if (E.channel >= 0) continue;
                for (int u = 0; u < E.upd_count; ++u) {
                    const smc_update &U = n.updates[E.upd_first + u];
                    VarUse &vu = use[U.var];
                    double cv = 0.0;
                    const int f = form(U, &cv);
                    if (f == SMC_U_ADD && whole(cv)) ++vu.add;
                    else if (f == SMC_U_SET) {
                        if (vu.set && cv != vu.value) vu.one_value = false;
                        vu.value = cv;
                        ++vu.set;
                    } else ++vu.other;
                    vu.writer = (vu.writer == -1 || vu.writer == c) ? c : -2;
                }
            }
    auto var_commutes = [&](int v) {
        const VarUse &vu = use[v];
        if (vu.other) return false;
        if (vu.writer >= 0) return true;
        return vu.set == 0 || (vu.add == 0 && vu.one_value);
    };

    // Clocks set to values far inside the doubles: a window under such a bound
    // is finite.  `most` bounds what a variable that is no clock holds; what a
    // run adds up, at most 1e20 terms, counts with the term.
    auto moderate = [](double v) { return std::fabs(v) <= 1e300; };
    std::vector<double> most(n.n_vars);
    std::function<double(int)> reach = [&](int x) -> double {
        if (x < 0) return HUGE_VAL;
        const smc_expr_node &e = n.exprs[x];
        double v = HUGE_VAL;
        switch (e.op) {
        case SMC_E_LIT: v = std::fabs(e.value); break;
        case SMC_E_VAR: v = n.var_kind[e.var] == SMC_VAR_CLOCK ? HUGE_VAL : most[e.var]; break;
        case SMC_E_ADD: case SMC_E_SUB: v = reach(e.a) + reach(e.b); break;
        case SMC_E_MUL: v = reach(e.a) * reach(e.b); break;
        case SMC_E_NEG: v = reach(e.a); break;
        case SMC_E_COND: v = std::max(reach(e.b), reach(e.c)); break;
        case SMC_E_RANDOM: case SMC_E_NOT: case SMC_E_AND: case SMC_E_OR: case SMC_E_LE: case SMC_E_GE:
        case SMC_E_LT: case SMC_E_GT: case SMC_E_EQ: case SMC_E_NE: v = 1.0; break;
        default: break;
        }
        return moderate(v) ? v : HUGE_VAL;
    };
    for (int v = 0; v < n.n_vars; ++v) most[v] = std::fabs(n.var_init[v]);
    bool grows = false;  // (needed for clocks set to expressions only)
    for (int u = 0; u < n.n_updates; ++u) {
        double c;
        grows |= n.var_kind[n.updates[u].var] == SMC_VAR_CLOCK && !literal(n.updates[u].expr, &c);
    }
    for (int round = 0; grows; ++round) {
        std::vector<double> set(n.n_vars), sum(n.n_vars, 0.0);
        for (int v = 0; v < n.n_vars; ++v) set[v] = std::fabs(n.var_init[v]);
        for (int u = 0; u < n.n_updates; ++u) {
            const int v = n.updates[u].var, x = n.updates[u].expr;
            const smc_expr_node *e = x >= 0 ? &n.exprs[x] : nullptr;
            if (n.var_kind[v] == SMC_VAR_CLOCK) continue;
            if (e && (e->op == SMC_E_ADD || e->op == SMC_E_SUB) && is_var(e->a, v)) sum[v] = std::max(sum[v], reach(e->b));
            else if (e && e->op == SMC_E_ADD && is_var(e->b, v)) sum[v] = std::max(sum[v], reach(e->a));
            else set[v] = std::max(set[v], reach(x));
        }
        grows = false;
        for (int v = 0; v < n.n_vars; ++v) {
            const double now = set[v] + 1e20 * sum[v];
            if (!(now > most[v])) continue;
            most[v] = round < 8 ? now : HUGE_VAL;
            grows = true;
        }
        // (a long chain of variables: one link a round)
        if (round < 64) continue;
        for (int u = 0; u < n.n_updates; ++u) {
            double c;
            if (!literal(n.updates[u].expr, &c)) most[n.updates[u].var] = HUGE_VAL;
        }
        break;
    }
    std::vector<uint8_t> clock_moderate(n.n_vars);
    for (int v = 0; v < n.n_vars; ++v) clock_moderate[v] = moderate(n.var_init[v]);
    for (int u = 0; u < n.n_updates; ++u)
        if (!moderate(reach(n.updates[u].expr))) clock_moderate[n.updates[u].var] = 0;

    // Null racers leave an all-exponential race only while every rate is
    // constant between transitions (a rate reading a clock changes at each
    // null step of the reference's race).
    bool clock_rate = false;
    for (int l = 0; l < n.n_locations; ++l)
        if (reads_clock(n.locations[l].rate)) clock_rate = true;
    img.freeze = !clock_rate;

    int n_rates = 0;  // distinct rate expressions (2: several, or one that reads private variables)
    std::vector<RawLoc> raw(n.n_locations);
    img.info.resize(n.n_locations);
    img.loc_edge0.assign(n.n_locations, 0);
    for (int comp = 0; comp < n.n_components; ++comp) {
        lw.set_component(comp);
        for (int l = n.comp_first_loc[comp]; l < n.comp_first_loc[comp + 1]; ++l) {
            const smc_location &L = n.locations[l];
            RawLoc &R = raw[l];
            DevLoc &d = R.loc;
            LocInfo &info = img.info[l];
            d.type = (uint8_t)L.type;
            d.rate = lw.ref(L.rate, 1.0);
            int inv_clock = -1;
            for (int k = 0; k < L.inv_count; ++k) {
                const smc_constraint &C = n.constraints[L.inv_first + k];
                if (!C.uses_variable) continue;
                if (n.var_kind[C.var] != SMC_VAR_CLOCK) continue;
                if (C.op != SMC_C_LE && C.op != SMC_C_LT) continue;
                DevInv iv{};
                iv.var = lw.field(C.var);
                inv_clock = C.var;
                iv.strict = C.op == SMC_C_LT;
                iv.bound = lw.ref(C.rhs, 0.0);
                if (SMC_REF_KIND(iv.bound) == SMC_REF_CONST) {
                    iv.bound_const = 1;
                    iv.bound_value = img.consts[iv.bound & 0x3FFFFFFFu];
                }
                R.invs.push_back(iv);
            }
            if (R.invs.size() > 65535) throw std::runtime_error("limit: more than 65535 invariants on a location");
            d.n_inv = (uint16_t)R.invs.size();
            d.klass = L.type > SMC_LOC_GOAL ? SMC_K_ZERO : (d.n_inv > 0 ? SMC_K_BOUNDED : SMC_K_EXP);
            if (L.edge_count > SMC_MAX_EDGES_PER_LOC)
                throw std::runtime_error("limit: a location has more than 64 outgoing edges");
            d.edge_n = (uint16_t)L.edge_count;
            img.loc_edge0[l] = L.edge_first;
            if (SMC_REF_KIND(d.rate) == SMC_REF_CONST) {
                d.rate_const = 1;
                d.rate_value = img.consts[d.rate & 0x3FFFFFFFu];
            }
            info.klass = d.klass;
            info.type = d.type;
            info.n_inv = d.n_inv;
            const uint32_t rate_plain = lw_plain.ref(L.rate, 1.0);
            if (d.rate_const) memcpy(&info.rate_key, &d.rate_value, 8);
            else info.rate_key = (int64_t)rate_plain ^ ((int64_t)1 << 62);

            for (int k = 0; k < L.edge_count; ++k) {
                const smc_edge &E = n.edges[L.edge_first + k];
                RawEdge re;
                DevEdge &e = re.e;
                e.dst = E.dst - l;
                re.dst_loc = E.dst;
                e.channel = E.channel;
                info.edges.push_back({e.dst, e.channel});
                e.weight = lw.ref(E.weight, 1.0);
                if (SMC_REF_KIND(e.weight) == SMC_REF_CONST) {
                    const int w = smc_to_int(img.consts[e.weight & 0x3FFFFFFFu]);
                    e.weight = w > 0 ? (uint32_t)w : 0u;
                    e.flags |= SMC_EF_WEIGHT_CONST;
                }
                if (n.locations[E.dst].type == SMC_LOC_GOAL) e.flags |= SMC_EF_GOAL;
                for (int g = 0; g < E.guard_count; ++g) {
                    const smc_constraint &C = n.constraints[E.guard_first + g];
                    if (!C.uses_variable) continue;
                    if (C.op == SMC_C_NE) { e.flags |= SMC_EF_NEVER; continue; }
                    if (C.var > 65535) throw std::runtime_error("limit: guarded variable index above 65535");
                    DevGuard G{};
                    G.var = lw.field(C.var);
                    G.op = (uint8_t)C.op;
                    G.flags = (uint8_t)((n.var_kind[C.var] != SMC_VAR_CLOCK && !reads_clock(C.rhs) ? SMC_GF_CLOCK_FREE : 0) |
                                        (n.var_kind[C.var] == SMC_VAR_CLOCK ? SMC_GF_CLOCK : 0));
                    G.rhs = lw.ref(C.rhs, 0.0);
                    if (SMC_REF_KIND(G.rhs) == SMC_REF_CONST) {
                        G.flags |= SMC_GF_RANGE;
                        range_of(C.op, img.consts[G.rhs & 0x3FFFFFFFu], &G.lo, &G.hi);
                    }
                    re.guards.push_back(G);
                }
                if (re.guards.size() > 65535) throw std::runtime_error("limit: more than 65535 guards on an edge");
                for (int k2 = 0; k2 < E.upd_count; ++k2) {
                    const smc_update &U = n.updates[E.upd_first + k2];
                    if (U.var > 65535) throw std::runtime_error("limit: assigned variable index above 65535");
                    DevUpd u{};
                    u.var = lw.field(U.var);
                    u.clock = n.var_kind[U.var] == SMC_VAR_CLOCK ? 1 : 0;
                    u.expr = lw.ref(U.expr, 0.0);
                    double cv = 0.0;
                    u.kind = (uint8_t)form(U, &cv);
                    if (u.kind != SMC_U_EXPR) u.value = cv;
                    re.upds.push_back(u);
                }
                if (E.upd_count > 65535) throw std::runtime_error("limit: more than 65535 updates on an edge");
                R.edges.push_back(std::move(re));
            }

            // time_free: the location's rate and its spontaneous edges'
            // guards read no clock, so between transitions neither its
            // enabled edges nor its rate change
            bool tf = !reads_clock(L.rate);
            for (int k = 0; k < L.edge_count && tf; ++k) {
                const smc_edge &E = n.edges[L.edge_first + k];
                if (E.channel < 0) continue;
                for (int g = 0; g < E.guard_count; ++g) {
                    const smc_constraint &G = n.constraints[E.guard_first + g];
                    if (!G.uses_variable) continue;
                    if (n.var_kind[G.var] == SMC_VAR_CLOCK || reads_clock(G.rhs)) tf = false;
                }
            }
            // blocking: always (every spontaneous edge has `!=`, or none),
            // by the variables (every other spontaneous edge has a
            // clock-free conjunct that may be false), or never
            int kind = 1;
            for (int k = 0; k < L.edge_count && kind != 0; ++k) {
                const smc_edge &E = n.edges[L.edge_first + k];
                if (E.channel < 0) continue;
                bool never = false, clock_free = false;
                for (int g = 0; g < E.guard_count; ++g) {
                    const smc_constraint &G = n.constraints[E.guard_first + g];
                    if (!G.uses_variable) continue;
                    if (G.op == SMC_C_NE) never = true;
                    else if (n.var_kind[G.var] != SMC_VAR_CLOCK && !reads_clock(G.rhs)) clock_free = true;
                }
                if (never) continue;
                kind = clock_free ? 2 : 0;
            }
            d.flags = (uint8_t)((tf ? SMC_LF_TIME_FREE : 0) | (kind == 1 ? SMC_LF_DEAD : 0) |
                                (kind == 2 ? SMC_LF_GUARDED : 0));
            if (kind == 2) {
                // the blocking test: clock-free conjuncts, edge after edge
                for (const RawEdge &re : R.edges) {
                    if (re.e.channel < 0 || (re.e.flags & SMC_EF_NEVER)) continue;
                    const size_t first = R.block.size();
                    for (const DevGuard &G : re.guards)
                        if (G.flags & SMC_GF_CLOCK_FREE) R.block.push_back(G);
                    if (R.block.size() == first)
                        throw std::runtime_error("internal: guarded edge without a clock-free conjunct");
                    R.block.back().flags |= SMC_GF_END_EDGE;
                }
                R.block.back().flags |= SMC_GF_END_LOC;
            }

            // receive edges
            bool fast = true, plain_recv = true;
            int chan = 0, n_recv = 0;
            int64_t weight = 0, low = 0;
            bool idle[2] = {true, true};
            for (int k = 0; k < L.edge_count; ++k) {
                const smc_edge &E = n.edges[L.edge_first + k];
                if (E.channel >= 0) continue;
                const RawEdge &re = R.edges[k];
                std::vector<int> seen;
                if (!(re.e.flags & SMC_EF_WEIGHT_CONST)) fast = false;
                else weight += re.e.weight;
                for (int k2 = 0; k2 < E.upd_count; ++k2) {
                    const smc_update &U = n.updates[E.upd_first + k2];
                    const DevUpd &u = re.upds[k2];
                    if (u.kind == SMC_U_EXPR || (u.kind == SMC_U_ADD && !whole(u.value)) || !var_commutes(U.var) ||
                        std::find(seen.begin(), seen.end(), U.var) != seen.end())
                        fast = false;
                    seen.push_back(U.var);
                }
                if (k >= 32) fast = false;
                if ((re.e.flags & SMC_EF_NEVER) || !re.guards.empty() || (chan && chan != -E.channel)) plain_recv = false;
                chan = -E.channel;
                if (k < 32) d.recv_mask |= 1u << k;
                idle[n_recv != 0] = re.e.dst == 0 && E.upd_count == 0 && !(re.e.flags & SMC_EF_GOAL);
                if (n_recv++ == 0) low = re.e.weight;
            }
            if (fast) d.flags |= SMC_LF_RECV_FAST;
            if (n_recv == 0) d.recv_chan = 0;
            else if (fast && plain_recv) {
                d.recv_chan = chan;
                d.recv_flags = (n_recv == 2 ? SMC_RF_TWO : n_recv > 2 ? SMC_RF_MORE : 0u) |
                               (idle[0] ? SMC_RF_LOW_IDLE : 0u) | (idle[1] ? SMC_RF_HIGH_IDLE : 0u);
                if (n_recv == 2) {
                    // the higher edge is picked unless the draw, of the sum of
                    // the weights, falls below the lower one's: monotone in
                    // the draw's 32 bits, and true of the largest
                    uint32_t from = 0, to = 0xFFFFFFFFu;
                    while (from < to) {
                        const uint32_t mid = from + (to - from) / 2;
                        if (low <= (int64_t)((double)weight * smc_u01_32(mid))) to = mid;
                        else from = mid + 1;
                    }
                    d.recv_split = to;
                }
            } else {
                d.recv_chan = -1;
                d.recv_mask = 0;
                img.recv_tested = std::max(img.recv_tested, L.edge_count);
            }

            // spontaneous edges with constant weights
            int64_t pick_sum = 0;
            bool pick = true;
            for (int k = 0; k < L.edge_count; ++k) {
                const RawEdge &re = R.edges[k];
                if (re.e.channel < 0) continue;
                if (k >= 32 || !(re.e.flags & SMC_EF_WEIGHT_CONST)) { pick = false; break; }
                d.pick_mask |= 1u << k;
                pick_sum += re.e.weight;
            }
            if (!pick || pick_sum >= 2147483648ll) d.pick_mask = 0;
            if (d.pick_mask) d.pick_weight = (uint32_t)pick_sum;

            // what a race step looks at
            DevHot &h = R.hot;
            uint32_t hf = 0;
            uint16_t hot_at = (uint16_t)(n.n_vars * 8u), hot_local = 0;  // the constant 0
            h.a = -HUGE_VAL;
            h.b = HUGE_VAL;
            if (d.klass == SMC_K_ZERO) {
                h.rate = -0.0;
            } else {
                if (img.freeze && kind == 1) {
                    hf |= SMC_HF_DEAD;
                } else if (d.rate_const) {
                    h.rate = d.rate_value > 0.0 ? d.rate_value : 0.0;
                } else {
                    const bool own = reads_local(L.rate);
                    hf |= SMC_HF_EXPR | (own ? SMC_HF_EXPR_LOCAL : 0);
                    if (own || (n_rates && img.one_rate != d.rate)) n_rates = 2;
                    else n_rates = std::max(n_rates, 1);
                    img.one_rate = d.rate;
                }
                if (d.n_inv == 1 && R.invs[0].bound_const) {
                    hf |= SMC_HF_INV;
                    inline_var(R.invs[0].var, &hot_at, &hot_local);
                    h.a = R.invs[0].bound_value;
                    h.b = R.invs[0].strict ? 1e-6 : 0.0;
                    if (!moderate(h.a) || !clock_moderate[inv_clock]) hf |= SMC_HF_WINDOW;
                } else if (d.n_inv) {
                    hf |= SMC_HF_XINV | SMC_HF_WINDOW;
                }
                if (img.freeze && kind == 2) {
                    if (R.block.size() == 1 && (R.block[0].flags & SMC_GF_RANGE) && !(hf & SMC_HF_INV)) {
                        hf |= SMC_HF_GUARD;
                        inline_var(R.block[0].var, &hot_at, &hot_local);
                        h.a = R.block[0].lo;
                        h.b = R.block[0].hi;
                    } else {
                        hf |= SMC_HF_XBLK;
                    }
                }
            }
            h.what = (uint32_t)hot_at | (hf << 16);
            h.base = (hot_local ? 0x1FFFu : 0u) | (hf & SMC_HF_EXPR ? SMC_HB_EXPR : 0u);
            for (RawEdge &re : R.edges) inline_edge(re);
            img.tests |= hf;
        }
    }

    if (n_rates != 1) img.one_rate = SMC_NO_REF;

    // classes of equal locations, and their records; record 0 is a slot
    // without a component (no edge, rate 0)
    uint32_t n_cls = 0;
    const std::vector<uint32_t> cls = classes_of(n, raw, &n_cls);
    // a state word holds the class and the base; with more classes than fit
    // beside a base, the class alone
    if (use_locals && n_cls >= (1u << 18)) return lower(n, false);
    img.rec_shift = use_locals ? 13 : 0;
    img.hots.assign(n_cls + 1, DevHot{});
    img.hots[0].a = -HUGE_VAL;
    img.hots[0].b = HUGE_VAL;
    img.hots[0].what = (uint16_t)(n.n_vars * 8u);
    img.locs.assign(n_cls + 1, DevLoc{});
    std::vector<uint8_t> done(n_cls, 0);
    std::unordered_map<std::string, uint32_t> gmap, umap, emap, imap;
    for (int l = 0; l < n.n_locations; ++l) {
        img.loc_rec.push_back(cls[l] + 1);
        if (done[cls[l]]) continue;
        done[cls[l]] = 1;
        RawLoc &R = raw[l];
        std::vector<DevEdge> run;
        for (RawEdge &re : R.edges) {
            re.e.guard_first = intern(img.guards, gmap, re.guards.data(), re.guards.size());
            re.e.upd_first = intern(img.upds, umap, re.upds.data(), re.upds.size());
            re.e.dst_rec = cls[re.dst_loc] + 1;
            run.push_back(re.e);
        }
        R.loc.edge_first = intern(img.edges, emap, run.data(), run.size());
        R.loc.inv_first = intern(img.invs, imap, R.invs.data(), R.invs.size());
        R.loc.block_first = intern(img.guards, gmap, R.block.data(), R.block.size());
        img.hots[cls[l] + 1] = R.hot;
        img.locs[cls[l] + 1] = R.loc;
    }
    for (int c = 0; c < n.n_components; ++c)
        img.comp_word.push_back((img.loc_rec[n.comp_init_loc[c]] << img.rec_shift) | (uint32_t)base[c]);
    // keep every table non-empty so device pointers are valid
    if (img.invs.empty()) img.invs.push_back(DevInv{});
    if (img.edges.empty()) img.edges.push_back(DevEdge{});
    if (img.guards.empty()) img.guards.push_back(DevGuard{});
    if (img.upds.empty()) img.upds.push_back(DevUpd{});
    if (img.consts.empty()) img.consts.push_back(0.0);
    if (img.code.empty()) img.code.push_back(DevInsn{});
    if (img.var_init.empty()) img.var_init.push_back(0.0);
    if (img.var_clock.empty()) img.var_clock.push_back(0);
    return img;
}

}  // namespace

ModelImage compile_model(const smc_network &n) {
    std::string err = validate(n);
    if (!err.empty()) throw std::runtime_error(err);
    // networks of SMC_MAX_LOCAL_VARS variables or more exceed the run
    // kernel's LDS budget at every launch shape; they keep plain indices
    return lower(n, n.n_vars < SMC_MAX_LOCAL_VARS);
}

}  // namespace smc
