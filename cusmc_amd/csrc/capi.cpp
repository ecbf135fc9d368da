// capi.cpp — the C ABI (include/smc_capi.h).
#include "smc_capi.h"

#include <hip/hip_runtime.h>

#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <filesystem>
#include <map>
#include <memory>
#include <stdexcept>
#include <string>
#include <unordered_set>
#include <tuple>
#include <vector>

#include "capi_internal.hpp"
#include "noalloc.hpp"
#include "uppaal.hpp"

namespace smc::capi {
thread_local std::string g_last_error;
}  // namespace smc::capi
using namespace smc::capi;

struct smc_parsed {
    std::unique_ptr<smc::Parsed> p;
    smc_network view{};
};

namespace {

// Launch shape for one group of instances.
struct Plan {
    int S = 1, C = 1, R = 64, stride = 1;
    int occ = 0;  // run-kernel build: 0 registers unrestricted, 3 three waves per SIMD
    bool tab = false;     // tables staged in LDS
    int group_waves = 1;  // waves per workgroup
    uint32_t table_bytes = 0, wave_lds = 0;
    size_t lds = 0;
    int waves = 1, per_cu = 1;
    int64_t resident = 1;  // waves that run side by side
    uint32_t chunk_runs = 1;
    int segments = 64;  // segments of a wave that take runs
};

constexpr size_t kLdsStatic = 64;  // the run kernel's own

int tree_levels(int S) {
    int levels = 0;
    while ((1 << levels) < S) ++levels;
    return levels;
}

// LDS of one wave (sim_body.h): variables of its R runs, state words and,
// with digests, locations.
size_t wave_lds_bytes(int R, int stride, int C, bool trace) {
    return ((size_t)R * stride * 8 + (size_t)C * 256 * (trace ? 2 : 1) + 15) & ~(size_t)15;
}

// The most variables a packing may hold: those of the packed runs, a clock
// time each and two doubles per lane and race-tree level, in 60,000 bytes.
bool vars_fit(int R, int n_vars, int levels) {
    return (size_t)R * ((n_vars + 1) | 1) * 8 + (size_t)levels * 1024 <= 60000;
}

// What a launch that names table staging is held to where the tables do not
// fit: with a record per location, 48 bytes each, and edges, guards and updates in
// their shortest form, 32, 8 and 16 bytes, equal runs of them shared (also by
// edges that only lead to different classes), they have to fit beside four
// waves.  Such tables were always accepted, though they may take several times
// as much; they are read from global memory then.
size_t named_tables_bytes(const smc_model *m, bool locations) {
    const smc::ModelImage &im = m->img;
    std::unordered_set<std::string> seen;
    const auto fresh = [&](char kind, const void *p, size_t n) {
        return seen.insert(kind + std::string((const char *)p, n)).second;
    };
    size_t edges = 0, guards = 0, upds = 0;
    for (const DevLoc &L : im.locs) {
        std::vector<DevEdge> run(im.edges.begin() + L.edge_first, im.edges.begin() + L.edge_first + L.edge_n);
        for (DevEdge &e : run) {
            e.dst_rec = 0;
            DevEdge g{}, u{};  // its guards, and its updates
            g.lo = e.lo, g.hi = e.hi, g.g_var = e.g_var, g.g_flags = e.g_flags;
            g.guard_first = e.guard_first, g.guard_n = e.guard_n, g.flags = e.flags & SMC_EF_NO_GUARD;
            u.u0_value = e.u0_value, u.u0_var = e.u0_var, u.u0_flags = e.u0_flags;
            u.u1_value = e.u1_value, u.u1_var = e.u1_var, u.u1_flags = e.u1_flags;
            u.upd_first = e.upd_first, u.upd_n = e.upd_n;
            if (fresh('g', &g, sizeof g)) guards += e.guard_n + ((e.flags & SMC_EF_NO_GUARD) ? 0 : 1);
            if (fresh('u', &u, sizeof u)) upds += e.upd_n + (e.u0_flags >= SMC_EU_ADD) + (e.u1_flags >= SMC_EU_ADD);
        }
        if (fresh('e', run.data(), run.size() * sizeof(DevEdge))) edges += run.size();
        if ((L.flags & SMC_LF_GUARDED) && fresh('b', &L.block_first, sizeof L.block_first)) {
            size_t k = L.block_first;
            while (!(im.guards[k].flags & SMC_GF_END_LOC)) ++k;
            guards += k + 1 - L.block_first;
        }
    }
    size_t total = 0;
    for (size_t part : {locations ? im.loc_rec.size() * 48 : 0, im.invs.size() * 16, edges * 32, guards * 8, upds * 16,
                        im.consts.size() * 8, im.code.size() * 8})
        total += align_up(part, 256);
    return total;
}

// Waves per CU that the registers of a run-kernel build allow (a property of
// the built code, asked for once per build).
int register_waves(int C, bool trace, int occ, bool tab) {
    static std::atomic<int> known[5][2][2][2];
    int c = 0;
    while ((1 << c) < C) ++c;
    std::atomic<int> &k = known[c][trace][occ == 3][tab];
    int v = k.load(std::memory_order_relaxed);
    if (!v) {
        int blocks = 0;
        hip_check(smc::sim_occupancy(C, trace, occ, tab, 1, 0, &blocks), "occupancy query");
        v = std::max(1, blocks);
        k.store(v, std::memory_order_relaxed);
    }
    return v;
}

// The launch of a call that asks for none on a model without a tuned one:
// the fewest lanes per run at which two waves per SIMD have their runs and
// their LDS, tables staged, and three waves per SIMD where sixteen slots a
// lane leave registers for two and there are runs for more.  A step costs a wave
// much the same whether it advances one run or many, so many runs are packed; few
// runs are spread, for the shortest steps.  Against the widest packing and tables in
// global memory (kernel ms): covid-350, 16384 runs, 32 lanes 17.6 for 34.4; SIR-77,
// 5e4 runs, 8 lanes 1.52 for 5.06; Fischer-32, 2e5 runs, 2 lanes 7.2 for 25.1;
// at 2000 runs Fischer-32 takes 0.82 at 32 lanes, 0.88 at 16 and 1.64 at 2.
// Where slots are tested one after another (invariants and blocking tests of
// several records) a lane gets as few as there are: csma-100, 16384 runs, 4.8
// at 64 lanes and 10.7 at 32.  Receivers tested edge by edge have at most four to
// a lane where the lists are longer than that (5, 20 and 34 edges on two channels, 70
// components, 2e4 runs: 1.25, 2.58 and 3.72 ms; at sixteen 1.86, 4.13 and 6.56); with
// two edges on 300 components sixteen are better, 2.1 ms for 2.9, and where the
// choice is eight or sixteen, 400 components: 6, 10 and 20 edges 5.26, 6.06 and 7.6 ms,
// at eight 6.30, 6.71 and 7.5.
smc_launch default_launch(const smc_model *m, uint64_t total_runs, bool trace) {
    const int P = m->img.n_leaves, stride = (m->img.n_vars + 1) | 1;
    const uint64_t simds = 4ull * (uint64_t)m->cu_count;
    smc_launch d{};
    int S = std::min(P, 64);
    const int most = m->img.recv_tested > 4 && P <= 256 ? 4 : 16;
    if (!(m->img.tests & (SMC_HF_XINV | SMC_HF_XBLK)))
        while (S > 1 && P / (S / 2) <= most) {
            const int s = S / 2, R = 64 / s;
            if (total_runs / (uint64_t)R < 2 * simds) break;
            if (!vars_fit(R, m->img.n_vars, tree_levels(s))) break;
            if (8 * (wave_lds_bytes(R, stride, P / s, trace) + kLdsStatic) > kLdsPerCu) break;
            S = s;
        }
    d.lanes_per_run = S;
    d.occupancy = P / S == 16 && total_runs / (uint64_t)(64 / S) > 2 * simds ? 3 : 0;
    d.tables = 2;  // staged if they fit
    return d;
}

// Half of a wave's even share of what is left, as a power of two.
int share_shift(int waves) {
    int s = 1;
    while (s < 62 && (1ll << (s - 1)) < waves) ++s;
    return s;
}

Plan plan_launch(const smc_model *m, const smc_launch *use, uint64_t total_runs, bool trace) {
    Plan pl;
    const int P = m->img.n_leaves;
    const smc_launch want = use ? *use : default_launch(m, total_runs, trace);
    if (want.occupancy != 0 && want.occupancy != 3) throw std::runtime_error("occupancy must be 0 or 3");
    if (want.tables < 0 || want.tables > 2) throw std::runtime_error("tables must be 0, 1 or 2");
    pl.occ = want.occupancy;
    int S = want.lanes_per_run ? want.lanes_per_run : (P < 64 ? P : 64);
    if (S <= 0 || S > 64 || (S & (S - 1))) throw std::runtime_error("lanes_per_run must be a power of two <= 64");
    if (S > P) S = P;
    pl.S = S;
    pl.C = P / S;
    if (pl.C > 16) throw std::runtime_error("limit: more than 16 components per lane; use more lanes per run");
    pl.R = 64 / S;
    pl.stride = (m->img.n_vars + 1) | 1;  // the variables and a constant 0
    const int levels = tree_levels(S);
    if (!vars_fit(pl.R, m->img.n_vars, levels))
        throw std::runtime_error("limit: variables of the packed runs exceed the LDS budget");
    const size_t wave = wave_lds_bytes(pl.R, pl.stride, pl.C, trace);
    pl.wave_lds = (uint32_t)wave;
    // with fewer runs than one wave on every SIMD can hold, spread over the
    // SIMDs instead, segments left idle: a lone wave's step takes the longer
    // the more runs differ in it
    const uint64_t spread = (total_runs + 4ull * m->cu_count - 1) / (4ull * m->cu_count);
    pl.segments = (int)std::min<uint64_t>(spread, (uint64_t)pl.R);
    const uint64_t most_waves = (total_runs + pl.segments - 1) / pl.segments;
    // Waves a CU holds: what the registers allow, and with staged tables
    // (one copy per workgroup) the LDS, for g waves per workgroup, as many on
    // each of the CU's four SIMDs.
    int per_cu = register_waves(pl.C, trace, pl.occ, want.tables != 0);
    const auto staged = [&](int g) {
        return std::min(groups_per_cu(m->table_bytes + (size_t)g * wave + kLdsStatic), std::max(per_cu / g, 1)) * g;
    };
    const int unstaged = std::min(per_cu, (int)(kLdsPerCu / (wave + kLdsStatic)));
    if (want.tables) {
        // (left to choose: where their bytes cost no waves.  What LDS rounds up may
        // cost one of ten; 150 components with a clock each, 5e4 runs: eleven waves a
        // CU 22.0 ms, ten that stage 19.4)
        int best = 0, by_bytes = 0;
        for (int g = 1; g <= SMC_MAX_GROUP_WAVES; g *= 2) {
            best = std::max(best, staged(g));
            by_bytes = std::max(by_bytes, std::min((int)(kLdsPerCu / (m->table_bytes + (size_t)g * wave + kLdsStatic)),
                                                   std::max(per_cu / g, 1)) * g);
        }
        pl.tab = best > 0 && (use || by_bytes >= unstaged);
        if (pl.tab) {
            // the smallest workgroups that hold what the runs ask for: few
            // runs then spread over the CUs evenly
            const int64_t cus = m->cu_count;
            int64_t need = best;
            if (want.waves > 0) need = std::min(need, (want.waves + cus - 1) / cus);
            else if (want.waves_per_cu > 0) need = std::min<int64_t>(need, want.waves_per_cu);
            need = std::min(need, (int64_t)((most_waves + (uint64_t)cus - 1) / (uint64_t)cus));
            pl.group_waves = 1;
            while (staged(pl.group_waves) < need) pl.group_waves *= 2;
            pl.table_bytes = m->table_bytes;
            per_cu = staged(pl.group_waves);
        } else {
            // a launch that names them is refused, but for what never was:
            // with digests, and tables that take little by the record
            if (use && !trace && named_tables_bytes(m, want.tables == 1) +
                                         4 * align_up((size_t)pl.R * pl.stride * 8 + (size_t)levels * 1024, 16) > kLdsPerCu)
                throw std::runtime_error("limit: the model tables do not fit in LDS");
            per_cu = register_waves(pl.C, trace, pl.occ, false);
        }
    }
    if (!pl.tab) per_cu = std::max(1, std::min(per_cu, groups_per_cu(wave + kLdsStatic)));
    pl.resident = (int64_t)m->cu_count * per_cu;
    if (want.waves_per_cu > 0 && want.waves_per_cu < per_cu) per_cu = want.waves_per_cu;
    pl.per_cu = per_cu;
    int waves = want.waves > 0 ? want.waves : m->cu_count * per_cu;
    // chunks: a wave takes as many as it has segments to start, and sixteen
    // times that on its way; what is left of a chunk waits in the wave, so
    // the waves end together only with small ones
    pl.chunk_runs = (uint32_t)std::min<uint64_t>(total_runs / (16ull * (uint64_t)waves * (uint64_t)pl.R) + 1, 256);
    waves = (int)std::min<uint64_t>((uint64_t)waves, most_waves);
    pl.lds = pl.table_bytes + (size_t)pl.group_waves * wave;
    pl.waves = (int)(((int64_t)waves + pl.group_waves - 1) / pl.group_waves * pl.group_waves);
    return pl;
}

void validate_query(const smc_query *q, int n_vars) {
    if (q->kind != SMC_QUERY_REACH && q->kind != SMC_QUERY_VAR) throw std::runtime_error("unknown query kind");
    if (q->kind == SMC_QUERY_VAR && (q->var < 0 || q->var >= n_vars))
        throw std::runtime_error("query variable id out of range");
    if (!(q->time_bound >= 0.0)) throw std::runtime_error("time bound must be a non-negative number");
}

SimParams make_params(const smc_query *q, const smc::ModelImage &img, uint64_t seed, uint64_t run_begin,
                      uint64_t n_runs, const RunBuffers &b, bool want_time, bool trace) {
    SimParams p{};
    p.seed = seed;
    p.run_begin = run_begin;
    p.n_runs = n_runs;
    p.bound = q->time_bound;
    p.threshold = q->threshold;
    p.reach = q->kind == SMC_QUERY_REACH;
    p.qvar = q->kind == SMC_QUERY_VAR ? q->var : -1;
    p.qinit = (p.qvar >= 0 && img.var_kind[p.qvar] == SMC_VAR_INT) ? img.var_init[p.qvar] : 0.0;
    p.is_max = q->is_max ? 1 : 0;
    p.max_steps = q->max_steps ? q->max_steps : SMC_DEFAULT_MAX_STEPS;
    p.flag = b.flag;
    p.value = b.value;
    p.steps = b.steps;
    p.trans = b.trans;
    p.digest = trace ? b.digest : nullptr;
    p.time = want_time ? b.time : nullptr;
    return p;
}

void fill_result(const smc_query *q, const ReducePartial &t, uint64_t n_runs, smc_result *out) {
    const double N = (double)n_runs;
    out->n_runs = n_runs;
    out->hits = t.hits;
    out->sum = t.sum;
    out->sumsq = t.sumsq;
    out->vmin = t.vmin;
    out->vmax = t.vmax;
    out->steps = t.steps;
    out->transitions = t.trans;
    out->truncated = t.truncated;
    out->ch_eps = smc_ch_epsilon(n_runs, 0.05);
    if (q->kind == SMC_QUERY_VAR && q->is_estimate) {
        out->estimate = t.sum / N;
        double var = n_runs > 1 ? std::max(0.0, (t.sumsq - t.sum * t.sum / N) / (N - 1.0)) : 0.0;
        out->clt_half = 1.959963984540054 * std::sqrt(var / N);
    } else {
        double pr = (double)t.hits / N;
        out->estimate = pr;
        out->clt_half = 1.959963984540054 * std::sqrt(pr * (1.0 - pr) / N);
    }
}

uint32_t reduce_blocks(uint64_t n_runs) {
    uint64_t b = (n_runs + 4095) / 4096;
    if (b < 1) b = 1;
    if (b > 1024) b = 1024;
    return (uint32_t)b;
}

}  // namespace

extern "C" {

const char *smc_last_error(void) { return g_last_error.c_str(); }
const char *smc_version(void) { return "cusmc_amd 0.1 (gfx950)"; }

double smc_ch_epsilon(uint64_t n, double delta) {
    if (n == 0 || !(delta > 0.0) || !(delta < 1.0)) return NAN;
    return std::sqrt(std::log(2.0 / delta) / (2.0 * (double)n));
}

// ------------------------------------------------------------ front end

static int parse_common(bool from_file, const char *src, const char *loc_query, smc_parsed **out) {
    if (!src || !out) return fail(SMC_E_INVALID, "null argument");
    *out = nullptr;
    try {
        auto res = std::make_unique<smc_parsed>();
        std::string q = loc_query ? loc_query : "";
        res->p = from_file ? smc::parse_uppaal_file(src, q) : smc::parse_uppaal_string(src, q);
        res->view = res->p->net.view();
        *out = res.release();
        return SMC_OK;
    } catch (const std::bad_alloc &) {
        return fail(SMC_E_ALLOC, "out of host memory");
    } catch (const std::exception &e) {
        return fail(SMC_E_PARSE, e.what());
    }
}

int smc_parse_uppaal(const char *path, const char *loc_query, smc_parsed **out) {
    return parse_common(true, path, loc_query, out);
}
int smc_parse_uppaal_string(const char *xml, const char *loc_query, smc_parsed **out) {
    return parse_common(false, xml, loc_query, out);
}
const smc_network *smc_parsed_network(const smc_parsed *p) { return p ? &p->view : nullptr; }
static const char *name_at(const std::vector<std::string> &v, int i) {
    return (i >= 0 && i < (int)v.size()) ? v[i].c_str() : "";
}
const char *smc_parsed_component_name(const smc_parsed *p, int c) { return p ? name_at(p->p->net.comp_names, c) : ""; }
const char *smc_parsed_location_name(const smc_parsed *p, int l) { return p ? name_at(p->p->net.loc_names, l) : ""; }
const char *smc_parsed_variable_name(const smc_parsed *p, int v) { return p ? name_at(p->p->net.var_names, v) : ""; }
int smc_parsed_goal_count(const smc_parsed *p) { return p ? p->p->goal_count : 0; }
void smc_parsed_destroy(smc_parsed *p) { delete p; }

// ------------------------------------------------------------ models

int smc_model_create(const smc_network *net, int device, smc_model **out) {
    if (!net || !out) return fail(SMC_E_INVALID, "null argument");
    *out = nullptr;
    return guarded([&]() -> int {
        auto m = std::make_unique<smc_model>();
        m->img = smc::compile_model(*net);
        if (m->img.n_leaves > 1024) throw std::runtime_error("limit: more than 1024 components per network");
        int ndev = 0;
        if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0)
            throw HipError("no HIP device available");
        if (device < 0 || device >= ndev) throw std::runtime_error("device index out of range");
        m->device = device;
        hip_check(hipSetDevice(device), "hipSetDevice");
        hipDeviceProp_t prop;
        hip_check(hipGetDeviceProperties(&prop, device), "hipGetDeviceProperties");
        m->cu_count = prop.multiProcessorCount;
        hip_check(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking), "hipStreamCreate");
        for (auto &e : m->ev) hip_check(hipEventCreate(&e), "hipEventCreate");

        // one arena for every table; variables start in their stored form
        // (a clock x = v0 as the reset stamp -v0)
        const smc::ModelImage &im = m->img;
        std::vector<double> var_start(im.var_init);
        for (size_t v = 0; v < var_start.size() && v < im.var_clock.size(); ++v)
            if (im.var_clock[v]) var_start[v] = -var_start[v];
        struct Part { const void *src; size_t bytes; size_t off; };
        std::vector<Part> parts = {
            {im.hots.data(), im.hots.size() * sizeof(DevHot), 0},
            {im.locs.data(), im.locs.size() * sizeof(DevLoc), 0},
            {im.edges.data(), im.edges.size() * sizeof(DevEdge), 0},
            {im.invs.data(), im.invs.size() * sizeof(DevInv), 0},
            {im.upds.data(), im.upds.size() * sizeof(DevUpd), 0},
            {im.guards.data(), im.guards.size() * sizeof(DevGuard), 0},
            {im.consts.data(), im.consts.size() * sizeof(double), 0},
            {im.code.data(), im.code.size() * sizeof(DevInsn), 0},
            {var_start.data(), var_start.size() * sizeof(double), 0},
            {im.comp_word.data(), im.comp_word.size() * sizeof(uint32_t), 0},
            {im.comp_init_loc.data(), im.comp_init_loc.size() * sizeof(int32_t), 0},
            {im.var_clock.data(), im.var_clock.size() * sizeof(uint8_t), 0},
            {im.comp_first_loc.data(), im.comp_first_loc.size() * sizeof(int32_t), 0},
            {im.loc_edge0.data(), im.loc_edge0.size() * sizeof(int32_t), 0},
            {im.loc_rec.data(), im.loc_rec.size() * sizeof(uint32_t), 0},
        };
        constexpr size_t kStaged = 8;  // hots .. code: what the run kernel reads every step
        size_t total = 0;
        for (size_t i = 0; i < parts.size(); ++i) {
            // the staged tables lie close together (16-byte records)
            total = align_up(total, i > 0 && i < kStaged ? 16 : 256);
            parts[i].off = total;
            total += parts[i].bytes;
        }
        total = align_up(total, 256);
        std::vector<uint8_t> host(total, 0);
        for (auto &p : parts) if (p.bytes) memcpy(host.data() + p.off, p.src, p.bytes);
        hip_check(hipMalloc(&m->arena, total), "hipMalloc model arena");
        hip_check(hipMemcpy(m->arena, host.data(), total, hipMemcpyHostToDevice), "upload model");
        auto at = [&](int i) { return (const void *)((const uint8_t *)m->arena + parts[i].off); };
        m->table_bytes = (uint32_t)align_up(parts[kStaged - 1].off + parts[kStaged - 1].bytes, 16);
        DevModel &d = m->dm;
        d.hots = (decltype(d.hots))at(0);
        d.locs = (decltype(d.locs))at(1);
        d.edges = (decltype(d.edges))at(2);
        d.invs = (decltype(d.invs))at(3);
        d.upds = (decltype(d.upds))at(4);
        d.guards = (decltype(d.guards))at(5);
        d.consts = (decltype(d.consts))at(6);
        d.code = (decltype(d.code))at(7);
        d.var_init = (decltype(d.var_init))at(8);
        d.comp_word = (decltype(d.comp_word))at(9);
        d.comp_init_loc = (decltype(d.comp_init_loc))at(10);
        d.var_clock = (decltype(d.var_clock))at(11);
        d.comp_first_loc = (decltype(d.comp_first_loc))at(12);
        d.loc_edge0 = (decltype(d.loc_edge0))at(13);
        d.loc_rec = (decltype(d.loc_rec))at(14);
        d.n_comp = im.n_comp;
        d.n_vars = im.n_vars;
        d.n_leaves = im.n_leaves;
        d.n_locs = (int)im.loc_rec.size();
        d.rec_shift = im.rec_shift;
        d.base_mask = (1u << im.rec_shift) - 1u;
        d.tests = im.tests;
        d.one_rate = im.one_rate;
        d.freeze = im.freeze ? 1 : 0;
        hip_check(hipMalloc(&m->d_inst, sizeof(InstDesc)), "hipMalloc instance");
        hip_check(hipMalloc(&m->d_counter, sizeof(unsigned long long)), "hipMalloc counter");
        hip_check(hipMalloc(&m->d_partials, 1024 * sizeof(ReducePartial)), "hipMalloc partials");
        *out = m.release();
        return SMC_OK;
    });
}

void smc_model_destroy(smc_model *m) { delete m; }

int smc_run(smc_model *m, const smc_query *q, uint64_t seed, uint64_t run_begin, uint64_t n_runs,
            const smc_launch *launch, smc_run_outputs *outputs, smc_result *out) {
    if (!m || !q || !out) return fail(SMC_E_INVALID, "null argument");
    return guarded([&]() -> int {
        auto wall0 = std::chrono::steady_clock::now();
        memset(out, 0, sizeof *out);
        validate_query(q, m->img.n_vars);
        if (n_runs == 0) throw std::runtime_error("n_runs must be positive");
        if (n_runs > (1ull << 32) - 1) throw std::runtime_error("limit: at most 2^32-1 runs per call");
        if (run_begin > (~0ull) - n_runs) throw std::runtime_error("run range overflows");
        const bool trace = outputs && outputs->digest;
        const smc_launch *use =
            (launch && (launch->lanes_per_run || launch->waves || launch->waves_per_cu || launch->occupancy ||
                        launch->tables))
                ? launch : (m->has_tuned ? &m->tuned : nullptr);
        hip_check(hipSetDevice(m->device), "hipSetDevice");
        Plan pl = plan_launch(m, use, n_runs, trace);
        m->runs.ensure(n_runs);
        // the totals are written straight to host memory
        if (!m->totals)
            hip_check(hipHostMalloc((void **)&m->totals, sizeof(ReducePartial), hipHostMallocDefault), "hipHostMalloc totals");
        const int waves = pl.waves;

        m->h_inst.m = m->dm;
        m->h_inst.p = make_params(q, m->img, seed, run_begin, n_runs, m->runs, outputs && outputs->time, trace);
        m->h_inst.chunk_first = 0;
        m->h_inst.chunk_runs = pl.chunk_runs;
        m->h_inst.lanes = pl.S;
        LaunchParams lp{};
        lp.inst = m->d_inst;
        lp.n_inst = 1;
        lp.total_chunks = (n_runs + pl.chunk_runs - 1) / pl.chunk_runs;
        lp.segments = pl.segments;
        lp.share_shift = share_shift(waves);
        lp.first = ((uint32_t)pl.segments + pl.chunk_runs - 1) / pl.chunk_runs;
        lp.handed = (uint64_t)lp.first * (uint64_t)std::min<int64_t>(waves, pl.resident);
        lp.counter = m->d_counter;
        lp.round = nullptr;
        lp.tables = pl.tab ? (decltype(lp.tables))m->arena : nullptr;
        lp.table_bytes = pl.table_bytes;
        lp.wave_lds = pl.wave_lds;
        const uint32_t blocks = reduce_blocks(n_runs);

        hip_check(smc::launch_setup(m->h_inst, m->d_inst, m->d_counter, m->stream), "setup kernel launch");
        hip_check(hipEventRecord(m->ev[0], m->stream), "event");
        hip_check(smc::launch_sim(lp, pl.C, trace, pl.occ, waves, pl.group_waves, pl.lds, m->stream), "run kernel launch");
        hip_check(hipEventRecord(m->ev[1], m->stream), "event");
        hip_check(smc::launch_reduce(m->d_inst, 1, blocks, m->d_partials, m->totals, 0, m->stream), "reduce kernel launch");
        hip_check(hipEventRecord(m->ev[2], m->stream), "event");
        // per-run outputs: small ones through pinned memory (a copy to memory
        // that is not waits for the device, each one some 25 us)
        struct Output { void *to; const void *from; size_t bytes; const char *what; };
        std::vector<Output> outs;
        size_t staged = 0;
        if (outputs) {
            const RunBuffers &b = m->runs;
            const Output all[] = {{outputs->flag, b.flag, n_runs, "copy flags"},
                                  {outputs->value, b.value, n_runs * 8, "copy values"},
                                  {outputs->steps, b.steps, n_runs * 4, "copy steps"},
                                  {outputs->transitions, b.trans, n_runs * 4, "copy transitions"},
                                  {outputs->digest, b.digest, n_runs * 8, "copy digests"},
                                  {outputs->time, b.time, n_runs * 8, "copy times"}};
            for (const Output &o : all)
                if (o.to) {
                    outs.push_back(o);
                    staged += align_up(o.bytes, 64);
                }
        }
        uint8_t *stage = nullptr;
        if (staged && staged <= smc_model::kStageBytes) {
            if (!m->stage && hipHostMalloc((void **)&m->stage, smc_model::kStageBytes, hipHostMallocDefault) != hipSuccess) {
                (void)hipGetLastError();  // without it the copies go straight to the caller's arrays
                m->stage = nullptr;
            }
            stage = m->stage;
        }
        size_t at = 0;
        for (const Output &o : outs) {
            hip_check(hipMemcpyAsync(stage ? stage + at : o.to, o.from, o.bytes, hipMemcpyDeviceToHost, m->stream), o.what);
            at += align_up(o.bytes, 64);
        }
        hip_check(hipStreamSynchronize(m->stream), "run");
        at = 0;
        for (const Output &o : outs) {
            if (stage) memcpy(o.to, stage + at, o.bytes);
            at += align_up(o.bytes, 64);
        }
        float k_ms = 0.f, r_ms = 0.f;
        hip_check(hipEventElapsedTime(&k_ms, m->ev[0], m->ev[1]), "event time");
        hip_check(hipEventElapsedTime(&r_ms, m->ev[1], m->ev[2]), "event time");
        fill_result(q, *m->totals, n_runs, out);
        out->kernel_ms = k_ms;
        out->reduce_ms = r_ms;
        out->lanes_per_run = pl.S;
        out->waves = waves;
        out->wall_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - wall0).count();
        return SMC_OK;
    });
}

int smc_run_noalloc(smc_model *m, const smc_query *q, uint64_t seed, uint64_t run_begin, uint64_t n_runs,
                    const smc_launch *launch, smc_result *out) {
    if (!m || !q || !out) return fail(SMC_E_INVALID, "null argument");
    return guarded([&]() -> int {
        auto wall0 = std::chrono::steady_clock::now();
        memset(out, 0, sizeof *out);
        validate_query(q, m->img.n_vars);
        if (n_runs == 0) throw std::runtime_error("n_runs must be positive");
        if (n_runs > SMC_NOALLOC_MAX_RUNS)
            throw std::runtime_error("limit: smc_run_noalloc takes at most 1048576 runs per call (its scratch is fixed)");
        if (run_begin > (~0ull) - n_runs) throw std::runtime_error("run range overflows");
        const smc_launch *use =
            (launch && (launch->lanes_per_run || launch->waves || launch->waves_per_cu || launch->occupancy ||
                        launch->tables))
                ? launch : (m->has_tuned ? &m->tuned : nullptr);
        hip_check(hipSetDevice(m->device), "hipSetDevice");
        void *scr = nullptr;
        hip_check(smc::noalloc_scratch(m->device, &scr), "scratch address");
        uint8_t *base = (uint8_t *)scr;
        Plan pl = plan_launch(m, use, n_runs, false);
        const int waves = pl.waves;

        // the per-run buffers are the scratch's (the whole run range of
        // this call is written by the run kernel before the reduction reads)
        RunBuffers b;
        b.flag = base + smc::kNoallocFlag;
        b.value = (double *)(base + smc::kNoallocValue);
        b.steps = (uint32_t *)(base + smc::kNoallocSteps);
        b.trans = (uint32_t *)(base + smc::kNoallocTrans);
        InstDesc *d_inst = (InstDesc *)(base + smc::kNoallocInst);
        unsigned long long *d_counter = (unsigned long long *)(base + smc::kNoallocCounter);
        ReducePartial *d_acc = (ReducePartial *)(base + smc::kNoallocAcc);
        ReducePartial *d_partials = (ReducePartial *)(base + smc::kNoallocPartials);
        const uint32_t blocks = reduce_blocks(n_runs);
        if (blocks > smc::kNoallocPartialsMax) throw std::runtime_error("internal: reduction blocks");

        m->h_inst.m = m->dm;
        m->h_inst.p = make_params(q, m->img, seed, run_begin, n_runs, b, false, false);
        m->h_inst.chunk_first = 0;
        m->h_inst.chunk_runs = pl.chunk_runs;
        m->h_inst.lanes = pl.S;
        LaunchParams lp{};
        lp.inst = d_inst;
        lp.n_inst = 1;
        lp.total_chunks = (n_runs + pl.chunk_runs - 1) / pl.chunk_runs;
        lp.segments = pl.segments;
        lp.share_shift = share_shift(waves);
        lp.first = ((uint32_t)pl.segments + pl.chunk_runs - 1) / pl.chunk_runs;
        lp.handed = (uint64_t)lp.first * (uint64_t)std::min<int64_t>(waves, pl.resident);
        lp.counter = d_counter;
        lp.round = nullptr;
        lp.tables = pl.tab ? (decltype(lp.tables))m->arena : nullptr;
        lp.table_bytes = pl.table_bytes;
        lp.wave_lds = pl.wave_lds;

        hip_check(smc::launch_setup(m->h_inst, d_inst, d_counter, m->stream), "setup kernel launch");
        hip_check(hipEventRecord(m->ev[0], m->stream), "event");
        hip_check(smc::launch_sim(lp, pl.C, false, pl.occ, waves, pl.group_waves, pl.lds, m->stream), "run kernel launch");
        hip_check(hipEventRecord(m->ev[1], m->stream), "event");
        hip_check(smc::launch_reduce(d_inst, 1, blocks, d_partials, d_acc, 0, m->stream), "reduce kernel launch");
        hip_check(hipEventRecord(m->ev[2], m->stream), "event");
        hip_check(hipMemcpyAsync(&m->h_acc, d_acc, sizeof(ReducePartial), hipMemcpyDeviceToHost, m->stream), "copy totals");
        hip_check(hipStreamSynchronize(m->stream), "run");
        float k_ms = 0.f, r_ms = 0.f;
        hip_check(hipEventElapsedTime(&k_ms, m->ev[0], m->ev[1]), "event time");
        hip_check(hipEventElapsedTime(&r_ms, m->ev[1], m->ev[2]), "event time");
        fill_result(q, m->h_acc, n_runs, out);
        out->kernel_ms = k_ms;
        out->reduce_ms = r_ms;
        out->lanes_per_run = pl.S;
        out->waves = waves;
        out->wall_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - wall0).count();
        return SMC_OK;
    });
}

}  // extern "C"

namespace {

// Persisted autotuner choices: one line per (model, query, device, library
// build, sample size) key in a text file — SMC_TUNE_CACHE names it (default
// $XDG_CACHE_HOME/cusmc_amd/tune.txt or ~/.cache/cusmc_amd/tune.txt;
// SMC_TUNE_CACHE=off disables it).
uint64_t fnv1a(uint64_t h, const void *p, size_t n) {
    const uint8_t *b = (const uint8_t *)p;
    for (size_t i = 0; i < n; ++i) h = (h ^ b[i]) * 1099511628211ull;
    return h;
}
template <class T>
uint64_t fnv_vec(uint64_t h, const std::vector<T> &v) {
    return fnv1a(h, v.data(), v.size() * sizeof(T));
}

std::string tune_cache_path() {
    const char *e = std::getenv("SMC_TUNE_CACHE");
    if (e && *e) return (std::string(e) == "off" || std::string(e) == "0") ? std::string() : std::string(e);
    const char *x = std::getenv("XDG_CACHE_HOME");
    const char *home = std::getenv("HOME");
    if (x && *x) return std::string(x) + "/cusmc_amd/tune.txt";
    if (home && *home) return std::string(home) + "/.cache/cusmc_amd/tune.txt";
    return std::string();
}

uint64_t tune_key(const smc_model *m, const smc_query *q, uint64_t sample_runs) {
    const smc::ModelImage &im = m->img;
    uint64_t h = 1469598103934665603ull;
    h = fnv_vec(h, im.hots); h = fnv_vec(h, im.locs); h = fnv_vec(h, im.invs); h = fnv_vec(h, im.edges); h = fnv_vec(h, im.guards);
    h = fnv_vec(h, im.upds); h = fnv_vec(h, im.consts); h = fnv_vec(h, im.code); h = fnv_vec(h, im.var_init);
    h = fnv_vec(h, im.comp_word);
    const int32_t qi[4] = {q->kind, q->var, q->is_max, q->is_estimate};
    const double qd[2] = {q->threshold, q->time_bound};
    h = fnv1a(h, qi, sizeof qi); h = fnv1a(h, qd, sizeof qd);
    h = fnv1a(h, &sample_runs, sizeof sample_runs);
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, m->device) == hipSuccess) {
        h = fnv1a(h, prop.gcnArchName, strnlen(prop.gcnArchName, sizeof prop.gcnArchName));
        h = fnv1a(h, &prop.multiProcessorCount, sizeof prop.multiProcessorCount);
    }
    static const char build[] = __DATE__ " " __TIME__;  // kernels of another build may rank differently
    return fnv1a(h, build, sizeof build);
}

bool tune_lookup(const std::string &path, uint64_t key, smc_launch *out) {
    if (path.empty()) return false;
    FILE *f = std::fopen(path.c_str(), "r");
    if (!f) return false;
    unsigned long long k;
    int S, wpc, occ, tab;
    bool found = false;
    while (std::fscanf(f, "%llx %d %d %d %d", &k, &S, &wpc, &occ, &tab) == 5)
        if (k == key) { *out = smc_launch{S, 0, wpc, occ, tab}; found = true; }
    std::fclose(f);
    return found;
}

void tune_store(const std::string &path, uint64_t key, const smc_launch &c) {
    if (path.empty()) return;
    const size_t slash = path.rfind('/');
    if (slash != std::string::npos) {
        std::error_code ec;
        std::filesystem::create_directories(path.substr(0, slash), ec);
    }
    if (FILE *f = std::fopen(path.c_str(), "a")) {
        std::fprintf(f, "%016llx %d %d %d %d\n", (unsigned long long)key, c.lanes_per_run, c.waves_per_cu, c.occupancy,
                     c.tables);
        std::fclose(f);
    }
}

}  // namespace

extern "C" {

int smc_autotune(smc_model *m, const smc_query *q, uint64_t seed, uint64_t sample_runs, smc_launch *best) {
    if (!m || !q) return fail(SMC_E_INVALID, "null argument");
    return guarded([&]() -> int {
        if (sample_runs == 0) sample_runs = 65536;
        validate_query(q, m->img.n_vars);
        const std::string cache = tune_cache_path();
        const uint64_t key = tune_key(m, q, sample_runs);
        smc_launch cached{};
        if (tune_lookup(cache, key, &cached)) {
            m->tuned = cached;
            m->has_tuned = true;
            if (best) *best = cached;
            return SMC_OK;
        }
        const int P = m->img.n_leaves;
        // lanes per run x register policy x table placement x waves per CU
        // (all the occupancy allows, or half of it: fewer waves contend less
        // for the caches and LDS)
        std::vector<smc_launch> cands;
        for (int S = P < 64 ? P : 64; S >= 1; S >>= 1) {
            if (P / S > 16) break;
            for (int occ : {0, 3})
                for (int tab : {0, 1}) {
                    const smc_launch c{S, 0, 0, occ, tab};
                    try {
                        const Plan pl = plan_launch(m, &c, sample_runs, false);
                        if (pl.tab != (tab == 1)) continue;  // the same as without
                        cands.push_back(c);
                        if (pl.per_cu >= 2) cands.push_back(smc_launch{S, 0, pl.per_cu / 2, occ, tab});
                    } catch (const std::exception &) {  // e.g. LDS budget exceeded at this packing
                    }
                }
        }
        if (cands.empty()) throw std::runtime_error("no launch shape could run this model");
        // each candidate runs at least twice the runs its grid holds at once,
        // so the sample measures the steady state rather than the tail
        double best_cost = 1e300;
        smc_launch pick = cands.front();
        for (const smc_launch &c : cands) {
            uint64_t n = sample_runs;
            const Plan pl = plan_launch(m, &c, sample_runs, false);
            n = std::max<uint64_t>(n, 2ull * (uint64_t)(pl.per_cu * m->cu_count) * (uint64_t)pl.R);
            smc_result r;
            int rc = smc_run(m, q, seed, 0, std::min<uint64_t>(n, 4096), &c, nullptr, &r);  // warm
            if (rc != SMC_OK) continue;
            rc = smc_run(m, q, seed + 1, 0, n, &c, nullptr, &r);
            const double cost = r.kernel_ms / (double)n;
            if (rc == SMC_OK && cost < best_cost) { best_cost = cost; pick = c; }
        }
        if (!(best_cost < 1e300)) throw std::runtime_error("no launch shape could run this model");
        m->tuned = pick;
        m->has_tuned = true;
        if (best) *best = pick;
        tune_store(cache, key, pick);
        return SMC_OK;
    });
}

// ------------------------------------------------------------ batches

}  // extern "C"

struct smc_batch {
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    std::vector<smc_batch_item> items;
    std::vector<RunBuffers> bufs;
    int C = 8, occ = 0, waves = 1, max_vars = 1;  // the one launch: slots per lane, register policy
    size_t lds = 0;
    InstDesc *d_all = nullptr;
    unsigned long long *d_counter = nullptr;
    ReducePartial *d_partials = nullptr, *d_acc = nullptr;
    uint64_t *d_round = nullptr;
    uint32_t blocks = 1;
    LaunchParams lp{};
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;

    ~smc_batch() {
        hipSetDevice(device);
        if (exec) hipGraphExecDestroy(exec);
        if (graph) hipGraphDestroy(graph);
        for (auto &b : bufs) b.release();
        for (void *p : {(void *)d_all, (void *)d_counter, (void *)d_partials, (void *)d_acc, (void *)d_round})
            if (p) hipFree(p);
        for (hipEvent_t e : {ev0, ev1}) if (e) hipEventDestroy(e);
        if (stream) hipStreamDestroy(stream);
    }
};

namespace {

// The instance records of one batch launch with C slots per lane: lanes per
// run S_i = next_pow2(components_i) / C (at least 1), R_i = 64 / S_i runs per
// wave and as many per chunk; returns the LDS bytes one wave needs (the
// largest instance) and the total of the chunks.  `runs_override` overrides every instance's n_runs
// (tuning samples).
struct BatchShape {
    std::vector<InstDesc> inst;
    size_t wave_lds = 0;
    uint64_t chunks = 0;
};

// Lanes per run of an instance at C slots per lane.
int batch_lanes(const smc_batch_item &it, int C) { return std::max(it.model->img.n_leaves / C, 1); }

bool batch_fits(const smc_batch &b, int C) {
    for (const smc_batch_item &it : b.items) {
        const int S = batch_lanes(it, C);
        if (!vars_fit(64 / S, b.max_vars, tree_levels(S))) return false;
    }
    return true;
}

// Waves that the runs fill at C slots per lane.
uint64_t batch_chunks(const smc_batch &b, int C) {
    uint64_t n = 0;
    for (const smc_batch_item &it : b.items) n += it.n_runs * (uint64_t)batch_lanes(it, C) / 64;
    return n;
}

BatchShape batch_shape(smc_batch *b, int C, uint64_t runs_override) {
    BatchShape sh;
    if (!batch_fits(*b, C)) throw std::runtime_error("limit: variables of the packed runs exceed the LDS budget");
    for (size_t i = 0; i < b->items.size(); ++i) {
        const smc_batch_item &it = b->items[i];
        const int P = it.model->img.n_leaves;
        if (P > 64 * C) throw std::runtime_error("internal: instance wider than the launch's packing");
        const int S = batch_lanes(it, C);
        const int R = 64 / S;
        sh.wave_lds = std::max(sh.wave_lds, wave_lds_bytes(R, (it.model->img.n_vars + 1) | 1, C, false));
        const uint64_t n = runs_override ? std::min<uint64_t>(runs_override, it.n_runs) : it.n_runs;
        InstDesc d{};
        d.m = it.model->dm;
        d.p = make_params(&it.query, it.model->img, it.seed, it.run_begin, n, b->bufs[i], false, false);
        d.chunk_first = sh.chunks;
        d.lanes = S;
        d.chunk_runs = (uint32_t)R;
        sh.chunks += (n + R - 1) / R;
        sh.inst.push_back(d);
    }
    return sh;
}

// Waves of one launch at C slots per lane and register policy occ: every
// CU filled to its occupancy (or to waves_per_cu when that is lower).
int batch_waves(int C, int occ, size_t wave_lds, int waves_per_cu, int cu_count) {
    int blocks = 0;
    hip_check(smc::sim_occupancy(C, false, occ, false, 1, wave_lds, &blocks), "occupancy query");
    int per_cu = std::min(blocks, groups_per_cu(wave_lds + kLdsStatic));
    if (waves_per_cu > 0 && waves_per_cu < per_cu) per_cu = waves_per_cu;
    return std::max(1, per_cu) * cu_count;
}

}  // namespace

extern "C" {

int smc_batch_create(const smc_batch_item *items, int n_items, int tune, smc_batch **out) {
    if (!items || n_items <= 0 || !out) return fail(SMC_E_INVALID, "null argument or empty batch");
    *out = nullptr;
    return guarded([&]() -> int {
        auto b = std::make_unique<smc_batch>();
        b->items.assign(items, items + n_items);
        b->device = items[0].model ? items[0].model->device : 0;
        int maxP = 1, max_vars = 1;
        for (int i = 0; i < n_items; ++i) {
            const smc_batch_item &it = items[i];
            if (!it.model) throw std::runtime_error("batch item without a model");
            if (it.model->device != b->device) throw std::runtime_error("batch items on different devices");
            validate_query(&it.query, it.model->img.n_vars);
            if (it.n_runs == 0 || it.n_runs > (1ull << 32) - 1) throw std::runtime_error("batch item n_runs out of range");
            maxP = std::max(maxP, it.model->img.n_leaves);
            max_vars = std::max(max_vars, it.model->img.n_vars);
        }
        hip_check(hipSetDevice(b->device), "hipSetDevice");
        hip_check(hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking), "hipStreamCreate");
        for (hipEvent_t *e : {&b->ev0, &b->ev1}) hip_check(hipEventCreate(e), "hipEventCreate");
        const int cu = items[0].model->cu_count;
        b->max_vars = max_vars;
        b->bufs.resize(n_items);
        uint64_t maxr = 0;
        for (int i = 0; i < n_items; ++i) {
            b->bufs[i].ensure(items[i].n_runs);
            maxr = std::max<uint64_t>(maxr, items[i].n_runs);
        }
        b->blocks = std::min<uint32_t>(reduce_blocks(maxr), 64);
        hip_check(hipMalloc(&b->d_all, n_items * sizeof(InstDesc)), "hipMalloc instances");
        hip_check(hipMalloc(&b->d_counter, sizeof(unsigned long long)), "hipMalloc counter");
        hip_check(hipMalloc(&b->d_partials, (size_t)n_items * b->blocks * sizeof(ReducePartial)), "hipMalloc partials");
        hip_check(hipMalloc(&b->d_acc, n_items * sizeof(ReducePartial)), "hipMalloc totals");
        hip_check(hipMalloc(&b->d_round, sizeof(uint64_t)), "hipMalloc round");
        hip_check(hipMemset(b->d_round, 0, sizeof(uint64_t)), "clear round");

        // the launch's slots per lane: left to choose (below), or (tune) the
        // fastest of the smallest that holds the widest instance in 64 lanes
        // and wider packings under both register policies on a sample of
        // every instance's runs
        int Cmin = 1;
        while (64 * Cmin < maxP) Cmin <<= 1;
        if (Cmin > 16) throw std::runtime_error("limit: more than 1024 components per network");
        auto set_launch = [&](const BatchShape &sh, int C, int occ, int waves) {
            b->C = C;
            b->occ = occ;
            b->waves = (int)std::min<uint64_t>((uint64_t)waves, std::max<uint64_t>(sh.chunks, 1));
            b->lds = sh.wave_lds;
            b->lp = LaunchParams{};
            b->lp.inst = b->d_all;
            b->lp.n_inst = n_items;
            b->lp.total_chunks = sh.chunks;
            b->lp.segments = 64;
            b->lp.share_shift = share_shift(b->waves);
            b->lp.first = 1;
            b->lp.handed = (uint64_t)b->waves;
            b->lp.counter = b->d_counter;
            b->lp.round = b->d_round;
            b->lp.tables = nullptr;
            b->lp.table_bytes = 0;
            b->lp.wave_lds = (uint32_t)sh.wave_lds;
            hip_check(hipMemcpy(b->d_all, sh.inst.data(), n_items * sizeof(InstDesc), hipMemcpyHostToDevice),
                      "upload instances");
        };
        // (a batch that does not fit at eight slots is refused)
        int bestC = std::max(Cmin, 8), best_occ = 0;
        batch_shape(b.get(), bestC, 0);
        // eight slots per lane where that leaves every SIMD two waves' runs,
        // else the fewest that hold the widest instance, for shorter steps: 34
        // instances of 1000 runs take 3.7 ms at 8 slots, 4.0 at 4, 4.9 at 2
        // and 4.7 at 16, 16 of 600 runs 2.7 ms at 8 and 1.8 at 4
        if (!tune && batch_fits(*b, Cmin) && batch_chunks(*b, bestC) < 8ull * (uint64_t)cu) bestC = Cmin;
        if (tune) {
            double best_ms = 1e300;
            uint64_t sample = 0;
            for (auto &it : b->items) sample = std::max<uint64_t>(sample, std::min<uint64_t>(it.n_runs, 2048));
            for (int C = Cmin; C <= 16; C <<= 1)
                for (int occ : {0, 3}) {
                    BatchShape sh = batch_shape(b.get(), C, sample);
                    const int waves = batch_waves(C, occ, sh.wave_lds, 0, cu);
                    set_launch(sh, C, occ, waves);
                    float ms = 0.f;
                    for (int rep = 0; rep < 2; ++rep) {  // the first launch warms the code
                        hip_check(smc::launch_prep(b->d_counter, nullptr, 0, b->stream), "prep");
                        hip_check(hipEventRecord(b->ev0, b->stream), "event");
                        hip_check(smc::launch_sim(b->lp, C, false, occ, b->waves, 1, b->lds, b->stream), "tune launch");
                        hip_check(hipEventRecord(b->ev1, b->stream), "event");
                        hip_check(hipStreamSynchronize(b->stream), "tune");
                        hip_check(hipEventElapsedTime(&ms, b->ev0, b->ev1), "event time");
                    }
                    if (ms < best_ms) { best_ms = ms; bestC = C; best_occ = occ; }
                }
        }
        {
            BatchShape sh = batch_shape(b.get(), bestC, 0);
            const int waves = batch_waves(bestC, best_occ, sh.wave_lds, 0, cu);
            set_launch(sh, bestC, best_occ, waves);
        }
        hip_check(hipDeviceSynchronize(), "batch setup");

        // capture one round: the run kernel over every instance, the
        // reduction accumulates, then the counter is cleared and the round
        // advances
        hip_check(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal), "begin capture");
        hip_check(smc::launch_prep(b->d_counter, nullptr, 0, b->stream), "capture prep");
        hip_check(smc::launch_sim(b->lp, b->C, false, b->occ, b->waves, 1, b->lds, b->stream), "capture run kernel");
        hip_check(smc::launch_reduce(b->d_all, n_items, b->blocks, b->d_partials, b->d_acc, 1, b->stream), "capture reduce");
        hip_check(smc::launch_prep(b->d_counter, b->d_round, 1, b->stream), "capture advance");
        hip_check(hipStreamEndCapture(b->stream, &b->graph), "end capture");
        hip_check(hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0), "instantiate graph");
        *out = b.release();
        return SMC_OK;
    });
}

int smc_batch_run(smc_batch *b, int rounds, smc_result *results, smc_batch_stats *stats) {
    if (!b || rounds <= 0) return fail(SMC_E_INVALID, "null batch or non-positive rounds");
    return guarded([&]() -> int {
        const int n = (int)b->items.size();
        hip_check(hipSetDevice(b->device), "hipSetDevice");
        std::vector<ReducePartial> init(n);
        for (auto &t : init) { t = ReducePartial{}; t.vmin = HUGE_VAL; t.vmax = -HUGE_VAL; }
        hip_check(hipMemcpyAsync(b->d_acc, init.data(), n * sizeof(ReducePartial), hipMemcpyHostToDevice, b->stream), "init totals");
        hip_check(hipEventRecord(b->ev0, b->stream), "event");
        for (int r = 0; r < rounds; ++r) hip_check(hipGraphLaunch(b->exec, b->stream), "graph launch");
        hip_check(hipEventRecord(b->ev1, b->stream), "event");
        std::vector<ReducePartial> acc(n);
        hip_check(hipMemcpyAsync(acc.data(), b->d_acc, n * sizeof(ReducePartial), hipMemcpyDeviceToHost, b->stream), "copy totals");
        hip_check(hipStreamSynchronize(b->stream), "batch run");
        float ms = 0.f;
        hip_check(hipEventElapsedTime(&ms, b->ev0, b->ev1), "event time");
        uint64_t runs = 0, steps = 0, trans = 0;
        for (int i = 0; i < n; ++i) {
            const uint64_t nr = b->items[i].n_runs * (uint64_t)rounds;
            runs += nr;
            steps += acc[i].steps;
            trans += acc[i].trans;
            if (results) {
                memset(&results[i], 0, sizeof(smc_result));
                fill_result(&b->items[i].query, acc[i], nr, &results[i]);
                results[i].kernel_ms = ms;
            }
        }
        if (stats) {
            stats->graph_ms = ms;
            stats->runs = runs;
            stats->steps = steps;
            stats->transitions = trans;
            stats->groups = 1;
            stats->rounds = rounds;
        }
        return SMC_OK;
    });
}

void smc_batch_destroy(smc_batch *b) { delete b; }

}  // extern "C"
