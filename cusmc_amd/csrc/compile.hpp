// compile.hpp — smc_network -> device model tables and register bytecode.
#pragma once

#include <string>
#include <vector>
#include "devmodel.h"
#include "smc_network.h"

namespace smc {

// A location of the network as written (tilt groups of importance sampling).
struct LocInfo {
    uint8_t klass = 0, type = 0;
    int n_inv = 0;
    int64_t rate_key = 0;  // the constant's bits, or the identity of the expression
    struct Edge { int32_t dst, channel; };  // dst relative to the location
    std::vector<Edge> edges;
};

struct ModelImage {
    std::vector<DevHot> hots;           // per record class
    std::vector<DevLoc> locs;           // per record class
    std::vector<DevInv> invs;
    std::vector<DevEdge> edges;
    std::vector<DevGuard> guards;
    std::vector<DevUpd> upds;
    std::vector<double> consts;
    std::vector<DevInsn> code;
    std::vector<double> var_init;
    std::vector<uint32_t> comp_word;    // initial state word of each component
    std::vector<int32_t> comp_init_loc;
    std::vector<int32_t> comp_first_loc;
    std::vector<uint8_t> var_clock;     // per variable: 1 for a clock
    std::vector<int32_t> var_kind;
    std::vector<int32_t> loc_edge0;     // per location: the network's index of its first edge
    std::vector<uint32_t> loc_rec;      // per location: its record class
    std::vector<LocInfo> info;          // per location
    int n_comp = 0, n_vars = 0, n_leaves = 1;
    int rec_shift = 13;
    uint32_t tests = 0;   // every SMC_HF_* flag in use
    uint32_t one_rate = SMC_NO_REF;  // the one rate expression, if there is just one
    bool freeze = true;   // no location's rate reads a clock
    int recv_tested = 0;  // most edges of a location whose receive edges are tested one by one (DevLoc.recv_chan -1)
};

// Throws std::runtime_error (message prefixed "limit:" for size limits).
ModelImage compile_model(const smc_network &net);

}  // namespace smc
