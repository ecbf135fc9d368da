// Lowers UPPAAL models to the run kernel's tables on the CPU and prints what
// came out: one line per file with its sizes, then one per edge whose first
// guard is an interval.  Built by test_compile_tables.py with the sanitiser for
// undefined behaviour.
#include <cstdio>

#include "compile.hpp"
#include "uppaal.hpp"

int main(int argc, char **argv) {
    for (int i = 1; i < argc; ++i) {
        const auto p = smc::parse_uppaal_file(argv[i], "");
        const smc::ModelImage im = smc::compile_model(p->net.view());
        std::printf("model locations %zu classes %zu edges %zu\n", im.loc_rec.size(), im.locs.size(), im.edges.size());
        for (const DevLoc &L : im.locs)
            if (L.recv_chan) std::printf("receives %s chan %d\n", L.flags & SMC_LF_RECV_FAST ? "together" : "in turn", L.recv_chan);
        for (const DevHot &h : im.hots)
            if ((h.what >> 16) & SMC_HF_INV) std::printf("window %s\n", (h.what >> 16) & SMC_HF_WINDOW ? "general" : "inline");
        for (const DevEdge &e : im.edges)
            if (!(e.flags & SMC_EF_NO_GUARD)) std::printf("interval %a %a\n", e.lo, e.hi);
    }
}
