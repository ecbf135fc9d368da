// sim_variant.hip — one build of the run kernel (sim_body.h): SMC_C
// component slots per lane, register policy SMC_OCC (0 unrestricted, 3 at
// most 168 registers: three waves per SIMD), with and without digests, with
// the tables in global memory or staged in LDS.
// The build compiles this file once per pair, in parallel.
#include "sim_body.h"

#if !defined(SMC_C) || !defined(SMC_OCC)
#error "SMC_C and SMC_OCC must be defined"
#endif

#define SMC_JOIN2(a, b, c, d) a##b##c##d
#define SMC_JOIN(a, b, c, d) SMC_JOIN2(a, b, c, d)

namespace {

#if SMC_OCC == 3
#define SMC_KERNEL sim_kernel_o3
#else
#define SMC_KERNEL sim_kernel
#endif

const void *kernel_fn(bool trace, bool tab) {
    if (trace) return tab ? (const void *)SMC_KERNEL<SMC_C, true, true> : (const void *)SMC_KERNEL<SMC_C, true, false>;
    return tab ? (const void *)SMC_KERNEL<SMC_C, false, true> : (const void *)SMC_KERNEL<SMC_C, false, false>;
}

hipError_t launch(const LaunchParams &lp, bool trace, bool tab, int waves, int group_waves, size_t lds,
                  hipStream_t s) {
    const dim3 grid(waves / group_waves), block(64 * group_waves);
    if (trace && tab) hipLaunchKernelGGL((SMC_KERNEL<SMC_C, true, true>), grid, block, lds, s, lp);
    else if (trace) hipLaunchKernelGGL((SMC_KERNEL<SMC_C, true, false>), grid, block, lds, s, lp);
    else if (tab) hipLaunchKernelGGL((SMC_KERNEL<SMC_C, false, true>), grid, block, lds, s, lp);
    else hipLaunchKernelGGL((SMC_KERNEL<SMC_C, false, false>), grid, block, lds, s, lp);
    return hipGetLastError();
}

hipError_t occupancy(bool trace, bool tab, int group_waves, size_t lds, int *blocks_per_cu) {
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, kernel_fn(trace, tab), 64 * group_waves, lds);
}

}  // namespace

namespace smc {
SimVariant SMC_JOIN(sim_variant_c, SMC_C, _o, SMC_OCC)() { return SimVariant{&launch, &occupancy}; }
}  // namespace smc
