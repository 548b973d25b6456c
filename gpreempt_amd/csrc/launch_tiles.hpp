// Launch of a kernel built around tile_loop.hpp's dispatchers on a one-dimensional list of tiles, shared by the
// operators, the stencil and the graph kernels.
#pragma once
#include <algorithm>
#include "common.hpp"

namespace gp {

// the three instantiations of one kernel: general dispatcher loop, no counters, fixed claims
template <class Kernel> struct KernelSet { Kernel any, plain, fixed; bool long_tiles = false; };  // (long_tiles: see plan_launch)
template <class Kernel> static KernelSet<Kernel> kernel_set(Kernel a, Kernel p, Kernel f) { return {a, p, f, false}; }
#define GP_KSET(...) kernel_set(__VA_ARGS__, LOOP_ANY>, __VA_ARGS__, LOOP_PLAIN>, __VA_ARGS__, LOOP_FIXED>)

// `more`: kernel arguments between the operator's parameters and the dispatcher's
template <class Kernel, class Arg, class... More>
static int launch_tiles(KernelSet<Kernel> ks, int sx, int sy, const gp_preempt_ctx *ctx, gp_stream s, gp_launch_info *info, const Arg &arg, size_t lds_bytes = 0, int max_batch = 16, int block = 256, More... more) {
    BlpArgs blp;
    int grid = 0;
    // several tiles per claim once there are far more tiles than workgroups that could hold them
    const long tiles = (long)sx * sy;
    const int batch = (int)std::min<long>(max_batch, std::max<long>(1, tiles / (32L * device_cus())));
    if (lds_bytes > 48 * 1024) {
        static thread_local size_t allowed = 0;  // (of this kernel: one instantiation of this function per kernel type,
        static thread_local const void *of = nullptr;  // and the kernels of one type share it)
        if (of != (const void *)ks.any || allowed < lds_bytes) {
            for (Kernel k : {ks.any, ks.plain, ks.fixed}) GP_HIP(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes));
            of = (const void *)ks.any; allowed = lds_bytes;
        }
    }
    // planned for the general form; the special ones need no more resources
    int rc = plan_launch(ks.any, block, lds_bytes, sx, sy, 1, ctx, &blp, &grid, info, batch, batch == 1 ? 4 : 1, ks.long_tiles && batch == 1);
    if (rc) return rc;
    Kernel kern = ks.any;
    if (batch == 1) {  // the special forms call the body once: one tile per claim only
        if (!ctx) kern = ks.plain;
        else if (fixed_claims(true, blp.groups, grid - blp.front, blp.total)) kern = ks.fixed;
    }
    hipLaunchKernelGGL(kern, dim3(grid), dim3(block), lds_bytes, native(s), arg, more..., blp);
    GP_HIP(hipGetLastError());
    return GP_SUCC;
}

}  // namespace gp
