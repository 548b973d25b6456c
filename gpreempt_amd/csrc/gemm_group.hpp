// Several convolutions of a network's level that do not read each other (the branches of an Inception block), as one launch.
//
// Why: at a batch of a few images each of them is 30-100 tiles on 256 compute units and, like every dependent launch, costs 5 us and more
// whatever it computes; run side by side they cost that once.  Inception-v3 has 94 convolutions in 52 levels.
//
// Structure: the tiles of the members stand one behind the other in the launch's tile order; a workgroup finds the member its tile
// belongs to and runs that member's own body (one of the forms, GEMM, convolution, convolution whose blocks straddle taps,
// convolution with its window in LDS, of one tile shape, which is all a kernel can hold), so sums and bits are those of launches of their own.
// Claims, claim counters and the kernel index are the launch's: a stop inside it resumes there.
#pragma once
#include "gemm_narrow.hpp"
#include "gemm_window.hpp"

namespace gp {

constexpr int kGroupMax = 4;
struct GroupMember {
    MatArgs g;
    int first, sx, sy, order, form;  // first tile in the launch's order, tile grid, order and body form (0, 1, 2: WideKernel's CONV, 3: WindowKernel)
    unsigned inv_sx, inv_sy;
};
struct GroupArgs {
    GroupMember m[kGroupMax];
    int first[kGroupMax];  // as in m; beyond the last member: no tile is that far
};

// F0 .. F3: the bodies of the forms; F3 == F1: there is no form 3
template <int LOOP, class F0, class F1, class F2, class F3>
__global__ __launch_bounds__(F0::NT) void group_kernel(GroupArgs a, BlpArgs blp) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    using T = typename F0::elem;
    T *lds = reinterpret_cast<T *>(lds_raw);
    constexpr bool SINGLE = LOOP != LOOP_ANY;
    auto tile = [&](TileIdx at, int *stop, auto asked) -> bool {
        const int idx = __builtin_amdgcn_readfirstlane(at.x);
        int which = 0;
#pragma unroll
        for (int i = 1; i < kGroupMax; ++i) which += idx >= a.first[i];
        // (the member's arguments where they lie, at the front of the kernel's: indexed as a by-value argument, the compiler would
        // copy all of them to scratch memory first)
        typedef const __attribute__((address_space(4))) GroupMember *MemberPtr;
        typedef const __attribute__((address_space(4))) unsigned long long *WordPtr;
        const MemberPtr m = (MemberPtr)__builtin_amdgcn_kernarg_segment_ptr() + which;
        struct Words { unsigned long long w[sizeof(MatArgs) / 8]; } words;
        static_assert(sizeof(MatArgs) % 8 == 0 && alignof(MatArgs) == 8, "whole words");
#pragma unroll
        for (unsigned i = 0; i < sizeof(MatArgs) / 8; ++i) words.w[i] = ((WordPtr)&m->g)[i];
        const MatArgs g = __builtin_bit_cast(MatArgs, words);
        const TileIdx t = decode_tile(idx - m->first, m->sx, m->sy, m->order, m->inv_sx, m->inv_sy);
        const CkptCtx cc{stop, nullptr, nullptr, 0};
        const int form = m->form;
        if (form == 0) return F0::template run<false, SINGLE>(g, t, lds, cc, asked);
        if constexpr (F3::window)
            if (form == 3) return F3::template run<false, SINGLE>(g, t, lds, cc, asked);
        if (form == 1) return F1::template run<false, SINGLE>(g, t, lds, cc, asked);
        return F2::template run<false, SINGLE>(g, t, lds, cc, asked);
    };
    if constexpr (LOOP == LOOP_FIXED) tile_fixed_early<F0::NT>(blp, [&](TileIdx t, int *stop) { return tile(t, stop, [&] { late_claim<F0::NT>(blp); }); });
    else tiles<LOOP>(blp, [&](TileIdx t) { tile(t, nullptr, NoneAsked{}); });
}

template <class F0, class F1, class F2, class F3 = F1>
static int launch_group(const MatPlan *pl, int n, const gp_preempt_ctx *ctx, gp_stream s, gp_launch_info *info) {
    static_assert(F0::NT == F1::NT && F0::NT == F2::NT && F0::NT == F3::NT, "one kernel");
    constexpr size_t rings = std::max(F0::LDS_BYTES, std::max(F1::LDS_BYTES, F2::LDS_BYTES)), most = F3::window ? std::max(rings, kWindowMaxLds) : rings;
    size_t lds = rings;
    constexpr auto any = group_kernel<LOOP_ANY, F0, F1, F2, F3>, plain = group_kernel<LOOP_PLAIN, F0, F1, F2, F3>, fixed = group_kernel<LOOP_FIXED, F0, F1, F2, F3>;
    static std::once_flag once;
    static hipError_t once_rc = hipSuccess;
    std::call_once(once, [] {
        for (const void *f : {(const void *)any, (const void *)plain, (const void *)fixed}) {
            hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)most);
            if (e != hipSuccess) once_rc = e;
        }
    });
    GP_HIP(once_rc);
    GroupArgs a = {};
    int total = 0;
    for (int i = 0; i < kGroupMax; ++i) {
        a.first[i] = i < n ? total : 0x7fffffff;
        if (i >= n) continue;
        GroupMember &m = a.m[i];
        const int tiles = pl[i].sx * pl[i].sy;
        m.g = pl[i].g;
        m.first = total; m.sx = pl[i].sx; m.sy = pl[i].sy; m.order = pl[i].order;
        m.form = !pl[i].conv ? 0 : F3::window && pl[i].window ? 3 : straddles_taps<typename F0::elem>(pl[i]) ? 2 : 1;
        if (m.form == 3) lds = std::max(lds, F3::LDS_BYTES + window_bytes(m.g, F3::bm, (int)sizeof(typename F0::elem)));
        m.inv_sx = inverse_of(m.sx, tiles); m.inv_sy = inverse_of(m.sy, tiles);
        total += tiles;
    }
    BlpArgs blp;
    int grid = 0;
    int rc = plan_launch(any, F0::NT, lds, total, 1, 1, ctx, &blp, &grid, info, 1, 2);
    if (rc) return rc;
    auto kern = !ctx ? plain : fixed_claims(true, blp.groups, grid - blp.front, blp.total) ? fixed : any;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(F0::NT), lds, native(s), a, blp);
    GP_HIP(hipGetLastError());
    return GP_SUCC;
}

}  // namespace gp
