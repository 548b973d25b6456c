// The matrix kernels' launchers by element type.  Instantiated in a unit of its own per type (gemm_f32.hip, gemm_f16.hip,
// gemm_bf16.hip), which the compiler can work on side by side; gemm.hip plans and picks.
#pragma once
#include <cstdlib>
#include <mutex>
#include "gemm_tile.hpp"
#include "gemm_pipe.hpp"
#include "gemm_wide.hpp"
#include "gemm_ln.hpp"
#include "gemm_narrow.hpp"
#include "plans.hpp"

namespace gp {
// whether a convolution's K-blocks (128 bytes) straddle filter taps
template <typename T> static bool straddles_taps(const MatPlan &pl) { return pl.g.Cin % (128 / (int)sizeof(T)) != 0; }
}  // namespace gp
#include "gemm_group.hpp"

namespace gp {

// Asks for the arguments that stand in front of a tile's first load, and for those of its epilogue, in one go.  Left to itself
// the compiler reads them where they are used, in four or five batches one behind the other, each a trip of 0.2 us.
// (INVERSES: of the channels and window columns too, for the form that finds its taps by them.)
template <bool CONV, bool INVERSES> __device__ __forceinline__ void read_args(const MatArgs &g, const BlpArgs &b) {
    asm volatile("" ::"s"(b.total), "s"(b.sx), "s"(b.sy), "s"(b.order), "s"(b.inv_sx), "s"(b.inv_sy), "s"(b.grid), "s"(b.front), "s"(b.executed), "s"(b.stop_index), "s"(g.M), "s"(g.N), "s"(g.K),
                 "s"(g.A), "s"(g.lda), "s"(g.B), "s"(g.ldb), "s"(g.batch_inner), "s"(g.C), "s"(g.ldc), "s"(g.bias), "s"(g.alpha), "s"(g.act));
    if (CONV) asm volatile("" ::"s"(g.H), "s"(g.W), "s"(g.Cin), "s"(g.S), "s"(g.Ho), "s"(g.Wo), "s"(g.sh), "s"(g.sw), "s"(g.ph), "s"(g.pw), "s"(g.R), "s"(g.rcp_hw), "s"(g.rcp_wo));
    if (INVERSES) asm volatile("" ::"s"(g.inv_cin), "s"(g.inv_s));
}

template <class K> struct K_divides { static constexpr bool value = false; };
template <typename T, int BM, int BN, int ST> struct K_divides<PipeKernel<T, BM, BN, ST, 3, false>> { static constexpr bool value = true; };
// LOOP: which dispatcher loop the instantiation is built around (tile_loop.hpp)
constexpr int LOOP_LOOKS = 3;
template <class TK, int LOOP>
__global__ __launch_bounds__(TK::NT) void mat_kernel(MatArgs g, BlpArgs blp) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    auto *lds = reinterpret_cast<typename TK::elem *>(lds_raw);
    if constexpr (LOOP != LOOP_ANY) read_args<TK::conv, K_divides<TK>::value>(g, blp);
    if constexpr (LOOP == LOOP_LOOKS)  // long tiles: fixed claims, and the body looks at the stop word every few K-stages
        tile_fixed_early<TK::NT, true>(blp, [&](TileIdx t, int *stop) {
            CkptCtx cc{stop, nullptr, nullptr, 0};
            if (stop && blp.done) cc.announce = done_counter(blp);
            return TK::template run<true, true>(g, t, lds, cc, [&] { late_claim<TK::NT>(blp); });
        });
    else if constexpr (LOOP == LOOP_FIXED && TK::early_stop)
        tile_fixed_early<TK::NT>(blp, [&](TileIdx t, int *stop) { return TK::template run<false, true>(g, t, lds, CkptCtx{stop, nullptr, nullptr, 0}, [&] { late_claim<TK::NT>(blp); }); });
    else if constexpr (LOOP == LOOP_PLAIN && TK::early_stop)
        tile_plain(blp, [&](TileIdx t) { TK::template run<false, true>(g, t, lds); });
    else
        tiles<LOOP>(blp, [&](TileIdx t) { TK::run(g, t, lds); });
}

// bodies that can leave a tile between two K-steps (tile_loop_ckpt)
template <class TK>
__global__ __launch_bounds__(TK::NT) void mat_kernel_ckpt(MatArgs g, BlpArgs blp) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    auto *lds = reinterpret_cast<typename TK::elem *>(lds_raw);
    const CkptCtx cc = {blp.executed && blp.ckpt ? blp.stop_index : nullptr, blp.flag, blp.ckpt, blp.kernel_id, blp.stamps};
    tile_loop_ckpt(blp, [&](TileIdx t, int tile_index, int kt0) { return TK::run(g, t, lds, cc, NoneAsked{}, tile_index, kt0); });
}

// Long tiles (1.8 * 10^7 multiply-adds of the 16-bit rate and more, 10-40 us depending on how many workgroups share a
// compute unit): what a stopped tenant would otherwise finish before it leaves.  The bodies that look at the stop
// word every few K-stages can give such a tile up (tile_fixed_early).  Measured with the threshold at 0.8 / 2 / 4 * 10^7:
// ResNet-50 fp32 b1 under a 500 req/s probe drains in 35 / 42 / 57 us (p99) and keeps 1046 / 1095 / 1094 req/s
// (a launch in this mode is about a microsecond longer).  The 64x64 tiles with K = 4608 and the 128x128 tiles with
// K = 1152 of VGG-16 have 1.89 * 10^7 each: with them in, BERT's drains of VGG-16 end within 48 us (p99) instead of
// 60, and a VGG-16 pass takes 4 % longer (those launches 13 %: the instantiation that looks runs its K-steps that
// much slower than the one that does not, although the two execute the same instructions per K-step to within a
// few scalar ones).  GPREEMPT_LONG_TILE_MACS overrides it.
inline bool tile_is_long(int bm, int bn, int K, int dtype) {
    static const double long_macs = [] { const char *e = getenv("GPREEMPT_LONG_TILE_MACS"); return e && atof(e) > 0 ? atof(e) : 1.8e7; }();
    return (double)bm * bn * K * (dtype == GP_F32 ? 8.0 : 1.0) >= long_macs;
}

template <typename T, int BM, int BN, int BK, int WGM, int WGN, bool CONV, bool B_KN>
using TK = TileKernel<T, BM, BN, BK, WGM, WGN, CONV, B_KN>;

template <class K> struct K_is_ckpt { static constexpr bool value = false; };
template <typename T, int BM, int BN, int ST, int CV, int W, bool PH> struct K_is_ckpt<PipeKernel<T, BM, BN, ST, CV, false, true, W, false, PH>> { static constexpr bool value = true; };
template <class K> struct KernelOf {
    static constexpr auto fn = mat_kernel<K, LOOP_ANY>;
    static constexpr auto plain = mat_kernel<K, LOOP_PLAIN>;
    static constexpr auto fixed = mat_kernel<K, LOOP_FIXED>;
#ifdef GP_NO_LOOKS  // (experiment switch: no instantiations that look more than once)
    static constexpr auto looks = fixed;
#else
    static constexpr auto looks = mat_kernel<K, K::can_look ? LOOP_LOOKS : LOOP_FIXED>;
#endif
};
template <typename T, int BM, int BN, int ST, int CV, int W, bool PH> struct KernelOf<PipeKernel<T, BM, BN, ST, CV, false, true, W, false, PH>> {
    static constexpr auto fn = mat_kernel_ckpt<PipeKernel<T, BM, BN, ST, CV, false, true, W, false, PH>>;
    static constexpr auto plain = fn;
    static constexpr auto fixed = fn;
    static constexpr auto looks = fn;
};

// bytes of checkpoint workspace a launch of body K needs (0: the body always finishes its tiles)
inline size_t ckpt_workspace_bytes(size_t slot_bytes, int workgroups) {
    return (size_t)CKPT_MAX_WGS * CKPT_HEADER_INTS * 4 + (size_t)workgroups * slot_bytes;
}

template <class K>
static int launch_mat(const MatPlan &pl, const gp_preempt_ctx *ctx, gp_stream s, gp_launch_info *info) {
    BlpArgs blp;
    int grid = 0;
    auto kern = KernelOf<K>::fn;  // the launch is planned for the general form; the others need no more resources
    constexpr int es = (int)sizeof(typename K::elem);
    const size_t lds_bytes = K::LDS_BYTES + (K::pre ? pre_table_bytes(pl.g.K, es) : 0) + (K::window ? window_bytes(pl.g, K::bm, es) : 0);
    constexpr size_t max_lds = K::pre ? pre_max_lds(K::LDS_BYTES) : K::window ? kWindowMaxLds : K::LDS_BYTES;
    if (max_lds > 48 * 1024) {
        // several tenant threads launch concurrently: the attribute is set by exactly one of them
        static std::once_flag once;
        static hipError_t once_rc = hipSuccess;
        std::call_once(once, [] {
            for (const void *f : {(const void *)KernelOf<K>::fn, (const void *)KernelOf<K>::plain, (const void *)KernelOf<K>::fixed, (const void *)KernelOf<K>::looks}) {
                hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)max_lds);
                if (e != hipSuccess) once_rc = e;
            }
        });
        GP_HIP(once_rc);
    }
    const bool long_tiles = K::can_look && tile_is_long(K::bm, K::bn, pl.g.K, pl.dtype);
    int rc = plan_launch(kern, K::NT, lds_bytes, pl.sx, pl.sy, pl.batch, ctx, &blp, &grid, info, 1, pl.rounds ? pl.rounds : K::LDS_BYTES <= 32 * 1024 ? 2 : K::LDS_BYTES <= 64 * 1024 ? 4 : 1, long_tiles);
    if (rc) return rc;
    if (pl.or_smaller && ctx && !blp.done) return kTileTooLong;
    if (pl.or_deeper && ctx && blp.done) {
        int per_cu = 0;
        rc = occupancy_of((const void *)kern, K::NT, lds_bytes, &per_cu);
        if (rc) return rc;
        if (front_costs_a_round(blp.total, (long)per_cu * device_cus())) return kFrontCostsARound;
    }
    blp.order = pl.order;
    if constexpr (K_is_ckpt<K>::value) {
        if (info) info->fixed_claims = 0;  // tile_loop_ckpt always claims through the counters
        if (blp.spare || blp.front) { grid -= blp.spare + blp.front; blp.grid = grid; blp.spare = blp.front = 0; blp.done = nullptr; set_poll_slices(&blp, grid); if (info) { info->grid = grid; info->front = 0; } }
        // mid-tile checkpoints need the caller's workspace and a slot per workgroup
        if (ctx && ctx->ckpt && ctx->ckpt_bytes >= ckpt_workspace_bytes(K::CKPT_SLOT_BYTES, grid) && grid <= CKPT_MAX_WGS) blp.ckpt = ctx->ckpt;
    }
    // one tile per claim here (plan_launch's default), which is what the two special forms assume
    if (!ctx) kern = KernelOf<K>::plain;
    else if (fixed_claims(true, blp.groups, grid - blp.front, blp.total)) kern = blp.done ? KernelOf<K>::looks : KernelOf<K>::fixed;  // (not for checkpointing bodies: theirs is fn)
    hipLaunchKernelGGL(kern, dim3(grid), dim3(K::NT), lds_bytes, native(s), pl.g, blp);
    GP_HIP(hipGetLastError());
    return GP_SUCC;
}

// ring depth per tile size (deeper rings were measured: no gain, lower occupancy)
#ifndef GP_S128
#define GP_S128 3
#endif
#ifndef GP_W256
#define GP_W256 8  // wavefronts of the 256 x 256 body
#endif
#ifndef GP_S64
#define GP_S64 4
#endif
#ifndef GP_S32
#define GP_S32 4
#endif
// The large-GEMM body.  Experiment switch GP_BIG_BM / GP_BIG_BN / GP_BIG_STAGES: another tile shape and ring depth
// for it (128 x 256 with three stages has a prefetch distance of two stages in 144 KB of LDS).
#ifndef GP_BIG_BM
#define GP_BIG_BM 256
#define GP_BIG_BN 256
#define GP_BIG_STAGES 2
#endif
template <typename T, bool CK, bool PHASED = false> using BigPipe = PipeKernel<T, GP_BIG_BM, GP_BIG_BN, GP_BIG_STAGES, false, false, CK, GP_W256, false, PHASED>;
// From which K on 16-bit tiles of 256 x 256 take a K-step in four phases.  Those fetch two K-steps ahead, and so two beyond the last one, and take
// longer to begin and to end.  Stage by stage -> in phases, f16, us, plain: 8192 x 8192 x 256 81.9 -> 88.5, x 512 107.3 -> 110.7, x 896 148.8 -> 150.1, x 1024
// 161.1 -> 162.0, x 2048 266.5 -> 264.6, x 8192 928 -> 894; 2600 x 8000 x 640 50.8 -> 51.1, x 1024 67.0 -> 66.1; with claim counters 5000 x 6000 x 512 61.5 -> 63.0, x 1024
// 85.7 -> 86.1, x 2048 138.4 -> 137.3; 4096 x 4096 x 256 24.9 -> 25.1, x 1024 44.3 -> 43.8.  Later with checkpoints, where more of a tile's state goes through scratch memory
// around the loop: 8192 x 8192 x 256 95.6 -> 109.5, x 1280 209.1 -> 210.3, x 1792 268.5 -> 265.8, x 2560 358.8 -> 350.8; 4096 x 4096 x 1024 54.4 -> 56.2,
// x 1792 77.0 -> 77.4, x 4096 144.1 -> 140.6.
constexpr int kPhasedK = 1024, kPhasedCkptK = 1792;
template <typename T, int TILE, int STAGES, bool SPLITK>
static int pipe_case(const MatPlan &pl, const gp_preempt_ctx *ctx, gp_stream s, gp_launch_info *info) {
    if constexpr (TILE == 64 && !SPLITK)
        if (pl.pre) return launch_mat<PipeKernel<T, TILE, TILE, STAGES, 0, false, false, 4, true>>(pl, ctx, s, info);
    if constexpr (sizeof(T) == 2 && TILE == 64 && STAGES == 2) {
        if (pl.tall && pl.taps) return launch_mat<PipeKernel<T, 128, 64, 2, 2, false>>(pl, ctx, s, info);
        if (pl.tall) return launch_mat<PipeKernel<T, 128, 64, 2, 3, false>>(pl, ctx, s, info);
    }
    if constexpr (sizeof(T) == 2)
        if (pl.taps) return launch_mat<PipeKernel<T, TILE, TILE, STAGES, 2, SPLITK>>(pl, ctx, s, info);
    if constexpr (TILE >= 64 && !SPLITK)
        if (pl.straddles) return launch_mat<PipeKernel<T, TILE, TILE, STAGES, 3, false>>(pl, ctx, s, info);
    if (pl.conv) return launch_mat<PipeKernel<T, TILE, TILE, STAGES, 1, SPLITK>>(pl, ctx, s, info);
    return launch_mat<PipeKernel<T, TILE, TILE, STAGES, 0, SPLITK>>(pl, ctx, s, info);
}
size_t plan_ckpt_bytes(const MatPlan &pl);  // gemm.hip
// the instantiation that can leave a tile between two K-steps, when the caller brought a workspace big enough for it
template <typename T, int TILE, int STAGES>
static int pipe_case_ckpt(const MatPlan &pl, const gp_preempt_ctx *ctx, gp_stream s, gp_launch_info *info) {
    if (!(ctx && ctx->ckpt && ctx->ckpt_bytes >= plan_ckpt_bytes(pl))) return pipe_case<T, TILE, STAGES, false>(pl, ctx, s, info);
    if constexpr (sizeof(T) == 2)
        if (pl.taps) return launch_mat<PipeKernel<T, TILE, TILE, STAGES, 2, false, true>>(pl, ctx, s, info);
    if (pl.conv) return launch_mat<PipeKernel<T, TILE, TILE, STAGES, 1, false, true>>(pl, ctx, s, info);
    return launch_mat<PipeKernel<T, TILE, TILE, STAGES, 0, false, true>>(pl, ctx, s, info);
}

// Ring depth of a wide body: three stages, four for the GEMM form of the 32 x 32 tile on 16 wavefronts (a
// stage is (WAVES / 4) K-blocks of BM + BN rows of 128 bytes: 32 KB there).  128 x 768 x 3072 went from
// 7.96 to 7.67 us per launch with the fourth stage; given to every body that has room for it, it cost the
// convolution chain of ResNet-152 1 us per launch (10.2 -> 11.2), and so did two stages instead of three for
// the convolution form (10.05 -> 10.98).
constexpr int wide_stages(int bm, int bn, int waves, bool conv) { return (!conv && bm == 32 && bn == 32 && waves == 16) ? 4 : 3; }
template <typename T, int BM, int BN, int WAVES, int CONV = 0>
using WideK = WideKernel<T, BM, BN, WAVES, wide_stages(BM, BN, WAVES, CONV != 0), CONV>;

template <typename T, int BM, int BN, int WAVES>
static int wide_case(const MatPlan &pl, const gp_preempt_ctx *ctx, gp_stream s, gp_launch_info *info) {
    if constexpr (sizeof(T) == 2 && BM == 32 && WAVES == 16)
        if (pl.window) return launch_mat<WindowKernel<T, BM, BN, 4>>(pl, ctx, s, info);
    if (pl.pre) return launch_mat<WideKernel<T, BM, BN, WAVES, wide_stages(BM, BN, WAVES, false), 0, true>>(pl, ctx, s, info);
    if (pl.conv && straddles_taps<T>(pl)) return launch_mat<WideK<T, BM, BN, WAVES, 2>>(pl, ctx, s, info);
    if (pl.conv) return launch_mat<WideK<T, BM, BN, WAVES, 1>>(pl, ctx, s, info);
    return launch_mat<WideK<T, BM, BN, WAVES, 0>>(pl, ctx, s, info);
}

template <int BM>
static int narrow_case(const MatPlan &pl, const gp_preempt_ctx *ctx, gp_stream s, gp_launch_info *info) {
    if (pl.pre) return launch_mat<NarrowKernel<BM, 3, 0, true>>(pl, ctx, s, info);
    if (pl.conv && straddles_taps<float>(pl)) return launch_mat<NarrowKernel<BM, 3, 2>>(pl, ctx, s, info);
    if (pl.conv) return launch_mat<NarrowKernel<BM, 3, 1>>(pl, ctx, s, info);
    return launch_mat<NarrowKernel<BM, 3, 0>>(pl, ctx, s, info);
}

template <typename T>
int launch_typed(const MatPlan &pl, const gp_preempt_ctx *ctx, gp_stream s, gp_launch_info *info) {
    constexpr int SBK = sizeof(T) == 4 ? 16 : 32;
    switch (pl.body) {
        case MB_PIPE256:  // GEMM only: the gathered A operand of a convolution does not fit its register budget
            if constexpr (sizeof(T) == 2) {
                if (pl.near && ctx && ctx->ckpt && pl.g.K >= kPhasedCkptK) return launch_mat<BigPipe<T, true, true>>(pl, ctx, s, info);
                if (pl.near && !(ctx && ctx->ckpt) && pl.g.K >= kPhasedK) return launch_mat<BigPipe<T, false, true>>(pl, ctx, s, info);
            }
            if (ctx && ctx->ckpt) return launch_mat<BigPipe<T, true>>(pl, ctx, s, info);
            return launch_mat<BigPipe<T, false>>(pl, ctx, s, info);
        // The depth of the ring decides how many workgroups a compute unit holds (160 KB of LDS).  A launch that gives it
        // more workgroups than fit with the deep ring is better off with two stages and twice the workgroups: one's
        // prologue, barriers and epilogue hide under the others' MFMAs.  Launch to launch, fp16, deep -> two stages:
        // 128 x 128: 3 x 3 at 56 x 56 x 256 batch 16 126 -> 83 us, at 28 x 28 x 512 110 -> 75; 64 x 64: at 224 x 224 x 64
        // 176 -> 119 us, 4096 x 1024 x 1024 17.3 -> 14.6.  A launch that fits at once keeps the depth: 3 x 3 at 14 x 14 x
        // 512 (392 tiles of 64 x 64) 33 us against 44, 2048^3 (256 of 128 x 128) 25 against 33 (choose_body has the line).
        // fp32 the same way: 3 x 3 at 56 x 56 x 256 650 -> 591 us, at 28 x 28 x 512 634 -> 586, at 224 x 224 x 64 batch 4 176 ->
        // 150 preemptible, 4096 x 2048 x 1024 150 -> 138.  Not where tiles fill the device to the last place and a
        // preemptible launch's front workgroup makes a round for one of them: 4096 x 2048 x 2048, 512 tiles, 77 us for 62 in fp16 and 344 for
        // 289 in fp32.
        case MB_PIPE128:
            if (pl.ring == 2 && !(ctx && ctx->ckpt && ctx->ckpt_bytes >= plan_ckpt_bytes(pl))) {
                MatPlan shallow = pl;
                shallow.or_deeper = true;
                const int rc = pipe_case<T, 128, 2, false>(shallow, ctx, s, info);
                if (rc != kFrontCostsARound) return rc;
            }
            return pipe_case_ckpt<T, 128, GP_S128>(pl, ctx, s, info);
        case MB_PIPE64:
            // A layer of at most four K-steps is all prologue and epilogue: two stages for any number of tiles.
            // 25088 x 256 x 64 with a residual (ResNet-152 b8, 56 x 56): 15.5 -> 10.7 us plain, 19.4 -> 13.6 us
            // preemptible; 6272 x 512 x 128: 10.0 -> 7.6 us.
            if (pl.ring == 2 || pl.g.K <= 256) return pipe_case<T, 64, 2, false>(pl, ctx, s, info);
            return pipe_case<T, 64, GP_S64, false>(pl, ctx, s, info);
        case MB_PIPE64_SK: return pipe_case<T, 64, GP_S64, true>(pl, ctx, s, info);
        case MB_PIPE32_SK: return pipe_case<T, 32, GP_S32, true>(pl, ctx, s, info);
        case MB_WIDE32x32_16: return wide_case<T, 32, 32, 16>(pl, ctx, s, info);
        case MB_WIDE32x32_8: return wide_case<T, 32, 32, 8>(pl, ctx, s, info);
        case MB_WIDE64x32_16: return wide_case<T, 64, 32, 16>(pl, ctx, s, info);
        case MB_WIDE64x64_8: return wide_case<T, 64, 64, 8>(pl, ctx, s, info);
        case MB_NARROW16x16:
            if constexpr (sizeof(T) == 4) return narrow_case<16>(pl, ctx, s, info);
            break;
        case MB_NARROW32x16:
            if constexpr (sizeof(T) == 4) return narrow_case<32>(pl, ctx, s, info);
            break;
        case MB_LNWIDE32x64_16:
            if constexpr (sizeof(T) == 2) return launch_mat<LnWideKernel<T, 32, 64, 16, 3>>(pl, ctx, s, info);
            break;
        case MB_STAGED128:
            if (pl.conv) return launch_mat<TK<T, 128, 128, SBK, 2, 2, true, false>>(pl, ctx, s, info);
            return pl.b_kn ? launch_mat<TK<T, 128, 128, SBK, 2, 2, false, true>>(pl, ctx, s, info)
                           : launch_mat<TK<T, 128, 128, SBK, 2, 2, false, false>>(pl, ctx, s, info);
        case MB_STAGED64:
            if (pl.conv) return launch_mat<TK<T, 64, 64, SBK, 2, 2, true, false>>(pl, ctx, s, info);
            return pl.b_kn ? launch_mat<TK<T, 64, 64, SBK, 2, 2, false, true>>(pl, ctx, s, info)
                           : launch_mat<TK<T, 64, 64, SBK, 2, 2, false, false>>(pl, ctx, s, info);
    }
    set_error("unknown matrix kernel body %d", pl.body);
    return GP_FAIL;
}

template <typename T>
int launch_group_typed(const MatPlan *pl, int n, const gp_preempt_ctx *ctx, gp_stream s, gp_launch_info *info) {
    if constexpr (sizeof(T) == 4) {
        if (pl[0].body == MB_NARROW16x16) return launch_group<NarrowKernel<16, 3, 0>, NarrowKernel<16, 3, 1>, NarrowKernel<16, 3, 2>>(pl, n, ctx, s, info);
    } else {
        if (pl[0].body == MB_WIDE32x32_16) return launch_group<WideK<T, 32, 32, 16, 0>, WideK<T, 32, 32, 16, 1>, WideK<T, 32, 32, 16, 2>, WindowKernel<T, 32, 32, 4>>(pl, n, ctx, s, info);
    }
    set_error("matrix kernel body %d does not run in groups", pl[0].body);
    return GP_FAIL;
}

}  // namespace gp
