// Preemptible GEMM and implicit-GEMM convolution on the gfx950 matrix cores.
//
// One workgroup owns one BM x BN output tile for the whole K range and walks K in a fixed
// order with fp32 accumulation, so the value of a tile does not depend on which workgroup or
// which launch computes it: a preempted-then-resumed run is bit-identical to an uninterrupted
// one.  Tiles are handed out by gp::tile_loop (tile_loop.hpp).
//
// Data movement: both operands are staged K-contiguous in LDS ([rows][BK + pad]) with 16-byte
// global loads that are issued one K-step ahead of the MFMAs (register prefetch).  A lane feeds
// v_mfma_f32_32x32x16_{f16,bf16} with one 16-byte LDS read per operand; for fp32 the same
// 16-byte read feeds four v_mfma_f32_32x32x2_f32 (K is consumed in a permuted but fixed order).
//
// The convolution is the same main loop with a gathered A operand: row m is output pixel
// (n, ho, wo) and column k is (r, s, ci) of an NHWC input, zero-filled outside the image.
#include <algorithm>
#include "gemm_launch.hpp"

namespace gp {

extern template int launch_typed<float>(const MatPlan &, const gp_preempt_ctx *, gp_stream, gp_launch_info *);
extern template int launch_typed<_Float16>(const MatPlan &, const gp_preempt_ctx *, gp_stream, gp_launch_info *);
extern template int launch_typed<__bf16>(const MatPlan &, const gp_preempt_ctx *, gp_stream, gp_launch_info *);

extern template int launch_group_typed<float>(const MatPlan *, int, const gp_preempt_ctx *, gp_stream, gp_launch_info *);
extern template int launch_group_typed<_Float16>(const MatPlan *, int, const gp_preempt_ctx *, gp_stream, gp_launch_info *);
extern template int launch_group_typed<__bf16>(const MatPlan *, int, const gp_preempt_ctx *, gp_stream, gp_launch_info *);

int launch_mat_plan(const MatPlan &pl, const gp_preempt_ctx *ctx, gp_stream s, gp_launch_info *info) {
    switch (pl.dtype) {
        case GP_F32: return launch_typed<float>(pl, ctx, s, info);
        case GP_F16: return launch_typed<_Float16>(pl, ctx, s, info);
        case GP_BF16: return launch_typed<__bf16>(pl, ctx, s, info);
    }
    set_error("unsupported dtype %d for matrix kernels", pl.dtype);
    return GP_OUTOFRANGE;
}

static size_t body_lds_bytes(int body, int dtype) {
    const size_t es = dtype == GP_F32 ? 4 : 2;
    switch (body) {
        case MB_PIPE256: return BigPipe<_Float16, false>::LDS_BYTES;
        case MB_PIPE128: return GP_S128 * (128 + 128) * 128;
        case MB_PIPE64: return GP_S64 * (64 + 64) * 128;
        case MB_PIPE64_SK: return GP_S64 * (64 + 64) * 128;   // at least the reduction buffer (4 waves x 4 blocks x 16 x 64 x 4 = 64 KB)
        case MB_PIPE32_SK: return GP_S32 * (32 + 32) * 128;
        case MB_WIDE32x32_16: return WideK<_Float16, 32, 32, 16>::LDS_BYTES;
        case MB_WIDE32x32_8: return WideK<_Float16, 32, 32, 8>::LDS_BYTES;
        case MB_WIDE64x32_16: return WideK<_Float16, 64, 32, 16>::LDS_BYTES;
        case MB_WIDE64x64_8: return WideK<_Float16, 64, 64, 8>::LDS_BYTES;
        case MB_NARROW16x16: return NarrowKernel<16, 3>::LDS_BYTES;
        case MB_NARROW32x16: return NarrowKernel<32, 3>::LDS_BYTES;
        case MB_LNWIDE32x64_16: return LnWideKernel<_Float16, 32, 64, 16, 3>::LDS_BYTES;
        case MB_STAGED128: return (128 + 128) * ((es == 4 ? 16 : 32) + (es == 4 ? 4 : 8)) * es;
        case MB_STAGED64: return (64 + 64) * ((es == 4 ? 16 : 32) + (es == 4 ? 4 : 8)) * es;
    }
    return 0;
}

// Kernel and tile choice.  B stored K x N needs the transposing, register-staged kernel.
// Otherwise the pipelined kernel is used with the largest tile that still gives every compute
// unit work; problems too small for that split K across the waves of a workgroup so that the
// serial K loop shrinks instead.
// the wide split-K bodies (gemm_wide.hpp) and their tiles
struct WideChoice { int body, bm, bn, waves; size_t lds; };
static const WideChoice kWide[6] = {
    {MB_NARROW16x16, 16, 16, 16, NarrowKernel<16, 3>::LDS_BYTES},
    {MB_NARROW32x16, 32, 16, 16, NarrowKernel<32, 3>::LDS_BYTES},
    {MB_WIDE32x32_16, 32, 32, 16, WideK<_Float16, 32, 32, 16>::LDS_BYTES},
    {MB_WIDE32x32_8, 32, 32, 8, WideK<_Float16, 32, 32, 8>::LDS_BYTES},
    {MB_WIDE64x32_16, 64, 32, 16, WideK<_Float16, 64, 32, 16>::LDS_BYTES},
    {MB_WIDE64x64_8, 64, 64, 8, WideK<_Float16, 64, 64, 8>::LDS_BYTES}};
static const WideChoice *wide_of(int body) {
    for (const WideChoice &w : kWide) if (w.body == body) return &w;
    return nullptr;
}
// Which wide body, if any: measured on MI355X (launch to launch, fp16, against the best of the
// four-wavefront bodies): they win where one round of workgroups covers the problem and K is deep
// enough to pay for the larger first stage.  128 x 768 x 3072: 10.2 -> 7.9 us; 392 x 512 x 4608:
// 14.0 -> 10.4; 1568 x 256 x 2304: 10.0 -> 8.3; 1568 x 256 x 1024: 6.6 -> 6.1; 128 x 768 x 768: 5.1 -> 4.7;
// 6272 x 128 x 1152: 8.9 -> 8.0; 392 x 2048 x 512: 6.4 -> 5.9.
static int wide_pick(const MatArgs &g, int batch, long cus, int dtype) {
    auto tiles = [&](int tm, int tn) { return (long)((g.M + tm - 1) / tm) * ((g.N + tn - 1) / tn) * batch; };
    // fp32 runs on MFMAs an eighth as fast, so a small layer is bound by them and not by its operands: as many
    // tiles as there are compute units to take them (ResNet-50 b1 fp32, launch to launch: 7 x 7 x 512 -> 2048
    // 13.1 -> 6.7 us, 3 x 3 at 56 x 56 x 64 16.2 -> 9.1 us; these tiles are also what a preempted tenant
    // finishes before it leaves)
    // (deep ones in tiles of a quarter and a half while those still run side by side, gemm_narrow.hpp: ResNet-50 b1 735 -> 584 us a pass,
    // DenseNet-201 b1 2458 -> 1907, Inception-v3 b2 1303 -> 1130, BERT b1 s64 871 -> 758; K from 128 or 256 on: level)
    if (dtype == GP_F32 && g.K >= 512 && tiles(16, 16) <= cus) return MB_NARROW16x16;
    if (dtype == GP_F32 && g.K >= 512 && tiles(32, 16) <= cus) return MB_NARROW32x16;
    if (dtype == GP_F32 && tiles(32, 32) <= cus) return g.K >= 768 ? MB_WIDE32x32_16 : MB_WIDE32x32_8;
    if (g.K >= 768 && tiles(32, 32) <= cus) return MB_WIDE32x32_16;
    if (g.K >= 768 && tiles(64, 32) <= cus) return MB_WIDE64x32_16;
    if (g.K >= 512 && tiles(64, 64) <= cus && g.N > 32) return MB_WIDE64x64_8;
    return -1;
}

// The wide bodies address their operands by 32-bit offsets in buffers of 2 GB.  (Beyond, the four-wavefront split-K bodies
// of gemm_pipe.hpp stand in for them: pointers of 64 bits, the same sums in the same order.)
static bool buffer_ok(const MatArgs &g, bool conv, int dtype) {
    const double limit = 2147483648.0 / (double)dtype_size(dtype);
    const double pixels = conv ? (double)(g.M / ((long)g.Ho * g.Wo)) * g.H * g.W + (double)(g.ph + g.K / (g.Cin * g.S)) * (g.W + g.S) : (double)g.M;
    return pixels * g.lda + g.K < limit && (double)g.N * g.ldb + g.K < limit;
}

static int choose_body(MatPlan *pl, int tile, int tile_n, int variant) {
    const MatArgs &g = pl->g;
    auto tiles = [&](int t) { return (long)((g.M + t - 1) / t) * ((g.N + t - 1) / t) * pl->batch; };
    const long cus = device_cus();
    // both operands K-contiguous; a convolution, whose A operand is gathered, when a bit per tap fits a word and, where K-blocks
    // straddle two filter taps, a lane can find its tap by multiplication (inverse_of is 0 from (K + 1) * Cin = 2^32 on)
    const int wide_bk = pl->dtype == GP_F32 ? 32 : 64;
    const bool whole_taps = pl->conv && g.Cin % wide_bk == 0;
    const bool wide_taps = !pl->conv || (g.K / g.Cin <= 32 && g.S < 32 && (whole_taps || (g.inv_cin && g.inv_s)));
    // (a caller that asks for a wide body gets one only where no block straddles two taps, as ever)
    const bool wide_shape = !pl->b_kn && wide_taps && (!pl->conv || whole_taps);
    const bool wide_ok = !pl->b_kn && wide_taps && buffer_ok(g, pl->conv, pl->dtype);
    int body = -1;
    if (g.ln_gamma) body = MB_LNWIDE32x64_16;  // (plan_gemm has checked that the shape fits)
    else if (pl->b_kn || variant == GP_MAT_STAGED) {
        int tm = tile ? tile : (tiles(128) >= cus ? 128 : 64);
        body = tm == 128 ? MB_STAGED128 : tm == 64 ? MB_STAGED64 : -1;
    } else if (variant == GP_MAT_PIPE) {
        int tm = tile ? tile : (tiles(128) >= cus ? 128 : 64);
        body = (tm == 256 && !pl->conv) ? MB_PIPE256 : tm == 128 ? MB_PIPE128 : tm == 64 ? MB_PIPE64 : -1;
    } else if (variant == GP_MAT_PIPE_SPLITK) {
        int tm = tile ? tile : (tiles(64) >= cus / 2 ? 64 : 32);
        body = tm == 64 ? MB_PIPE64_SK : tm == 32 ? MB_PIPE32_SK : -1;
    } else if (variant == GP_MAT_WIDE || variant == GP_MAT_WIDE8) {
        if (wide_shape) {
            const int tn = tile_n ? tile_n : tile;
            if (tile == 32 && tn == 32) body = !wide_ok ? MB_PIPE32_SK : variant == GP_MAT_WIDE ? MB_WIDE32x32_16 : MB_WIDE32x32_8;
            else if (tile == 64 && tn == 32) body = wide_ok ? MB_WIDE64x32_16 : MB_PIPE32_SK;
            else if (tile == 64 && tn == 64) body = wide_ok ? MB_WIDE64x64_8 : MB_PIPE64_SK;
        }
    } else if (variant == GP_MAT_AUTO) {
        // a tile wider than the problem multiplies zero columns: N <= 64 never takes the larger tiles
        if (!pl->conv && (tile == 256 || (tile == 0 && tiles(256) >= cus && g.N > 128 && g.M > 128))) body = MB_PIPE256;
        // (a problem of one or two K-steps is all epilogue, i.e. memory-bound: the 128 x 128 body runs one or two
        // workgroups per CU, too few threads for that; 25088 x 256 x 64 with a residual: 19.8 us on 128 x 128, 15.0 on 64 x 64)
        // (... and with hardly more tiles than compute units a shallow one is better cut into tiles of 64 x 64, several
        // to a compute unit: 4096 x 1024 x 1024 17.1 -> 14.6 us; 2048^3 25.4 on 128 x 128, 26.2 on 64 x 64; in fp32
        // 5000 x 1000 x 768 105 -> 78, 3000 x 1500 x 256 42 -> 30, 4096 x 1024 x 1024 77 -> 81 but 149 -> 101 preemptible)
        else if (tile == 128 || (tile == 0 && tiles(128) >= (g.K <= 1024 ? cus + cus / 2 : cus) && g.N > 64 && g.M > 64 && g.K > 128)) body = MB_PIPE128;
        else if (tile == 0 && wide_ok && wide_pick(g, pl->batch, cus, pl->dtype) >= 0) body = wide_pick(g, pl->batch, cus, pl->dtype);
        else if (tile == 64 || (tile == 0 && (tiles(64) >= cus || g.K < 512))) body = MB_PIPE64;
        else if (tile == 0 && tiles(64) >= cus / 2) body = MB_PIPE64_SK;
        else if (tile == 0 || tile == 32) body = MB_PIPE32_SK;
    }
    if (body < 0) {
        set_error("no matrix kernel for tile %d x %d with variant %d (tiles: 256, 128, 64; 64, 32 with split K; wide: 32x32, 64x32, 64x64, N x K operands; convolutions with Cin a multiple of the K-block and at most 32 taps)", tile, tile_n ? tile_n : tile, variant);
        return GP_OUTOFRANGE;
    }
    // (the phases of the 16-bit body of 256 x 256 have no registers left for addresses of 64 bits)
    pl->near = body == MB_PIPE256 && pl->dtype != GP_F32 && 256.0 * (double)std::max(g.lda, g.ldb) + g.K < 1073741823.0;
    int t = body == MB_PIPE256 ? GP_BIG_BM : (body == MB_PIPE128 || body == MB_STAGED128) ? 128 : (body == MB_PIPE32_SK ? 32 : 64);
    int tn = body == MB_PIPE256 ? GP_BIG_BN : t;
    if (const WideChoice *w = wide_of(body)) { t = w->bm; tn = w->bn; }
    if (body == MB_LNWIDE32x64_16) { t = 32; tn = 64; }
    pl->body = body;
    pl->sx = (g.N + tn - 1) / tn;
    pl->sy = (g.M + t - 1) / t;
    pl->lds_bytes = body_lds_bytes(body, pl->dtype);
    // (what the 16-bit pipelined bodies' form for whole taps assumes)
    pl->taps = whole_taps && pl->dtype != GP_F32 && wide_ok;
    // (... and their form for K-steps that straddle taps: inverses, and factors of 24 bits)
    pl->straddles = pl->conv && !whole_taps && g.inv_cin && g.inv_s && g.K + 64 < (1 << 24) && (double)(g.R + 64) * g.W < 16777216.0 && buffer_ok(g, true, pl->dtype);
    // A convolution whose tiles' input windows are runs of consecutive pixels that fit in LDS fetches them once (gemm_window.hpp; where the
    // launcher picks the body itself; 16-bit, fp32 being bound by its arithmetic; 32 x 32 tiles: with 64 x 32 the four multiplying wavefronts,
    // which work out where a lane's row lies, are what a stage waits for, 0.76 us for the gather's 0.53, ResNet-152 b8 1530 -> 1560).
    pl->window = pl->conv && variant == GP_MAT_AUTO && tile == 0 && pl->dtype != GP_F32 && body == MB_WIDE32x32_16 && g.Cin % 64 == 0 && g.sh == 1 && g.sw == 1 &&
                 g.Ho == g.H && g.Wo == g.W && WindowKernel<_Float16, 32, 32, 4>::LDS_BYTES + window_bytes(g, 32, 2) <= kWindowMaxLds;
    // (a caller that names the tile gets that body at its own depth)
    if (tile == 0 && variant == GP_MAT_AUTO && ((body == MB_PIPE128 && tiles(128) > cus) || (body == MB_PIPE64 && tiles(64) > 2 * cus))) pl->ring = 2;
    // Tiles of a few microseconds: claimed through the counters, a tile waits 1-2 us for its claim, and the kernel around
    // the general loop fits a compute unit three times where the others fit four or five times.  With a workgroup per claim a 3 x 3 layer
    // of 12544 tiles at 224 x 224 x 64, seventeen rounds of them, takes 152 us instead of 182 (plain launch 136); behind
    // a stop its workgroups still have to start and leave, about a microsecond per thousand.  (fp32, whose tiles take eight times as long and
    // wait no longer: 3136 tiles there 150 us either way.)
    if (tile == 0 && variant == GP_MAT_AUTO && body == MB_PIPE64 && g.K <= 640) pl->rounds = 20;
    // Layers of at most 64 channels over many pixels (the first ones of a VGG) in tiles of 128 x 64: half the workgroups, each of which takes about as
    // long from its claim to its first operands and from its last to its store, and half the weights through LDS.  Preemptible, fp16, batch 16 at
    // 224 x 224: 8 -> 64 channels 75 -> 65 us, 64 -> 64 138 -> 120; batch 8 72 -> 64.  From sixteen tiles of 64 x 64 to a compute unit on: batch 4,
    // twelve, is level.  (bf16 125 -> 109; plain, f16 and bf16: 64 -> 64 115 -> 103 and 111 -> 100, batch 8 60 -> 56 and 56 -> 55.)
    if (pl->ring == 2 && body == MB_PIPE64 && pl->dtype != GP_F32 && (pl->taps || pl->straddles) && g.N > 32 && g.N <= 64 && g.K <= 640 && tiles(64) >= 16 * cus) {
        pl->tall = true;
        pl->sy = (g.M + 127) / 128;
    }
    // Each XCD works on a contiguous eighth of the tile order (util/slice_map.h).  With x fastest
    // that is a band of tile rows: every XCD fetches its share of A and all of B; with y fastest
    // it is a band of tile columns: all of A and a share of B.  Take the cheaper one.
    const double a_elems = pl->conv ? (double)(g.M / (g.Ho * g.Wo > 0 ? g.Ho * g.Wo : 1)) * g.H * g.W * g.Cin : (double)g.M * g.K;
    const double b_elems = (double)g.N * g.K;
    pl->order = b_elems > a_elems ? 1 : 0;
    // Large GEMMs on the 256 x 256 tiles: an XCD runs 32 of them side by side, and a single tile row
    // with 32 column panels means 33 distinct operand panels streaming through its 4 MB L2; taken
    // as bands of two tile rows it is 18.  Measured at 8192^3 bf16, plain launches: constant
    // operands 889 -> 718 us, U[-1,1) operands 956 -> 928 us (those are bounded by power, see the
    // profile of this kernel); bands of 4, 8 and 16 rows were level or worse.
    if (!pl->conv && body == MB_PIPE256 && pl->sx >= 16 && pl->sy >= 16) pl->order = 2;
    return GP_SUCC;
}

static bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

// shapes the layer-norm prologue body takes (the tile count bounds how often a row is re-normalised)
static bool ln_shape_ok(const gp_gemm_params *p) {
    if (!p || (p->dtype != GP_F16 && p->dtype != GP_BF16) || p->batch > 1 || !p->b_is_nk) return false;
    if (p->M <= 0 || p->N <= 0 || p->K <= 0 || p->lda != p->K || p->K % 64 != 0 || p->K > LnWideKernel<_Float16, 32, 64, 16, 3>::MAXK) return false;
    // one round of workgroups: every workgroup normalises its own 32 rows, which pays while that hides
    // behind the fetch of B and not when a compute unit does it twice
    const long tiles = (long)((p->M + 31) / 32) * ((p->N + 63) / 64);
    return tiles <= device_cus() && (double)p->ldb < 16777216.0;  // (a tile's 64 rows of B in a buffer of 2 GB)
}
int plan_gemm(const gp_gemm_params *p, MatPlan *out);
// ... and the body the launcher would pick for the plain GEMM sums K in the prologue body's order (K-steps
// dealt to four wavefronts, partial tiles added in wavefront order), so that fusing changes no bit
extern "C" int gp_gemm_ln_supported(const gp_gemm_params *p) {
    if (!ln_shape_ok(p)) return 0;
    gp_gemm_params q = *p;
    q.ln_gamma = q.ln_beta = nullptr; q.ln_out = nullptr;
    q.tile_m = q.tile_n = q.variant = 0;
    MatPlan pl;
    KeepLastError keep;
    if (!q.A || !q.B || !q.C || plan_gemm(&q, &pl) != GP_SUCC) return 0;
    return (is_wide_body(pl.body) || pl.body == MB_PIPE64_SK || pl.body == MB_PIPE32_SK) ? 1 : 0;
}

int plan_gemm(const gp_gemm_params *p, MatPlan *out) {
    GP_REQUIRE(p != nullptr, "null gemm params");
    GP_REQUIRE(p->dtype == GP_F32 || p->dtype == GP_F16 || p->dtype == GP_BF16, "gemm dtype %d", p->dtype);
    const int vec = p->dtype == GP_F32 ? 4 : 8;
    GP_REQUIRE(p->M > 0 && p->N > 0 && p->K > 0, "gemm shape %dx%dx%d", p->M, p->N, p->K);
    GP_REQUIRE(p->A && p->B && p->C, "gemm needs A, B and C");
    GP_REQUIRE(p->K % vec == 0 && p->lda % vec == 0 && p->ldb % vec == 0, "gemm: K, lda, ldb must be multiples of %d elements", vec);
    GP_REQUIRE(!p->b_is_nk ? (p->N % vec == 0) : true, "gemm: N must be a multiple of %d when B is K x N", vec);
    GP_REQUIRE(aligned16(p->A) && aligned16(p->B), "gemm: A and B must be 16-byte aligned");
    const int batch = p->batch > 0 ? p->batch : 1;
    if (batch > 1) {
        GP_REQUIRE(p->stride_a % vec == 0 && p->stride_b % vec == 0, "gemm: batch strides of A and B must be multiples of %d elements", vec);
        if (p->batch_inner > 0)
            GP_REQUIRE(p->stride_a_outer % vec == 0 && p->stride_b_outer % vec == 0, "gemm: outer batch strides must be multiples of %d elements", vec);
    }
    GP_REQUIRE(p->lda >= p->K && p->ldc >= p->N && p->ldb >= (p->b_is_nk ? p->K : p->N), "gemm: leading dimension smaller than the row");
    GP_REQUIRE(p->tile_m == p->tile_n || p->variant == GP_MAT_WIDE || p->variant == GP_MAT_WIDE8, "gemm: square tiles only (the wide variants also take 64 x 32)");
    MatPlan &pl = *out;
    pl = MatPlan{};
    MatArgs &g = pl.g;
    g.M = p->M; g.N = p->N; g.K = p->K;
    g.A = p->A; g.lda = p->lda; g.stride_a = p->stride_a; g.stride_a_outer = p->stride_a_outer;
    g.B = p->B; g.ldb = p->ldb; g.stride_b = p->stride_b; g.stride_b_outer = p->stride_b_outer;
    g.C = p->C; g.ldc = p->ldc; g.stride_c = p->stride_c; g.stride_c_outer = p->stride_c_outer;
    g.bias = p->bias; g.residual = p->residual; g.ldr = p->ldc;
    g.alpha = p->alpha == 0.f ? 1.f : p->alpha;
    g.act = p->act; g.batch_inner = batch > 1 ? p->batch_inner : 0;
    pl.dtype = p->dtype; pl.conv = 0; pl.b_kn = !p->b_is_nk; pl.batch = batch;
    if (p->ln_gamma) {
        GP_REQUIRE(ln_shape_ok(p), "gemm: no layer-norm prologue for this shape (16-bit, batch 1, B as N x K, lda == K, K a multiple of 64 up to %d)", LnWideKernel<_Float16, 32, 64, 16, 3>::MAXK);
        GP_REQUIRE(p->ln_beta && p->ln_out, "gemm: the layer-norm prologue needs gamma, beta and ln_out");
        GP_REQUIRE(aligned16(p->ln_gamma) && aligned16(p->ln_beta) && aligned16(p->ln_out), "gemm: ln_gamma, ln_beta and ln_out must be 16-byte aligned");
        g.ln_gamma = p->ln_gamma; g.ln_beta = p->ln_beta; g.ln_out = p->ln_out; g.ln_eps = p->ln_eps;
    }
    return choose_body(&pl, p->tile_m, p->tile_n, p->variant);
}

int plan_conv2d(const gp_conv_params *p, MatPlan *out) {
    GP_REQUIRE(p != nullptr, "null conv params");
    GP_REQUIRE(p->dtype == GP_F32 || p->dtype == GP_F16 || p->dtype == GP_BF16, "conv dtype %d", p->dtype);
    const int vec = p->dtype == GP_F32 ? 4 : 8;
    GP_REQUIRE(p->N > 0 && p->H > 0 && p->W > 0 && p->Cin > 0 && p->Cout > 0 && p->R > 0 && p->S > 0, "conv shape");
    GP_REQUIRE(p->stride_h > 0 && p->stride_w > 0 && p->pad_h >= 0 && p->pad_w >= 0, "conv stride/pad");
    GP_REQUIRE(p->Cin % vec == 0, "conv: Cin must be a multiple of %d (pad the channels)", vec);
    GP_REQUIRE(p->in && p->weight && p->out, "conv needs in, weight and out");
    GP_REQUIRE(p->in_pix_stride >= p->Cin && p->in_pix_stride % vec == 0, "conv: input pixel stride");
    GP_REQUIRE(p->out_pix_stride >= p->Cout, "conv: output pixel stride");
    GP_REQUIRE(aligned16(p->in) && aligned16(p->weight), "conv: in and weight must be 16-byte aligned");
    int Ho = (p->H + 2 * p->pad_h - p->R) / p->stride_h + 1, Wo = (p->W + 2 * p->pad_w - p->S) / p->stride_w + 1;
    GP_REQUIRE(Ho > 0 && Wo > 0, "conv: empty output");
    long M = (long)p->N * Ho * Wo;
    GP_REQUIRE(M < (1L << 31), "conv: too many output pixels");
    GP_REQUIRE((long)p->N * (p->H + 2L * p->pad_h) * (p->W + 2L * p->pad_w) < (1L << 31), "conv: too many input pixels");
    GP_REQUIRE(!p->residual || p->res_pix_stride >= p->Cout, "conv: residual pixel stride");
    GP_REQUIRE(p->tile_m == p->tile_n || p->variant == GP_MAT_WIDE || p->variant == GP_MAT_WIDE8, "conv: square tiles only (the wide variants also take 64 x 32)");
    MatPlan &pl = *out;
    pl = MatPlan{};
    MatArgs &g = pl.g;
    if (p->R == 1 && p->S == 1 && p->stride_h == 1 && p->stride_w == 1 && p->pad_h == 0 && p->pad_w == 0) {
        // A pointwise convolution IS a GEMM over the pixels (rows in_pix_stride apart); the GEMM
        // bodies need no window arithmetic and were measured about 1 us per launch faster at
        // ResNet-152's shapes (1568 x 256 x 1024: 7.7 -> 6.6 us with the same tile body).
        g.M = (int)M; g.N = p->Cout; g.K = p->Cin;
        g.A = p->in; g.lda = p->in_pix_stride;
        g.B = p->weight; g.ldb = g.K;
        g.C = p->out; g.ldc = p->out_pix_stride;
        g.bias = p->bias; g.residual = p->residual; g.ldr = p->residual ? p->res_pix_stride : 0;
        g.alpha = 1.f; g.act = p->act; g.batch_inner = 0;
        pl.dtype = p->dtype; pl.conv = 0; pl.b_kn = 0; pl.batch = 1;
        // an explicit variant keeps its meaning; the staged variant of a convolution has no K x N weights
        return choose_body(&pl, p->tile_m, p->tile_n, p->variant);
    }
    g.M = (int)M; g.N = p->Cout; g.K = p->R * p->S * p->Cin;
    g.A = p->in; g.lda = p->in_pix_stride;
    g.B = p->weight; g.ldb = g.K;
    g.C = p->out; g.ldc = p->out_pix_stride;
    g.bias = p->bias; g.residual = p->residual; g.ldr = p->residual ? p->res_pix_stride : 0;
    g.alpha = 1.f; g.act = p->act; g.batch_inner = 0;
    g.H = p->H; g.W = p->W; g.Cin = p->Cin; g.S = p->S; g.Ho = Ho; g.Wo = Wo;
    g.sh = p->stride_h; g.sw = p->stride_w; g.ph = p->pad_h; g.pw = p->pad_w;
    g.R = p->R; g.inv_cin = inverse_of(g.Cin, g.K); g.inv_s = inverse_of(g.S, g.K / g.Cin);
    g.rcp_hw = 1.0f / (float)(Ho * Wo); g.rcp_wo = 1.0f / (float)Wo;
    pl.dtype = p->dtype; pl.conv = 1; pl.b_kn = 0; pl.batch = 1;
    return choose_body(&pl, p->tile_m, p->tile_n, p->variant);
}

// The bodies that take a scale, shift and ReLU on A: those that a pointwise layer of a batch of a few images gets.
static bool takes_pre(const MatPlan &pl) { return !pl.conv && !pl.b_kn && (pl.body == MB_PIPE64 || is_wide_body(pl.body)); }

// An element-wise layer and the pointwise convolution that reads its output, as one launch of the body (and with the sums, so
// that no bit changes) that the convolution alone would get.
int plan_eltwise_conv2d(const gp_eltwise_params *e, const gp_conv_params *c, MatPlan *out) {
    EltPlan elt;
    if (int rc = plan_eltwise(e, &elt)) return rc;
    if (int rc = plan_conv2d(c, out)) return rc;
    GP_REQUIRE(e->scale && e->shift && !e->b && (e->act == GP_ACT_NONE || e->act == GP_ACT_RELU), "eltwise + conv: a scale, a shift and possibly a ReLU");
    GP_REQUIRE(e->dtype == c->dtype && c->in == e->out && c->in_pix_stride == e->out_stride && c->Cin == e->cols && (long)c->N * c->H * c->W == e->rows, "eltwise + conv: the convolution does not read the layer's output");
    GP_REQUIRE(c->out != e->a && c->residual != e->out, "eltwise + conv: overlapping operands");
    GP_REQUIRE(e->a_stride >= 0, "eltwise + conv: the matrix bodies count a row's bytes from the first one up");
    MatPlan &pl = *out;
    MatArgs alone = pl.g;
    alone.A = e->a; alone.lda = e->a_stride;
    GP_REQUIRE(c->tile_m == 0 && c->variant == 0 && takes_pre(pl) && (pl.body == MB_PIPE64 || buffer_ok(alone, false, pl.dtype)) &&
                   pl.lds_bytes + pre_table_bytes(alone.K, (unsigned)dtype_size(pl.dtype)) <= pre_max_lds(pl.lds_bytes),
               "eltwise + conv: no matrix body that takes a scale and shift for this shape");
    pl.g = alone;
    pl.g.pre_scale = e->scale; pl.g.pre_shift = e->shift; pl.g.pre_relu = e->act == GP_ACT_RELU;
    pl.pre = true;
    return GP_SUCC;
}

// Convolutions that run as one launch (gemm_group.hpp): each with the body it would get alone, which is the same for all, and tiles
// too short to be given up (the group's kernel does not look at the stop word inside a tile); together no more tiles than compute
// units.  (Layers that fill the device alone gain nothing beside each other: with up to two rounds of tiles Inception-v3 b2 fp32 takes 1167 us
// for 1105, b8 bf16 1227 for 1163.)  That leaves the smallest tiles of either kind: a layer gets the next larger ones (64 x 32, 32 x 16) from
// more tiles than half of the compute units on, and two of them are too many.
static int group_body(int dtype) { return dtype == GP_F32 ? MB_NARROW16x16 : MB_WIDE32x32_16; }
int plan_conv2d_group(const gp_conv_params *p, int n, MatPlan *out) {
    GP_REQUIRE(p && n >= 2 && n <= kGroupMax, "conv group of %d: two to %d", n, kGroupMax);
    long total = 0;
    for (int i = 0; i < n; ++i) {
        if (int rc = plan_conv2d(p + i, out + i)) return rc;
        const MatPlan &pl = out[i];
        GP_REQUIRE(p[i].tile_m == 0 && p[i].variant == 0 && pl.dtype == out[0].dtype && pl.body == group_body(pl.dtype) &&
                       !tile_is_long(wide_of(pl.body)->bm, wide_of(pl.body)->bn, pl.g.K, pl.dtype),
                   "conv group: member %d has no body that runs in a group with the first one's", i);
        total += (long)pl.sx * pl.sy;
    }
    GP_REQUIRE(total <= device_cus(), "conv group of %ld tiles", total);
    return GP_SUCC;
}

}  // namespace gp

using namespace gp;

extern "C" int gp_conv2d_group_supported(const gp_conv_params *p, int n) {
    MatPlan pl[kGroupMax];
    KeepLastError keep;
    return plan_conv2d_group(p, n, pl) == GP_SUCC ? 1 : 0;
}
extern "C" int gp_launch_conv2d_group(const gp_conv_params *p, int n, const gp_preempt_ctx *ctx, gp_stream s, gp_launch_info *info) {
    MatPlan pl[kGroupMax];
    int rc = plan_conv2d_group(p, n, pl);
    if (rc) return rc;
    switch (pl[0].dtype) {
        case GP_F32: return launch_group_typed<float>(pl, n, ctx, s, info);
        case GP_F16: return launch_group_typed<_Float16>(pl, n, ctx, s, info);
        default: return launch_group_typed<__bf16>(pl, n, ctx, s, info);
    }
}

extern "C" int gp_eltwise_conv2d_supported(const gp_eltwise_params *e, const gp_conv_params *c) {
    MatPlan pl;
    KeepLastError keep;
    return plan_eltwise_conv2d(e, c, &pl) == GP_SUCC ? 1 : 0;
}
extern "C" int gp_launch_eltwise_conv2d(const gp_eltwise_params *e, const gp_conv_params *c, const gp_preempt_ctx *ctx, gp_stream s, gp_launch_info *info) {
    MatPlan pl;
    int rc = plan_eltwise_conv2d(e, c, &pl);
    return rc ? rc : launch_mat_plan(pl, ctx, s, info);
}

extern "C" int gp_launch_gemm(const gp_gemm_params *p, const gp_preempt_ctx *ctx, gp_stream s, gp_launch_info *info) {
    MatPlan pl;
    int rc = plan_gemm(p, &pl);
    return rc ? rc : launch_mat_plan(pl, ctx, s, info);
}

extern "C" int gp_launch_conv2d(const gp_conv_params *p, const gp_preempt_ctx *ctx, gp_stream s, gp_launch_info *info) {
    MatPlan pl;
    int rc = plan_conv2d(p, &pl);
    if (rc) return rc;
    // A preemptible launch that cannot give its tiles up finishes the ones it holds before it leaves, so a tenant's
    // preemption latency is its longest tile.  A 128 x 128 tile of a deep layer runs 45-65 us (VGG-16 b16: K = 2304 at
    // 56 x 56, K = 4608 at 28 x 28); four 64 x 64 tiles in its place finish one by one; same summation per element, so
    // the bits do not change.  Where plan_launch finds that the tiles can be given up (counters of leavers, several
    // claim counters, a flag that is not read at every claim, at most eight rounds of workgroups), the larger ones, which are 8 (K =
    // 2304) and 24 % (K = 4608) faster, stay.  Not when the caller chose the tile, and not when it brought a checkpoint
    // workspace (then long tiles are left between two K-steps).
    pl.or_smaller = ctx && ctx->flag && pl.body == MB_PIPE128 && pl.g.K >= 2304 && p->tile_m == 0 && p->variant == 0 && !(ctx->ckpt && ctx->ckpt_bytes >= plan_ckpt_bytes(pl));
    rc = launch_mat_plan(pl, ctx, s, info);
    if (rc == kTileTooLong) {
        gp_conv_params q = *p;
        q.tile_m = q.tile_n = 64;
        q.variant = GP_MAT_PIPE;
        rc = plan_conv2d(&q, &pl);
        if (rc) return rc;
        pl.ring = (long)pl.sx * pl.sy > 2 * device_cus() ? 2 : 0;
        rc = launch_mat_plan(pl, ctx, s, info);
    }
    return rc;
}

#ifdef GP_TILE_PROF
extern "C" int gp_debug_tile_prof(unsigned long long *out, int n) {
    GP_HIP(hipDeviceSynchronize());
    const int body = n < 256 * 8 ? n : 256 * 8;
    GP_HIP(hipMemcpyFromSymbol(out, HIP_SYMBOL(gp::g_tile_prof), sizeof(unsigned long long) * (size_t)body));
    if (n > body) GP_HIP(hipMemcpyFromSymbol(out + body, HIP_SYMBOL(gp::g_disp_prof), sizeof(unsigned long long) * (size_t)std::min(n - body, 256 * 8)));
    return GP_SUCC;
}
#endif

// Checkpoint workspace of the bodies that can leave a tile half-way (the 256 x 256 and 128 x 128
// bodies): headers plus one accumulator slot per resident workgroup.
namespace gp {
size_t plan_ckpt_bytes(const MatPlan &pl) {
    if (pl.body == MB_PIPE256) return ckpt_workspace_bytes(BigPipe<float, true>::CKPT_SLOT_BYTES, (int)device_cus());
    if (pl.body == MB_PIPE128) return ckpt_workspace_bytes(PipeKernel<float, 128, 128, GP_S128, false, false, true>::CKPT_SLOT_BYTES, 2 * (int)device_cus());
    return 0;
}
}  // namespace gp
extern "C" int gp_gemm_ckpt_bytes(const gp_gemm_params *p, size_t *bytes) {
    GP_REQUIRE(bytes != nullptr, "null bytes");
    MatPlan pl;
    int rc = plan_gemm(p, &pl);
    if (rc) return rc;
    *bytes = plan_ckpt_bytes(pl);
    return GP_SUCC;
}
extern "C" int gp_conv2d_body(const gp_conv_params *p, char *name, size_t len) {
    GP_REQUIRE(name && len, "null name");
    MatPlan pl;
    if (int rc = plan_conv2d(p, &pl)) return rc;
    static const char *const names[] = {"pipe128", "pipe64", "pipe64_splitk", "pipe32_splitk", "staged128", "staged64", "pipe256", "wide32x32_16", "wide32x32_8", "wide64x32_16",
                                        "wide64x64_8", "lnwide32x64_16", "narrow16x16", "narrow32x16"};
    static_assert(MB_PIPE128 == 0 && MB_PIPE64 == 1 && MB_PIPE64_SK == 2 && MB_PIPE32_SK == 3 && MB_STAGED128 == 4 && MB_STAGED64 == 5 && MB_PIPE256 == 6 && MB_NARROW32x16 == 13, "names");
    const bool blocks_straddle = pl.conv && pl.g.Cin % (pl.dtype == GP_F32 ? 32 : 64) != 0;
    // (the wide bodies multiply as well; those of four wavefronts do where the launcher takes that form of them, gemm_launch.hpp)
    const bool divides = !is_wide_body(pl.body) && !((pl.body == MB_PIPE64 || pl.body == MB_PIPE128) && pl.straddles);
    snprintf(name, len, "%s%s", pl.tall ? "pipe128x64" : names[pl.body],
             !pl.conv ? "" : pl.window ? " window" : blocks_straddle ? divides ? " divided" : " straddling" : pl.taps ? " taps" : " gathered");
    return GP_SUCC;
}
extern "C" int gp_conv_ckpt_bytes(const gp_conv_params *p, size_t *bytes) {
    GP_REQUIRE(bytes != nullptr, "null bytes");
    MatPlan pl;
    int rc = plan_conv2d(p, &pl);
    if (rc) return rc;
    *bytes = plan_ckpt_bytes(pl);
    return GP_SUCC;
}

extern "C" int gp_ckpt_reset_async(void *ckpt, gp_stream s) {
    GP_REQUIRE(ckpt != nullptr, "null checkpoint workspace");
    return gp_fill32_async(ckpt, 0, (size_t)CKPT_MAX_WGS * CKPT_HEADER_INTS, s);
}

// ---- a preemptible GEMM launch that allocates nothing -----------------------------------------------
// gp_launch_gemm takes its claim counters and stop index from the caller's context, which somebody
// had to allocate.  Callers that cannot allocate (code under HIP graph capture, tight serving loops,
// harnesses that forbid it) get the same launch with that state in a file-scope device array: 64
// kernel slots of 32 counters (one per 64-byte line), then one line that holds the stop index.
// The array exists once per GPU for the life of the process; every call on a GPU shares it and it
// keeps the last call's contents, so calls that overlap on one GPU race.
namespace gp {
constexpr int kStaticSlots = 64;      // kernels whose counters the array can hold at once
constexpr int kStaticGroups = 32;     // claim counters per kernel, as BLPExecutor uses
constexpr int kStaticSlotInts = kStaticGroups * COUNTER_STRIDE;
constexpr int kStaticInts = kStaticSlots * kStaticSlotInts + COUNTER_STRIDE;   // 131 136 bytes
constexpr int kStaticMaxDevices = 16;
static __device__ __align__(256) int scratch[kStaticInts];

// `scratch` is only a host-side stand-in here: the array's address on each device comes from
// hipGetSymbolAddress, once per device, with that device current.
static std::mutex g_scratch_mu;
static int *g_scratch_ptr[kStaticMaxDevices] = {nullptr};

int static_scratch_setup(int **out) {
    int dev = -1;
    GP_HIP(hipGetDevice(&dev));
    GP_REQUIRE(dev >= 0 && dev < kStaticMaxDevices, "device %d is beyond the %d the static scratch serves", dev, kStaticMaxDevices);
    std::lock_guard<std::mutex> g(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        GP_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        GP_REQUIRE(p != nullptr, "hipGetSymbolAddress returned no address for the static scratch");
        g_scratch_ptr[dev] = (int *)p;
    }
    if (out) *out = g_scratch_ptr[dev];
    return GP_SUCC;
}

// Clears one slot's counter lines and re-arms the stop index (a kernel, not a memset: the call may
// be recorded into a graph).
__global__ void static_reset_kernel(int *counters, int n, int *stop) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (counters && i < n) counters[i] = 0;
    if (stop && i == 0) *stop = -1;
}
__global__ void static_report_kernel(const int *stop, int *out) {
    if (threadIdx.x == 0) __hip_atomic_store(out, *stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
}  // namespace gp

extern "C" int gp_launch_gemm_noalloc(const gp_gemm_params *p, int *flag, int slot, int mode, int inject_at, int *stop_index_out,
                                      gp_stream s, gp_launch_info *info) {
    GP_REQUIRE(mode >= 0 && mode <= (GP_NOALLOC_CLEAR | GP_NOALLOC_REARM), "mode %d", mode);
    GP_REQUIRE(slot >= 0 && slot < kStaticSlots, "slot %d: the static scratch holds the counters of %d kernels (slots 0..%d)", slot, kStaticSlots, kStaticSlots - 1);
    MatPlan pl;
    int rc = plan_gemm(p, &pl);
    if (rc) return rc;
    // every claim must be countable in the slot: the tile grid is bounded like a launch's
    GP_REQUIRE((long)pl.sx * pl.sy * pl.batch <= (1L << 24), "gemm of %ld tiles: the static scratch serves at most %ld per launch", (long)pl.sx * pl.sy * pl.batch, 1L << 24);
    int *base = nullptr;
    rc = static_scratch_setup(&base);
    if (rc) return rc;
    int *counters = base + (size_t)slot * kStaticSlotInts, *stop = base + (size_t)kStaticSlots * kStaticSlotInts;
    if (mode) {
        hipLaunchKernelGGL(static_reset_kernel, dim3((kStaticSlotInts + 255) / 256), dim3(256), 0, native(s),
                           (mode & GP_NOALLOC_CLEAR) ? counters : (int *)nullptr, kStaticSlotInts, (mode & GP_NOALLOC_REARM) ? stop : (int *)nullptr);
        GP_HIP(hipGetLastError());
    }
    gp_preempt_ctx ctx{};
    ctx.flag = flag; ctx.stop_index = stop; ctx.executed = counters; ctx.kernel_id = slot; ctx.inject_at = inject_at;
    ctx.counter_groups = kStaticGroups;
    ctx.fresh = (mode & GP_NOALLOC_CLEAR) != 0;
    rc = launch_mat_plan(pl, &ctx, s, info);
    if (rc) return rc;
    if (stop_index_out) {
        hipLaunchKernelGGL(static_report_kernel, dim3(1), dim3(64), 0, native(s), (const int *)stop, stop_index_out);
        GP_HIP(hipGetLastError());
    }
    return GP_SUCC;
}
