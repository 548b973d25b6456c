// Layer-norm + GEMM in one kernel, for small deep-learning shapes where a launch costs more than the
// arithmetic: C = act(LN(A) * B^T + bias [+ residual]), with LN(A) also written out once.
//
// Why: in a transformer layer at batch 1 the layer-norm kernel in front of the QKV and the first FFN
// projection moves 0.4 MB and takes as long as any dependent launch takes on this GPU (about 5 us),
// a fifth of the request.  The projection's workgroups read their rows of A anyway, and a row is
// short (K elements), so every workgroup normalises its own BM rows before it multiplies them:
// the rows go from global memory through registers into LDS, where they stay for the whole tile
// (BM x K elements: 48 KB for 32 rows of 768 halves), and only B streams through the ring of
// gemm_wide.hpp.  The workgroups of tile column 0 also store the normalised rows, for the later
// kernels that read them (the residual additions).
//
// Same bits as the two-kernel form: a row is normalised by one wavefront through ln_rows_math, the
// function the stand-alone layer-norm kernel uses, with the same lane-to-chunk assignment, and
// rounded to the storage type before it is multiplied, as it would be on its way through memory;
// the main loop and the reduction are those of WideKernel (wavefront w multiplies MFMA k-step w of
// every K-block, partial tiles summed in wavefront order).
#pragma once
#include <type_traits>
#include "elementwise_bodies.hpp"
#include "gemm_wide.hpp"

namespace gp {

// Two rows of 65 to 96 chunks by one wavefront, with the bits of ln_rows_math.  There a lane holds chunks l and l + 64 of each row, and at 96
// chunks every second instruction runs for half of the lanes.  Sixteen wavefronts, four to a SIMD, normalise the rows of a tile, and the
// prologue's time is the number of vector instructions: so the chunks behind the 64th share a register, row 0's in the lower half of the
// wavefront and row 1's in the upper.  A lane adds up its chunk l first and its chunk l + 64 behind it, as there: the upper half's sums of row 0
// and the lower half's of row 1 change places in between.  430 -> 240 vector instructions with f16; BERT-base b1 s128 fp16 467 -> 456 us,
// b2 s211 bf16 level (its conversions are instructions of their own, and its launches have more tiles than compute units).
__device__ __forceinline__ void swap_halves(float &row0, float &row1) {  // row 0's upper half <-> row 1's lower half
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, row0), __builtin_bit_cast(unsigned, row1), false, false);
    const unsigned lo = r[0], hi = r[1];
    row0 = __builtin_bit_cast(float, lo);
    row1 = __builtin_bit_cast(float, hi);
}
// x + the value in a half of `word`, and with f16 no conversion of its own (exact, so the sum is rounded once either way)
template <typename T, int HALF> __device__ __forceinline__ float add_half(unsigned word, float x) {
    if constexpr (std::is_same<T, _Float16>::value) {
        float y;
        if constexpr (HALF == 0) asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(y) : "v"(word), "v"(x));
        else asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(y) : "v"(word), "v"(x));
        return y;
    } else {
        return __builtin_bit_cast(float, HALF ? word & 0xFFFF0000u : word << 16) + x;
    }
}
template <typename T> __device__ __forceinline__ void ln_pair_math(const out_u32x4 (&x)[3], int tail, int lane, int cols, float eps,
                                                                   const out_u32x4 (&gamma)[2], const out_u32x4 (&beta)[2], out_u32x4 (&y)[3]) {
#pragma clang fp contract(off)
    static_assert(sizeof(T) == 2, "two values to a word");
    const bool behind = (lane & 31) < tail;  // this lane has a chunk behind the 64th
    float sum[2], sq[2];
    auto add_chunk = [](const out_u32x4 &c, float s) {
#pragma unroll
        for (int w = 0; w < 4; ++w) s = add_half<T, 1>(c[w], add_half<T, 0>(c[w], s));
        return s;
    };
    sum[0] = add_chunk(x[0], 0.f);
    sum[1] = add_chunk(x[1], 0.f);
    swap_halves(sum[0], sum[1]);
    sum[0] = add_chunk(x[2], sum[0]);  // (zeros where there is no chunk)
    swap_halves(sum[0], sum[1]);
    wave_sum_rows<2>(sum);
    // x / cols with the bits of the division, in three instructions for ten, from the rounded reciprocal: its product, corrected by the exact
    // remainder (Markstein).  With f16 only, whose sums of squares cannot overflow: of an infinity the remainder makes NaN.
    const float n = (float)cols, c = 1.0f / n;
    auto over_cols = [&](float v) {
        if constexpr (!std::is_same<T, _Float16>::value) return v / n;
        const float q = v * c;
        return __builtin_fmaf(__builtin_fmaf(-q, n, v), c, q);
    };
    const float mean[2] = {over_cols(sum[0]), over_cols(sum[1])};
    const float mean_behind = lane < 32 ? mean[0] : mean[1];
    float d[3][8];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float m = c < 2 ? mean[c] : mean_behind;
            d[c][2 * w] = add_half<T, 0>(x[c][w], -m);
            d[c][2 * w + 1] = add_half<T, 1>(x[c][w], -m);
        }
    // (the first product of a row is the fused one and its second the rounded one, as there)
    auto first_squares = [](const float (&v)[8]) {
        float s = __builtin_fmaf(v[0], v[0], v[1] * v[1]);
#pragma unroll
        for (int j = 2; j < 8; ++j) s = __builtin_fmaf(v[j], v[j], s);
        return s;
    };
    sq[0] = first_squares(d[0]);
    sq[1] = first_squares(d[1]);
    swap_halves(sq[0], sq[1]);
    float with = sq[0];
#pragma unroll
    for (int j = 0; j < 8; ++j) with = __builtin_fmaf(d[2][j], d[2][j], with);
    sq[0] = behind ? with : sq[0];
    swap_halves(sq[0], sq[1]);
    wave_sum_rows<2>(sq);
    const float inv[2] = {rsqrtf(over_cols(sq[0]) + eps), rsqrtf(over_cols(sq[1]) + eps)};
    const float inv_behind = lane < 32 ? inv[0] : inv[1];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        float ga[8], be[8], o[8];
        VecIO<T>::unpack(gamma[c / 2], ga);
        VecIO<T>::unpack(beta[c / 2], be);
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = __builtin_fmaf(d[c][j] * (c < 2 ? inv[c] : inv_behind), ga[j], be[j]);
        y[c] = VecIO<T>::pack(o);
    }
}

template <typename T, int BM, int BN, int WAVES, int STAGES>
struct LnWideKernel {
    using elem = T;
    static constexpr int bm = BM, bn = BN;
    static constexpr bool conv = false, pre = false, window = false;
    static constexpr int VEC = Elem<T>::VEC;
    static constexpr int NT = WAVES * 64;
    static constexpr int RB = 128;                         // row bytes of a block in LDS
    static constexpr int BK = RB / (int)sizeof(T);         // K elements per block
    static constexpr int KB = WAVES / 4;                   // blocks per stage
    static constexpr int LPW = BN / 8 / 4;                 // B row groups a wavefront fetches per stage
    static constexpr int MAXK = 832;                       // longest row: BM x MAXK elements stay resident (104 KB of the 160)
    static constexpr int MAXC = 2;                         // 16-byte chunks of a row per lane (ln_rows_math): K <= 128 * VEC
    static constexpr int A_BLK_BYTES = BM * RB;            // one K-block of the resident rows
    static constexpr int B_BLK_BYTES = BN * RB, STAGE_BYTES = KB * B_BLK_BYTES;
    static constexpr int MI = BM / 32, NI = BN / 32;
    // wavefront group kb < G multiplies for the output blocks kb, kb + G, ... (WideKernel keeps G = 1; here two
    // groups, one per 32 x 32 block of the 32 x 64 tile, took 0.25-0.3 us off a launch: 7.87 -> 7.62, 8.43 -> 8.13)
    static constexpr int G = MI * NI < KB ? MI * NI : KB, BPW = MI * NI / G;
    static_assert(MI * NI % G == 0, "output blocks divide among the multiplying groups");
    static constexpr int SLICES = MI * NI * 16;
    static constexpr size_t RED_BYTES = (size_t)4 * SLICES * 64 * 4;
    static constexpr size_t RING_BYTES = (size_t)STAGES * STAGE_BYTES;
    static constexpr size_t A_RES_BYTES = (size_t)BM * MAXK * sizeof(T);
    // the reduction buffer reuses the ring, which lies in front of the resident rows
    static constexpr size_t RING_REGION = RING_BYTES > RED_BYTES ? RING_BYTES : RED_BYTES;
    static constexpr size_t LDS_BYTES = RING_REGION + A_RES_BYTES;
    static constexpr size_t CKPT_SLOT_BYTES = 0;
    static constexpr bool ckpt = false;
    static constexpr bool early_stop = true;
    static constexpr bool can_look = false;
    static constexpr int PRE = GP_WIDE_PREFILL ? STAGES : STAGES - 1;
    static_assert(sizeof(T) == 2, "16-bit element types");
    static_assert(WAVES == 16 && BM % WAVES == 0 && BN % 32 == 0 && BM % 32 == 0, "tile shape");
    static_assert(STAGES >= 2 && STAGES <= 4 && (STAGES - 1) * LPW < 64, "pipeline depth");
    static_assert(LDS_BYTES <= 160 * 1024, "LDS budget");

    template <bool LOOKS = false, bool SINGLE = false, class Asked = NoneAsked>  // (as in PipeKernel)
    static __device__ __forceinline__ bool run(const MatArgs &g, TileIdx t, T *lds_t, CkptCtx cc = CkptCtx{nullptr, nullptr, nullptr, 0}, Asked &&asked = Asked{}) {
        GP_PROBE(0);
        __shared__ int early_slot[64];
        const bool early = __builtin_amdgcn_readfirstlane((int)(cc.stop_index != nullptr)) != 0;
        const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) void *)lds_t;
        char *lds_c = (char *)lds_t;
        char *a_res = lds_c + RING_REGION;
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int kb = wave >> 2, wv = wave & 3;
        const int l32 = lane & 31, half = lane >> 5;
        const int m0 = t.y * BM, n0 = t.x * BN;
        const T *A = (const T *)g.A, *B = (const T *)g.B;
        const int KT = g.K / BK;                        // blocks along K (K is a multiple of BK: checked by the planner)
        const int NS = (KT + KB - 1) / KB;              // stages of B

        // ---- B loader slots, as in WideKernel ---------------------------------------------------
        const int rig = lane >> 3, cpos = lane & 7;
        const u32x4 rsrc_b = buffer_of(B + (long)n0 * g.ldb);  // (from the tile's first row: the planner bounds 64 rows, not all of B)
        unsigned off[LPW];
#pragma unroll
        for (int j = 0; j < LPW; ++j) {
            const int r = (wv * LPW + j) * 8 + rig;
            off[j] = n0 + r < g.N ? ((unsigned)r * (unsigned)g.ldb + (unsigned)(cpos ^ ((r >> 1) & 7)) * VEC) * (unsigned)sizeof(T) : kBufferEnd;
        }
        auto issue = [&](int s) {
            const int k0 = (s * KB + kb) * BK;
            const unsigned sbase = lds0 + ((unsigned)s % STAGES) * STAGE_BYTES + (unsigned)kb * B_BLK_BYTES;
#pragma unroll
            for (int j = 0; j < LPW; ++j)  // (whole blocks past the last one, when the stage is not full: zeros)
                load_lds16_buffer<SINGLE>(rsrc_b, k0 < g.K ? off[j] : kBufferEnd, (unsigned)k0 * (unsigned)sizeof(T), sbase + (unsigned)((wv * LPW + j) * 8 * RB));
        };

        if (!SINGLE) __syncthreads();  // the previous tile of this workgroup may still be reading LDS

        // ---- the rows of A: normalise, keep in LDS, store once -------------------------------------
        // wavefront w takes rows w, w + WAVES, ...; lane l holds chunks l and l + 64 of a row.  B is asked for behind the rows, so that the
        // arithmetic on them covers its way from memory.  (It takes longer than that: 128 x 2304 x 768 spends 5000 ticks until the rows
        // and the first stage are there, and 1900 more on the rows; 3300 more before ln_pair_math.)
        constexpr int RPW = BM / WAVES;
        const int chunks = g.K / VEC, tail = chunks - 64;
        auto first_stages = [&]() {
#pragma unroll
            for (int s = 0; s < PRE; ++s) {
                if (s < NS) issue(s);
                if (s == 0 && early && wave == 0) load_lds4(cc.stop_index, (unsigned)(size_t)(__attribute__((address_space(3))) void *)early_slot);
            }
            asked();
        };
        // chunk ch of row r is chunk ch % 8 of K-block ch / 8, at the swizzled position
        auto keep = [&](int r, int ch, const out_u32x4 &y) {
            *(out_u32x4 *)(a_res + (size_t)(ch >> 3) * A_BLK_BYTES + r * RB + ((ch & 7) ^ ((r >> 1) & 7)) * 16) = y;
        };
        if (RPW == 2 && tail > 0 && tail <= 32) {
            // No branch stands around these loads and what is computed from them, so the compiler waits for each where it is used.  It counts the seven loads here
            // and not B's, which come behind them: its wait for the rows, four loads of gamma and beta outstanding, lets four of B be on their way, which is
            // all of them where two stages are asked for.  Those for gamma and beta let two and none, so B has landed before the first row is kept.
            const int m = m0 + wave, over = lane >> 5, ch = 64 + (lane & 31);
            const int r0 = m < g.M ? m : g.M - 1, r1 = m + WAVES < g.M ? m + WAVES : g.M - 1;
            const bool behind = (lane & 31) < tail;
            const int at = behind ? ch : 0;  // (a chunk of the row for the lanes that have none)
            const T *a0 = A + (long)r0 * g.lda, *a1 = A + (long)r1 * g.lda;
            out_u32x4 x[3] = {*(const out_u32x4 *)(a0 + lane * VEC), *(const out_u32x4 *)(a1 + lane * VEC), *(const out_u32x4 *)((over ? a1 : a0) + at * VEC)};
            const T *ga = (const T *)g.ln_gamma, *be = (const T *)g.ln_beta;
            const out_u32x4 gamma[2] = {*(const out_u32x4 *)(ga + lane * VEC), *(const out_u32x4 *)(ga + at * VEC)};
            const out_u32x4 beta[2] = {*(const out_u32x4 *)(be + lane * VEC), *(const out_u32x4 *)(be + at * VEC)};
            __builtin_amdgcn_sched_barrier(0);
            first_stages();
            __builtin_amdgcn_sched_barrier(0);
            if (tail < 32) {
#pragma unroll
                for (int w = 0; w < 4; ++w) x[2][w] = behind ? x[2][w] : 0u;
            }
            out_u32x4 y[3];
            ln_pair_math<T>(x, tail, lane, g.K, g.ln_eps, gamma, beta, y);
            keep(wave, lane, y[0]);
            keep(wave + WAVES, lane, y[1]);
            if (behind) keep(wave + over * WAVES, ch, y[2]);
        } else {  // (the waits stand inside branches here, and the compiler's for the rows would be one for B too: B is asked for when they are there)
            out_u32x4 rx[RPW][MAXC];
#pragma unroll
            for (int q = 0; q < RPW; ++q) {
                const int m = m0 + wave + q * WAVES;
                const T *x = A + (long)(m < g.M ? m : g.M - 1) * g.lda;
#pragma unroll
                for (int i = 0; i < MAXC; ++i) {
                    const int ch = lane + i * 64;
                    rx[q][i] = out_u32x4{0, 0, 0, 0};
                    if (ch < chunks) rx[q][i] = *(const out_u32x4 *)(x + ch * VEC);
                }
            }
            // gamma and beta with them: a wait for them later would be a wait for B as well
            out_u32x4 graw[MAXC], braw[MAXC];
#pragma unroll
            for (int i = 0; i < MAXC; ++i) {
                const int ch = lane + i * 64;
                graw[i] = braw[i] = out_u32x4{0, 0, 0, 0};
                if (ch < chunks) {
                    graw[i] = *(const out_u32x4 *)((const T *)g.ln_gamma + ch * VEC);
                    braw[i] = *(const out_u32x4 *)((const T *)g.ln_beta + ch * VEC);
                }
            }
#pragma unroll
            for (int i = 0; i < MAXC; ++i) {
#pragma unroll
                for (int q = 0; q < RPW; ++q) asm volatile("" : "+v"(rx[q][i]) :: "memory");  // the rows have arrived
                asm volatile("" : "+v"(graw[i]), "+v"(braw[i]) :: "memory");
            }
            first_stages();
            float v[RPW][MAXC][VEC];
#pragma unroll
            for (int q = 0; q < RPW; ++q)
#pragma unroll
                for (int i = 0; i < MAXC; ++i) {
                    const int ch = lane + i * 64;
                    if (ch < chunks) VecIO<T>::unpack(rx[q][i], v[q][i]);
                }
            out_u32x4 y[RPW][MAXC];
            ln_rows_math<T, MAXC, RPW, true>(v, chunks, lane, g.K, g.ln_eps, (const T *)g.ln_gamma, (const T *)g.ln_beta, graw, braw, y);
#pragma unroll
            for (int q = 0; q < RPW; ++q) {
                const int r = wave + q * WAVES;
#pragma unroll
                for (int i = 0; i < MAXC; ++i) {
                    const int ch = lane + i * 64;
                    if (ch < chunks) keep(r, ch, y[q][i]);
                }
            }
        }

        GP_PROBE(1);
        f32x16 acc[BPW];
#pragma unroll
        for (int q = 0; q < BPW; ++q)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[q][v] = 0.f;
        auto frag_a = [&](int blk, int row, int chunk) -> u32x4 {
            const int phys = chunk ^ ((row >> 1) & 7);
            return *(const u32x4 *)(a_res + (size_t)blk * A_BLK_BYTES + row * RB + phys * 16);
        };
        auto frag_b = [&](int stage, int blk, int row, int chunk) -> u32x4 {
            const int phys = chunk ^ ((row >> 1) & 7);
            return *(const u32x4 *)(lds_c + (size_t)stage * STAGE_BYTES + (size_t)blk * B_BLK_BYTES + row * RB + phys * 16);
        };

        // ---- main loop: B streams, A is there ------------------------------------------------------
        for (int s = 0; s < NS; ++s) {
            if (s == 0) wait_stages<LPW>((NS < PRE ? NS : PRE) - 1);
            else if (s + STAGES - 2 < NS) wait_vmcnt<(STAGES - 2) * LPW>();
            else wait_vmcnt<0>();
            __syncthreads();  // stage s of B (and, the first time, the rows of A) visible; the buffer of stage s-1 is free
            if (s == 0) GP_PROBE(2);
            if (s == 0 && early && __builtin_amdgcn_readfirstlane(read_lds_word(early_slot)) != -1) {
                wait_vmcnt<0>();  // loads still landing in LDS must not outlive the workgroup
                return true;
            }
            // The workgroups of tile column 0 store the normalised rows, and only now: a launch that started
            // eagerly behind a stopped kernel normalised rows of an incomplete x, and must leave (above) without
            // having written anything.  Every wavefront stores the rows it normalised, from their copy in LDS.
            if (s == 0 && t.x == 0) {
#pragma unroll
                for (int q = 0; q < BM / WAVES; ++q) {
                    const int r = wave + q * WAVES, m = m0 + r;
#pragma unroll
                    for (int i = 0; i < MAXC; ++i) {
                        const int ch = lane + i * 64;
                        if (ch < chunks && m < g.M) {
                            const int blk = ch >> 3, phys = (ch & 7) ^ ((r >> 1) & 7);
                            st_out128((T *)g.ln_out + (long)m * g.K + ch * VEC, *(const out_u32x4 *)(a_res + (size_t)blk * A_BLK_BYTES + r * RB + phys * 16));
                        }
                    }
                }
            }
            if (s >= PRE - (STAGES - 1) && s + STAGES - 1 < NS) issue(s + STAGES - 1);
            if (kb >= G) continue;  // (uniform) the other wavefronts only fetch
            const int stage = (int)((unsigned)s % STAGES);
#pragma unroll
            for (int b = 0; b < KB; ++b) {
                if (s * KB + b >= KT) break;
#pragma unroll
                for (int q = 0; q < BPW; ++q) {
                    const int blk = kb + q * G, i = blk / NI, j = blk % NI;
                    const u32x4 fa = frag_a(s * KB + b, i * 32 + l32, wv * 2 + half);
                    const u32x4 fb = frag_b(stage, b, j * 32 + l32, wv * 2 + half);
                    Elem<T>::mma(fa, fb, acc[q]);
                }
            }
        }
        GP_PROBE(3);
        wide_reduce_store<T, BM, BN, NT, G>(g, (float *)lds_t, acc, m0, n0, 0, tid, wv, lane, kb);
#ifdef GP_TILE_PROF
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        GP_PROBE(5);
#endif
        return false;
    }
};

}  // namespace gp
