// Split-K GEMM and convolution bodies with 16 x 16 and 32 x 16 output tiles, for fp32 layers of few rows and columns.
//
// Why: fp32 runs on MFMAs an eighth as fast as the 16-bit types, so a deep layer cut into fewer 32 x 32 tiles than there are compute
// units is bound by the matrix cores of the few that have a tile: 3 x 3 at 7 x 7 x 512, one image, is 32 tiles of 9.4 MFLOP, 16 us at a
// compute unit's 0.6 TFLOP/s.  Tiles of a quarter and a half give that work to four times and twice as many.  What they pay is
// operand traffic, 16 instead of 32 multiplications per element fetched, which at this rate of arithmetic still keeps up.
//
// Structure: as gemm_wide.hpp (sixteen wavefronts fetch, wavefronts 0..3 multiply one MFMA k-step each of every K-block, partial tiles
// summed in wavefront order), with two wavefronts to a block, eight blocks to a stage, and 16x16x4 MFMAs.  Their four products are
// added one after the other, so with the lanes' K elements dealt out to match, a sum has the order and the bits of two
// 32x32x2 MFMAs, i.e. of the 32 x 32 bodies and of the whole-model program (tests/test_narrow_gpu.py).
#pragma once
#include "gemm_wide.hpp"

namespace gp {

template <int BM, int STAGES, int CONV = 0, bool SCALED = false>  // (as WideKernel)
struct NarrowKernel {
    using T = float;
    using elem = float;
    static constexpr int BN = 16, WAVES = 16;
    static constexpr int bm = BM, bn = BN;
    static constexpr bool conv = CONV != 0, pre = SCALED, window = false;
    static_assert(!SCALED || !CONV, "GEMM rows only");
    static constexpr int VEC = 4, NT = WAVES * 64, RB = 128, BK = RB / 4;
    static constexpr int KB = WAVES / 2;                   // blocks per stage
    static constexpr int LPW_A = BM / 16, LPW_B = BN / 16, LPW = LPW_A + LPW_B;  // 8-row groups of its block that a wavefront fetches
    static constexpr int A_BYTES = BM * RB, BLK_BYTES = (BM + BN) * RB, STAGE_BYTES = KB * BLK_BYTES;
    static constexpr int MI = BM / 16;
    static constexpr int PART = MI * 4 * 64;               // floats of a wavefront's partial tile
    static constexpr size_t RED_BYTES = (size_t)4 * PART * 4, RING_BYTES = (size_t)STAGES * STAGE_BYTES;
    static constexpr size_t LDS_BYTES = RING_BYTES > RED_BYTES ? RING_BYTES : RED_BYTES;
    static constexpr size_t CKPT_SLOT_BYTES = 0;
    static constexpr bool ckpt = false, early_stop = true, can_look = true;  // (as WideKernel)
    static_assert(BM == 16 || BM == 32, "tile shape");
    static_assert(STAGES >= 2 && STAGES <= 4 && LDS_BYTES <= 160 * 1024, "LDS budget");

    // Returns true when the early look found a stop recorded: the tile was not run.
    template <bool LOOKS = false, bool SINGLE = false, class Asked = NoneAsked>
    static __device__ __forceinline__ bool run(const MatArgs &g, TileIdx t, T *lds_t, CkptCtx cc = CkptCtx{nullptr, nullptr, nullptr, 0}, Asked &&asked = Asked{}) {
        GP_PROBE(0);
        __shared__ int early_slot[64];
        const bool early = __builtin_amdgcn_readfirstlane((int)(cc.stop_index != nullptr)) != 0;
        constexpr int LOOK_EVERY = 4;  // (see WideKernel)
        static_assert(LOOK_EVERY >= STAGES, "a look is read before the next one is fetched");
        const bool looking = LOOKS && early;
        const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) void *)lds_t;
        const char *lds_c = (const char *)lds_t;
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int kb = wave >> 1, member = wave & 1;
        const int m0 = t.y * BM, n0 = t.x * BN;
        long offa, offb, offc;
        if (g.batch_inner > 0) {
            int zo = t.z / g.batch_inner, zi = t.z - zo * g.batch_inner;
            offa = zo * g.stride_a_outer + zi * g.stride_a;
            offb = zo * g.stride_b_outer + zi * g.stride_b;
            offc = zo * g.stride_c_outer + zi * g.stride_c;
        } else {
            offa = t.z * g.stride_a; offb = t.z * g.stride_b; offc = t.z * g.stride_c;
        }
        const T *A = (const T *)g.A + offa, *B = (const T *)g.B + offb;

        // ---- loader slots: the wavefront's row groups member, member + 2, .. of A and its group of B ------------
        const int rig = lane >> 3, cpos = lane & 7;
        __shared__ unsigned row_off[CONV ? BM : 1], row_taps[CONV ? BM : 1];  // (see WideKernel)
        if (CONV && tid < BM) {
            const int m = m0 + tid, hw = g.Ho * g.Wo;
            const bool in = m < g.M, small = g.M < kSmallDivLimit;
            const int mm = in ? m : 0;
            const int n = small ? small_div(mm, hw, g.rcp_hw) : mm / hw, rem = mm - n * hw;
            const int ho = small ? small_div(rem, g.Wo, g.rcp_wo) : rem / g.Wo, wo = rem - ho * g.Wo;
            row_off[CONV ? tid : 0] = (unsigned)((n * g.H + ho * g.sh) * g.W + wo * g.sw) * (unsigned)g.lda;
            row_taps[CONV ? tid : 0] = in ? window_tap_mask(ho * g.sh - g.ph, wo * g.sw - g.pw, g.H, g.W, g.R, g.S) : 0u;
        }
        const u32x4 rsrc_a = buffer_of(CONV ? A - (long)(g.ph * g.W + g.pw) * g.lda : A), rsrc_b = buffer_of(B);
        auto group_of = [&](int j) { return j < LPW_A ? member + 2 * j : BM / 8 + member; };
        unsigned off[LPW], taps[CONV ? LPW_A : 1], row[CONV ? LPW_A : 1];
        int kc[LPW];
#pragma unroll
        for (int j = 0; j < LPW; ++j) {
            const bool is_a = j < LPW_A;
            const int r = (is_a ? group_of(j) : member) * 8 + rig;  // row in its region
            kc[j] = (cpos ^ ((r >> 1) & 7)) * VEC;
            if (!is_a || !CONV) {
                const int x = (is_a ? m0 : n0) + r;
                off[j] = x < (is_a ? g.M : g.N) ? ((unsigned)x * (unsigned)(is_a ? g.lda : g.ldb) + (unsigned)kc[j]) * 4u : kBufferEnd;
            }
        }
        const int KT = (g.K + BK - 1) / BK;  // blocks along K
        const int NS = (KT + KB - 1) / KB;   // stages
        int nx_tap = 0, nx_r = 0, nx_s = 0, nx_ci = 0;
        auto advance = [&](int elems) {
            nx_ci += elems;
            while (nx_ci >= g.Cin) {
                nx_ci -= g.Cin;
                ++nx_tap;
                if (++nx_s == g.S) { nx_s = 0; ++nx_r; }
            }
        };
        if (CONV) advance(kb * BK);
        constexpr bool straddles = CONV == 2;
        auto issue_part = [&](int s, auto first, auto last) {
            const int k0 = (s * KB + kb) * BK;
            const unsigned sbase = lds0 + ((unsigned)s % STAGES) * STAGE_BYTES + (unsigned)kb * BLK_BYTES;
            const unsigned tap_bit = (k0 < g.K && nx_tap < 32) ? 1u << nx_tap : 0u;
            const unsigned tap_off = (unsigned)((nx_r * g.W + nx_s) * (int)g.lda + nx_ci) * 4u;
            const bool whole = k0 + BK <= g.K;
#pragma unroll
            for (int j = first; j < last; ++j) {
                const unsigned to = sbase + (unsigned)(group_of(j) * 8 * RB);
                if (CONV && j < LPW_A && straddles) {
                    const int k = k0 + kc[j], tap = (int)__umulhi((unsigned)k + 1u, g.inv_cin), ci = k - tap * g.Cin, r = (int)__umulhi((unsigned)tap + 1u, g.inv_s), s2 = tap - r * g.S;
                    const unsigned at = row[CONV ? j : 0] + (unsigned)((r * g.W + s2) * (int)g.lda + ci) * 4u;
                    load_lds16_buffer<SINGLE>(rsrc_a, k < g.K && (taps[CONV ? j : 0] >> tap & 1u) ? at : kBufferEnd, 0u, to);
                } else if (CONV && j < LPW_A) load_lds16_buffer<SINGLE>(rsrc_a, (taps[CONV ? j : 0] & tap_bit) ? off[j] : kBufferEnd, tap_off, to);
                else load_lds16_buffer<SINGLE>(j < LPW_A ? rsrc_a : rsrc_b, whole || k0 + kc[j] < g.K ? off[j] : kBufferEnd, (unsigned)k0 * 4u, to);
            }
            if (CONV && last == LPW_A) advance(KB * BK);
        };
        auto issue_a = [&](int s) { issue_part(s, IntC<0>{}, IntC<LPW_A>{}); };
        auto issue_b = [&](int s) { issue_part(s, IntC<LPW_A>{}, IntC<LPW>{}); };
        auto issue = [&](int s) { issue_b(s); issue_a(s); };

        f32x4 acc[MI];
#pragma unroll
        for (int i = 0; i < MI; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        // Lane l multiplies row (column) l % 16 and, of the four products of an MFMA, number l / 16 = q: element q / 2 (and q / 2 + 2 in the
        // second MFMA) of the k-step's chunk q % 2, as the lanes of half q % 2 do with the elements of a chunk one after the other.
        const int l16 = lane & 15, q = lane >> 4;
        struct Pair { float lo, hi; };
        auto frag = [&](int stage, int blk, int region_bytes, int row) -> Pair {
            const int phys = (wave * 2 + (q & 1)) ^ ((row >> 1) & 7);
            const float *p = (const float *)(lds_c + (size_t)stage * STAGE_BYTES + (size_t)blk * BLK_BYTES + region_bytes + row * RB + phys * 16) + (q >> 1);
            return Pair{p[0], p[2]};
        };

        // ---- main loop ------------------------------------------------------------------------
        GP_PROBE(1);
        constexpr bool B_FIRST = SINGLE && CONV;  // (the weights of the first stage need no row table)
        if (B_FIRST) issue_b(0);
        if (CONV || !SINGLE) __syncthreads();  // the row table; the previous tile of this workgroup may still be reading LDS
        if constexpr (SCALED) pre_fetch_table<T, WAVES>(g, lds0 + (unsigned)LDS_BYTES, wave, lane);
        if (CONV) {
#pragma unroll
            for (int j = 0; j < LPW_A; ++j) {
                const int r = group_of(j) * 8 + rig;
                row[CONV ? j : 0] = row_off[CONV ? r : 0] * 4u;
                off[j] = row[CONV ? j : 0] + (unsigned)kc[j] * 4u;
                taps[CONV ? j : 0] = row_taps[CONV ? r : 0];
            }
        }
#pragma unroll
        for (int s = 0; s < STAGES - 1; ++s) {
            if (B_FIRST && s == 0) issue_a(s);
            else if (s < NS) issue(s);
            if (s == 0 && early && wave == 0) load_lds4(cc.stop_index, (unsigned)(size_t)(__attribute__((address_space(3))) void *)early_slot);
        }
        asked();
        for (int s = 0; s < NS; ++s) {
            if (s == 0) wait_stages<LPW>((NS < STAGES - 1 ? NS : STAGES - 1) - 1);
            else if (s + STAGES - 2 < NS) wait_vmcnt<(STAGES - 2) * LPW>();
            else wait_vmcnt<0>();
            if constexpr (SCALED) {
                if (s == 0) __syncthreads();  // everyone's part of the table
                const int k0 = (s * KB + kb) * BK;
                char *blk = (char *)lds_t + (size_t)((unsigned)s % STAGES) * STAGE_BYTES + (size_t)kb * BLK_BYTES + lane * 16;
                if (k0 < g.K) {
#pragma unroll
                    for (int j = 0; j < LPW_A; ++j) pre_apply<T>(g, blk + group_of(j) * 8 * RB, lds_c + LDS_BYTES, k0 + kc[j]);
                }
            }
            __syncthreads();  // everyone's part of stage s is visible; the buffer of stage s-1 is free
            if (s == 0) GP_PROBE(2);
            if (((s == 0 && early) || (looking && s > 0 && (s & (LOOK_EVERY - 1)) == 0)) && __builtin_amdgcn_readfirstlane(read_lds_word(early_slot)) != -1) {
                wait_vmcnt<0>();  // loads still landing in LDS must not outlive the workgroup
                return true;      // the tile is given up: the caller withdraws the claim
            }
            if constexpr (LOOKS) {  // (the last stage: the workgroup counts itself, see WideKernel)
                if (looking && cc.announce && s == NS - 1 && tid == 0)
                    __hip_atomic_fetch_add(cc.announce, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            if (s + STAGES - 1 < NS) {
                if (looking && wave == 0 && ((s + STAGES - 1) & (LOOK_EVERY - 1)) == 0)
                    load_lds4(cc.stop_index, (unsigned)(size_t)(__attribute__((address_space(3))) void *)early_slot);
                issue(s + STAGES - 1);
            }
            if (wave >= 4) continue;  // (uniform) the other wavefronts only fetch
            const int stage = (int)((unsigned)s % STAGES);
            Pair fa[KB][MI], fb[KB];
#pragma unroll
            for (int b = 0; b < KB; ++b) {
#pragma unroll
                for (int i = 0; i < MI; ++i) fa[b][i] = frag(stage, b, 0, i * 16 + l16);
                fb[b] = frag(stage, b, A_BYTES, l16);
            }
#pragma unroll
            for (int b = 0; b < KB; ++b) {
                if (s * KB + b >= KT) break;  // a block past the last one is skipped (see WideKernel)
#pragma unroll
                for (int i = 0; i < MI; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[b][i].lo, fb[b].lo, acc[i], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < MI; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[b][i].hi, fb[b].hi, acc[i], 0, 0, 0);
            }
        }

        GP_PROBE(3);
        // partial tiles as [wavefront][block][register][lane]: register v of lane l is row 4 * (l / 16) + v, column l % 16
        float *red = (float *)lds_t;
        __syncthreads();  // all wavefronts are done reading the stage buffers
        if (wave < 4) {
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int v = 0; v < 4; ++v) red[(size_t)wave * PART + (i * 4 + v) * 64 + lane] = acc[i][v];
        }
        __syncthreads();
        GP_PROBE(4);
        wide_finish<T, BM, BN, NT, PART>(g, red, m0, n0, offc, tid, [&](int row, int column) { return (size_t)((row >> 4) * 4 + (row & 3)) * 64 + ((row & 15) >> 2) * 16 + column; });
#ifdef GP_TILE_PROF
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        GP_PROBE(5);
#endif
        return false;
    }
};

}  // namespace gp
