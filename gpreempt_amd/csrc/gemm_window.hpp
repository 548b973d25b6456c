// Convolution bodies of the wide kind that keep their input window in LDS.
//
// Why: as an implicit GEMM a 3 x 3 layer fetches every input pixel nine times, and a row's window has to be worked out in front of its first
// load.  At stride 1 and with an output as large as the input, the pixels that a tile's rows read at a tap are consecutive ones
// (consecutive pixels of the flattened images, moved by the tap), so all taps together read BM + 2 * (ph * W + pw) consecutive pixels:
// 62 for 32 rows of a 14 x 14 image.  They are fetched once, in front of the first stage, only the weights stream through the ring, and
// the rows' masks are worked out while the loads are under way.  Launches of 32 x 32 tiles: 4 x 14 x 14 x 128 -> 32 channels 7.3 -> 6.3 us,
// 8 x 7 x 7 x 512 13.1 -> 12.0, 1 x 17 x 17 x 192 7.7 -> 7.2.  Not for 64 x 32 tiles, where the instruction stream of the four
// multiplying wavefronts bounds a stage and a fragment's address costs more than the ring's: ResNet-152 b8 1530 -> 1560 us with them.
//
// Structure: as gemm_wide.hpp (sixteen wavefronts fetch, 0..3 multiply one MFMA k-step each of every block, the same sums in the same
// order, hence the same bits).  The window lies behind the ring, K-block after K-block of Cin, rows of 128 bytes swizzled like the
// ring's; a lane's row at a tap is its own row moved by the tap, or a row of zeros where the tap is outside the image.
#pragma once
#include "gemm_wide.hpp"

namespace gp {

constexpr size_t kWindowMaxLds = 156 * 1024;  // of the 160 KB, with the ring (the rest is for the bodies' and the dispatcher's own words)
// rows of the window in LDS (whole groups of eight), and its bytes with the row of zeros
inline __host__ __device__ int window_rows(const MatArgs &g, int bm) { return (bm + 2 * (g.ph * g.W + g.pw) + 7) & ~7; }
inline __host__ __device__ size_t window_bytes(const MatArgs &g, int bm, int es) { return (size_t)window_rows(g, bm) * (size_t)g.Cin * (size_t)es + 128; }

template <typename T, int BM, int BN, int STAGES>
struct WindowKernel {
    using elem = T;
    static constexpr int bm = BM, bn = BN;
    static constexpr bool conv = true, pre = false, window = true;
    static constexpr int VEC = Elem<T>::VEC, WAVES = 16, NT = WAVES * 64, RB = 128, BK = RB / (int)sizeof(T), KB = WAVES / 4;
    static constexpr int LPW = BN / 8 / 4;                 // B row groups a wavefront fetches per stage
    static constexpr int BLK_BYTES = BN * RB, STAGE_BYTES = KB * BLK_BYTES;
    static constexpr int MI = BM / 32, NI = BN / 32;
    static constexpr size_t RED_BYTES = (size_t)4 * MI * NI * 16 * 64 * 4, RING_BYTES = (size_t)STAGES * STAGE_BYTES;
    static constexpr size_t LDS_BYTES = RING_BYTES > RED_BYTES ? RING_BYTES : RED_BYTES;  // without the window
    static constexpr size_t CKPT_SLOT_BYTES = 0;
    static constexpr bool ckpt = false, early_stop = true, can_look = true;  // (as WideKernel)
    static_assert(BM % 32 == 0 && BN % 32 == 0 && LPW >= 1 && STAGES >= 2 && STAGES <= 4, "tile shape");

    template <bool LOOKS = false, bool SINGLE = false, class Asked = NoneAsked>
    static __device__ __forceinline__ bool run(const MatArgs &g, TileIdx t, T *lds_t, CkptCtx cc = CkptCtx{nullptr, nullptr, nullptr, 0}, Asked &&asked = Asked{}) {
        GP_PROBE(0);
        __shared__ int early_slot[64];
        __shared__ unsigned row_taps[BM];  // bit t: tap t of the row's window is inside the image
        const bool early = __builtin_amdgcn_readfirstlane((int)(cc.stop_index != nullptr)) != 0;
        constexpr int LOOK_EVERY = 4;  // (see WideKernel)
        static_assert(LOOK_EVERY >= STAGES, "a look is read before the next one is fetched");
        const bool looking = LOOKS && early;
        const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) void *)lds_t;
        const char *lds_c = (const char *)lds_t;
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int kb = wave >> 2, wv = wave & 3;
        const int l32 = lane & 31, half = lane >> 5;
        const int m0 = t.y * BM, n0 = t.x * BN;
        const T *A = (const T *)g.A, *B = (const T *)g.B;
        const int rows = window_rows(g, BM), origin = m0 - g.ph * g.W - g.pw;  // window row r is pixel origin + r of the flattened images
        const int blocks = g.Cin / BK;
        const unsigned win = (unsigned)LDS_BYTES, zeros = win + (unsigned)(blocks * rows * RB);

        // ---- weights: as WideKernel's B ---------------------------------------------------------------------
        const int rig = lane >> 3, cpos = lane & 7;
        const u32x4 rsrc_a = buffer_of(A), rsrc_b = buffer_of(B);
        unsigned off[LPW];
#pragma unroll
        for (int j = 0; j < LPW; ++j) {
            const int r = (wv * LPW + j) * 8 + rig, x = n0 + r;
            off[j] = x < g.N ? ((unsigned)x * (unsigned)g.ldb + (unsigned)((cpos ^ ((r >> 1) & 7)) * VEC)) * (unsigned)sizeof(T) : kBufferEnd;
        }
        const int KT = g.K / BK;             // blocks along K (Cin is a multiple of BK)
        const int NS = (KT + KB - 1) / KB;   // stages
        auto issue = [&](int s) {
            const int k0 = (s * KB + kb) * BK;
            const unsigned sbase = lds0 + ((unsigned)s % STAGES) * STAGE_BYTES + (unsigned)kb * BLK_BYTES;
#pragma unroll
            for (int j = 0; j < LPW; ++j)  // (whole blocks past the last one, when the stage is not full: zeros)
                load_lds16_buffer<SINGLE>(rsrc_b, k0 < g.K ? off[j] : kBufferEnd, (unsigned)k0 * (unsigned)sizeof(T), sbase + (unsigned)((wv * LPW + j) * 8 * RB));
        };

        if (!SINGLE) __syncthreads();  // the previous tile of this workgroup may still be reading LDS
        // ---- the window: groups of eight rows of a block, dealt out to the wavefronts -------------------------------
        const int groups = rows >> 3;
        for (int blk = 0, gi = wave; blk < blocks; gi += WAVES) {
            while (gi >= groups) { gi -= groups; ++blk; }
            if (blk >= blocks) break;
            const int r = gi * 8 + rig, pixel = origin + r;
            const unsigned at = ((unsigned)pixel * (unsigned)g.lda + (unsigned)((cpos ^ ((r >> 1) & 7)) * VEC)) * (unsigned)sizeof(T);
            load_lds16_buffer<SINGLE>(rsrc_a, (unsigned)pixel < (unsigned)g.M ? at : kBufferEnd, (unsigned)(blk * RB), lds0 + win + (unsigned)((blk * rows + gi * 8) * RB));
        }
#pragma unroll
        for (int s = 0; s < STAGES - 1; ++s) {
            if (s < NS) issue(s);
            if (s == 0 && early && wave == 0) load_lds4(cc.stop_index, (unsigned)(size_t)(__attribute__((address_space(3))) void *)early_slot);
        }
        asked();
        if (tid < 32) *(int *)((char *)lds_t + zeros + tid * 4) = 0;
        if (tid < BM) {
            const int m = m0 + tid, hw = g.Ho * g.Wo;
            const bool in = m < g.M, small = g.M < kSmallDivLimit;
            const int mm = in ? m : 0;
            const int n = small ? small_div(mm, hw, g.rcp_hw) : mm / hw, rem = mm - n * hw;
            const int ho = small ? small_div(rem, g.Wo, g.rcp_wo) : rem / g.Wo, wo = rem - ho * g.Wo;
            row_taps[tid] = in ? window_tap_mask(ho - g.ph, wo - g.pw, g.H, g.W, g.R, g.S) : 0u;
        }

        f32x16 acc[MI * NI];
#pragma unroll
        for (int q = 0; q < MI * NI; ++q)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[q][v] = 0.f;
        unsigned taps[MI];
        int nx_tap = 0, nx_s = 0, nx_shift = 0, nx_blk = 0;  // of the next block: tap, its column, how far it moves a row, and K-block of Cin

        // ---- main loop ------------------------------------------------------------------------
        GP_PROBE(1);
        for (int s = 0; s < NS; ++s) {
            if (s == 0) wait_stages<LPW>((NS < STAGES - 1 ? NS : STAGES - 1) - 1);
            else if (s + STAGES - 2 < NS) wait_vmcnt<(STAGES - 2) * LPW>();
            else wait_vmcnt<0>();
            __syncthreads();  // everyone's part of stage s (and, the first time, of the window) is visible; the buffer of stage s-1 is free
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
            if (kb >= 1) continue;  // (uniform) the other wavefronts only fetch
            if (s == 0) {
#pragma unroll
                for (int i = 0; i < MI; ++i) taps[i] = row_taps[i * 32 + l32];
            }
            const int stage = (int)((unsigned)s % STAGES);
            // every block's fragments are asked for before the first is multiplied
            u32x4 fa[KB][MI], fb[KB][NI];
#pragma unroll
            for (int b = 0; b < KB; ++b) {
#pragma unroll
                for (int i = 0; i < MI; ++i) {
                    const int row = i * 32 + l32 + nx_shift;
                    const unsigned at = win + (unsigned)((nx_blk * rows + row) * RB + ((wv * 2 + half) ^ ((row >> 1) & 7)) * 16);
                    fa[b][i] = *(const u32x4 *)(lds_c + (s * KB + b < KT && (taps[i] >> nx_tap & 1u) ? at : zeros));
                }
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    const int row = j * 32 + l32;
                    fb[b][j] = *(const u32x4 *)(lds_c + (size_t)stage * STAGE_BYTES + (size_t)b * BLK_BYTES + row * RB + ((wv * 2 + half) ^ ((row >> 1) & 7)) * 16);
                }
                if (++nx_blk == blocks) {
                    nx_blk = 0;
                    ++nx_tap;
                    ++nx_shift;
                    if (++nx_s == g.S) { nx_s = 0; nx_shift += g.W - g.S; }
                }
            }
#pragma unroll
            for (int b = 0; b < KB; ++b) {
                if (s * KB + b >= KT) break;  // a block past the last one is skipped (see WideKernel)
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int j = 0; j < NI; ++j) Elem<T>::mma(fa[b][i], fb[b][j], acc[i * NI + j]);
            }
        }

        GP_PROBE(3);
        wide_reduce_store<T, BM, BN, NT, 1>(g, (float *)lds_t, acc, m0, n0, 0, tid, wv, lane, kb);
#ifdef GP_TILE_PROF
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        GP_PROBE(5);
#endif
        return false;
    }
};

}  // namespace gp
