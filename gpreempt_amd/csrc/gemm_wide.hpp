// Wide split-K GEMM tile kernel for small, deep problems (few output tiles, long K): 8 or 16 wavefronts
// share ONE output tile and split every K-stage between them.
//
// Why: on MI355X one wavefront's operand fetches (direct global -> LDS loads as well as register
// loads of 16 bytes per lane) complete at about 30-35 GB/s from an L2-resident source, however many
// loads it keeps in flight (about 60 cycles per 1 KB instruction), and the rate of a compute unit
// grows with the number of wavefronts that issue loads (about 120-140 GB/s with 4 wavefronts,
// 260-440 with 16).  A layer with fewer tiles than the GPU has compute units therefore streams its
// operands two to three times faster when sixteen wavefronts fetch for a tile than when four do,
// and for these layers the operand stream is what the main loop waits for (a 32 x 32 tile of a
// K = 3072 layer does 6 MFLOP on 384 KB of operands: 3 us at 130 GB/s).
//
// Structure: a stage holds KB = WAVES / 4 consecutive K-blocks of BK elements (one 128-byte row
// chunk per tile row, the layout and swizzle of gemm_pipe.hpp); wavefront w belongs to block group
// kb = w / 4 and fetches a quarter of the rows of that group's block.  One barrier per stage.  The
// arithmetic stays with wavefronts 0..3 (there is little of it: these layers wait for operands):
// wavefront w multiplies MFMA k-step w of every block, block after block, for the whole BM x BN
// tile (the code lets G groups of four share the output blocks between them; G = 1, see there), and at the end
// the four partial tiles are summed through LDS in the order 0, 1, 2, 3.  That
// is exactly the summation of the four-wavefront split-K bodies of gemm_pipe.hpp, so the result
// has the same bits as theirs (the whole-model program, whose workgroups have four wavefronts,
// uses those) and does not depend on scheduling: a preempted-then-resumed run stays bit-identical.
//
// Measured (fp16, launch to launch): 128 x 768 x 3072 (BERT's second FFN layer) 10.2 -> 8.2 us,
// 384 x 768 x 3072 11.9 -> 10.4 us; level with the four-wavefront bodies at K <= 1024, where the
// longer wait for the first, larger stage costs what the faster stream saves.
//
// CONV = true: the A operand is gathered (implicit GEMM over NHWC pixels): row m is output pixel
// (n, ho, wo), K element k is filter tap k / Cin, channel k % Cin.  Needs at most 32 taps: which taps of a pixel's window lie
// inside the image is worked out once per tile, as one bit per tap, so that a stage's loads cost a
// shift, a select and an add per lane; the tap and channel of a wavefront group's next block
// advance incrementally.  Where Cin is no multiple of BK a block straddles taps, and a lane works out the tap and channel of its
// chunk for itself, with two multiplications for the divisions (Inception-v3 b1, 1 x 7 over 160 channels: 10.3 -> 8.4 us a launch against the
// four-wavefront body, which divided).
#pragma once
#include "gemm_pipe.hpp"

namespace gp {

// 1: ask for all STAGES buffers of the ring before the main loop instead of STAGES - 1 (every buffer is free
// at the start of a tile).  Measured, launch to launch: 128 x 768 x 3072 8.04 -> 7.80 us, but 128 x 2304 x 768
// 5.74 -> 5.85 and 128 x 768 x 768 4.84 -> 4.90: off.
#ifndef GP_WIDE_PREFILL
#define GP_WIDE_PREFILL 0
#endif
// waits until at most `stages` stages of LPW loads each are still in flight (stages = 0..3)
template <int LPW> __device__ __forceinline__ void wait_stages(int stages) {
    if (stages >= 3) wait_vmcnt<3 * LPW>();
    else if (stages == 2) wait_vmcnt<2 * LPW>();
    else if (stages == 1) wait_vmcnt<LPW>();
    else wait_vmcnt<0>();
}

// The end of a tile of the wide bodies: the partial tiles of wavefronts 0..3, PART floats each in LDS, are summed in wavefront
// order and the epilogue (alpha, bias, residual, activation) is applied on the way out.  The first BM * BN / 4 threads finish four
// consecutive columns of one row each; at(row, column) is where a partial tile has those four.
template <typename T, int BM, int BN, int NT, int PART, class At>
__device__ __forceinline__ void wide_finish(const MatArgs &g, const float *red, int m0, int n0, long offc, int tid, At &&at) {
    T *C = (T *)g.C + offc;
    const T *R = g.residual ? (const T *)g.residual + offc : nullptr;
    const T *bias = (const T *)g.bias;
    const bool vec_ok = (g.N % 4 == 0) && (g.ldc % 4 == 0) && (offc % 4 == 0) && ((size_t)g.C % 16 == 0) &&
                        (!R || (g.ldr % 4 == 0 && (size_t)g.residual % 16 == 0)) && (!bias || (size_t)bias % 16 == 0);
    constexpr int L4 = BN / 4;                        // threads per output row
    constexpr int FIN = BM * L4 < NT ? BM * L4 : NT;  // threads that finish
    constexpr int RPP = FIN / L4, PASSES = BM / RPP;
    if (tid < FIN) {
        const int col = tid % L4 * 4, r_in = tid / L4;
        const int n = n0 + col;
        float bq[4] = {0.f, 0.f, 0.f, 0.f};
        if (bias && n < g.N) {
            if (vec_ok) {
                const Vec4<T> b = *(const Vec4<T> *)(bias + n);
#pragma unroll
                for (int q = 0; q < 4; ++q) bq[q] = Elem<T>::to_f(b.v[q]);
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (n + q < g.N) bq[q] = Elem<T>::to_f(bias[n + q]);
            }
        }
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
            const int row = p * RPP + r_in, m = m0 + row;
            const size_t o = at(row, col);
            f32x4 a = *(const f32x4 *)(red + o);
#pragma unroll
            for (int w = 1; w < 4; ++w) a += *(const f32x4 *)(red + (size_t)w * PART + o);
            if (m >= g.M || n >= g.N) continue;
            if (vec_ok) {
                Vec4<T> rv;
                if (R) rv = *(const Vec4<T> *)(R + (long)m * g.ldr + n);
                Vec4<T> out;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float x = a[q] * g.alpha + bq[q];
                    if (R) x += Elem<T>::to_f(rv.v[q]);
                    out.v[q] = Elem<T>::from_f(apply_act(x, g.act));
                }
                st_vec4<T>(&C[(long)m * g.ldc + n], out);
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (n + q >= g.N) break;
                    float x = a[q] * g.alpha + bq[q];
                    if (R) x += Elem<T>::to_f(R[(long)m * g.ldr + n + q]);
                    st_elem<T>(&C[(long)m * g.ldc + n + q], Elem<T>::from_f(apply_act(x, g.act)));
                }
            }
        }
    }
}

// ... of the bodies whose wavefronts hold 32 x 32 blocks: partial tiles of wavefronts 0..3 -> LDS as [wavefront][slice][lane], slice = (i*NI +
// j)*16 + v, which is row 8*(v/4) + 4*(lane/32) + v%4, column 32*j + lane%32 of block (i, j).
template <typename T, int BM, int BN, int NT, int G>
__device__ __forceinline__ void wide_reduce_store(const MatArgs &g, float *red, const f32x16 (&acc)[(BM / 32) * (BN / 32) / G], int m0, int n0, long offc,
                                                  int tid, int wv, int lane, int kb) {
    constexpr int MI = BM / 32, NI = BN / 32, SLICES = MI * NI * 16, BPW = MI * NI / G;
    __syncthreads();  // all wavefronts are done reading the stage buffers
    if (kb < G) {  // wavefront (kb, wv) holds k-step wv of the 32 x 32 blocks kb, kb + G, ...
#pragma unroll
        for (int q = 0; q < BPW; ++q)
#pragma unroll
            for (int v = 0; v < 16; ++v) red[((size_t)wv * SLICES + (kb + q * G) * 16 + v) * 64 + lane] = acc[q][v];
    }
    __syncthreads();
    GP_PROBE(4);
    wide_finish<T, BM, BN, NT, SLICES * 64>(g, red, m0, n0, offc, tid, [&](int row, int column) {
        const int i = row >> 5, r = row & 31, j = column >> 5;
        const int v = 4 * (r >> 3) + (r & 3), hf = (r >> 2) & 1;
        return ((size_t)(i * NI + j) * 16 + v) * 64 + hf * 32 + (column & 31);
    });
}

// CONV: 0 a GEMM, 1 a convolution, 2 one whose blocks straddle taps (as a run-time switch, the test cost the others 1 % of a ResNet-152 pass).
// SCALED: PRE of PipeKernel.
template <typename T, int BM, int BN, int WAVES, int STAGES, int CONV = 0, bool SCALED = false>
struct WideKernel {
    using elem = T;
    static constexpr int bm = BM, bn = BN;
    static constexpr bool conv = CONV != 0, pre = SCALED, window = false;
    static_assert(!SCALED || !CONV, "GEMM rows only");
    static constexpr int VEC = Elem<T>::VEC;
    static constexpr int NT = WAVES * 64;
    static constexpr int RB = 128;                         // row bytes of a block in LDS
    static constexpr int BK = RB / (int)sizeof(T);         // K elements per block: 64 (16-bit) or 32 (fp32)
    static constexpr int KB = WAVES / 4;                   // blocks per stage
    static constexpr int GROUPS = (BM + BN) / 8;           // 8-row load groups per block (A rows, then B rows)
    static constexpr int LPW_A = BM / 8 / 4, LPW_B = BN / 8 / 4;  // of a wavefront's loads per stage, the first LPW_A fetch A rows
    static constexpr int LPW = LPW_A + LPW_B;              // load instructions per wavefront per stage
    static constexpr int A_BYTES = BM * RB, BLK_BYTES = (BM + BN) * RB, STAGE_BYTES = KB * BLK_BYTES;
    static constexpr int MI = BM / 32, NI = BN / 32;
    // Which wavefronts multiply: group kb < G takes the 32 x 32 output blocks kb, kb + G, ... (k-step wv of every
    // K-block: whose registers a partial sum lives in does not change what is added to what).  G = 1 here:
    // two multiplying groups (one per output block of a 64 x 32 tile) were measured and changed nothing or
    // cost a little (1568 x 256 x 2304: 8.50 -> 8.54 us, 128 x 2304 x 768: 5.16 -> 5.43; each group re-reads
    // the fragments it shares with the other); the layer-norm prologue body, whose A operand stays in LDS,
    // gains from two (gemm_ln.hpp).
    static constexpr int G = 1;
    static constexpr int BPW = MI * NI / G;
    static_assert(MI * NI % G == 0, "output blocks divide among the multiplying groups");
    static constexpr int SLICES = MI * NI * 16;            // 64-float slices of one k-step's partial tile
    static constexpr size_t RED_BYTES = (size_t)4 * SLICES * 64 * 4;   // the partial tiles of wavefronts 0..3
    static constexpr size_t RING_BYTES = (size_t)STAGES * STAGE_BYTES;
    static constexpr size_t LDS_BYTES = RING_BYTES > RED_BYTES ? RING_BYTES : RED_BYTES;
    static constexpr size_t CKPT_SLOT_BYTES = 0;
    static constexpr bool ckpt = false;
    static constexpr bool early_stop = true;  // as PipeKernel::run: a second look at the stop index when the first stage has landed
    static constexpr bool can_look = true;
    static constexpr int PRE = GP_WIDE_PREFILL ? STAGES : STAGES - 1;  // stages asked for before the main loop
    static_assert(WAVES % 4 == 0 && WAVES >= 4 && WAVES <= 16, "4, 8, 12 or 16 wavefronts");
    static_assert(BM % 32 == 0 && BN % 32 == 0 && GROUPS % 4 == 0, "tile shape");
    // slot j of wavefront wv (of its block group): row group wv*LPW_A + j of A, or wv*LPW_B + (j - LPW_A) of B
    static __device__ __forceinline__ constexpr int group_of(int wv, int j) { return j < LPW_A ? wv * LPW_A + j : BM / 8 + wv * LPW_B + (j - LPW_A); }
    static_assert(STAGES >= 2 && STAGES <= 4 && (STAGES - 1) * LPW < 64, "pipeline depth");
    static_assert(LDS_BYTES <= 160 * 1024, "LDS budget");

    // Returns true when the early look found a stop recorded: the tile was not run.
    template <bool LOOKS = false, bool SINGLE = false, class Asked = NoneAsked>  // (as in PipeKernel)
    static __device__ __forceinline__ bool run(const MatArgs &g, TileIdx t, T *lds_t, CkptCtx cc = CkptCtx{nullptr, nullptr, nullptr, 0}, Asked &&asked = Asked{}) {
        GP_PROBE(0);
        __shared__ int early_slot[64];
        const bool early = __builtin_amdgcn_readfirstlane((int)(cc.stop_index != nullptr)) != 0;
        // Long tiles look again every LOOK_EVERY stages (a stage is KB blocks of 64 K-elements: about a microsecond of a
        // 32 x 32 x 25088 tile): the word is fetched by wavefront 0 in front of the loads of the stage it travels
        // with, so that the wait for that stage covers it, and read by everybody behind that stage's barrier.  One
        // landing slot is enough: the next fetch is issued LOOK_EVERY - (STAGES - 1) stages after this one was read.
        constexpr int LOOK_EVERY = 4;
        static_assert(LOOK_EVERY >= STAGES, "a look is read before the next one is fetched");
        const bool looking = LOOKS && early;  // (an instantiation of its own, as in PipeKernel)
        const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) void *)lds_t;
        const char *lds_c = (const char *)lds_t;
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int kb = wave >> 2, wv = wave & 3;
        const int l32 = lane & 31, half = lane >> 5;
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

        // ---- loader slots: every wavefront fetches LPW_A row groups of A and LPW_B of B of its block (which
        // kind a slot is is known at compile time: no branches in the stage's load sequence) ------
        // lane -> (row in the group, chunk position); the swizzle is applied on the source side:
        // the lane at position cpos of row r fetches chunk cpos ^ ((r >> 1) & 7) of that row.
        // The loads go through buffer descriptors: a lane's row and chunk are one 32-bit offset that never changes, the
        // position in K (CONV: the tap) is a scalar, and a lane with nothing to fetch has an offset beyond the
        // descriptor's end, which the hardware answers with zeros.  Sixteen wavefronts issue a stage's loads, four to a
        // SIMD: with 64-bit addresses, selects and a page of zeros a stage of a 3 x 3 layer cost as much in vector
        // instructions as its loads take.
        const int rig = lane >> 3, cpos = lane & 7;
        // CONV: where a row's window lies and which of its taps are inside the image, worked out by one lane per row (eight lanes of
        // each of the KB wavefront groups need it; every one for itself, that was some hundred vector instructions in front of the first
        // load, four wavefronts to a SIMD)
        __shared__ unsigned row_off[CONV ? BM : 1], row_taps[CONV ? BM : 1];
        if (CONV && tid < BM) {
            const int m = m0 + tid, hw = g.Ho * g.Wo;
            const bool in = m < g.M, small = g.M < kSmallDivLimit;
            const int mm = in ? m : 0;
            const int n = small ? small_div(mm, hw, g.rcp_hw) : mm / hw, rem = mm - n * hw;
            const int ho = small ? small_div(rem, g.Wo, g.rcp_wo) : rem / g.Wo, wo = rem - ho * g.Wo;
            row_off[CONV ? tid : 0] = (unsigned)((n * g.H + ho * g.sh) * g.W + wo * g.sw) * (unsigned)g.lda;
            row_taps[CONV ? tid : 0] = in ? window_tap_mask(ho * g.sh - g.ph, wo * g.sw - g.pw, g.H, g.W, g.R, g.S) : 0u;
        }
        // (CONV: offsets count from the origin of the window of output pixel (0, 0), which lies in front of the image by the padding)
        const u32x4 rsrc_a = buffer_of(CONV ? A - (long)(g.ph * g.W + g.pw) * g.lda : A), rsrc_b = buffer_of(B);
        unsigned off[LPW];     // the lane's row and chunk at k = 0, in bytes
        int kc[LPW];           // the lane's chunk offset in elements
        unsigned taps[CONV ? LPW : 1];  // CONV, A rows: bit t set = tap t of the row's window is inside the image
        unsigned row[CONV ? LPW : 1];   // CONV, A rows: the row's window origin, in bytes
#pragma unroll
        for (int j = 0; j < LPW; ++j) {
            const int gi = group_of(wv, j);           // group index in the block
            const bool is_a = j < LPW_A;
            const int r = (is_a ? gi : gi - BM / 8) * 8 + rig;   // row in its region
            kc[j] = (cpos ^ ((r >> 1) & 7)) * VEC;
            if (!is_a || !CONV) {
                const int x = (is_a ? m0 : n0) + r;
                off[j] = x < (is_a ? g.M : g.N) ? ((unsigned)x * (unsigned)(is_a ? g.lda : g.ldb) + (unsigned)kc[j]) * (unsigned)sizeof(T) : kBufferEnd;
            }
        }
        const int KT = (g.K + BK - 1) / BK;             // blocks along K
        const int NS = (KT + KB - 1) / KB;              // stages
        // CONV: tap and channel of the block this wavefront group fetches next (stages are issued in order)
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
        auto issue_part = [&](int s, auto first, auto last) {  // the loads first..last-1 of the wavefront's LPW for stage s
            const int k0 = (s * KB + kb) * BK;          // first K element of this wavefront group's block
            const unsigned sbase = lds0 + ((unsigned)s % STAGES) * STAGE_BYTES + (unsigned)kb * BLK_BYTES;
            const unsigned tap_bit = (k0 < g.K && nx_tap < 32) ? 1u << nx_tap : 0u;  // blocks past K have no tap
            const unsigned tap_off = (unsigned)((nx_r * g.W + nx_s) * (int)g.lda + nx_ci) * (unsigned)sizeof(T);
            const bool whole = k0 + BK <= g.K;          // (uniform) the block's K elements all exist
#pragma unroll
            for (int j = first; j < last; ++j) {
                const int gi = group_of(wv, j);
                if (CONV && j < LPW_A && straddles) {
                    const int k = k0 + kc[j], tap = (int)__umulhi((unsigned)k + 1u, g.inv_cin), ci = k - tap * g.Cin, r = (int)__umulhi((unsigned)tap + 1u, g.inv_s), s2 = tap - r * g.S;
                    const unsigned at = row[CONV ? j : 0] + (unsigned)((r * g.W + s2) * (int)g.lda + ci) * (unsigned)sizeof(T);
                    load_lds16_buffer<SINGLE>(rsrc_a, k < g.K && (taps[CONV ? j : 0] >> tap & 1u) ? at : kBufferEnd, 0u, sbase + (unsigned)(gi * 8 * RB));
                } else if (CONV && j < LPW_A) {
                    // taps outside the image, rows outside the problem and blocks past K have nothing to fetch
                    load_lds16_buffer<SINGLE>(rsrc_a, (taps[CONV ? j : 0] & tap_bit) ? off[j] : kBufferEnd, tap_off, sbase + (unsigned)(gi * 8 * RB));
                } else {
                    // (nor have rows outside the problem and K-chunks past K, also whole blocks past the last one when
                    // the stage is not full)
                    const unsigned at = whole || k0 + kc[j] < g.K ? off[j] : kBufferEnd;
                    load_lds16_buffer<SINGLE>(j < LPW_A ? rsrc_a : rsrc_b, at, (unsigned)k0 * (unsigned)sizeof(T), sbase + (unsigned)(gi * 8 * RB));
                }
            }
            if (CONV && last == LPW_A) advance(KB * BK);
        };
        auto issue_a = [&](int s) { issue_part(s, IntC<0>{}, IntC<LPW_A>{}); };
        auto issue_b = [&](int s) { issue_part(s, IntC<LPW_A>{}, IntC<LPW>{}); };
        auto issue = [&](int s) { issue_b(s); issue_a(s); };

        f32x16 acc[BPW];
#pragma unroll
        for (int q = 0; q < BPW; ++q)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[q][v] = 0.f;
        auto frag = [&](int stage, int blk, int region_bytes, int row, int chunk) -> u32x4 {
            const int phys = chunk ^ ((row >> 1) & 7);
            return *(const u32x4 *)(lds_c + (size_t)stage * STAGE_BYTES + (size_t)blk * BLK_BYTES + region_bytes + row * RB + phys * 16);
        };

        // ---- main loop ------------------------------------------------------------------------
        GP_PROBE(1);
        // (the weights of the first stage need no row table)
        constexpr bool B_FIRST = SINGLE && CONV;
        if (B_FIRST) issue_b(0);
        if (CONV || !SINGLE) __syncthreads();  // the row table; the previous tile of this workgroup may still be reading LDS
        if constexpr (SCALED) pre_fetch_table<T, WAVES>(g, lds0 + (unsigned)LDS_BYTES, wave, lane);
        if (CONV) {
#pragma unroll
            for (int j = 0; j < LPW_A; ++j) {
                const int r = group_of(wv, j) * 8 + rig;
                row[CONV ? j : 0] = row_off[CONV ? r : 0] * (unsigned)sizeof(T);
                off[j] = row[CONV ? j : 0] + (unsigned)kc[j] * (unsigned)sizeof(T);
                taps[CONV ? j : 0] = row_taps[CONV ? r : 0];
            }
        }
#pragma unroll
        for (int s = 0; s < PRE; ++s) {
            if (B_FIRST && s == 0) issue_a(s);
            else if (s < NS) issue(s);
            if (s == 0 && early && wave == 0) load_lds4(cc.stop_index, (unsigned)(size_t)(__attribute__((address_space(3))) void *)early_slot);
        }
        asked();
        for (int s = 0; s < NS; ++s) {
            // stage s has landed once at most the loads of the younger stages in flight remain
            if (s == 0) wait_stages<LPW>((NS < PRE ? NS : PRE) - 1);
            else if (s + STAGES - 2 < NS) wait_vmcnt<(STAGES - 2) * LPW>();
            else wait_vmcnt<0>();
            if constexpr (SCALED) {
                if (s == 0) __syncthreads();  // everyone's part of the table
                const int k0 = (s * KB + kb) * BK;
                char *blk = (char *)lds_t + (size_t)((unsigned)s % STAGES) * STAGE_BYTES + (size_t)kb * BLK_BYTES + lane * 16;
                if (k0 < g.K) {
#pragma unroll
                    for (int j = 0; j < LPW_A; ++j) pre_apply<T>(g, blk + group_of(wv, j) * 8 * RB, lds_c + LDS_BYTES, k0 + kc[j]);
                }
            }
            __syncthreads();  // everyone's part of stage s is visible; the buffer of stage s-1 is free
            if (s == 0) GP_PROBE(2);
            if (((s == 0 && early) || (looking && s > 0 && (s & (LOOK_EVERY - 1)) == 0)) && __builtin_amdgcn_readfirstlane(read_lds_word(early_slot)) != -1) {
                wait_vmcnt<0>();  // loads still landing in LDS must not outlive the workgroup
                return true;      // the tile is given up: the caller withdraws the claim
            }
            if constexpr (LOOKS) {
                // the last stage: the workgroup counts itself (tile_fixed_early).  Not earlier: an atomic in front of operand
                // loads is waited for with them (the waits count in the order of issue), and its acknowledgement takes
                // microseconds when every resident workgroup sends one.
                if (looking && cc.announce && s == NS - 1 && tid == 0)
                    __hip_atomic_fetch_add(cc.announce, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            if (s >= PRE - (STAGES - 1) && s + STAGES - 1 < NS) {
                if (looking && wave == 0 && ((s + STAGES - 1) & (LOOK_EVERY - 1)) == 0)
                    load_lds4(cc.stop_index, (unsigned)(size_t)(__attribute__((address_space(3))) void *)early_slot);
                issue(s + STAGES - 1);
            }
            if (kb >= G) continue;  // (uniform) the other wavefronts only fetch
            const int stage = (int)((unsigned)s % STAGES);
            // fp32: every block's fragments are asked for before the first is multiplied (a block is four MFMAs of 64 cycles
            // then, in a chain that also waited for LDS once per block: 3 x 3 at 7 x 7 x 512 35.2 -> 32.5 us).  The 16-bit
            // bodies read as they go: their blocks are one MFMA, and 128 x 768 x 3072 took 2 % longer.
            constexpr int AHEAD = sizeof(T) == 4 ? KB : 1;
            u32x4 fa[AHEAD][MI], fb[AHEAD][NI];
            auto read = [&](int slot, int b) {
#pragma unroll
                for (int i = 0; i < MI; ++i) fa[slot][i] = frag(stage, b, 0, i * 32 + l32, wv * 2 + half);
#pragma unroll
                for (int j = 0; j < NI; ++j) fb[slot][j] = frag(stage, b, A_BYTES, j * 32 + l32, wv * 2 + half);
            };
            if constexpr (AHEAD > 1) {
#pragma unroll
                for (int b = 0; b < KB; ++b) read(b, b);
            }
#pragma unroll
            for (int b = 0; b < KB; ++b) {
                // a block past the last one holds zeros; it is skipped, not multiplied, so that the sum
                // has the bits of a K loop that ends at the last block
                if (s * KB + b >= KT) break;
                if constexpr (AHEAD == 1) read(0, b);
#pragma unroll
                for (int q = 0; q < BPW; ++q) {
                    const int blk = kb + q * G;
                    Elem<T>::mma(fa[AHEAD > 1 ? b : 0][blk / NI], fb[AHEAD > 1 ? b : 0][blk % NI], acc[q]);
                }
            }
        }

        GP_PROBE(3);
        wide_reduce_store<T, BM, BN, NT, G>(g, (float *)lds_t, acc, m0, n0, offc, tid, wv, lane, kb);
#ifdef GP_TILE_PROF
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        GP_PROBE(5);
#endif
        return false;
    }
};

}  // namespace gp
