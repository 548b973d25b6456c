// Fused scaled-dot-product attention; a tile is one (batch, head, 64-query block):
//   O = softmax(Q K^T * scale) V      with head dimension 64, 16-bit operands, fp32 softmax.
//
// It replaces three launches (batched Q K^T, row softmax, batched P V) and the two S x S score
// tensors they pass through memory.  A wavefront takes 32 queries and a share of the keys and computes the
// transposed scores S^T = K Q^T with v_mfma_f32_32x32x16: in the accumulator layout a lane then holds, for
// ITS query (column lane%32), the scores of keys 8*(v/4) + 4*(lane/32) + v%4 of every 32-key
// block, so the row softmax is a reduction over the lane's own registers plus one exchange with
// lane^32, and the probabilities are already laid out as the B operand of O^T = V^T P^T:
// an MFMA only needs A and B to agree on which K indices a (lane, register) pair stands for,
// and V^T is staged in LDS so that the A fragments can be gathered in that same key order.
#pragma once
#include "mma.hpp"

namespace gp {

struct AttnArgs {
    gp_attention_params p;
};

constexpr int ATT_D = 64;        // head dimension
constexpr int ATT_QB = 64;       // query rows per tile
constexpr int ATT_OP = ATT_D + 4;  // floats from one row of a partial result to the next: 8 lanes' 16-byte writes cover all banks once
__host__ __device__ inline int attention_key_blocks(int seq) { return (seq + 31) / 32; }
// Wavefronts that share the keys of 32 queries, by the class of the sequence length.  Two up to 256 keys: with four, the partial results are most of what
// goes through LDS (12 heads x 128 keys x 32 sequences 14.1 us instead of 11.5, x 256 keys x 4 10.0 instead of 8.9).  Four beyond: a wavefront's scores
// and keys then fit into 128 registers, two workgroups share a compute unit, and a wavefront's chain is half as long (12 x 512 x 2 15.6 us with two, 12.6 with four).
__host__ __device__ constexpr int attention_parts(int nb) { return nb >= 12 ? 4 : 2; }
__host__ __device__ constexpr int attention_threads(int nb) { return 2 * attention_parts(nb) * 64; }
// V^T, and in its place afterwards the partial results; the maxima and sums of the parts
__host__ __device__ inline size_t attention_sums_at(int nb) {
    const size_t vt = (size_t)ATT_D * (nb * 32 + 4) * 2, o = (size_t)attention_parts(nb) * ATT_QB * ATT_OP * sizeof(float);
    return ((vt > o ? vt : o) + 15) / 16 * 16;
}
__host__ __device__ inline size_t attention_lds_bytes(int nb) { return attention_sums_at(nb) + attention_parts(nb) * ATT_QB * 2 * sizeof(float); }

// What bounds a tile is its chain of dependent steps (operands from memory, V through LDS, scores, exponentials, P V, the merge): BERT's
// twelve heads are 24 tiles at 128 tokens, and a tile's arithmetic is a few hundred cycles of one compute unit.  So the chain of a wavefront is kept short:
// two or four wavefronts share the keys of 32 queries, each with its own running maximum (probabilities left unnormalised), and all of them
// merge: O = sum_i a_i O_i / sum_i a_i sum_i, a_i = exp(m_i - max m).  Everything a wavefront needs from memory is asked for
// at the start, V first, since its way through LDS is the longest.  O is computed transposed, so that a lane holds values of one query: its
// partial results leave in 16-byte writes, and a result's factors are read once per eight of its values.
// In turn with two wavefronts to 32 queries, V fetched and staged in front of everything else, and one of the two merging (f16, us per launch):
// 12 heads x 128 keys 6.5 -> 6.0, x 211 x 2 sequences 8.7 -> 7.9, x 384 11.2 -> 10.4, x 512 14.1 -> 11.8; where the tiles fill the device, 12 x 512 x 8 45 -> 29,
// 16 x 512 x 64 472 -> 255 (270 TFLOP/s; bound by the vector instructions of the softmax), 12 x 256 x 64 64 -> 54.
template <typename T, int NB>
__device__ __forceinline__ void attention_tile(const AttnArgs &a, TileIdx t, T *lds) {
    // (products and sums are contracted where the code says so and nowhere else, so that the kernels and the whole-model program, which are built around
    // this body, give the same bits)
#pragma clang fp contract(off)
    constexpr int PARTS = attention_parts(NB), NBW = NB / PARTS, THREADS = attention_threads(NB);
    static_assert(NB % PARTS == 0, "key blocks are shared evenly");
    const gp_attention_params &p = a.p;
    // padded row of V^T: consecutive rows (d) start 2 banks apart, so the 8-byte fragment reads of 16
    // lanes cover all 32 banks once
    constexpr int SP = NB * 32 + 4;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, half = lane >> 5;
    const int part = wave % PARTS, qg = wave / PARTS;  // keys and query group (wave-uniform)
    const int S = p.seq;
    const int head = t.y % p.heads, bat = t.y / p.heads;  // tile grid: x = query block, y = batch * heads + head
    const long tok0 = (long)bat * S;
    const T *Q = (const T *)p.q + tok0 * p.ld_qkv + (long)head * ATT_D;
    const T *K = (const T *)p.k + tok0 * p.ld_qkv + (long)head * ATT_D;
    const T *V = (const T *)p.v + tok0 * p.ld_qkv + (long)head * ATT_D;
    T *O = (T *)p.out + tok0 * p.ld_out + (long)head * ATT_D;
    T *vt = lds;
    float *partial = (float *)lds;
    float *sums = (float *)((char *)lds + attention_sums_at(NB));
    const u32x4 zero4 = {0, 0, 0, 0};

    // ---- all fetches.  A thread moves NB * 32 * 8 / THREADS chunks of eight values of V; a wavefront takes 64 consecutive keys of
    // one chunk, so its transposing 2-byte writes are 128 contiguous bytes per d, free of bank conflicts ----
    constexpr int CHUNKS = NB * 32 * (ATT_D / 8) / THREADS;
    u32x4 raw[CHUNKS], ak[NBW][4], bq[4];
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int idx = tid + c * THREADS, key = idx % (NB * 32), dc = idx / (NB * 32);
        raw[c] = key < S ? *(const u32x4 *)(V + (long)key * p.ld_qkv + dc * 8) : zero4;
    }
    const int q = t.x * ATT_QB + qg * 32 + l32;  // this lane's query row
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) bq[ks] = q < S ? *(const u32x4 *)(Q + (long)q * p.ld_qkv + ks * 16 + half * 8) : zero4;
#pragma unroll
    for (int i = 0; i < NBW; ++i) {
        const int key = (part * NBW + i) * 32 + l32;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) ak[i][ks] = key < S ? *(const u32x4 *)(K + (long)key * p.ld_qkv + ks * 16 + half * 8) : zero4;
    }

    // ---- V^T into LDS (keys past the sequence are zero: their probability is 0, but 0 * garbage could be NaN) ----
    __syncthreads();  // the previous tile of this workgroup may still be reading the partial results
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int idx = tid + c * THREADS, key = idx % (NB * 32), dc = idx / (NB * 32);
        const unsigned short *e = (const unsigned short *)&raw[c];
#pragma unroll
        for (int j = 0; j < 8; ++j) ((unsigned short *)vt)[(dc * 8 + j) * SP + key] = e[j];
    }
    __syncthreads();

    // ---- scores (transposed): s[i][v] = <K[key], Q[query]> ----
    f32x16 s[NBW];
#pragma unroll
    for (int i = 0; i < NBW; ++i) {
#pragma unroll
        for (int v = 0; v < 16; ++v) s[i][v] = 0.f;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) Elem<T>::mma(ak[i][ks], bq[ks], s[i]);
    }
    // ---- softmax over the part's keys of this lane's query, in powers of two ----
    const float scale2 = p.scale * 1.44269504088896340736f;  // log2(e)
#pragma unroll
    for (int i = 0; i < NBW; ++i) {
#pragma unroll
        for (int v = 0; v < 16; ++v) s[i][v] *= scale2;
        const int key0 = (part * NBW + i) * 32;
        if (key0 + 32 > S) {  // (wave-uniform)
#pragma unroll
            for (int v = 0; v < 16; ++v)
                if (key0 + 8 * (v / 4) + 4 * half + (v % 4) >= S) s[i][v] = -INFINITY;
        }
    }
    float m = -INFINITY;
#pragma unroll
    for (int i = 0; i < NBW; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) m = fmaxf(m, s[i][v]);
    m = fmaxf(m, __shfl_xor(m, 32, 64));
    const float mm = m == -INFINITY ? 0.f : m;  // a part with no valid key contributes nothing (and no NaN)
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < NBW; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            s[i][v] = __builtin_amdgcn_exp2f(s[i][v] - mm);
            sum += s[i][v];
        }
    sum += __shfl_xor(sum, 32, 64);
    if (half == 0) *(f32x2 *)(sums + 2 * (part * ATT_QB + qg * 32 + l32)) = f32x2{m, sum};

    // ---- O^T = V^T P^T: A gathered from V^T, B = probabilities (already per query lane) ----
    f32x16 o[2];
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[db][v] = 0.f;
#pragma unroll
    for (int i = 0; i < NBW; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            // registers 8j..8j+7 of a block are its keys 16j + 4*half + {0..3} and + 8 + {0..3}
            typedef T tx8 __attribute__((ext_vector_type(8)));
            tx8 pb;
#pragma unroll
            for (int e = 0; e < 8; ++e) pb[e] = Elem<T>::from_f(s[i][8 * j + e]);
            const int kbase = (part * NBW + i) * 32 + 16 * j + 4 * half;
#pragma unroll
            for (int db = 0; db < 2; ++db) {
                const unsigned short *row = (const unsigned short *)vt + (db * 32 + l32) * SP + kbase;
                const unsigned long long lo = *(const unsigned long long *)row, hi = *(const unsigned long long *)(row + 8);
                u32x4 av = {(unsigned)lo, (unsigned)(lo >> 32), (unsigned)hi, (unsigned)(hi >> 32)};
                Elem<T>::mma(av, __builtin_bit_cast(u32x4, pb), o[db]);
            }
        }
    __syncthreads();  // V^T has been read by everybody
    // ---- partial results: o[db][v] = O[query lane%32][db*32 + 8*(v/4) + 4*half + v%4] ----
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int vq = 0; vq < 4; ++vq)
            *(f32x4 *)(partial + (part * ATT_QB + qg * 32 + l32) * ATT_OP + db * 32 + 8 * vq + 4 * half) =
                f32x4{o[db][4 * vq], o[db][4 * vq + 1], o[db][4 * vq + 2], o[db][4 * vq + 3]};
    __syncthreads();
    // ---- merge: a thread finishes eight consecutive values of one query ----
    const bool vec_out = p.ld_out % 8 == 0 && (size_t)p.out % 16 == 0;  // rows of 64 values start on 16-byte boundaries
#pragma unroll
    for (int it = 0; it < ATT_QB * (ATT_D / 8) / THREADS; ++it) {
        const int item = tid + it * THREADS, r = item >> 3, d8 = (item & 7) * 8;
        f32x2 ms[PARTS];
        float M = -INFINITY, den = 0.f, f[PARTS];
#pragma unroll
        for (int i = 0; i < PARTS; ++i) {
            ms[i] = *(const f32x2 *)(sums + 2 * (i * ATT_QB + r));
            M = fmaxf(M, ms[i][0]);
        }
#pragma unroll
        for (int i = 0; i < PARTS; ++i) {
            f[i] = ms[i][0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms[i][0] - M);
            den = __builtin_fmaf(f[i], ms[i][1], den);
        }
        f32x4 x[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int i = 0; i < PARTS; ++i) {
            const float w = f[i] / den;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const f32x4 y = *(const f32x4 *)(partial + (i * ATT_QB + r) * ATT_OP + d8 + 4 * h);
#pragma unroll
                for (int e = 0; e < 4; ++e) x[h][e] = __builtin_fmaf(w, y[e], x[h][e]);
            }
        }
        if (t.x * ATT_QB + r >= S) continue;
        T *dst = O + (long)(t.x * ATT_QB + r) * p.ld_out + d8;
        T out[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float r32 = x[e / 4][e % 4];
            asm("" : "+v"(r32));  // (rounded to fp32 first: the compiler makes one operation with a single rounding of the last sum and the conversion, for some of them)
            out[e] = Elem<T>::from_f(r32);
        }
        if (vec_out) st_out128(dst, *(const out_u32x4 *)out);
        else {
#pragma unroll
            for (int e = 0; e < 8; ++e) st_elem<T>(dst + e, out[e]);
        }
    }
}

// Key blocks the body is instantiated for: seq <= 128 / 256 / 384 / 512 keys.
__host__ __device__ inline int attention_nb_class(int seq) {
    const int nb = attention_key_blocks(seq);
    return nb <= 4 ? 4 : nb <= 8 ? 8 : nb <= 12 ? 12 : 16;
}

// One kernel per class: the score registers of the longest class would otherwise set the register budget of the short sequences too.
// 128 registers, so that 16 wavefronts share a compute unit (256 keys without the bound: 64 sequences 57.8 us instead of 54.2); the general loop, which holds
// more over a tile, would go to scratch memory for that.
template <typename T, int NB, int LOOP = LOOP_ANY>
__global__ __launch_bounds__(attention_threads(NB), LOOP == LOOP_ANY && NB > 4 ? 2 : 4) void attention_kernel(AttnArgs a, BlpArgs blp) {
    extern __shared__ __attribute__((aligned(16))) unsigned char att_lds[];
    tiles<LOOP>(blp, [&](TileIdx t) { attention_tile<T, NB>(a, t, reinterpret_cast<T *>(att_lds)); });
}

}  // namespace gp
