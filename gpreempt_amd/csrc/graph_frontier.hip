// The kernels the graph executors run: whole iterations of breadth-first search, single-source shortest paths and
// PageRank, and connected components by union-find, over 32-bit adjacency in vectors of four.
//
// Layout.  row[v] .. row[v+1] are offsets into `ids` (and `weights`) in units of four neighbours; a list's last vector
// is padded with the id vertex_count, whose label / cost / rank entry exists and makes every kernel pass it over.
// Against the 64-bit lists of the files this is half the bytes, every access is an aligned 16-byte load, and a list
// of 16 neighbours keeps four lanes busy for one load each (the 16-lane groups of graph_bodies.hpp started at a
// 128-byte boundary and left half of their lanes without an edge).
//
// Split.  A wavefront owns 64 consecutive vertices: lane l reads what belongs to vertex l (coalesced), and the four
// lanes of a quad walk the lists of the quad's four vertices one after the other, handing the offsets round with DPP
// quad broadcasts.  The first vectors of all four lists are requested before the first is used.  A list of more than
// kLongRow vectors is walked by the whole wavefront afterwards, so that a hub does not hold four lanes for long.
// A tile is 256 vertices; a preemptible launch hands tiles out through tile_loop.hpp like any other kernel.
//
// Several iterations are queued at once: an iteration whose predecessor changed nothing (*prev_changed == 0) leaves
// before its first claim.  A launch that starts says how the iteration before it went, so the host needs no look of its own.
#include "launch_tiles.hpp"

namespace gp {

constexpr int GF_TILE = 256;
constexpr unsigned GF_INF = 0xFFFFFFFFu;
constexpr unsigned kLongRow = 64;

template <int S> __device__ __forceinline__ unsigned quad_bcast(unsigned x) { return (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, S * 0x55, 0xf, 0xf, true); }
// sum over the four lanes of a quad, left in all of them
__device__ __forceinline__ float quad_sum(float x) {
    x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0xB1, 0xf, 0xf, true));  // lanes 1 0 3 2
    x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x4E, 0xf, 0xf, true));  // lanes 2 3 0 1
    return x;
}

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// Whether a stop has been recorded, looked at while a wavefront works on its tile: ask() sends a load out, told() waits for
// it, and the work between the two covers its way.  Reads of one address come back one every 11 ns, whoever asks (every
// wavefront asking the stop index itself made sssp at 2^20 vertices 7 % slower), so the front workgroup hands the stop on
// in GP_GRAPH_RELAYS words, a line apart, and a workgroup asks one of those.
struct StopLook {
    const unsigned *relay = nullptr;  // nullptr: nobody looks
    unsigned seen = 0;
    __device__ __forceinline__ void ask() { if (relay) seen = __hip_atomic_load(relay, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
    __device__ __forceinline__ bool told() const { return relay && __builtin_amdgcn_readfirstlane(seen) != 0; }
};
static_assert(GP_GRAPH_RELAYS == 64, "a lane per word");
constexpr unsigned kRelayStride = 32;

// The front workgroup of a launch whose claims are given back: as front_workgroup of tile_loop.hpp, with three differences.
// It hands a stop on to the wavefronts that are at work.  It stays until seven eighths of the workers have left, because
// what a frontier gives the workers to do is uneven.  And it reads the flag every ten microseconds only: while a read of
// host memory is under way, the loads of that XCD come back later, and kernels that walk chains of them feel every one
// (read back to back: flattening 40 -> 178 us, bfs at 2^20 vertices 320 -> 369, sssp 1.68 -> 1.80 ms).  Bounded like
// front_workgroup; true in a front workgroup.
__device__ __forceinline__ bool gf_front(const BlpArgs &b, unsigned *relay) {
    if ((int)blockIdx.x >= b.front) return false;
    if (blockIdx.x != 0) return true;
    __shared__ int front_leave;
    const int lane = threadIdx.x & 63, wave = threadIdx.x / 64;
    if (threadIdx.x == 0) front_leave = 0;
    __syncthreads();
    auto told = [&] { return __hip_atomic_load(&front_leave, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != 0; };
    if (wave == 0) {
        for (int look = 0; look < (1 << 15) && !told(); ++look) {
            int flag = 0;
            if (lane == 0) flag = __hip_atomic_load(b.flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            if (__builtin_amdgcn_readfirstlane(flag) != 0) {
                if (lane == 0) record_stop(b.stop_index, b.kernel_id, b.stamps);
                break;
            }
            for (int us = 0; us < 8 && !told(); ++us) __builtin_amdgcn_s_sleep(36);
        }
    } else if (wave == 1) {
        const int target = wg_count(b) - wg_count(b) / 8;
        for (int look = 0; look < (1 << 18); ++look) {  // about a microsecond each
            const int stop = __hip_atomic_load(b.stop_index, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            int n = 0;
            for (int g = lane; g < b.groups; g += 64) n += __hip_atomic_load(b.done + g * COUNTER_STRIDE, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int d = 32; d > 0; d >>= 1) n += __shfl_xor(n, d);
            if (__builtin_amdgcn_readfirstlane(stop) != -1) {
                __hip_atomic_store(relay + kRelayStride * lane, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
            if (__builtin_amdgcn_readfirstlane(n) >= target) break;
            __builtin_amdgcn_s_sleep(4);
        }
        if (lane == 0) __hip_atomic_store(&front_leave, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    return true;
}

// f(index of a vector of four neighbours, its ids, the owner's payload) for every vector of the 64 lists that this
// wavefront's lanes own; an empty range (begin == end) stands for a vertex that takes no part.  Returns true when it
// was left because of a stop, after some of the lists: the tile has to be walked again from the start.
template <class F>
__device__ __forceinline__ bool gf_walk(const u32x4 *ids, unsigned begin, unsigned end, unsigned payload, StopLook look, F &&f) {
    const unsigned sub = threadIdx.x & 3;
    const bool is_long = end - begin > kLongRow;
    const unsigned stop = is_long ? begin : end;
    const unsigned b0 = quad_bcast<0>(begin) + sub, b1 = quad_bcast<1>(begin) + sub, b2 = quad_bcast<2>(begin) + sub, b3 = quad_bcast<3>(begin) + sub;
    const unsigned e0 = quad_bcast<0>(stop), e1 = quad_bcast<1>(stop), e2 = quad_bcast<2>(stop), e3 = quad_bcast<3>(stop);
    const unsigned p0 = quad_bcast<0>(payload), p1 = quad_bcast<1>(payload), p2 = quad_bcast<2>(payload), p3 = quad_bcast<3>(payload);
    u32x4 i0{}, i1{}, i2{}, i3{};
    if (b0 < e0) i0 = ids[b0];
    if (b1 < e1) i1 = ids[b1];
    if (b2 < e2) i2 = ids[b2];
    if (b3 < e3) i3 = ids[b3];
    look.ask();
    if (b0 < e0) f(b0, i0, p0);
    if (look.told()) return true;
    look.ask();
    if (b1 < e1) f(b1, i1, p1);
    if (look.told()) return true;
    look.ask();
    if (b2 < e2) f(b2, i2, p2);
    if (look.told()) return true;
    if (b3 < e3) f(b3, i3, p3);
    for (unsigned c = b0 + 4; c < e0; c += 4) f(c, ids[c], p0);
    for (unsigned c = b1 + 4; c < e1; c += 4) f(c, ids[c], p1);
    for (unsigned c = b2 + 4; c < e2; c += 4) f(c, ids[c], p2);
    for (unsigned c = b3 + 4; c < e3; c += 4) f(c, ids[c], p3);
    for (unsigned long long m = __builtin_amdgcn_ballot_w64(is_long); m; m &= m - 1) {
        const int l = __builtin_ctzll(m);
        const unsigned lb = __builtin_amdgcn_readlane(begin, l), le = __builtin_amdgcn_readlane(end, l), lp = __builtin_amdgcn_readlane(payload, l);
        look.ask();
        for (unsigned c = lb + (threadIdx.x & 63); c < le; c += 64) f(c, ids[c], lp);
        if (look.told()) return true;
    }
    return false;
}

// The words in which the workgroups say how the iteration goes: a set of them, in lines of its own, per XCD where the caller has
// room for that (gp_graph_iter_params::sets).  In one set, the stores of all wavefronts go through eight L2s to a line that moves from
// one to the other, and with it what else it holds: in a line with claim counters or with the words that the launch's
// workgroups read first, every second pull over 2^20 vertices took 56 us for 46.  PageRank at 2^20 vertices of degree 16
// 3600 -> 3385 us, at 2^17 of degree 4 441 -> 392 (one set, in a line of its own: 3400 and 435).
constexpr unsigned kSetInts = 32;
static_assert(GP_GRAPH_SETS == kXcds, "a set per XCD");
__device__ __forceinline__ unsigned *own_words(const gp_graph_iter_params &p) { return p.changed + (p.sets == GP_GRAPH_IN_SETS ? blockIdx.x % kXcds * kSetInts : 0u); }
// What the launch before said: lane 8 * w + x reads word w of set x, for the first five words.
struct WordsBefore {
    unsigned mine = 0;
    __device__ __forceinline__ explicit WordsBefore(const gp_graph_iter_params &p) {
        const unsigned lane = threadIdx.x & 63, word = lane / kXcds, set = lane % kXcds;
        if (p.prev_changed && word < 5 && (p.sets == GP_GRAPH_IN_SETS || set == 0)) mine = p.prev_changed[set * kSetInts + word];
    }
    __device__ __forceinline__ bool any(unsigned word) const { return (__builtin_amdgcn_ballot_w64(mine != 0) >> word * kXcds & 0xFF) != 0; }
    // f over a word of all sets, the same in every lane
    template <class F> __device__ __forceinline__ unsigned fold(unsigned word, F &&f) const {
        unsigned x = mine;
#pragma unroll
        for (int d = 1; d < kXcds; d <<= 1) x = f(x, (unsigned)__shfl_xor((int)x, d));
        return (unsigned)__builtin_amdgcn_readlane((int)x, (int)(word * kXcds));
    }
};

__device__ __forceinline__ void raise_changed(unsigned *word, bool mine) {
    if (__builtin_amdgcn_ballot_w64(mine) && (threadIdx.x & 63) == 0) *word = 1;
}

// ---- connected components: union-find with the smaller id as the parent ---------------------------------------------
// (Afforest, Sutton et al.: hook every vertex to a neighbour, compress, link the remaining edges, compress; the linking
// by compare-and-swap on the larger root.)
// Parents only ever fall, so a stale read (the L2s of the eight XCDs do not see each other's stores within a launch)
// is an older ancestor and still an ancestor; a root is only hooked by a compare-and-swap, whose answer comes from
// memory.  Every turn replaces the larger of the two candidates by something smaller, so the loop ends.
__device__ __forceinline__ void cc_link(unsigned *parent, unsigned u, unsigned v) {
    unsigned a = parent[u], b = parent[v];
    while (a != b) {
        const unsigned hi = a > b ? a : b, lo = a > b ? b : a;
        unsigned p = parent[hi];
        if (p == lo) return;
        if (p == hi) {
            p = atomicCAS(&parent[hi], hi, lo);
            if (p == hi || p == lo) return;
        }
        a = p;
        b = lo;
    }
}
__device__ __forceinline__ unsigned cc_root(const unsigned *parent, unsigned v) {
    unsigned p = parent[v];
    for (unsigned g; (g = parent[p]) != p; p = g) { }
    return p;
}

// ---- PageRank -----------------------------------------------------------------------------------------------------------
// Many vertices over the tolerance (PR): residual[v] += the shares its in-neighbours hand out this iteration, then the
// update of the reference's pr_update on the spot.  Shares are double-buffered (0 where u has nothing to hand out).
// The push's 16.8 million float atomics of a 2^20-vertex iteration (207 us, and 14 us for the update) become a gather
// from an array of 4 MB: 40 us, of which 16 are the streams and the rest the 4.4 million lines asked of the L2s for
// the gather (1.2 million of them beyond; non-temporal streams keep fewer of those but lose the vector cache's reuse
// of a quad's line and take 52).
// Few (PR_STEP): one launch takes in what the iteration before pushed (gained), updates, and pushes what the vertices
// over the tolerance hand out into the next iteration's sums; the rest of the residual stays where it is, so only the
// vertices that gained something are touched at all.
__device__ __forceinline__ float pr_pull4(const float *share, const u32x4 &i) { return (share[i[0]] + share[i[1]]) + (share[i[2]] + share[i[3]]); }

__device__ __forceinline__ float pr_share(const gp_graph_iter_params &p, unsigned v, float r) {
    const float degree = p.degree[v];
    return degree > 0.f ? r * p.alpha / degree : 0.f;  // a sink has nobody to hand it to
}
// whether anybody was over the tolerance, and how many in one tile of GP_GRAPH_SAMPLED
__device__ __forceinline__ void pr_report(const gp_graph_iter_params &p, int tile, bool up) {
    const unsigned long long ups = __builtin_amdgcn_ballot_w64(up);
    if (ups == 0 || (threadIdx.x & 63) != 0) return;
    unsigned *words = own_words(p);
    words[0] = 1;
    if (tile % GP_GRAPH_SAMPLED == 0) atomicAdd(words + 1, (unsigned)__builtin_popcountll(ups));
}
__device__ __forceinline__ void pr_push(const gp_graph_iter_params &p, const u32x4 *ids, unsigned v, float share) {
    if (!__builtin_amdgcn_ballot_w64(share != 0.f)) return;
    unsigned begin = 0, end = 0;
    if (share != 0.f) { begin = p.row[v]; end = p.row[v + 1]; }
    gf_walk(ids, begin, end, __builtin_bit_cast(unsigned, share), StopLook{}, [&](unsigned, const u32x4 &i, unsigned from) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (i[j] < p.vertex_count) atomicAdd(&p.next_gained[i[j]], __builtin_bit_cast(float, from));
    });
}

// ---- shortest paths: delta-stepping with one bucket (Meyer and Sanders), or the near and far piles of Davidson et al. ----
// An iteration relaxes the marked vertices whose cost is below a limit; the others keep their mark.  The limit rises by
// one step whenever an iteration has left no marked vertex below it.  Vertices are then relaxed close to their final
// cost: on the generated graphs 1.1-1.4 times per vertex, where relaxing whatever is marked takes 4-5, for a fifth more
// iterations (weights uniform in 1..64, a step of the average weight).  The first iteration's limit is one step; the
// words of the iteration before say how it went on:
//   [1] somebody improved below the limit   [2] the limit   [3] somebody was below it   [4] ~(lowest marked cost)
// After an iteration that found nobody below its limit, an iteration of its own finds the lowest marked cost, and the
// limit goes one step beyond that: a gap in the costs (one heavy edge in a light graph) takes two iterations more,
// whatever its width, where step by step a bridge of 10^6 among unit weights took half a million.
__device__ __forceinline__ void sssp_lowest(const gp_graph_iter_params &p, unsigned cost) {
    for (int d = 32; d; d >>= 1) cost = min(cost, (unsigned)__shfl_xor((int)cost, d));
    // (a look first: it may be an old one, which is a higher cost; an atomic on one address takes 40 ns of everybody's time)
    if (cost != GF_INF && (threadIdx.x & 63) == 0 && __hip_atomic_load(own_words(p) + 4, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < ~cost)
        atomicMax(own_words(p) + 4, ~cost);
}

// What a tile is looked through for (the vertices on the frontier): read for several tiles at a time, and before the
// claim where the claim's answer is known, so that the reads of a claim's tiles are one trip to memory.
template <int KIND>
__device__ __forceinline__ unsigned gf_key(const gp_graph_iter_params &p, int tile) {
    const unsigned v = (unsigned)tile * GF_TILE + threadIdx.x;
    if (v >= p.vertex_count) return KIND == GP_GRAPH_IT_BFS ? GF_INF : 0;
    if constexpr (KIND == GP_GRAPH_IT_BFS) return p.label[v];
    else if constexpr (KIND == GP_GRAPH_IT_SSSP) return p.active[v];
    else if constexpr (KIND == GP_GRAPH_IT_PR_STEP) return __builtin_bit_cast(unsigned, p.gained[v]);
    else return 0;
}

// Kernels whose tiles can be left at any point and done again from the start: labels, costs and parents only fall, and a
// second look at a neighbour finds nothing left to do.  (PR and PR_PUSH add: a tile of theirs is done once.  One of
// PR_STEP that is done finds nothing gained when it is done again, but only if it does not leave its shares behind.)
template <int KIND>
__device__ __forceinline__ bool gf_repeatable(const gp_graph_iter_params &p) {
    return KIND == GP_GRAPH_IT_BFS || KIND == GP_GRAPH_IT_SSSP || KIND == GP_GRAPH_IT_CC_LINK || (KIND == GP_GRAPH_IT_PR_STEP && p.next_gained);
}

// true: a stop is recorded and the tile was left
template <int KIND>
__device__ __forceinline__ bool gf_tile(const gp_graph_iter_params &p, int tile, unsigned key, unsigned limit, bool find, StopLook look) {
    const unsigned n = p.vertex_count;
    const unsigned v = (unsigned)tile * GF_TILE + threadIdx.x;
    const bool in = v < n;
    const u32x4 *ids = reinterpret_cast<const u32x4 *>(p.ids);
    if constexpr (KIND == GP_GRAPH_IT_BFS) {
        const bool on = key == p.level;
        if (!__builtin_amdgcn_ballot_w64(on)) return false;
        unsigned begin = 0, end = 0;
        if (on) { begin = p.row[v]; end = p.row[v + 1]; }
        bool mine = false;
        const bool left = gf_walk(ids, begin, end, 0, look, [&](unsigned, const u32x4 &i, unsigned) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (p.label[i[j]] == GF_INF) { p.label[i[j]] = p.level + 1; mine = true; }
        });
        raise_changed(own_words(p), mine);
        return left;
    } else if constexpr (KIND == GP_GRAPH_IT_SSSP) {
        bool on = key != 0;
        if (!__builtin_amdgcn_ballot_w64(on)) return false;
        bool far = false;
        unsigned begin = 0, end = 0, cost = 0;
        if (on) {
            cost = p.cost[v];
            far = find || cost >= limit;
            on = !far;
            p.active[v] = 0;
            if (far) p.next_active[v] = 1;  // its turn comes with a later limit
        }
        if (find) sssp_lowest(p, far ? cost : GF_INF);
        else raise_changed(own_words(p) + 3, on);
        if (on) { begin = p.row[v]; end = p.row[v + 1]; }
        bool mine = far, near = false;
        const u32x4 *weights = reinterpret_cast<const u32x4 *>(p.weights);
        const bool left = gf_walk(ids, begin, end, cost, look, [&](unsigned c, const u32x4 &i, unsigned from) {
            const u32x4 w = weights[c];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                // (costs only fall, so a stale one is too large and never hides an improvement)
                const unsigned via = from + w[j];
                if (p.cost[i[j]] > via && atomicMin(&p.cost[i[j]], via) > via) {
                    p.next_active[i[j]] = 1;
                    mine = true;
                    near |= via < limit;
                }
            }
        });
        if (left && on) p.active[v] = 1;  // its turn again when the tile is done again
        raise_changed(own_words(p), mine);
        raise_changed(own_words(p) + 1, near);
        return left;
    } else if constexpr (KIND == GP_GRAPH_IT_PR) {
        unsigned begin = 0, end = 0;
        float r = 0.f, value = 0.f, degree = 0.f;
        // (value and degree are wanted at the end; asked for there, they were one more trip to memory: 5000 vertices of degree 8, 338 -> 325 us a run)
        if (in) { begin = p.row[v]; end = p.row[v + 1]; r = p.residual[v]; value = p.value[v]; degree = p.degree[v]; }
        const unsigned sub = threadIdx.x & 3, none = p.row_end;
        const bool is_long = end - begin > kLongRow;
        const unsigned stop = is_long ? begin : end;
        const unsigned b[4] = {quad_bcast<0>(begin) + sub, quad_bcast<1>(begin) + sub, quad_bcast<2>(begin) + sub, quad_bcast<3>(begin) + sub};
        const unsigned e[4] = {quad_bcast<0>(stop), quad_bcast<1>(stop), quad_bcast<2>(stop), quad_bcast<3>(stop)};
        // (no branches around these loads: a lane without a vector reads the one behind the last list, which names
        // only the neighbour that counts nothing; two vectors per lane and list, 32 neighbours, are in flight at once)
        const bool two = __builtin_amdgcn_ballot_w64(stop - begin > 4);
        u32x4 i[4], k[4];
        float g[4], h[4] = {0.f, 0.f, 0.f, 0.f}, sum[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) i[s] = ids[b[s] < e[s] ? b[s] : none];
        if (two) {
#pragma unroll
            for (int s = 0; s < 4; ++s) k[s] = ids[b[s] + 4 < e[s] ? b[s] + 4 : none];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 4; ++s) g[s] = pr_pull4(p.share, i[s]);
        if (two) {
#pragma unroll
            for (int s = 0; s < 4; ++s) h[s] = pr_pull4(p.share, k[s]);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            sum[s] = g[s] + h[s];
            for (unsigned c = b[s] + 8; c < e[s]; c += 4) sum[s] += pr_pull4(p.share, ids[c]);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) sum[s] = quad_sum(sum[s]);
        r += sub == 0 ? sum[0] : sub == 1 ? sum[1] : sub == 2 ? sum[2] : sum[3];
        for (unsigned long long m = __builtin_amdgcn_ballot_w64(is_long); m; m &= m - 1) {
            const int l = __builtin_ctzll(m);
            const unsigned lb = __builtin_amdgcn_readlane(begin, l), le = __builtin_amdgcn_readlane(end, l);
            float x = 0.f;
            for (unsigned c = lb + (threadIdx.x & 63); c < le; c += 64) x += pr_pull4(p.share, ids[c]);
            for (int d = 32; d; d >>= 1) x += __shfl_xor(x, d);
            if ((int)(threadIdx.x & 63) == l) r += x;
        }
        const bool up = in && r > p.tolerance;
        if (in) {
            __builtin_nontemporal_store(up && degree > 0.f ? r * p.alpha / degree : 0.f, p.next_share + v);
            __builtin_nontemporal_store(up ? 0.f : r, p.residual + v);
        }
        if (up) __builtin_nontemporal_store(value + r, p.value + v);
        pr_report(p, tile, up);
    } else if constexpr (KIND == GP_GRAPH_IT_PR_PUSH) {
        const float share = in ? p.share[v] : 0.f;
        pr_push(p, ids, v, share);
    } else if constexpr (KIND == GP_GRAPH_IT_PR_STEP) {
        // (next_gained == nullptr: the next iteration pulls; the shares are left for it instead of pushed)
        const float gained = __builtin_bit_cast(float, key);
        if (p.next_gained && !__builtin_amdgcn_ballot_w64(gained != 0.f)) return false;
        bool up = false;
        float share = 0.f;
        if (gained != 0.f) {
            const float r = p.residual[v] + gained;
            p.gained[v] = 0.f;
            up = r > p.tolerance;
            p.residual[v] = up ? 0.f : r;
            if (up) { p.value[v] += r; share = pr_share(p, v, r); }
        }
        pr_report(p, tile, up);
        if (p.next_gained) pr_push(p, ids, v, share);
        else if (in) p.next_share[v] = share;
    } else if constexpr (KIND == GP_GRAPH_IT_PR_INIT) {
        if (!in) return false;
        p.value[v] = 1.0f - p.alpha;
        p.next_share[v] = p.degree[v] > 0.f ? (1.0f - p.alpha) * p.alpha / p.degree[v] : 0.f;
        p.residual[v] = 0.f;
        p.gained[v] = 0.f;
        p.next_gained[v] = 0.f;
    } else if constexpr (KIND == GP_GRAPH_IT_BFS_INIT) {
        if (in) p.label[v] = v == 0 ? 0 : GF_INF;  // source = vertex 0
    } else if constexpr (KIND == GP_GRAPH_IT_SSSP_INIT) {
        if (!in) return false;
        p.cost[v] = v == 0 ? 0 : GF_INF;
        p.active[v] = v == 0;
        p.next_active[v] = 0;
    } else if constexpr (KIND == GP_GRAPH_IT_CC_INIT) {
        // hook every vertex to its first neighbour at once, if that is smaller (nobody reads a parent in this launch)
        if (!in) return false;
        unsigned first = v;
        if (p.row[v] < p.row[v + 1]) { first = p.ids[4ull * p.row[v]]; }
        p.parent[v] = first < v ? first : v;
    } else if constexpr (KIND == GP_GRAPH_IT_CC_FLATTEN) {
        if (in) p.parent[v] = cc_root(p.parent, v);
    } else if constexpr (KIND == GP_GRAPH_IT_CC_LINK) {
        // (every edge between two trees walks up to their roots, and tries to hook one that an L2 still takes for a root:
        // linking all edges of a graph at once takes 300-570 us at 2^20 vertices of degree 16, and what is in flight when a
        // stop comes is most of that.  So a few edges of everybody are linked first, and the trees are flattened again before
        // the others are: then both ends have the same root already, mostly)
        unsigned begin = 0, end = 0;
        if (in) { begin = p.row[v]; end = p.row[v + 1]; }
        if (p.level && p.level < 4) {
            for (unsigned j = 0; j < p.level; ++j) {
                const unsigned other = begin < end ? p.ids[4ull * begin + j] : n;
                if (other < n) cc_link(p.parent, v, other);
            }
            return false;
        }
        if (p.level) end = min(end, begin + 1);
        return gf_walk(ids, begin, end, v, look, [&](unsigned, const u32x4 &i, unsigned from) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (i[j] < n) cc_link(p.parent, from, i[j]);
        });
    } else {  // GP_GRAPH_IT_CC_LABEL
        if (in) p.comp[v] = cc_root(p.parent, v);
    }
    return false;
}

__device__ __forceinline__ unsigned sssp_limit(const gp_graph_iter_params &p, const WordsBefore &before, bool *find) {
    unsigned limit = p.step;
    *find = false;
    if (p.prev_changed) {
        auto above = [&](unsigned x) { return x + p.step < x ? GF_INF : x + p.step; };
        limit = (unsigned)__builtin_amdgcn_readlane((int)before.mine, 2 * kXcds);  // (set 0 has it: workgroup 0 wrote it)
        const bool near = before.any(1);
        if (before.any(4)) limit = above(~before.fold(4, [](unsigned a, unsigned b) { return max(a, b); }));
        else if (!near && before.any(3)) limit = above(limit);
        else *find = !near;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) p.changed[2] = limit;
    return limit;
}

// The launch tells the host that it has started, and how the iteration before it went (gp_graph_iter_params::started).
// One store to host memory that nobody waits for; the next launch is queued while this one works.
__device__ __forceinline__ void report_start(const gp_graph_iter_params &p, const WordsBefore &before, const BlpArgs &blp) {
    if (!p.started || blockIdx.x != 0 || threadIdx.x >= 64) return;
    const unsigned count = before.fold(1, [](unsigned a, unsigned b) { return a + b; });
    unsigned low = GP_GRAPH_START_CHANGED;
    if (p.prev_changed) low = before.any(0) ? GP_GRAPH_START_CHANGED | min(count, GP_GRAPH_START_COUNT) : 0u;
    if (threadIdx.x != 0) return;
    const int stop = blp.stop_index ? __hip_atomic_load(blp.stop_index, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : -1;
    if (stop != -1) low = GP_GRAPH_START_STOPPED | (unsigned)stop;
    __hip_atomic_store(p.started, (unsigned long long)p.seq << 32 | low, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A claim of a launch stands for `per` tiles of 256 vertices.  In a launch of all its workgroups at once every claim is
// made when it starts: from then on a stop waits for the whole launch, unless the workgroups give their claims back.  They
// do where the tiles can be done again and the launch is a long one (gp_launch_graph_iter): a wavefront looks whether it
// has to between the lists of a quad, a sixteenth of the launch apart.  Stops next to BERT's requests at 2^20 vertices, mean / p99: bfs 30 / 47 us,
// sssp 39 / 71 (118 / 256 without), pagerank 32 / 57 (51 / 120), connected components 48 / 134 (278 / 598, linked at once).
template <int KIND, int LOOP = LOOP_ANY>
__global__ __launch_bounds__(GF_TILE) void graph_iter_kernel(gp_graph_iter_params p, int per, BlpArgs blp) {
    const WordsBefore before(p);
    report_start(p, before, blp);
    if (p.prev_changed && !before.any(0)) return;  // converged before this iteration (the same answer for every workgroup)
    unsigned limit = 0;
    bool find = false;
    if constexpr (KIND == GP_GRAPH_IT_SSSP) limit = sssp_limit(p, before, &find);
    unsigned key[4];  // of the next tiles
    auto look = [&](int first, int count) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (j < count) key[j] = gf_key<KIND>(p, first + j);
    };
    const int known = LOOP == LOOP_ANY || wg_id(blp) < 0 || wg_id(blp) >= blp.total ? -1 : xcd_contiguous(wg_id(blp), blp.total);
    if (known >= 0) look(known * per, per);
    auto claim = [&](TileIdx t, StopLook stop) {
        bool left = false;
#pragma unroll 1
        for (int j = 0; j < per && !left; ++j) {
            if (j % 4 == 0 && (j || known < 0)) look(t.x * per + j, per - j);
            if (j) stop.ask();
            left = gf_tile<KIND>(p, t.x * per + j, key[0], limit, find, stop) || (j && stop.told());
            key[0] = key[1]; key[1] = key[2]; key[2] = key[3];
        }
        return left;
    };
    if constexpr (LOOP == LOOP_FIXED) {
        if (blp.done && gf_front(blp, p.relay)) return;
        tile_fixed_early(blp, [&](TileIdx t, int *) {
            const bool looks = blp.done && gf_repeatable<KIND>(p);
            const bool left = claim(t, StopLook{looks ? p.relay + kRelayStride * (blockIdx.x / kXcds % GP_GRAPH_RELAYS) : nullptr});
            return looks ? __syncthreads_or(left) != 0 : false;
        });
    } else
        tiles<LOOP>(blp, [&](TileIdx t) { claim(t, StopLook{}); });
}

// 64-bit neighbour ids (and weights) into padded vectors of four
__global__ __launch_bounds__(GF_TILE) void graph_pack_kernel(gp_graph_pack_params p) {
    const unsigned v = (unsigned)blockIdx.x * (GF_TILE / 4) + threadIdx.x / 4;
    if (v == 0) p.ids[4ull * p.row_end + (threadIdx.x & 3)] = p.vertex_count;  // behind the last list
    if (v >= p.vertex_count) return;
    const unsigned long long from = p.vertex_list[v], to = p.vertex_list[v + 1];
    for (unsigned c = p.row[v] + (threadIdx.x & 3); c < p.row[v + 1]; c += 4) {
        const unsigned long long at = from + 4ull * (c - p.row[v]);
        for (int j = 0; j < 4; ++j) {
            p.ids[4ull * c + j] = at + j < to ? (unsigned)p.edge_list[at + j] : p.vertex_count;
            if (p.weights) p.weights[4ull * c + j] = at + j < to ? p.weight_list[at + j] : 0u;
        }
    }
}

}  // namespace gp

using namespace gp;

extern "C" int gp_launch_graph_iter(const gp_graph_iter_params *p, const gp_preempt_ctx *ctx, gp_stream s, gp_launch_info *info) {
    GP_REQUIRE(p && p->row && p->ids, "null graph iteration params");
    GP_REQUIRE(p->vertex_count > 0 && p->vertex_count < (1u << 31), "graph: vertex count out of range");
    switch (p->kernel) {
        case GP_GRAPH_IT_BFS: GP_REQUIRE(p->label && p->changed, "bfs: operands missing"); break;
        case GP_GRAPH_IT_BFS_INIT: GP_REQUIRE(p->label, "bfs: label missing"); break;
        case GP_GRAPH_IT_SSSP: GP_REQUIRE(p->weights && p->cost && p->active && p->next_active && p->active != p->next_active && p->changed, "sssp: operands missing"); break;
        case GP_GRAPH_IT_SSSP_INIT: GP_REQUIRE(p->cost && p->active && p->next_active, "sssp: operands missing"); break;
        case GP_GRAPH_IT_PR: GP_REQUIRE(p->share && p->next_share && p->share != p->next_share && p->residual && p->value && p->degree && p->changed, "pagerank: operands missing"); break;
        case GP_GRAPH_IT_PR_PUSH: GP_REQUIRE(p->share && p->next_gained, "pagerank: operands missing"); break;
        case GP_GRAPH_IT_PR_STEP: GP_REQUIRE(p->gained && p->gained != p->next_gained && (p->next_gained || p->next_share) && p->residual && p->value && p->degree && p->changed, "pagerank: operands missing"); break;
        case GP_GRAPH_IT_PR_INIT: GP_REQUIRE(p->next_share && p->residual && p->value && p->degree && p->gained && p->next_gained, "pagerank: operands missing"); break;
        case GP_GRAPH_IT_CC_LABEL: GP_REQUIRE(p->comp, "cc: labels missing");  // fallthrough
        case GP_GRAPH_IT_CC_INIT: case GP_GRAPH_IT_CC_LINK: case GP_GRAPH_IT_CC_FLATTEN: GP_REQUIRE(p->parent, "cc: parents missing"); break;
    }
    const long tiles = ((long)p->vertex_count + GF_TILE - 1) / GF_TILE;
    // A launch's cost besides its edges is its workgroups (a claim, a barrier: 4096 of them take 12 us): up to eight
    // tiles per claim as long as that leaves four workgroups per compute unit.  The pull wants as many lists in flight
    // as the chip holds and takes one tile at a time.
    int per = p->kernel == GP_GRAPH_IT_PR ? 1 : (int)std::min<long>(8, std::max<long>(1, tiles / (4L * device_cus())));
    // A preemptible launch that may walk a million edges (20 us) is one whose claims are given back behind a stop.  Where
    // they cannot be (no counters for it, or more claims than a launch with fixed claims takes), they are as small as they
    // get.  (The other kernels are done in 40 us at 2^20 vertices.)
    const bool walks = p->kernel == GP_GRAPH_IT_BFS || p->kernel == GP_GRAPH_IT_SSSP || p->kernel == GP_GRAPH_IT_CC_LINK || p->kernel == GP_GRAPH_IT_PR || p->kernel == GP_GRAPH_IT_PR_STEP;
    const bool far = ctx && walks && p->row_end >= (1u << 18);
    const bool gives_back = far && ctx->done && p->relay && ctx->counter_groups > 1 && ctx->poll_every != 1 && tiles / per <= 32L * device_cus();
    if (far && !gives_back) per = 1;
    auto launch = [&](auto kernels) {
        kernels.long_tiles = gives_back;
        return launch_tiles(kernels, (int)((tiles + per - 1) / per), 1, ctx, s, info, *p, 0, far ? 1 : 4, GF_TILE, per);
    };
    switch (p->kernel) {
#define GP_GI(K) case K: return launch(GP_KSET(graph_iter_kernel<K));
        GP_GI(GP_GRAPH_IT_BFS) GP_GI(GP_GRAPH_IT_BFS_INIT) GP_GI(GP_GRAPH_IT_SSSP) GP_GI(GP_GRAPH_IT_SSSP_INIT) GP_GI(GP_GRAPH_IT_PR)
        GP_GI(GP_GRAPH_IT_PR_PUSH) GP_GI(GP_GRAPH_IT_PR_STEP) GP_GI(GP_GRAPH_IT_PR_INIT) GP_GI(GP_GRAPH_IT_CC_INIT) GP_GI(GP_GRAPH_IT_CC_LINK)
        GP_GI(GP_GRAPH_IT_CC_FLATTEN) GP_GI(GP_GRAPH_IT_CC_LABEL)
#undef GP_GI
    }
    set_error("graph iteration kernel %d", p->kernel);
    return GP_OUTOFRANGE;
}

extern "C" int gp_graph_pack_async(const gp_graph_pack_params *p, gp_stream s) {
    GP_REQUIRE(p && p->vertex_list && p->row && p->ids && (p->edge_list || p->row_end == 0), "null graph pack params");
    GP_REQUIRE(!p->weights == !p->weight_list, "graph pack: weights come together");
    GP_REQUIRE(p->vertex_count > 0 && p->vertex_count < (1u << 31), "graph: vertex count out of range");
    hipLaunchKernelGGL(graph_pack_kernel, dim3((p->vertex_count + GF_TILE / 4 - 1) / (GF_TILE / 4)), dim3(GF_TILE), 0, native(s), *p);
    GP_HIP(hipGetLastError());
    return GP_SUCC;
}
