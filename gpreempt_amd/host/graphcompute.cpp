// Host loops of the graph workloads (reference src/workloads/graphcompute.tr.cu:142-174, :257-285,
// :450-495, :635-675) and the graph file format (src/workloads/graphcompute.cu:16-45).
#include "workloads/graphcompute.h"

#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <deque>
#include <thread>

#include "numeric.h"

namespace GraphCompute {

using namespace foo::util;

namespace {

template <class T>
bool read_array(const std::string &path, std::vector<T> &out) {
    FILE *fp = std::fopen(path.c_str(), "rb");
    if (!fp) return false;
    uint64_t count = 0, tag = 0;
    bool ok = std::fread(&count, sizeof(count), 1, fp) == 1 && std::fread(&tag, sizeof(tag), 1, fp) == 1 && count < (1ULL << 36);
    if (ok) {  // the header's count must fit what is left of the file, before anything is allocated for it
        const long here = std::ftell(fp);
        ok = here >= 0 && std::fseek(fp, 0, SEEK_END) == 0;
        const long end = ok ? std::ftell(fp) : -1;
        ok = ok && end >= here && (uint64_t)(end - here) / sizeof(T) >= count && std::fseek(fp, here, SEEK_SET) == 0;
    }
    if (ok) {
        out.resize(count);
        ok = std::fread(out.data(), sizeof(T), count, fp) == count;
    }
    std::fclose(fp);
    return ok;
}
template <class T>
bool write_array(const std::string &path, const std::vector<T> &v) {
    FILE *fp = std::fopen(path.c_str(), "wb");
    if (!fp) return false;
    uint64_t count = v.size(), tag = sizeof(T);
    bool ok = std::fwrite(&count, sizeof(count), 1, fp) == 1 && std::fwrite(&tag, sizeof(tag), 1, fp) == 1 &&
              std::fwrite(v.data(), sizeof(T), v.size(), fp) == v.size();
    return std::fclose(fp) == 0 && ok;
}

size_t round4(size_t n) { return (n + 3) / 4 * 4; }

}  // namespace

Status read_graph(const std::string &base, CsrGraph &g, bool with_weights) {
    if (!read_array(base + ".col", g.vertexList) || !read_array(base + ".dst", g.edgeList)) return Status::NotFound;
    if (g.vertexList.size() < 2) return Status::Fail;
    g.vertex_count = g.vertexList.size() - 1;
    g.edge_count = g.edgeList.size();
    // a malformed file must not turn into out-of-bounds reads on the GPU
    if (g.vertexList.front() != 0 || g.vertexList.back() != g.edge_count) return Status::Fail;
    for (size_t i = 0; i + 1 < g.vertexList.size(); ++i)
        if (g.vertexList[i] > g.vertexList[i + 1]) return Status::Fail;
    for (uint64_t e : g.edgeList)
        if (e >= g.vertex_count) return Status::OutOfRange;
    g.weightList.clear();
    if (with_weights) {
        if (!read_array(base + ".val", g.weightList)) return Status::NotFound;
        if (g.weightList.size() != g.edge_count) return Status::Fail;
    }
    return Status::Succ;
}

Status write_graph(const std::string &base, const CsrGraph &g) {
    if (!write_array(base + ".col", g.vertexList) || !write_array(base + ".dst", g.edgeList)) return Status::Fail;
    if (!g.weightList.empty() && !write_array(base + ".val", g.weightList)) return Status::Fail;
    return Status::Succ;
}

// Edges are drawn once in order (the seed alone decides), counted into offsets and scattered; every list is then
// sorted by (neighbour, weight), lists in parallel.  2^20 vertices of degree 8: 0.3 s, where a vector per vertex took 2.
CsrGraph synthetic_graph(uint64_t n, unsigned degree, uint64_t seed) {
    foo::numeric::Rng rng(seed);
    CsrGraph g;
    g.vertex_count = n;
    g.symmetric = true;
    g.vertexList.assign(n + 1, 0);
    std::vector<uint64_t> drawn(n * degree);  // neighbour << 32 | weight, weight 0: a self-loop, left out
    for (uint64_t v = 0; v < n; ++v) {
        for (unsigned d = 0; d < degree; ++d) {
            // mostly short-range edges with a few long ones: several components are unlikely,
            // the diameter stays at tens of hops
            uint64_t u = (d % 4 == 0) ? rng.next() % n : (v + 1 + rng.next() % 64) % n;
            drawn[v * degree + d] = 0;
            if (u == v) continue;
            drawn[v * degree + d] = u << 32 | (1 + rng.next() % 64);
            ++g.vertexList[v + 1];
            ++g.vertexList[u + 1];
        }
    }
    for (uint64_t v = 0; v < n; ++v) g.vertexList[v + 1] += g.vertexList[v];
    g.edge_count = g.vertexList[n];
    std::vector<uint64_t> edge(g.edge_count), at(g.vertexList.begin(), g.vertexList.end() - 1);
    for (uint64_t v = 0; v < n; ++v) {
        for (unsigned d = 0; d < degree; ++d) {
            const uint64_t e = drawn[v * degree + d];
            if (!e) continue;
            edge[at[v]++] = e;
            edge[at[e >> 32]++] = v << 32 | (e & 0xFFFFFFFFu);
        }
    }
    g.edgeList.resize(g.edge_count);
    g.weightList.resize(g.edge_count);
    auto finish = [&](uint64_t from, uint64_t to) {
        for (uint64_t v = from; v < to; ++v) {
            std::sort(edge.begin() + g.vertexList[v], edge.begin() + g.vertexList[v + 1]);
            for (uint64_t i = g.vertexList[v]; i < g.vertexList[v + 1]; ++i) { g.edgeList[i] = edge[i] >> 32; g.weightList[i] = (uint32_t)edge[i]; }
        }
    };
    const unsigned workers = n < (1u << 14) ? 1 : std::max(1u, std::min(8u, std::thread::hardware_concurrency()));
    std::vector<std::thread> pool;
    for (unsigned w = 1; w < workers; ++w) pool.emplace_back(finish, n * w / workers, n * (w + 1) / workers);
    finish(0, n / workers);
    for (std::thread &t : pool) t.join();
    return g;
}

// ---- the workload ---------------------------------------------------------------------------
#define GC_CHECK(call)                                                                          \
    do {                                                                                        \
        if ((call) != 0) {                                                                      \
            std::fprintf(stderr, "%s failed: %s (%s:%d)\n", #call, gp_last_error(), __FILE__, __LINE__); \
            return Status::Fail;                                                                \
        }                                                                                       \
    } while (0)

std::unique_ptr<Workload> Workload::create(const std::string &kind, const CsrGraph &g) {
    if (kind != "cc" && kind != "bfs" && kind != "pagerank" && kind != "sssp") return nullptr;
    if (g.vertex_count == 0 || g.vertex_count >= (1ULL << 32) || g.vertexList.size() != g.vertex_count + 1) return nullptr;
    if (kind == "sssp" && g.weightList.size() != g.edge_count) return nullptr;
    std::unique_ptr<Workload> w(new Workload());
    w->kind_ = kind;
    w->n_ = g.vertex_count;
    w->m_ = g.edge_count;
    // lanes per neighbour list: the width nearest the average degree keeps most lanes busy
    const double avg_degree = (double)g.edge_count / (double)g.vertex_count;
    w->lanes_ = avg_degree <= 24 ? 16 : avg_degree <= 48 ? 32 : 64;
    const size_t n = g.vertex_count;
    auto dev = [](GPUdeviceptr *p, size_t bytes) { return gp_malloc(p, bytes ? bytes : 4) == 0; };
    auto up = [&](GPUdeviceptr *p, const void *src, size_t bytes) { return dev(p, bytes) && (bytes == 0 || gp_memcpy_h2d(*p, src, bytes) == 0); };
    bool ok = up(&w->vertex_list_, g.vertexList.data(), (n + 1) * 8) && up(&w->edge_list_, g.edgeList.data(), g.edge_count * 8);
    ok = ok && dev(&w->changed_, 4) && gp_host_alloc((void **)&w->host_words_, 2 * sizeof(int)) == 0;
    // (label_, cost_ and the shares carry one entry more, 0: the neighbour that fills up the last vector of a list)
    if (kind == "bfs") ok = ok && dev(&w->label_, (n + 1) * 4) && gp_fill32_async((uint32_t *)w->label_ + n, 0, 1, nullptr) == 0;
    if (kind == "cc") ok = ok && dev(&w->comp_, n * 8) && dev(&w->active_, round4(n)) && dev(&w->next_active_, round4(n)) && dev(&w->parent_, n * 4);
    if (kind == "pagerank") {
        ok = ok && dev(&w->active_, round4(n)) && dev(&w->delta_, (n + 1) * 4) && dev(&w->share_, (n + 1) * 4) && dev(&w->gained_, 2 * n * 4) && dev(&w->residual_, n * 4) && dev(&w->value_, n * 4);
        ok = ok && gp_fill32_async((uint32_t *)w->delta_ + n, 0, 1, nullptr) == 0 && gp_fill32_async((uint32_t *)w->share_ + n, 0, 1, nullptr) == 0;
        std::vector<float> degree(n);
        for (size_t v = 0; v < n; ++v) degree[v] = (float)(g.vertexList[v + 1] - g.vertexList[v]);
        ok = ok && up(&w->degree_, degree.data(), n * 4);
    }
    if (kind == "sssp") {
        uint64_t sum = 0;
        for (uint32_t x : g.weightList) sum += x;
        if (g.edge_count) w->step_ = (uint32_t)std::max<uint64_t>(1, sum / g.edge_count);
        ok = ok && up(&w->weight_list_, g.weightList.data(), g.edge_count * 4) && dev(&w->active_, round4(n)) && dev(&w->next_active_, round4(n)) &&
             dev(&w->cost_, (n + 1) * 4) && dev(&w->new_cost_, n * 4) && gp_fill32_async((uint32_t *)w->cost_ + n, 0, 1, nullptr) == 0;
    }
    // (beyond 32-bit offsets a graph is run one iteration at a time, on the 64-bit lists)
    if (n < (1ULL << 31) && g.edge_count / 4 + n < (1ULL << 32)) ok = ok && w->upload_packed(g, kind == "sssp");
    ok = ok && gp_host_alloc_coherent((void **)&w->starts_, &w->starts_dev_, (kRing + 1) * sizeof(unsigned long long)) == 0;
    if (!ok) {
        std::fprintf(stderr, "graph workload: allocation failed: %s\n", gp_last_error());
        return nullptr;
    }
    return w;
}

Workload::~Workload() {
    for (GPUdeviceptr p : {vertex_list_, edge_list_, weight_list_, label_, active_, next_active_, comp_, delta_, residual_, value_, cost_, new_cost_, changed_,
                           row_, ids_, weights_, parent_, share_, degree_, gained_, ring_})
        if (p) gp_free(p);
    if (starts_) gp_host_free((void *)starts_);
    if (host_words_) gp_host_free(host_words_);
}

// The adjacency the launches of gp_launch_graph_iter read.  PageRank pulls, so it gets the lists of in-neighbours:
// the same ones where the graph is known to be symmetric, their transpose otherwise.
bool Workload::upload_packed(const CsrGraph &g, bool with_weights) {
    const size_t n = g.vertex_count;
    const uint64_t *offsets = g.vertexList.data();
    GPUdeviceptr from_offsets = vertex_list_, from_edges = edge_list_, own_offsets = nullptr, own_edges = nullptr;
    std::vector<uint64_t> in_offsets;
    bool ok = true;
    if (kind_ == "pagerank" && !g.symmetric) {
        in_offsets.assign(n + 1, 0);
        for (uint64_t e : g.edgeList) ++in_offsets[e + 1];
        for (size_t v = 0; v < n; ++v) in_offsets[v + 1] += in_offsets[v];
        std::vector<uint64_t> at(in_offsets.begin(), in_offsets.end() - 1), in_edges(g.edge_count);
        for (size_t v = 0; v < n; ++v)
            for (uint64_t i = offsets[v]; i < offsets[v + 1]; ++i) in_edges[at[g.edgeList[i]]++] = v;
        offsets = in_offsets.data();
        ok = gp_malloc(&own_offsets, (n + 1) * 8) == 0 && gp_memcpy_h2d(own_offsets, offsets, (n + 1) * 8) == 0 &&
             gp_malloc(&own_edges, std::max<size_t>(8, g.edge_count * 8)) == 0 && (g.edge_count == 0 || gp_memcpy_h2d(own_edges, in_edges.data(), g.edge_count * 8) == 0);
        from_offsets = own_offsets; from_edges = own_edges;
    }
    std::vector<uint32_t> row(n + 1, 0);
    for (size_t v = 0; v < n; ++v) row[v + 1] = row[v] + (uint32_t)((offsets[v + 1] - offsets[v] + 3) / 4);
    const size_t bytes = (size_t)row[n] * 16 + 16;
    row_end_ = row[n];
    symmetric_ = g.symmetric;
    ok = ok && gp_malloc(&row_, (n + 1) * 4) == 0 && gp_memcpy_h2d(row_, row.data(), (n + 1) * 4) == 0 && gp_malloc(&ids_, bytes) == 0 &&
         (!with_weights || gp_malloc(&weights_, bytes) == 0);
    gp_graph_pack_params p;
    std::memset(&p, 0, sizeof(p));
    p.vertex_count = (unsigned)n; p.row_end = row[n];
    p.vertex_list = (const unsigned long long *)from_offsets; p.edge_list = (const unsigned long long *)from_edges;
    p.weight_list = with_weights ? (const unsigned *)weight_list_ : nullptr;
    p.row = (const unsigned *)row_; p.ids = (unsigned *)ids_; p.weights = (unsigned *)weights_;
    ok = ok && gp_graph_pack_async(&p, nullptr) == 0 && gp_stream_sync(nullptr) == 0;
    if (own_offsets) gp_free(own_offsets);
    if (own_edges) gp_free(own_edges);
    return ok;
}

// initial state of a stepwise run (the memsets and single-element copies at the top of each reference loop)
Status Workload::begin(GPUstream stream) {
    const size_t n = n_;
    const uint32_t zero = 0;
    const unsigned char one = 1;
    if (kind_ == "bfs") {
        GC_CHECK(gp_fill32_async(label_, 0xFFFFFFFFu, n, stream));
        GC_CHECK(gp_stream_sync(stream));
        GC_CHECK(gp_memcpy_h2d(label_, &zero, 4));  // source = vertex 0 (graphcompute.tr.cu:255)
        level_ = 0;
    } else if (kind_ == "sssp") {
        GC_CHECK(gp_fill32_async(cost_, 0xFFFFFFFFu, n, stream));
        GC_CHECK(gp_fill32_async(new_cost_, 0xFFFFFFFFu, n, stream));
        GC_CHECK(gp_fill32_async(active_, 0, round4(n) / 4, stream));
        GC_CHECK(gp_stream_sync(stream));
        GC_CHECK(gp_memcpy_h2d(active_, &one, 1));
        GC_CHECK(gp_memcpy_h2d(cost_, &zero, 4));
        GC_CHECK(gp_memcpy_h2d(new_cost_, &zero, 4));
    }
    return Status::Succ;
}

// A launch was stopped: stay off the GPU while a higher priority needs it, then re-arm the stop index.
Status Workload::wait_turn(GPUstream stream, const PreemptEnv *env) {
    ++preemptions_;
    if (flag_to_lower_) {  // nobody else will lower a flag the kernel raised itself
        GC_CHECK(gp_fill32_async(env->flag, 0, 1, stream));  // a device store, as the raise was
        GC_CHECK(gp_stream_sync(stream));
        flag_to_lower_ = false;
    }
    if (env->higher_priority_active) {
        while (env->higher_priority_active()) std::this_thread::yield();
    } else {
        // nobody to ask: give whoever raised the flag time to lower it instead of relaunching
        // kernels that would leave at once
        std::this_thread::sleep_for(std::chrono::microseconds(50));
    }
    GC_CHECK(gp_fill32_async(env->stop_index, 0xFFFFFFFFu, 1, stream));
    return Status::Succ;
}

// Launches `kernels` in order; when a stop was recorded, waits for the workload's turn and
// relaunches from the stopped kernel on, counters untouched, until the list has run to its end.
Status Workload::run_kernels(const std::vector<int> &kernels, GPUstream stream, const PreemptEnv *env, int iteration, bool *changed) {
    const int K = (int)kernels.size();
    const size_t per_kernel = env ? (size_t)env->counter_groups * env->counter_stride : 0;
    if (env) GC_CHECK(gp_fill32_async(env->executed, 0, per_kernel * K, stream));
    GC_CHECK(gp_fill32_async(changed_, 0, 1, stream));
    const bool inject = env && env->inject_iteration == iteration && env->inject_kernel >= 0 && env->inject_kernel < K;
    int from = 0;
    for (;;) {
        for (int k = from; k < K; ++k) {
            gp_graph_params p;
            std::memset(&p, 0, sizeof(p));
            p.kernel = kernels[k];
            p.level = level_;
            p.vertex_count = n_;
            p.vertex_list = (const unsigned long long *)vertex_list_;
            p.edge_list = (const unsigned long long *)edge_list_;
            p.weight_list = (const unsigned int *)weight_list_;
            p.label = (unsigned int *)label_;
            p.active = (unsigned char *)active_;
            p.next_active = (unsigned char *)next_active_;
            p.comp = (unsigned long long *)comp_;
            p.delta = (float *)delta_; p.residual = (float *)residual_; p.value = (float *)value_;
            p.alpha = 0.85f; p.tolerance = 0.001f;  // graphcompute.h:83-84
            p.cost = (unsigned int *)cost_; p.new_cost = (unsigned int *)new_cost_;
            p.changed = (unsigned int *)changed_;
            p.lanes_per_vertex = lanes_;
            if (env) {
                gp_preempt_ctx ctx;
                std::memset(&ctx, 0, sizeof(ctx));
                ctx.flag = (int *)env->flag; ctx.stop_index = (int *)env->stop_index;
                ctx.executed = (int *)env->executed + per_kernel * k;
                ctx.kernel_id = k;
                ctx.inject_at = (inject && !injected_ && k == env->inject_kernel) ? env->inject_claim : -1;
                if (ctx.inject_at >= 0) { injected_ = true; flag_to_lower_ = true; }
                ctx.poll_every = env->poll_every;
                ctx.counter_groups = env->counter_groups;
                GC_CHECK(gp_launch_graph(&p, &ctx, stream, nullptr));
            } else {
                GC_CHECK(gp_launch_graph(&p, nullptr, stream, nullptr));
            }
            ++launches_;
        }
        host_words_[0] = -1;
        if (env) GC_CHECK(gp_memcpy_d2h_async(&host_words_[0], env->stop_index, sizeof(int), stream));
        GC_CHECK(gp_memcpy_d2h_async(&host_words_[1], changed_, sizeof(int), stream));
        // polled, not a blocking wait: a blocked thread wakes up tens of microseconds late, which
        // is paid once per iteration and on every preemption
        for (;;) {
            int idle = 0;
            GC_CHECK(gp_stream_query(stream, &idle));
            if (idle) break;
        }
        const int stop = host_words_[0];
        if (!env || stop < 0) break;
        RETURN_STATUS(wait_turn(stream, env));
        from = stop < K ? stop : K - 1;
    }
    *changed = host_words_[1] != 0;
    return Status::Succ;
}

// A launch's slot: its words, the claim counters and as many counters of the workgroups that have left it
// (gp_preempt_ctx::done), each in lines of 128 bytes of its own.  Behind the slots, gp_graph_iter_params::relay.
static size_t per_kernel_ints(const PreemptEnv *env) { return (size_t)env->counter_groups * env->counter_stride; }
// (nobody waits for the words of connected components, and its few launches clear half a ring like everybody's: with a set of words per XCD
// 4096 vertices of degree 16 took 60.5 us for 54.6, 2^17 of degree 6 68.2 for 66.0)
static bool in_sets(const std::string &kind) { return kind != "cc"; }
static size_t word_ints(const std::string &kind) { return in_sets(kind) ? GP_GRAPH_SETS * 32 : 32; }
constexpr size_t kRelayInts = GP_GRAPH_RELAYS * 32;

Status Workload::launch_slot(int i, bool fresh, GPUstream stream, const PreemptEnv *env) {
    gp_graph_iter_params p = queued_[i % kRing];
    int *slot = (int *)ring_ + slot_ints_ * (i % kRing);
    p.changed = (unsigned *)slot;
    if (p.prev_changed) p.prev_changed = (const unsigned *)((int *)ring_ + slot_ints_ * ((i - (int)(uintptr_t)p.prev_changed) % kRing));
    p.started = (unsigned long long *)starts_dev_ + i % kRing;
    p.sets = in_sets(kind_) ? GP_GRAPH_IN_SETS : 0;
    p.seq = seq_of_[i % kRing] = ++seq_;
    gp_preempt_ctx ctx;
    if (env) {
        std::memset(&ctx, 0, sizeof(ctx));
        ctx.flag = (int *)env->flag; ctx.stop_index = (int *)env->stop_index;
        ctx.executed = slot + word_ints(kind_);
        ctx.kernel_id = i % kRing; ctx.inject_at = -1; ctx.fresh = fresh;
        ctx.poll_every = env->poll_every; ctx.counter_groups = env->counter_groups;
        ctx.done = slot + word_ints(kind_) + per_kernel_ints(env);
        p.relay = (unsigned *)ring_ + slot_ints_ * kRing;
    }
    GC_CHECK(gp_launch_graph_iter(&p, env ? &ctx : nullptr, stream, nullptr));
    ++launches_;
    return Status::Succ;
}

// Queues one launch behind the others.  The words and claim counters of half the ring are cleared at a time, in stream
// order behind the launches that used them last.
Status Workload::submit(const gp_graph_iter_params &p, GPUstream stream, const PreemptEnv *env) {
    const size_t slot_ints = word_ints(kind_) + (env ? 2 * per_kernel_ints(env) : 0);
    if (slot_ints != slot_ints_) {
        if (ring_) gp_free(ring_);
        ring_ = nullptr; slot_ints_ = 0;
        GC_CHECK(gp_malloc(&ring_, (slot_ints * kRing + kRelayInts) * sizeof(int)));
        slot_ints_ = slot_ints;
        GC_CHECK(gp_fill32_async((int *)ring_ + slot_ints * kRing, 0, kRelayInts, stream));
    }
    const int i = submitted_++;
    if (i % (kRing / 2) == 0) GC_CHECK(gp_fill32_async((int *)ring_ + slot_ints_ * (i % kRing), 0, slot_ints_ * (kRing / 2), stream));
    queued_[i % kRing] = p;
    return launch_slot(i, true, stream, env);
}

// Waits until everything queued has left the GPU; *stop receives the slot of the launch that was stopped, or -1.
Status Workload::drain(GPUstream stream, const PreemptEnv *env, int *stop) {
    GC_CHECK(gp_report_stop_async(env ? (const int *)env->stop_index : nullptr, (unsigned long long *)starts_dev_ + kRing, ++seq_, stream));
    unsigned long long report = 0;
    RETURN_STATUS(spin_until(stream, [&] { report = __atomic_load_n(starts_ + kRing, __ATOMIC_ACQUIRE); return (unsigned)report == seq_; }));
    *stop = (int)(report >> 32);
    return Status::Succ;
}

// A launch was stopped and this run has left the GPU: when it is this workload's turn again, that launch is
// queued once more, and the ones behind it with it (they left when they found the stop recorded).
Status Workload::restart(int stop, GPUstream stream, const PreemptEnv *env) {
    RETURN_STATUS(wait_turn(stream, env));
    int from = submitted_ - 1;
    while (from > 0 && from % kRing != stop) --from;
    GC_CHECK(gp_fill32_async((int *)ring_ + slot_ints_ * kRing, 0, kRelayInts, stream));
    for (int i = from; i < submitted_; ++i) {
        // (a launch that left in front of its first claim counted nobody: the count of leavers starts again)
        GC_CHECK(gp_fill32_async((int *)ring_ + slot_ints_ * (i % kRing) + word_ints(kind_) + per_kernel_ints(env), 0, per_kernel_ints(env), stream));
        RETURN_STATUS(launch_slot(i, false, stream, env));
    }
    return Status::Succ;
}

// The end of a run: everything queued is done, or had nothing to do, and has left.
Status Workload::settle(GPUstream stream, const PreemptEnv *env) {
    for (;;) {
        int stop = -1;
        RETURN_STATUS(drain(stream, env, &stop));
        if (stop < 0) return Status::Succ;
        RETURN_STATUS(restart(stop, stream, env));
    }
}

// Waits until launch `i` starts, i.e. until the ones before it are done.  *changed: the iteration before it changed
// something; *count: of how many vertices over the tolerance it knows.
Status Workload::await_start(int i, GPUstream stream, const PreemptEnv *env, bool *changed, unsigned *count) {
    auto start_of = [&](int k, unsigned *low) {
        return spin_until(stream, [&] {
            const unsigned long long word = __atomic_load_n(starts_ + k % kRing, __ATOMIC_ACQUIRE);
            *low = (unsigned)word;
            return (unsigned)(word >> 32) == seq_of_[k % kRing];
        });
    };
    for (;;) {
        unsigned low = 0;
        RETURN_STATUS(start_of(i, &low));
        if (!(low & GP_GRAPH_START_STOPPED)) {
            *changed = (low & GP_GRAPH_START_CHANGED) != 0;
            *count = low & GP_GRAPH_START_COUNT;
            return Status::Succ;
        }
        // A stop is recorded.  The GPU is vacated when the last launch queued has started, as it finds nothing to do.  (That
        // is known from what is in the queue already: a report submitted now can come to stand behind the work of whoever
        // raised the flag, where the two streams share a hardware queue.)
        unsigned other = 0;
        for (int k = i + 1; k < submitted_; ++k) RETURN_STATUS(start_of(k, &other));
        RETURN_STATUS(restart((int)(low & ~GP_GRAPH_START_STOPPED), stream, env));
    }
}

gp_graph_iter_params Workload::params(int kernel) const {
    gp_graph_iter_params p;
    std::memset(&p, 0, sizeof(p));
    p.kernel = kernel;
    p.vertex_count = (unsigned)n_; p.row_end = row_end_;
    p.row = (const unsigned *)row_; p.ids = (const unsigned *)ids_; p.weights = (const unsigned *)weights_;
    p.label = (unsigned *)label_; p.cost = (unsigned *)cost_; p.parent = (unsigned *)parent_;
    p.active = (unsigned char *)active_; p.next_active = (unsigned char *)next_active_;
    p.comp = (unsigned long long *)comp_;
    p.share = (const float *)share_; p.next_share = (float *)delta_;
    p.degree = (const float *)degree_; p.residual = (float *)residual_; p.value = (float *)value_;
    p.gained = (float *)gained_; p.next_gained = gained_ ? (float *)gained_ + n_ : nullptr;
    p.alpha = 0.85f; p.tolerance = 0.001f;  // graphcompute.h:83-84
    p.step = step_;
    return p;
}

// The iterations are those of the reference's loops.  Launches are queued a few ahead of the GPU: a launch tells the host
// when it starts and, since the ones before it are done then, whether the iteration before it changed anything, and the
// host queues the next one.  (A launch takes 3-4 us at least and the host's turn, from the word to a queued launch, as
// long; kAhead of them keep the GPU busy.  Those are what is still queued when the run converges or is stopped: each has
// to start and leave, 3-4 us, before the run can end or the GPU is vacated.)
Status Workload::compute(GPUstream stream, const PreemptEnv *env) {
    if (!row_ || (env && env->inject_kernel >= 0 && env->inject_iteration >= -1)) return compute_stepwise(stream, env);
    iterations_ = submitted_ = 0;
    if (kind_ == "cc") {
        iterations_ = 3;  // (linking, flattening, labels)
        // (a graph of a million edges and more in three steps, by the first two neighbours, the first four and all of them:
        // 2^20 vertices of degree 16 take 290 us, at once 500-600, of which a stop waited for half; on a small graph the
        // launches more cost 8 us)
        RETURN_STATUS(submit(params(GP_GRAPH_IT_CC_INIT), stream, env));
        for (unsigned neighbours : {2u, 4u, 0u}) {
            if (neighbours && row_end_ < (1u << 18)) continue;
            RETURN_STATUS(submit(params(GP_GRAPH_IT_CC_FLATTEN), stream, env));
            gp_graph_iter_params link = params(GP_GRAPH_IT_CC_LINK);
            link.level = neighbours;
            RETURN_STATUS(submit(link, stream, env));
        }
        RETURN_STATUS(submit(params(GP_GRAPH_IT_CC_LABEL), stream, env));
        return settle(stream, env);
    }
    const bool bfs = kind_ == "bfs", pagerank = kind_ == "pagerank";
    const int max_iter = pagerank ? 100 : 1 << 30;  // graphcompute.h:82
    RETURN_STATUS(submit(params(bfs ? GP_GRAPH_IT_BFS_INIT : pagerank ? GP_GRAPH_IT_PR_INIT : GP_GRAPH_IT_SSSP_INIT), stream, env));
    GPUdeviceptr share = delta_, other = share_;
    float *gained = (float *)gained_, *next_gained = gained + (gained ? n_ : 0);
    bool push = false, pushing = false;  // wanted; the shares of the iteration before have been pushed
    unsigned sampled = ~0u;              // vertices over the tolerance in the sampled tiles, of the last iteration that is known
    int next = 0, started = 0;           // the iteration to queue next; launches that have started
    std::deque<int> first_of;            // of the iterations queued and not started (next - 1 the last): their first launch
    for (;;) {
        while (next < max_iter && submitted_ - started <= kAhead) {
            gp_graph_iter_params p = params(bfs ? GP_GRAPH_IT_BFS : pagerank ? GP_GRAPH_IT_PR : GP_GRAPH_IT_SSSP);
            p.level = (unsigned)next;
            if (next & 1) std::swap(p.active, p.next_active);
            p.prev_changed = next ? (const unsigned *)(uintptr_t)1 : nullptr;  // (how many launches back that word is; launch_slot makes it an address)
            first_of.push_back(submitted_);
            // (2^20 vertices of degree 16: 46 us for the pull, as much for atomics from one vertex in thirty-five, and the count is
            // two launches old while the vertices become more by an eighth per iteration.  The push begins a little below that,
            // because going over to it takes a launch.  From one in twenty-five and back to it below one in 32: 1-2 % slower.)
            if (pagerank) push = symmetric_ && sampled < n_ / GP_GRAPH_SAMPLED / (push ? 32 : 36);
            if (pagerank && pushing) {
                p.kernel = GP_GRAPH_IT_PR_STEP;
                p.gained = gained;
                p.next_gained = push ? next_gained : nullptr;
                p.next_share = (float *)share;
                std::swap(gained, next_gained);
                pushing = push;
            } else if (pagerank) {
                p.share = (const float *)share;
                if (push) {  // the pull's shares go out; this iteration takes them in, and pushes its own
                    p.kernel = GP_GRAPH_IT_PR_PUSH;
                    p.next_gained = gained;
                    RETURN_STATUS(submit(p, stream, env));
                    p.kernel = GP_GRAPH_IT_PR_STEP;
                    p.prev_changed = next ? (const unsigned *)(uintptr_t)2 : nullptr;
                    p.gained = gained; p.next_gained = next_gained;
                    std::swap(gained, next_gained);
                    pushing = true;
                } else {
                    p.next_share = (float *)other;
                    std::swap(share, other);
                }
            }
            RETURN_STATUS(submit(p, stream, env));
            ++next;
        }
        if (started == submitted_) {  // all there may be
            iterations_ = max_iter;
            return settle(stream, env);
        }
        bool changed = true;
        unsigned count = 0;
        RETURN_STATUS(await_start(started, stream, env, &changed, &count));
        if (!first_of.empty() && first_of.front() == started) {  // the first launch of an iteration speaks of the iteration before
            iterations_ = next - (int)first_of.size();
            first_of.pop_front();
            if (!changed) return settle(stream, env);
            sampled = iterations_ ? count : ~0u;
        }
        ++started;
    }
}

Status Workload::compute_stepwise(GPUstream stream, const PreemptEnv *env) {
    iterations_ = 0;
    injected_ = false;
    RETURN_STATUS(begin(stream));
    bool changed = false;
    std::vector<int> loop;
    int max_iter = 1 << 30;
    if (kind_ == "bfs") loop = {GP_GRAPH_BFS_STEP};
    else if (kind_ == "cc") {
        loop = {GP_GRAPH_CC_STEP};
        // labels and frontier are set up by a kernel (the reference uploads 8 bytes per vertex
        // from the host on every run, graphcompute.tr.cu:143-146)
        RETURN_STATUS(run_kernels({GP_GRAPH_CC_INIT}, stream, env, -1, &changed));
    }
    else if (kind_ == "sssp") loop = {GP_GRAPH_SSSP_RELAX, GP_GRAPH_SSSP_UPDATE};
    else {
        loop = {GP_GRAPH_PR_PUSH, GP_GRAPH_PR_UPDATE};
        max_iter = 100;  // graphcompute.h:82
        RETURN_STATUS(run_kernels({GP_GRAPH_PR_INIT}, stream, env, -1, &changed));
    }
    do {
        RETURN_STATUS(run_kernels(loop, stream, env, iterations_, &changed));
        if (kind_ == "bfs") ++level_;
        if (kind_ == "cc") {  // the frontier just used is cleared and becomes the next one's buffer
            GC_CHECK(gp_fill32_async(active_, 0, round4(n_) / 4, stream));
            std::swap(active_, next_active_);
        }
        ++iterations_;
    } while (changed && iterations_ < max_iter);
    if (flag_to_lower_ && env) {  // raised by the very last claims: no later claim saw it
        GC_CHECK(gp_fill32_async(env->flag, 0, 1, stream));
        GC_CHECK(gp_stream_sync(stream));
        flag_to_lower_ = false;
    }
    return Status::Succ;
}

size_t Workload::result_bytes(const std::string &key) const {
    if (key == "comp" && comp_) return n_ * 8;
    if (key == "label" && label_) return n_ * 4;
    if (key == "value" && value_) return n_ * 4;
    if (key == "cost" && cost_) return n_ * 4;
    return 0;
}

Status Workload::read_result(const std::string &key, void *out, size_t len, bool pinned) const {
    const size_t bytes = result_bytes(key);
    if (bytes == 0) return Status::NotFound;
    if (len < bytes) return Status::OutOfRange;
    GPUdeviceptr src = key == "comp" ? comp_ : key == "label" ? label_ : key == "value" ? value_ : cost_;
    if (pinned) {
        GC_CHECK(gp_fetch(out, src, bytes, nullptr));  // (compute() has waited for its stream)
        return Status::Succ;
    }
    GC_CHECK(gp_stream_sync(nullptr));
    GC_CHECK(gp_memcpy_d2h(out, src, bytes));
    return Status::Succ;
}

}  // namespace GraphCompute
