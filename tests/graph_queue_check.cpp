// The host loop of the graph workloads (host/graphcompute.cpp) over a device made of threads: every stream is a thread
// that works off what was submitted to it, in order and slowly.  An iteration changes something until a level that the
// check chooses; what it does to its claim counters, its words and the stop index is what the kernels do.
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <new>
#include <thread>

#include "workloads/graphcompute.h"

// ---- memory in use, for the check that a long run keeps nothing per launch ------------------------------------------
static std::atomic<long> g_live{0}, g_peak{0};
void *operator new(size_t n) {
    size_t *p = (size_t *)std::malloc(n + 16);
    if (!p) throw std::bad_alloc();
    *p = n;
    const long live = g_live += (long)n;
    for (long peak = g_peak; live > peak && !g_peak.compare_exchange_weak(peak, live);) { }
    return (char *)p + 16;
}
void operator delete(void *p) noexcept {
    if (!p) return;
    p = (char *)p - 16;
    g_live -= (long)*(size_t *)p;
    std::free(p);
}
void operator delete(void *p, size_t) noexcept { operator delete(p); }

// ---- the device -----------------------------------------------------------------------------------------------------
struct gp_stream_s {
    std::mutex mu;
    std::condition_variable cv;
    std::deque<std::function<void()>> ops;
    std::atomic<int> pending{0};
    bool quit = false;
    std::thread worker{[this] {
        for (;;) {
            std::function<void()> op;
            {
                std::unique_lock<std::mutex> l(mu);
                cv.wait(l, [&] { return quit || !ops.empty(); });
                if (ops.empty()) return;
                op = std::move(ops.front());
                ops.pop_front();
            }
            op();
            pending.fetch_sub(1);
        }
    }};
    void submit(std::function<void()> op) {
        pending.fetch_add(1);
        std::lock_guard<std::mutex> l(mu);
        ops.push_back(std::move(op));
        cv.notify_one();
    }
    ~gp_stream_s() {
        { std::lock_guard<std::mutex> l(mu); quit = true; }
        cv.notify_one();
        worker.join();
    }
};
static gp_stream_s g_null;
static gp_stream_s *of(gp_stream s) { return s ? s : &g_null; }

static int g_delay_us = 0;        // what a launch takes
static int g_last_level = 0;      // the iteration that changes nothing
static int g_stop_at_level = -1;  // the iteration that finds the flag up, once
static std::vector<int> g_ran;    // levels in the order in which they ran
static std::atomic<int> g_in_flight{0};  // launches submitted and not done
static int g_left = 0;            // launches that left because of a recorded stop
static std::atomic<size_t> g_cleared{0};  // words
static void pause_us(int us) { if (us) std::this_thread::sleep_for(std::chrono::microseconds(us)); }

extern "C" {
const char *gp_last_error(void) { return ""; }
int gp_malloc(void **p, size_t n) { *p = std::malloc(n ? n : 1); return 0; }
int gp_free(void *p) { std::free(p); return 0; }
int gp_host_alloc(void **p, size_t n) { return gp_malloc(p, n); }
int gp_host_free(void *p) { return gp_free(p); }
int gp_host_alloc_coherent(void **h, void **d, size_t n) { *h = *d = std::calloc(1, n); return 0; }
int gp_memcpy_h2d(void *d, const void *h, size_t n) { std::memcpy(d, h, n); return 0; }
int gp_memcpy_d2h(void *h, const void *d, size_t n) { std::memcpy(h, d, n); return 0; }
int gp_memcpy_d2h_async(void *h, const void *d, size_t n, gp_stream s) { of(s)->submit([=] { std::memcpy(h, d, n); }); return 0; }
int gp_fetch(void *h, const void *d, size_t n, gp_stream s) { gp_stream_sync(s); std::memcpy(h, d, n); return 0; }
int gp_stream_sync(gp_stream s) { while (of(s)->pending) std::this_thread::yield(); return 0; }
int gp_stream_query(gp_stream s, int *idle) { *idle = of(s)->pending == 0; return 0; }
int gp_fill32_async(void *p, uint32_t v, size_t n, gp_stream s) {
    g_cleared += n;
    of(s)->submit([=] { for (size_t i = 0; i < n; ++i) ((uint32_t *)p)[i] = v; });
    return 0;
}
int gp_graph_pack_async(const gp_graph_pack_params *, gp_stream) { return 0; }
int gp_launch_graph(const gp_graph_params *, const gp_preempt_ctx *, gp_stream, gp_launch_info *) { return 1; }
int gp_report_stop_async(const int *stop_index, unsigned long long *word, unsigned seq, gp_stream s) {
    of(s)->submit([=] { __atomic_store_n(word, (unsigned long long)(unsigned)(stop_index ? *stop_index : -1) << 32 | seq, __ATOMIC_RELEASE); });
    return 0;
}
int gp_launch_graph_iter(const gp_graph_iter_params *pp, const gp_preempt_ctx *ctx, gp_stream s, gp_launch_info *) {
    const gp_graph_iter_params p = *pp;
    int *stop = ctx ? ctx->stop_index : nullptr, *claims = ctx ? ctx->executed : nullptr;
    const int id = ctx ? ctx->kernel_id : 0;
    const bool iteration = p.kernel == GP_GRAPH_IT_BFS || p.kernel == GP_GRAPH_IT_PR || p.kernel == GP_GRAPH_IT_PR_STEP || p.kernel == GP_GRAPH_IT_SSSP;
    ++g_in_flight;
    of(s)->submit([=] {
        struct Done { ~Done() { --g_in_flight; } } done;
        if (p.started) {
            unsigned low = !p.prev_changed ? GP_GRAPH_START_CHANGED : *p.prev_changed ? GP_GRAPH_START_CHANGED | p.prev_changed[1] : 0;
            if (stop && *stop != -1) low = GP_GRAPH_START_STOPPED | (unsigned)*stop;
            __atomic_store_n(p.started, (unsigned long long)p.seq << 32 | low, __ATOMIC_RELEASE);
        }
        pause_us(g_delay_us);
        if (p.prev_changed && *p.prev_changed == 0) return;
        if (stop && *stop != -1) { ++g_left; return; }
        if (iteration && stop && (int)p.level == g_stop_at_level) { g_stop_at_level = -1; *stop = id; return; }
        if (claims && claims[0]++) { std::printf("launch %d claimed twice\n", id); std::exit(1); }
        if (!iteration) return;
        g_ran.push_back((int)p.level);
        if ((int)p.level != g_last_level) { p.changed[0] = 1; p.changed[1] = 1000; }
    });
    return 0;
}
}

#define CHECK(cond, ...) do { if (!(cond)) { std::printf("%s: ", #cond); std::printf(__VA_ARGS__); std::printf("\n"); std::exit(1); } } while (0)

static GraphCompute::CsrGraph path_graph(uint64_t n) {
    GraphCompute::CsrGraph g;
    g.vertex_count = n;
    for (uint64_t v = 0; v < n; ++v) { g.vertexList.push_back(v); if (v + 1 < n) { g.edgeList.push_back(v + 1); g.weightList.push_back(1); } }
    g.vertexList.push_back(n - 1);
    g.edge_count = n - 1;
    return g;
}

static int g_flag = 0, g_stop = -1, g_claims[64];
static GraphCompute::PreemptEnv env_of() {
    GraphCompute::PreemptEnv env;
    env.flag = &g_flag; env.stop_index = &g_stop; env.executed = g_claims;
    return env;
}

static void run(const char *kind, int last_level, gp_stream s, const GraphCompute::PreemptEnv *env, GraphCompute::Workload &w) {
    g_last_level = last_level;
    g_ran.clear();
    CHECK(w.compute(s, env) == Status::Succ, "%s", kind);
    CHECK((int)g_ran.size() == last_level + 1 && w.iterations() == last_level + 1, "%s: %zu iterations ran, %d counted, of %d", kind, g_ran.size(), w.iterations(), last_level + 1);
    for (int i = 0; i <= last_level; ++i) CHECK(g_ran[i] == i, "%s: iteration %d ran as number %d", kind, g_ran[i], i);
}

// compute() is blocking: nothing of a run is left in its stream, whatever iteration ends it
static void check_nothing_left_behind() {
    g_delay_us = 300;
    for (const char *kind : {"bfs", "pagerank", "sssp"}) {
        auto w = GraphCompute::Workload::create(kind, path_graph(64));
        const GraphCompute::PreemptEnv env = env_of();
        gp_stream_s a, b;
        for (int last = 0; last < 26; last += 5)
            for (gp_stream s : {&a, &b}) {
                run(kind, last, s, &env, *w);
                CHECK(g_in_flight == 0, "%s ended by iteration %d: %d launches still in the stream", kind, last, g_in_flight.load());
            }
    }
    g_delay_us = 0;
}

// A stop, wherever it falls: when the workload gives way, nothing of it is on the GPU any more but a launch that is
// leaving, and few launches had to start and leave for that; every iteration still runs once, in order.
static void check_stops() {
    g_delay_us = 100;
    for (const char *kind : {"bfs", "pagerank", "sssp"})
        for (int last : {9, 40})
            for (int stop_at : {0, 1, 2, 5, last - 1, last}) {
                auto w = GraphCompute::Workload::create(kind, path_graph(64));
                gp_stream_s s;
                GraphCompute::PreemptEnv env = env_of();
                int gave_way = 0;
                g_left = 0;
                g_stop_at_level = stop_at;
                env.higher_priority_active = [&] {
                    ++gave_way;
                    CHECK(g_in_flight <= 1, "%s stopped at %d: %d launches still to come", kind, stop_at, g_in_flight.load());
                    CHECK(g_left <= 4, "%s stopped at %d: %d launches had to leave", kind, stop_at, g_left);
                    return false;
                };
                run(kind, last, &s, &env, *w);
                CHECK(gave_way == 1 && w->preemptions() == 1, "%s stopped at %d: gave way %d times", kind, stop_at, gave_way);
            }
    g_delay_us = 0;
}

// a run of many iterations keeps as much as a short one
static void check_long_run_keeps_nothing() {
    auto w = GraphCompute::Workload::create("bfs", path_graph(64));
    const GraphCompute::PreemptEnv env = env_of();
    const int iterations = 100000;
    g_ran.reserve(iterations + 64);
    gp_stream_s s;
    run("bfs", 100, &s, &env, *w);
    const long before = g_live;
    g_peak = before;
    run("bfs", iterations - 1, &s, &env, *w);
    // (what the fake device has queued at one time, and the loop's own lists)
    CHECK(g_peak - before < 256 << 10, "%ld bytes more in use during %d iterations", g_peak.load() - before, iterations);
}

// connected components is a handful of launches, and what it clears in front of them counts: half a ring of claim counters, and a line of words each
static void check_what_cc_clears() {
    auto w = GraphCompute::Workload::create("cc", path_graph(64));
    const GraphCompute::PreemptEnv env = env_of();
    gp_stream_s s;
    for (int i = 0; i < 2; ++i) {
        g_cleared = 0;
        CHECK(w->compute(&s, &env) == Status::Succ, "cc");
    }
    const size_t counters = 2 * (size_t)env.counter_groups * env.counter_stride;
    CHECK(g_cleared <= 32 * (counters + 32), "%zu words cleared, with %zu words of counters to a launch", g_cleared.load(), counters);
}

int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "blocking") check_nothing_left_behind();
    else if (what == "stops") check_stops();
    else if (what == "clears") check_what_cc_clears();
    else if (what == "memory") check_long_run_keeps_nothing();
    else return 2;
    std::printf("ok %s\n", what.c_str());
}
