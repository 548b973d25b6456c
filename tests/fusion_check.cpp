// foo::Model's launch fusions (scale-shift into the convolution behind it, convolutions side by side) over a device layer in host
// memory whose kernels compute the first row of what they write from the first row of what they read.  Every case runs on a model that
// merges launches and on one that does not, and looks at what a caller can see.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <string>
#include <vector>

#include "../gpreempt_amd/host/graph_builder.h"
#include "../gpreempt_amd/host/zoo.h"
#include "model.h"

using foo::GraphBuilder;
using foo::Model;
using foo::Tensor;

static int g_merged = 0, g_launches = 0;  // launches that did the work of several kernels, and all
static int g_capturing = 0;
static gp_stream g_scaled_on = nullptr;  // where the last scale-shift layer was launched
static std::vector<gp_stream> g_gone;

static uint32_t mix(uint32_t a, uint32_t b) { return (a ^ (b + 0x9E3779B9u + (a << 6) + (a >> 2))) * 0x85EBCA6Bu; }
static uint32_t hash(const void *p, long n, uint32_t h = 1) {
    if (!p) return h;
    for (long i = 0; i < n; ++i) h = mix(h, ((const uint32_t *)p)[i]);
    return h;
}
static void put(void *p, long n, uint32_t h) {
    for (long i = 0; i < n; ++i) ((uint32_t *)p)[i] = mix(h, (uint32_t)i);
}
static uint32_t scaled(const gp_eltwise_params *e, long i) {
    return mix(mix(((const uint32_t *)e->a)[i], ((const uint32_t *)e->scale)[i]), ((const uint32_t *)e->shift)[i]);
}
static void conv(const gp_conv_params *c, uint32_t in) { put(c->out, c->Cout, mix(mix(hash(c->weight, c->Cin), hash(c->bias, c->Cout)), mix(in, hash(c->residual, c->Cout)))); }
static std::vector<int> g_at;  // the kernel of each launch that a preemption was injected into
static int done(const gp_preempt_ctx *ctx, gp_launch_info *info) {
    if (ctx && ctx->inject_at >= 0) g_at.push_back(ctx->kernel_id);
    if (info) std::memset(info, 0, sizeof(*info));
    ++g_launches;
    return 0;
}

// (these take the place of the library's: the executable's symbols come first; every model here is fp32)
extern "C" {
int gp_malloc(void **p, size_t n) { *p = std::calloc(1, n ? n : 1); return 0; }
int gp_free(void *p) { std::free(p); return 0; }
int gp_memcpy_h2d(void *d, const void *h, size_t n) { std::memcpy(d, h, n); return 0; }
int gp_memcpy_h2d_async(void *d, const void *h, size_t n, gp_stream) { std::memcpy(d, h, n); return 0; }
int gp_memcpy_d2h_async(void *h, const void *d, size_t n, gp_stream) { std::memcpy(h, d, n); return 0; }
int gp_fetch(void *h, const void *d, size_t n, gp_stream) { std::memcpy(h, d, n); return 0; }
int gp_fill32_async(void *, uint32_t, size_t, gp_stream) { return 0; }
int gp_stream_sync(gp_stream) { return 0; }
int gp_stream_capturing(gp_stream, int *capturing) { *capturing = g_capturing; return 0; }
int gp_stream_exists(gp_stream s) { for (gp_stream g : g_gone) if (g == s) return 0; return 1; }
int gp_stage_create(gp_stage *out) { *out = (gp_stage)std::malloc(1); return 0; }
int gp_stage_destroy(gp_stage st) { std::free(st); return 0; }
int gp_stage_upload_async(gp_stage, void *d, const void *h, size_t n, gp_stream) { std::memcpy(d, h, n); return 0; }
int gp_launch_nchw_to_nhwc(const gp_layout_params *p, const gp_preempt_ctx *x, gp_stream, gp_launch_info *i) { put(p->out, p->c_pad, hash(p->in, p->C)); return done(x, i); }
int gp_launch_pool2d(const gp_pool_params *p, const gp_preempt_ctx *x, gp_stream, gp_launch_info *i) { put(p->out, p->C, hash(p->in, p->C)); return done(x, i); }
int gp_launch_softmax(const gp_softmax_params *p, const gp_preempt_ctx *x, gp_stream, gp_launch_info *i) { put(p->out, p->cols, hash(p->x, p->cols)); return done(x, i); }
int gp_launch_eltwise(const gp_eltwise_params *e, const gp_preempt_ctx *x, gp_stream s, gp_launch_info *info) {
    g_scaled_on = s;
    for (long i = 0; i < e->cols; ++i) ((uint32_t *)e->out)[i] = scaled(e, i);
    return done(x, info);
}
int gp_launch_conv2d(const gp_conv_params *c, const gp_preempt_ctx *x, gp_stream, gp_launch_info *info) {
    conv(c, hash(c->in, c->Cin));
    return done(x, info);
}
int gp_launch_eltwise_conv2d(const gp_eltwise_params *e, const gp_conv_params *c, const gp_preempt_ctx *x, gp_stream, gp_launch_info *info) {
    uint32_t in = 1;
    for (long i = 0; i < e->cols; ++i) in = mix(in, scaled(e, i));
    conv(c, in);
    ++g_merged;
    return done(x, info);
}
int gp_launch_conv2d_group(const gp_conv_params *p, int n, const gp_preempt_ctx *x, gp_stream, gp_launch_info *info) {
    for (int i = 0; i < n; ++i) conv(p + i, hash(p[i].in, p[i].Cin));
    ++g_merged;
    return done(x, info);
}
}

// Three scale-shift layers in front of pointwise convolutions, the way DenseNet has them; "group": three convolutions side by side;
// "rewritten": what the second layer reads is overwritten by a kernel behind its convolution; "beside": by one that writes the
// channels next to those; "residual": the second convolution also adds the second layer's output.
Status foo::zoo_build(Model &m, const std::string &name) {
    GraphBuilder b(m, "f32");
    auto is = [&](const char *s) { return name == s; };
    if (is("group")) {  // kernels: 0 layout, 1 stem, 2 left, 3 middle, 4 right (side by side), 5 join, 6 softmax
        Tensor t = b.conv("stem", b.input_nchw(1, 8, 2, 2), 512, 1, 1, 0, GP_ACT_RELU);
        Tensor left = b.conv("left", t, 512, 1, 1, 0, GP_ACT_RELU);
        b.conv("middle", t, 32, 3, 1, 1, GP_ACT_RELU);
        Tensor right = b.conv("right", t, 512, 1, 1, 0, GP_ACT_RELU);
        Tensor join = b.conv("join", left, 512, 1, 1, 0, GP_ACT_RELU, &right);
        size_t heads = b.add_storage("heads", 512, "float32");
        b.softmax(join.st, heads, 1, 512, 1.f);
        return Status::Succ;
    }
    Tensor t = b.input_nchw(1, 8, 2, 2);
    Tensor block = b.activation("block", 1, 2, 2, 64), first = GraphBuilder::slice(block, 0, 32), next = GraphBuilder::slice(block, 32, 32);
    b.conv("stem", t, 32, 1, 1, 0, GP_ACT_RELU, nullptr, &first);
    Tensor n1 = b.eltwise("norm1", first, nullptr, "norm1", GP_ACT_RELU);
    Tensor c1 = b.conv("conv1", n1, 32, 1, 1, 0, GP_ACT_RELU);
    Tensor n2 = b.eltwise("norm2", c1, nullptr, "norm2", GP_ACT_RELU);
    Tensor c2 = b.conv("conv2", n2, 32, 1, 1, 0, GP_ACT_RELU, is("residual") ? &n2 : nullptr);
    if (is("rewritten")) b.pool("over", c2, 1, 1, 0, 0, &c1);
    if (is("beside")) b.conv("grow", c2, 32, 3, 1, 1, GP_ACT_NONE, nullptr, &next);
    Tensor mid = b.pool("mid", c2, 1, 1, 0, 0);
    Tensor n3 = b.eltwise("norm3", mid, nullptr, "norm3", GP_ACT_NONE);
    Tensor c3 = b.conv("conv3", n3, 32, 1, 1, 0, GP_ACT_RELU);
    size_t heads = b.add_storage("heads", 32, "float32");
    b.softmax(c3.st, heads, 1, 32, 1.f);
    return Status::Succ;
}

// a model that merges launches beside one that does not
struct Pair {
    Model merged, apart;
    explicit Pair(const char *name) {
        for (int fuse = 0; fuse < 2; ++fuse) {
            setenv("GPREEMPT_FUSE_LN", fuse ? "1" : "0", 1);
            if ((fuse ? merged : apart).build(name) != Status::Succ) { std::printf("no model %s\n", name); std::exit(1); }
        }
        each([&](Model &m) {
            for (size_t i = 0; i < m.get_storage_num(); ++i) fill(m, i, 7);
        });
    }
    void each(const std::function<void(Model &)> &f) { f(apart); f(merged); }
    static void fill(Model &m, size_t idx, uint32_t seed) {
        std::vector<uint32_t> v(m.get_storage_size(idx) / 4);
        put(v.data(), (long)v.size(), mix(seed, (uint32_t)idx));
        if (m.set(idx, v.data(), v.size() * 4, nullptr) != Status::Succ) { std::printf("set %zu\n", idx); std::exit(1); }
    }
    static size_t at(Model &m, const char *name) {
        size_t idx = 0;
        if (m.find_storage_idx(name, idx) != Status::Succ) { std::printf("no storage %s\n", name); std::exit(1); }
        return idx;
    }
    static void launch(Model &m, size_t from, size_t to, gp_stream s = nullptr) {
        for (size_t i = from; i < to; ++i)
            if (m.launch(i, s) != Status::Succ) { std::printf("kernel %zu\n", i); std::exit(1); }
    }
    void pass(gp_stream s = nullptr) {
        each([&](Model &m) { launch(m, 0, m.get_kernel_num(), s); });
    }
    // `f` on both, then the same in every storage, before and after another pass, and on another pair from fresh values
    void then(const char *when, const std::function<void(Model &)> &f) {
        each(f);
        same(when);
        pass();
        same(when);
    }
    // what a pointer of before shows
    void same_at(GPUdeviceptr a, GPUdeviceptr b, size_t bytes, const char *when) {
        if (std::memcmp(a, b, bytes) == 0) return;
        std::printf("%s: the memory differs\n", when);
        std::exit(1);
    }
    // both models show the same in every storage
    void same(const char *when) {
        for (size_t i = 0; i < merged.get_storage_num(); ++i) {
            std::vector<uint32_t> a(merged.get_storage_size(i) / 4), b(a);
            if (merged.get(i, a.data(), a.size() * 4, nullptr) != Status::Succ || apart.get(i, b.data(), b.size() * 4, nullptr) != Status::Succ || a != b) {
                std::printf("%s: %s differs\n", when, merged.get_storage_info(i).name.c_str());
                std::exit(1);
            }
        }
    }
};

static void passes_merge(const char *name, int merged) {
    Pair p(name);
    for (int pass = 0; pass < 2; ++pass) {
        g_merged = 0;
        p.pass();
        if (g_merged != merged) { std::printf("%s: %d launches merged, not %d\n", name, g_merged, merged); std::exit(1); }
        p.same(name);
    }
}

// kernels of "plain": 0 layout, 1 stem, 2 norm1, 3 conv1, 4 norm2, 5 conv2, 6 pool, 7 norm3, 8 conv3, 9 softmax
static void storages() {
    auto index = [](Model &m, const char *key) { return Pair::at(m, key); };
    for (const char *key : {"norm2.out", "conv1.out", "norm2.scale", "norm2.shift", "block", "conv2.out", "data"}) {
        Pair p("plain");
        p.pass();
        p.then((std::string("set ") + key).c_str(), [&](Model &m) { Pair::fill(m, index(m, key), 21); });
        p.then("set twice", [&](Model &m) { Pair::fill(m, index(m, key), 22); Pair::fill(m, index(m, key), 23); });
        // ... and the convolution alone, which reads what was set
        p.then("the convolution alone", [&](Model &m) { Pair::fill(m, index(m, key), 24); Pair::launch(m, 5, 6); });
        p.then("the layer alone", [&](Model &m) { Pair::launch(m, 4, 5); });
        p.then("the layer, a value, the convolution", [&](Model &m) { Pair::launch(m, 4, 5); Pair::fill(m, index(m, key), 25); Pair::launch(m, 5, 6); });
        p.then("pinned", [&](Model &m) {
            std::vector<uint32_t> v(m.get_storage_size(index(m, key)) / 4, 26);
            if (m.set_pinned(index(m, key), v.data(), v.size() * 4, nullptr) != Status::Succ) std::exit(1);
            Pair::launch(m, 5, 6);
        });
        g_merged = 0;
        p.pass();
        if (g_merged != 3) { std::printf("set %s: %d launches merged afterwards\n", key, g_merged); std::exit(1); }
    }
    // the convolution alone, before any pass: the layer has not run
    Pair fresh("plain");
    fresh.then("the convolution first", [](Model &m) { Pair::launch(m, 5, 6); });
    // pointers, to the layer's output and to what it reads, taken before the first pass or behind one
    for (const char *key : {"norm2.out", "conv1.out", "norm2.scale"})
        for (int passes = 0; passes < 2; ++passes)
            for (int by_name = 0; by_name < 2; ++by_name) {
                Pair p("plain");
                const size_t out = index(p.merged, "norm2.out"), bytes = p.merged.get_storage_size(out), at = index(p.merged, key);
                for (int i = 0; i < passes; ++i) p.pass((gp_stream)64);
                g_scaled_on = nullptr;
                GPUdeviceptr a = nullptr, b = nullptr;
                if (by_name) {
                    if (p.apart.get_global_ptr(key, &a) != Status::Succ || p.merged.get_global_ptr(key, &b) != Status::Succ) std::exit(1);
                } else { a = p.apart.get_storage_ptr(at); b = p.merged.get_storage_ptr(at); }
                if (passes && g_scaled_on != (gp_stream)64) { std::printf("not on the stream of the pass\n"); std::exit(1); }
                for (int i = 0; i < 2; ++i) {
                    p.same_at(a, b, p.merged.get_storage_size(at), "a pointer");
                    p.same("a pointer");
                    put(a, 4, 31 + (uint32_t)i);  // the caller writes through it
                    put(b, 4, 31 + (uint32_t)i);
                    p.same("a value through a pointer");
                    p.each([](Model &m) { Pair::launch(m, 5, 6); });
                    p.same("a value through a pointer, and the convolution");
                    p.pass();
                }
                p.same_at(p.apart.get_storage_ptr(out), p.merged.get_storage_ptr(out), bytes, "the output");
            }
    // the stream of the pass is gone
    Pair p("plain");
    p.pass((gp_stream)64);
    g_gone = {(gp_stream)64};
    p.same_at(p.apart.get_storage_ptr(Pair::at(p.apart, "norm2.out")), p.merged.get_storage_ptr(Pair::at(p.merged, "norm2.out")), 32 * 4, "a stream that is gone");
    if (g_scaled_on != nullptr) { std::printf("on a stream that is gone\n"); std::exit(1); }
    g_gone.clear();
}

// a recorded pass writes everything, since its replays cannot be followed
static void recorded() {
    Pair p("plain");
    p.pass();
    g_capturing = 1;
    g_merged = 0;
    p.pass();
    if (g_merged) { std::printf("%d recorded launches merged\n", g_merged); std::exit(1); }
    g_capturing = 0;
    p.each([](Model &m) { Pair::fill(m, Pair::at(m, "norm2.scale"), 41); });
    p.same("recorded");
}

// A kernel that is stopped and launched again has the form of its first launch, whatever has been asked for in between.
static void stopped() {
    for (int first_merged = 0; first_merged < 2; ++first_merged) {
        Pair p("plain");
        static int counters[10 * 32 * 16], flag, stop;
        GPUdeviceptr pf = &flag, ps = &stop;
        Model &m = p.merged;
        m.batchAddParam(&pf);
        m.batchAddParam(&ps);
        if (m.add_block_preemption_param(counters, 32) != Status::Succ) std::exit(1);
        m.counters_cleared(true);
        g_capturing = !first_merged;
        Pair::launch(m, 0, 6);
        g_capturing = 0;
        g_merged = g_launches = 0;
        if (first_merged) m.get_storage_ptr(Pair::at(m, "norm2.out"));  // (runs the layer)
        else if (m.launch(2, nullptr) != Status::Succ) std::exit(1);    // (resumes a layer that was launched itself)
        const int layers = g_launches;
        Pair::launch(m, 5, 6);
        if (g_merged != first_merged || layers != 1) { std::printf("%d layers, %d of %d merged when launched again\n", layers, g_merged, first_merged); std::exit(1); }
        m.counters_cleared(true);
        g_merged = 0;
        Pair::launch(m, 0, m.get_kernel_num());
        if (g_merged != (first_merged ? 2 : 3)) { std::printf("%d merged in a fresh run\n", g_merged); std::exit(1); }
        // a replayed graph has launched every kernel by itself
        m.launched_once_more();
        g_merged = 0;
        Pair::launch(m, 3, 4);
        if (g_merged) { std::printf("merged behind a replay\n"); std::exit(1); }
    }
}

static void groups() {
    passes_merge("group", 1);
    Pair p("group");
    p.pass();
    // a member alone, behind a pass and from new values, in front of any launch of the group
    for (size_t k = 2; k < 5; ++k)
        for (const char *key : {"stem.out", "left.weight", "middle.weight", "middle.out", "right.bias", "left.out"}) {
            p.then("a new value, a member alone", [&](Model &m) { Pair::fill(m, Pair::at(m, key), 50 + (uint32_t)k); Pair::launch(m, k, k + 1); if (k == 2) Pair::launch(m, 3, 5); });
            p.then("a new value between the members", [&](Model &m) { Pair::launch(m, 2, 3); Pair::fill(m, Pair::at(m, key), 60 + (uint32_t)k); Pair::launch(m, 3, 5); });
        }
    Pair fresh("group");
    fresh.then("a member first", [](Model &m) { Pair::launch(m, 3, 4); });
    g_launches = 0;
    Pair::launch(p.merged, 0, p.merged.get_kernel_num());
    if (g_launches != 5) { std::printf("%d launches of seven kernels, three of them side by side\n", g_launches); std::exit(1); }

    // a preemption injected at a member is launched with that member, and the kernels launched again keep their form
    static int counters[7 * 32 * 16], flag, stop;
    GPUdeviceptr pf = &flag, ps = &stop;
    Model &m = p.merged;
    m.batchAddParam(&pf);
    m.batchAddParam(&ps);
    if (m.add_block_preemption_param(counters, 32) != Status::Succ) std::exit(1);
    auto run = [&](size_t from, int inject) {
        g_merged = g_launches = 0;
        g_at.clear();
        m.keep_apart(inject);
        for (size_t i = from; i < 7; ++i)
            if (m.launch(i, nullptr, (int)i == inject ? 0 : -1) != Status::Succ) std::exit(1);
    };
    for (int inject = 0; inject < 7; ++inject) {
        const int apart = inject == 3 || inject == 4;
        m.counters_cleared(true);
        run(0, inject);
        if (g_at != std::vector<int>{inject} || g_merged != !apart) { std::printf("injected at %d: %zu launches, %d merged\n", inject, g_at.size(), g_merged); std::exit(1); }
        if (inject > 4) continue;
        run(apart ? 2 : (size_t)(inject < 2 ? inject : 2), -1);  // resumed at or in front of the group
        if (g_merged != !apart) { std::printf("injected at %d and resumed: %d merged\n", inject, g_merged); std::exit(1); }
    }
    // recorded in a group, launched apart since, replayed, resumed: in a group
    m.counters_cleared(false);
    run(0, -1);
    m.launches_recorded();
    m.counters_cleared(true);
    run(0, 3);
    m.counters_cleared(false);
    m.launched_once_more();
    run(2, -1);
    if (g_merged != 1) { std::printf("a replay resumed: %d merged\n", g_merged); std::exit(1); }
    // a run given up behind the group's first kernel: the next one's members are launched
    m.counters_cleared(true);
    Pair::launch(m, 2, 3);
    m.counters_cleared(true);
    g_launches = 0;
    Pair::launch(m, 3, 4);
    if (g_launches != 1) { std::printf("a member of a run given up is not launched\n"); std::exit(1); }
}

int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "writers") {
        passes_merge("plain", 3);
        passes_merge("beside", 3);
        passes_merge("rewritten", 2);
        passes_merge("residual", 2);
    } else if (what == "storages") storages();
    else if (what == "groups") groups();
    else if (what == "recorded") recorded();
    else if (what == "stopped") stopped();
    else return 1;
    std::printf("ok %s\n", what.c_str());
}
