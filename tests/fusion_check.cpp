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
static int done(const gp_preempt_ctx *, gp_launch_info *info) {
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
int gp_stage_create(gp_stage *out) { *out = (gp_stage)std::malloc(1); return 0; }
int gp_stage_destroy(gp_stage st) { std::free(st); return 0; }
int gp_stage_upload_async(gp_stage, void *d, const void *h, size_t n, gp_stream) { std::memcpy(d, h, n); return 0; }
int gp_launch_nchw_to_nhwc(const gp_layout_params *p, const gp_preempt_ctx *x, gp_stream, gp_launch_info *i) { put(p->out, p->c_pad, hash(p->in, p->C)); return done(x, i); }
int gp_launch_pool2d(const gp_pool_params *p, const gp_preempt_ctx *x, gp_stream, gp_launch_info *i) { put(p->out, p->C, hash(p->in, p->C)); return done(x, i); }
int gp_launch_softmax(const gp_softmax_params *p, const gp_preempt_ctx *x, gp_stream, gp_launch_info *i) { put(p->out, p->cols, hash(p->x, p->cols)); return done(x, i); }
int gp_launch_eltwise(const gp_eltwise_params *e, const gp_preempt_ctx *x, gp_stream, gp_launch_info *info) {
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

// Three scale-shift layers in front of pointwise convolutions, the way DenseNet has them; "group": two convolutions side by side;
// "rewritten": what the second layer reads is overwritten by a kernel behind its convolution; "beside": by one that writes the
// channels next to those; "residual": the second convolution also adds the second layer's output.
Status foo::zoo_build(Model &m, const std::string &name) {
    GraphBuilder b(m, "f32");
    auto is = [&](const char *s) { return name == s; };
    Tensor t = b.input_nchw(1, 8, 2, 2);
    Tensor block = b.activation("block", 1, 2, 2, 64), first = GraphBuilder::slice(block, 0, 32), next = GraphBuilder::slice(block, 32, 32);
    b.conv("stem", t, 32, 1, 1, 0, GP_ACT_RELU, nullptr, &first);
    Tensor n1 = b.eltwise("norm1", first, nullptr, "norm1", GP_ACT_RELU);
    Tensor c1 = b.conv("conv1", n1, 32, 1, 1, 0, GP_ACT_RELU);
    Tensor n2 = b.eltwise("norm2", c1, nullptr, "norm2", GP_ACT_RELU);
    Tensor c2 = b.conv("conv2", n2, 32, 1, 1, 0, GP_ACT_RELU, is("residual") ? &n2 : nullptr);
    if (is("rewritten")) b.pool("over", c2, 1, 1, 0, 0, &c1);
    if (is("beside")) b.conv("grow", c2, 32, 3, 1, 1, GP_ACT_NONE, nullptr, &next);
    Tensor n3 = b.eltwise("norm3", c2, nullptr, "norm3", GP_ACT_NONE);
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
    void pass() {
        each([](Model &m) {
            for (size_t i = 0; i < m.get_kernel_num(); ++i)
                if (m.launch(i, nullptr) != Status::Succ) { std::printf("kernel %zu\n", i); std::exit(1); }
        });
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

int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "writers") {
        passes_merge("plain", 3);
        passes_merge("beside", 3);
        passes_merge("rewritten", 2);
        passes_merge("residual", 2);
    } else return 1;
    std::printf("ok %s\n", what.c_str());
}
