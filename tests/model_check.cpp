// foo::Model over a device layer in host memory that counts: two threads' first inputs make one ring, and what a sweep
// needs is allocated by the first sweep.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>

#include "model.h"

static std::atomic<int> g_made{0}, g_gone{0}, g_uploads{0};
static long g_allocated = 0, g_blocks = 0;

// (these take the place of the library's: the executable's symbols come first)
extern "C" {
int gp_malloc(void **p, size_t n) { *p = std::calloc(1, n ? n : 1); g_allocated += (long)n; ++g_blocks; return 0; }
int gp_malloc_capturing(void **p, size_t n) { return gp_malloc(p, n); }
int gp_free(void *p) { if (p) --g_blocks; std::free(p); return 0; }
int gp_memcpy_h2d(void *d, const void *h, size_t n) { std::memcpy(d, h, n); return 0; }
int gp_fill32_async(void *, uint32_t, size_t, gp_stream) { return 0; }
int gp_stream_sync(gp_stream) { return 0; }
int gp_stage_create(gp_stage *out) {
    std::this_thread::sleep_for(std::chrono::milliseconds(50));
    ++g_made;
    *out = (gp_stage)std::malloc(1);
    return 0;
}
int gp_stage_destroy(gp_stage st) { ++g_gone; std::free(st); return 0; }
int gp_stage_upload_async(gp_stage st, void *d, const void *h, size_t n, gp_stream) {
    if (!st) return 1;
    std::memcpy(d, h, n);
    ++g_uploads;
    return 0;
}
int gp_launch_miniweather(const gp_miniweather_params *p, const gp_preempt_ctx *, gp_stream, gp_launch_info *) { return p->state ? 0 : 1; }
int gp_launch_miniweather_sweep(const gp_mw_sweep_params *p, const gp_preempt_ctx *, gp_stream, gp_launch_info *) {
    return p->in && p->out && p->in != p->out && (p->in == p->state || p->out == p->state) ? 0 : 1;
}
}

static int sweeps() {
    foo::Model m;
    if (m.load_model("./miniweather@nx=40,nz=20/mod.json", "./miniweather@nx=40,nz=20/host.json", "") != Status::Succ) { std::printf("no model\n"); return 1; }
    long storages = 0;
    for (size_t i = 0; i < m.get_storage_num(); ++i) storages += (long)m.get_storage_size(i);
    for (size_t i = 0; i < m.get_kernel_num(); ++i)
        if (m.launch(i, nullptr) != Status::Succ) { std::printf("kernel %zu\n", i); return 1; }
    if (g_allocated != storages) { std::printf("%ld bytes allocated for %ld of storages\n", g_allocated, storages); return 1; }
    const long blocks = g_blocks;
    for (int run = 0; run < 2; ++run)
        for (size_t g = 0; g < 4; ++g)
            if (m.launch_sweep(g, nullptr) != Status::Succ) { std::printf("sweep %zu\n", g); return 1; }
    if (g_blocks != blocks + 1) { std::printf("%ld blocks more for the sweeps\n", g_blocks - blocks); return 1; }
    m.clear();
    if (g_blocks != 0) { std::printf("%ld blocks left\n", g_blocks); return 1; }
    std::printf("ok sweeps\n");
    return 0;
}

int main(int argc, char **) {
    if (argc > 1) return sweeps();
    foo::Model m;
    if (m.load_model("./toy@rows=8,cols=8,n=1,dtype=f32/mod.json", "./toy@rows=8,cols=8,n=1,dtype=f32/host.json", "") != Status::Succ) { std::printf("no model\n"); return 1; }
    float x[64] = {1.f};
    std::thread a([&] { m.set("data", x, sizeof(x), nullptr); }), b([&] { m.set("data", x, sizeof(x), nullptr); });
    a.join();
    b.join();
    m.clear();
    if (g_uploads != 2 || g_made != 1 || g_gone != 1) { std::printf("%d uploads, %d rings made, %d destroyed\n", g_uploads.load(), g_made.load(), g_gone.load()); return 1; }
    std::printf("ok first input\n");
}
