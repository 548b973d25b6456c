// Two threads' first inputs to one model, over a device layer that takes its time to make the ring: there is one of it.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>

#include "model.h"

static std::atomic<int> g_made{0}, g_gone{0}, g_uploads{0};

// (these take the place of the library's: the executable's symbols come first)
extern "C" {
int gp_malloc(void **p, size_t n) { *p = std::calloc(1, n ? n : 1); return 0; }
int gp_free(void *p) { std::free(p); return 0; }
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
}

int main() {
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
