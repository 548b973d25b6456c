// Device, stream, event, memory, flag, gate and graph entry points of the C ABI.
#include "common.hpp"
#include <atomic>
#include <ctime>
#include <mutex>
#include <unordered_set>
#include <vector>

namespace gp {

static thread_local char g_err[512] = "";
void set_error(const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

int static_scratch_setup(int **out);  // gemm.hip
static std::atomic<int> g_cus{0};
static std::atomic<int> g_device{-1};
int device_cus() {
    int c = g_cus.load(std::memory_order_relaxed);
    if (c > 0) return c;
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess) {
        g_cus.store(prop.multiProcessorCount);
        return prop.multiProcessorCount;
    }
    return 256;
}

__global__ void fill32_kernel(uint32_t *p, uint32_t v, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// One wave polls *stop with system-scope loads; bounded so that a lost release cannot hang the
// device (the reference's gpu_block spins forever, src/block.cu:1-3).
__global__ void gate_kernel(const int *stop, unsigned long long spin_limit, int *timed_out) {
    if (threadIdx.x != 0) return;
    for (unsigned long long i = 0; i < spin_limit; ++i) {
        if (__hip_atomic_load(stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) != 0) return;
        __builtin_amdgcn_s_sleep(8);
    }
    if (timed_out) __hip_atomic_store(timed_out, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void noop_kernel() {}

// Copies between pinned host memory and device memory; the last workgroup to finish stores `seq` where the host spins
// (the one whose arrival is number `last`: nobody clears the counter, the host knows how many there have been).
// Bound by PCIe (50-55 GB/s from 200 KB on) or, below, by the way there and back; against hipMemcpyAsync on pinned
// memory and a stream synchronisation: 16 KB 6 us for 12, 200 KB 10 for 13, 800 KB 23 either way; on ordinary memory
// those take 28, 80 and 44 us.
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
// TO_HOST: the host reads the values when it sees the word, so they are released at system scope first, once per
// workgroup (an XCD's L2 is written back for it, which whoever else runs there notices).  Towards the device the word
// only says that the host's memory has been read, and the kernels that use the values come later on the stream.
template <bool TO_HOST>
__global__ __launch_bounds__(256) void host_copy_kernel(unsigned char *dst, const unsigned char *src, size_t bytes, unsigned *arrived, unsigned last, unsigned *done, unsigned seq) {
    const size_t vecs = bytes / 16, step = (size_t)gridDim.x * blockDim.x, first = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    u32x4 *d = (u32x4 *)dst;
    const u32x4 *s = (const u32x4 *)src;
    size_t i = first;
    for (; i + 3 * step < vecs; i += 4 * step) {  // four trips in flight per lane
        const u32x4 a = s[i], b = s[i + step], c = s[i + 2 * step], e = s[i + 3 * step];
        d[i] = a; d[i + step] = b; d[i + 2 * step] = c; d[i + 3 * step] = e;
    }
    for (; i < vecs; i += step) d[i] = s[i];
    if (first < bytes % 16) dst[vecs * 16 + first] = src[vecs * 16 + first];
    // (the acknowledgement of a store to host memory alone does not say that a store from another XCD, the word's, will
    // not overtake it, hence a release and not just the wait for it; towards the device, a value that is being stored has been read)
    if constexpr (TO_HOST) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x != 0) return;
    constexpr int order = TO_HOST ? __ATOMIC_ACQ_REL : __ATOMIC_RELAXED;
    if constexpr (TO_HOST) __threadfence_system();
    if (gridDim.x > 1 && __hip_atomic_fetch_add(arrived, 1u, order, __HIP_MEMORY_SCOPE_AGENT) != last) return;
    __hip_atomic_store(done, seq, TO_HOST ? __ATOMIC_RELEASE : __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// hands the stop index to a host that spins on the word: one store, so nothing has to be released in front of it, which
// would write an XCD's L2 back under whoever has the GPU by now
__global__ void report_stop_kernel(const int *stop_index, unsigned long long *host_word, unsigned seq) {
    if (threadIdx.x != 0) return;
    const int stop = stop_index ? __hip_atomic_load(stop_index, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : -1;
    __hip_atomic_store(host_word, (unsigned long long)(unsigned)stop << 32 | seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// stores the device's constant-rate clock where the host can see it
__global__ void clock_probe_kernel(unsigned long long *host_word) {
    if (threadIdx.x == 0) __hip_atomic_store(host_word, (unsigned long long)wall_clock64(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// stores a value where the host can see it: a marker that says "everything before me on this stream has left the GPU"
__global__ void store_word_kernel(int *host_word, int value) {
    if (threadIdx.x == 0) __hip_atomic_store(host_word, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

struct RelayArgs { const int *flags[8]; int *mirror; int n; const int *quit; unsigned long long spin_limit; };

// Lane i mirrors flag word i into device memory; lane 0 also watches the quit word.
__global__ void flag_relay_kernel(RelayArgs a) {
    const int lane = threadIdx.x;
    int last = 0;
    for (unsigned long long it = 0; it < a.spin_limit; ++it) {
        if (lane < a.n) {
            int v = __hip_atomic_load(a.flags[lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            if (v != last) {
                __hip_atomic_store(a.mirror + lane, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                last = v;
            }
        }
        int q = 0;
        if (lane == 0) q = __hip_atomic_load(a.quit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (__builtin_amdgcn_readfirstlane(q) != 0) break;
        __builtin_amdgcn_s_sleep(4);
    }
    // leave the mirror lowered so that nothing stays stopped because the relay is gone
    if (lane < a.n && last != 0) __hip_atomic_store(a.mirror + lane, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace gp

using namespace gp;

// what gp_stream_create has made and gp_stream_destroy has not taken back
struct LiveStreams { std::mutex mu; std::unordered_set<gp_stream> all; };
static LiveStreams &live_streams() {
    static LiveStreams *l = new LiveStreams;  // (never destroyed: streams may be, behind the library's statics)
    return *l;
}

extern "C" const char *gp_last_error(void) { return g_err; }

extern "C" int gp_init(int device) {
    int n = 0;
    GP_HIP(hipGetDeviceCount(&n));
    GP_REQUIRE(device >= 0 && device < n, "device %d not present (%d visible)", device, n);
    GP_HIP(hipSetDevice(device));
    // address of the library's static scratch on this device (gp_launch_gemm_noalloc)
    if (int rc = static_scratch_setup(nullptr)) return rc;
    if (g_device.load() != device) {
        hipDeviceProp_t prop;
        GP_HIP(hipGetDeviceProperties(&prop, device));
        g_cus.store(prop.multiProcessorCount);
        g_device.store(device);
    }
    return GP_SUCC;
}

extern "C" int gp_device_info(int *compute_units, int *clock_khz, char *name, size_t name_len) {
    int dev = 0;
    GP_HIP(hipGetDevice(&dev));
    hipDeviceProp_t prop;
    GP_HIP(hipGetDeviceProperties(&prop, dev));
    if (compute_units) *compute_units = prop.multiProcessorCount;
    if (clock_khz) *clock_khz = prop.clockRate;
    if (name && name_len) { strncpy(name, prop.name, name_len - 1); name[name_len - 1] = 0; }
    return GP_SUCC;
}

extern "C" int gp_stream_create(int priority, gp_stream *out) {
    GP_REQUIRE(out != nullptr, "null stream out");
    hipStream_t s;
    GP_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    *out = new gp_stream_s{s, priority};
    LiveStreams &live = live_streams();
    std::lock_guard<std::mutex> g(live.mu);
    live.all.insert(*out);
    return GP_SUCC;
}
extern "C" int gp_stream_exists(gp_stream s) {
    LiveStreams &live = live_streams();
    std::lock_guard<std::mutex> g(live.mu);
    return !s || live.all.count(s) ? 1 : 0;
}
extern "C" int gp_stream_destroy(gp_stream s) {
    if (!s) return GP_SUCC;
    {
        LiveStreams &live = live_streams();
        std::lock_guard<std::mutex> g(live.mu);
        live.all.erase(s);
    }
    hipError_t e = hipStreamDestroy(s->s);
    delete s;
    if (e != hipSuccess) { set_error("hipStreamDestroy: %s", hipGetErrorString(e)); return GP_FAIL; }
    return GP_SUCC;
}
extern "C" int gp_stream_sync(gp_stream s) { GP_HIP(hipStreamSynchronize(native(s))); return GP_SUCC; }
extern "C" int gp_stream_query(gp_stream s, int *idle) {
    hipError_t e = hipStreamQuery(native(s));
    if (e == hipSuccess) { if (idle) *idle = 1; return GP_SUCC; }
    if (e == hipErrorNotReady) { if (idle) *idle = 0; return GP_SUCC; }
    set_error("hipStreamQuery: %s", hipGetErrorString(e));
    return GP_FAIL;
}
extern "C" int gp_stream_capturing(gp_stream s, int *capturing) {
    GP_REQUIRE(capturing != nullptr, "null out pointer");
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    GP_HIP(hipStreamIsCapturing(native(s), &st));
    *capturing = st != hipStreamCaptureStatusNone;
    return GP_SUCC;
}
extern "C" int gp_stream_priority(gp_stream s, int *priority) {
    GP_REQUIRE(s && priority, "null stream");
    *priority = s->priority;
    return GP_SUCC;
}
extern "C" int gp_stream_set_priority(gp_stream s, int priority) {
    GP_REQUIRE(s != nullptr, "null stream");
    GP_REQUIRE(priority >= 0, "priority %d", priority);
    s->priority = priority;
    return GP_SUCC;
}
extern "C" void *gp_stream_native(gp_stream s) { return (void *)native(s); }

extern "C" int gp_event_create(gp_event *out) {
    GP_REQUIRE(out != nullptr, "null event out");
    hipEvent_t e;
    GP_HIP(hipEventCreate(&e));
    *out = new gp_event_s{e};
    return GP_SUCC;
}
extern "C" int gp_event_destroy(gp_event e) {
    if (!e) return GP_SUCC;
    hipError_t r = hipEventDestroy(e->e);
    delete e;
    if (r != hipSuccess) { set_error("hipEventDestroy: %s", hipGetErrorString(r)); return GP_FAIL; }
    return GP_SUCC;
}
extern "C" int gp_event_record(gp_event e, gp_stream s) { GP_REQUIRE(e, "null event"); GP_HIP(hipEventRecord(e->e, native(s))); return GP_SUCC; }
extern "C" int gp_event_sync(gp_event e) { GP_REQUIRE(e, "null event"); GP_HIP(hipEventSynchronize(e->e)); return GP_SUCC; }
extern "C" int gp_event_query(gp_event e, int *done) {
    GP_REQUIRE(e && done, "null event");
    hipError_t r = hipEventQuery(e->e);
    if (r == hipSuccess) { *done = 1; return GP_SUCC; }
    if (r == hipErrorNotReady) { *done = 0; return GP_SUCC; }
    set_error("hipEventQuery: %s", hipGetErrorString(r));
    return GP_FAIL;
}
extern "C" int gp_event_elapsed_ms(gp_event a, gp_event b, float *ms) {
    GP_REQUIRE(a && b && ms, "null event");
    GP_HIP(hipEventElapsedTime(ms, a->e, b->e));
    return GP_SUCC;
}

extern "C" int gp_malloc(void **dev, size_t bytes) {
    GP_REQUIRE(dev != nullptr, "null out pointer");
    GP_HIP(hipMalloc(dev, bytes ? bytes : 1));
    return GP_SUCC;
}
extern "C" int gp_malloc_capturing(void **dev, size_t bytes) {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    GP_HIP(hipThreadExchangeStreamCaptureMode(&mode));
    const int rc = gp_malloc(dev, bytes);
    GP_HIP(hipThreadExchangeStreamCaptureMode(&mode));
    return rc;
}
extern "C" int gp_free(void *dev) { if (dev) GP_HIP(hipFree(dev)); return GP_SUCC; }
extern "C" int gp_host_alloc(void **host, size_t bytes) {
    GP_REQUIRE(host != nullptr, "null out pointer");
    GP_HIP(hipHostMalloc(host, bytes ? bytes : 1, hipHostMallocDefault));
    return GP_SUCC;
}
extern "C" int gp_host_free(void *host) { if (host) GP_HIP(hipHostFree(host)); return GP_SUCC; }
extern "C" int gp_host_alloc_coherent(void **host, void **dev, size_t bytes) {
    GP_REQUIRE(host && dev && bytes, "null out pointer");
    GP_HIP(hipHostMalloc(host, bytes, hipHostMallocCoherent | hipHostMallocMapped));
    memset(*host, 0, bytes);
    GP_HIP(hipHostGetDevicePointer(dev, *host, 0));
    return GP_SUCC;
}
extern "C" int gp_memcpy_h2d(void *dev, const void *host, size_t bytes) { GP_HIP(hipMemcpy(dev, host, bytes, hipMemcpyHostToDevice)); return GP_SUCC; }
extern "C" int gp_memcpy_d2h(void *host, const void *dev, size_t bytes) { GP_HIP(hipMemcpy(host, dev, bytes, hipMemcpyDeviceToHost)); return GP_SUCC; }
extern "C" int gp_memcpy_h2d_async(void *dev, const void *host, size_t bytes, gp_stream s) { GP_HIP(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, native(s))); return GP_SUCC; }
extern "C" int gp_memcpy_d2h_async(void *host, const void *dev, size_t bytes, gp_stream s) { GP_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, native(s))); return GP_SUCC; }
extern "C" int gp_memcpy_d2d_async(void *dst, const void *src, size_t bytes, gp_stream s) { GP_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, native(s))); return GP_SUCC; }
extern "C" int gp_fill32_async(void *dev, uint32_t value, size_t count, gp_stream s) {
    if (count == 0) return GP_SUCC;
    GP_REQUIRE(dev && ((uintptr_t)dev & 3) == 0, "fill32 needs a 4-byte aligned device pointer");
    unsigned grid = (unsigned)((count + 255) / 256);
    hipLaunchKernelGGL(fill32_kernel, dim3(grid), dim3(256), 0, native(s), (uint32_t *)dev, value, count);
    GP_HIP(hipGetLastError());
    return GP_SUCC;
}

namespace {
// what a host_copy_kernel reports through: a word in host memory and a counter on the device
struct CopyDone {
    unsigned *word = nullptr, *word_dev = nullptr, *arrived = nullptr;
    unsigned seq = 0, arrivals = 0;
    int create() {
        int rc = gp_host_alloc_coherent((void **)&word, (void **)&word_dev, 64);
        if (rc) return rc;
        GP_HIP(hipMalloc((void **)&arrived, 4));
        return gp_fill32_async(arrived, 0, 1, nullptr) || gp_stream_sync(nullptr) ? GP_FAIL : GP_SUCC;
    }
    void destroy() {
        if (word) hipHostFree(word);
        if (arrived) hipFree(arrived);
    }
    bool reached(unsigned s) const { return (int)(__atomic_load_n(word, __ATOMIC_ACQUIRE) - s) >= 0; }
    // `asked` is the copy's own stream, or null where that may be gone by now.  An error of the device ends the wait; besides,
    // while the host has nothing else to do the runtime takes note of the launches that have ended (left to the next device-wide
    // synchronisation, that makes it 35 us behind a BERT request instead of 6).
    int wait(unsigned s, hipStream_t asked = nullptr) const {
        for (unsigned spins = 1; !reached(s); ++spins) {
            if (spins % (1u << 16)) continue;
            const hipError_t e = hipStreamQuery(asked);
            if (e != hipSuccess && e != hipErrorNotReady) { set_error("host copy: %s", hipGetErrorString(e)); return GP_FAIL; }
        }
        return GP_SUCC;
    }
    template <bool TO_HOST>
    int launch(void *dst, const void *src, size_t bytes, hipStream_t stream) {
        const unsigned grid = (unsigned)(bytes <= (16u << 10) ? 1 : bytes >= (1u << 20) ? 64 : bytes / (16u << 10));
        hipLaunchKernelGGL(host_copy_kernel<TO_HOST>, dim3(grid), dim3(256), 0, stream, (unsigned char *)dst, (const unsigned char *)src, bytes, arrived,
                           arrivals + grid - 1, word_dev, seq + 1);
        GP_HIP(hipGetLastError());
        ++seq;
        if (grid > 1) arrivals += grid;
        return GP_SUCC;
    }
};
std::mutex g_copies_mu;
std::vector<CopyDone> g_copies;  // free ones: as many as there have been fetches at one time
}  // namespace

extern "C" int gp_fetch(void *host, const void *dev, size_t bytes, gp_stream s) {
    GP_REQUIRE(host && dev, "gp_fetch: null pointer");
    if (bytes >= (8u << 20) || ((uintptr_t)dev & 15) || ((uintptr_t)host & 15)) {  // the copy engine is as fast, and leaves the compute units alone
        GP_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, native(s)));
        GP_HIP(hipStreamSynchronize(native(s)));
        return GP_SUCC;
    }
    CopyDone c;
    {
        std::lock_guard<std::mutex> lock(g_copies_mu);
        if (!g_copies.empty()) { c = g_copies.back(); g_copies.pop_back(); }
    }
    int rc = c.word ? GP_SUCC : c.create();
    if (rc == GP_SUCC) rc = c.launch<true>(host, dev, bytes, native(s));
    if (rc == GP_SUCC) rc = c.wait(c.seq, native(s));
    if (rc) return rc;  // (a copy that may still be under way keeps its words)
    std::lock_guard<std::mutex> lock(g_copies_mu);
    g_copies.push_back(c);
    return GP_SUCC;
}

// A ring whose pieces report for themselves: a piece is free again when its own copy has read it, whatever stream that was
// on and whatever the others do.  It starts with eight pieces and grows while its streams are held up (behind a gate, a
// suspended tenant), up to kMost bytes; from there on an upload waits for the piece that has been in use longest.
struct gp_stage_s {
    static constexpr size_t kPiece = 1u << 20, kMost = 64u << 20;
    static constexpr int kPerBlock = 8;
    struct Piece { unsigned char *host, *dev; size_t room; CopyDone done; unsigned long long turn; };
    struct Block { void *host; void *arrived; };
    std::mutex mu;
    std::vector<Piece> pieces;
    std::vector<Block> blocks;
    size_t total = 0;
    unsigned long long turns = 0;

    // eight pieces of `room` bytes, with the words they report through (the counters are cleared here and now: the stream that
    // asks may be held up while another one takes the next piece)
    int grow(size_t room) {
        Block b{};
        unsigned char *dev = nullptr;
        const size_t words = kPerBlock * 64;
        if (int rc = gp_host_alloc_coherent(&b.host, (void **)&dev, room * kPerBlock + words)) return rc;
        int rc = gp_malloc(&b.arrived, kPerBlock * 64);
        if (rc == GP_SUCC) rc = gp_fill32_async(b.arrived, 0, kPerBlock * 16, nullptr) || gp_stream_sync(nullptr) ? GP_FAIL : GP_SUCC;
        if (rc != GP_SUCC) { hipHostFree(b.host); if (b.arrived) hipFree(b.arrived); return rc; }
        for (int k = 0; k < kPerBlock; ++k) {
            Piece p{(unsigned char *)b.host + words + k * room, dev + words + k * room, room, {}, 0};
            p.done.word = (unsigned *)((unsigned char *)b.host + 64 * k);
            p.done.word_dev = (unsigned *)(dev + 64 * k);
            p.done.arrived = (unsigned *)b.arrived + 16 * k;
            pieces.push_back(p);
        }
        blocks.push_back(b);
        total += room * kPerBlock;
        return GP_SUCC;
    }
    // a piece for `want` bytes or, when there is nothing else to do, for fewer
    int piece_for(size_t want, Piece **out) {
        Piece *longest = nullptr;
        for (Piece &p : pieces) {
            if (p.room >= want && p.done.reached(p.done.seq)) { *out = &p; return GP_SUCC; }
            if (!longest || p.turn < longest->turn) longest = &p;
        }
        if (total + want * kPerBlock <= kMost || !longest) {
            if (int rc = grow(want)) return rc;
            *out = &pieces[pieces.size() - kPerBlock];
            return GP_SUCC;
        }
        *out = longest;
        return longest->done.wait(longest->done.seq);
    }
};
extern "C" int gp_stage_create(gp_stage *out) {
    GP_REQUIRE(out != nullptr, "null stage out");
    *out = new gp_stage_s();
    return GP_SUCC;
}
extern "C" int gp_stage_destroy(gp_stage st) {
    if (!st) return GP_SUCC;
    int rc = GP_SUCC;
    for (auto &p : st->pieces)
        if (rc == GP_SUCC) rc = p.done.wait(p.done.seq);
    if (rc == GP_SUCC)
        for (auto &b : st->blocks) { hipHostFree(b.host); hipFree(b.arrived); }
    delete st;
    return rc;
}
extern "C" int gp_stage_upload_async(gp_stage st, void *dev, const void *host, size_t bytes, gp_stream s) {
    GP_REQUIRE(st && dev && host, "gp_stage_upload_async: null pointer");
    std::lock_guard<std::mutex> lock(st->mu);
    // four pieces of a large input are copied to the ring while the one before is on its way; a small one is one piece
    size_t want = bytes <= (256u << 10) ? bytes : (bytes + 3) / 4;
    want = want > gp_stage_s::kPiece ? gp_stage_s::kPiece : (want + 4095) / 4096 * 4096;
    for (size_t at = 0; at < bytes;) {
        gp_stage_s::Piece *p = nullptr;
        if (int rc = st->piece_for(want, &p)) return rc;
        size_t n = bytes - at < want ? bytes - at : want;
        if (n > p->room) n = p->room;
        memcpy(p->host, (const char *)host + at, n);
        if (int rc = p->done.launch<false>((char *)dev + at, p->dev, n, native(s))) return rc;
        p->turn = ++st->turns;
        at += n;
    }
    return GP_SUCC;
}

extern "C" int gp_flag_create(volatile int **host_ptr, void **dev_ptr) {
    GP_REQUIRE(host_ptr && dev_ptr, "null out pointer");
    void *h = nullptr;
    // Coherent (fine-grained) pinned memory: a host store becomes visible to a running kernel.
    GP_HIP(hipHostMalloc(&h, 64, hipHostMallocCoherent | hipHostMallocMapped));
    memset(h, 0, 64);
    void *d = nullptr;
    GP_HIP(hipHostGetDevicePointer(&d, h, 0));
    *host_ptr = (volatile int *)h;
    *dev_ptr = d;
    return GP_SUCC;
}
extern "C" int gp_flag_destroy(volatile int *host_ptr) { if (host_ptr) GP_HIP(hipHostFree((void *)host_ptr)); return GP_SUCC; }

extern "C" int gp_flag_relay_start(void *const *flags_dev, int *mirror, int n, const int *quit_dev,
                                   unsigned long long spin_limit, gp_stream s) {
    GP_REQUIRE(flags_dev && mirror && quit_dev && s, "relay needs flags, mirror, quit flag and an explicit stream");
    GP_REQUIRE(n >= 1 && n <= 8, "relay handles 1..8 flag words");
    GP_REQUIRE(spin_limit > 0, "relay needs a finite spin limit");
    RelayArgs a{};
    for (int i = 0; i < n; ++i) { GP_REQUIRE(flags_dev[i] != nullptr, "null flag"); a.flags[i] = (const int *)flags_dev[i]; }
    a.mirror = mirror; a.n = n; a.quit = quit_dev; a.spin_limit = spin_limit;
    hipLaunchKernelGGL(flag_relay_kernel, dim3(1), dim3(64), 0, native(s), a);
    GP_HIP(hipGetLastError());
    return GP_SUCC;
}

extern "C" int gp_launch_gate(const int *stop, unsigned long long spin_limit, int *timed_out, gp_stream s) {
    GP_REQUIRE(stop != nullptr, "null gate flag");
    GP_REQUIRE(spin_limit > 0, "gate needs a finite spin limit");
    hipLaunchKernelGGL(gate_kernel, dim3(1), dim3(64), 0, native(s), stop, spin_limit, timed_out);
    GP_HIP(hipGetLastError());
    return GP_SUCC;
}
extern "C" int gp_launch_noop(gp_stream s) {
    hipLaunchKernelGGL(noop_kernel, dim3(1), dim3(64), 0, native(s));
    GP_HIP(hipGetLastError());
    return GP_SUCC;
}

// Device clock against the host's: a kernel stores wall_clock64() into fine-grained host memory and the
// host, spinning on the word, notes its own clock when the value appears.  host - device is the offset plus
// the store's way to the host; the minimum over the rounds keeps the shortest way (1-2 us).
extern "C" int gp_device_clock(gp_stream s, int rounds, double *tick_ns, double *offset_ns, unsigned long long *ticks) {
    GP_REQUIRE(tick_ns && offset_ns, "null clock out");
    if (rounds < 1) rounds = 16;
    int dev = 0, khz = 0;
    GP_HIP(hipGetDevice(&dev));
    GP_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
    GP_REQUIRE(khz > 0, "the device reports no wall clock rate");
    const double tick = 1e6 / (double)khz;
    volatile unsigned long long *word = nullptr;
    GP_HIP(hipHostMalloc((void **)&word, 64, hipHostMallocCoherent | hipHostMallocMapped));
    void *word_dev = nullptr;
    if (hipHostGetDevicePointer(&word_dev, (void *)word, 0) != hipSuccess) { hipHostFree((void *)word); set_error("gp_device_clock: no device address for the probe word"); return GP_FAIL; }
    double best = 0;
    unsigned long long best_ticks = 0;
    bool have = false;
    for (int r = 0; r < rounds; ++r) {
        *word = 0;
        hipLaunchKernelGGL(clock_probe_kernel, dim3(1), dim3(64), 0, native(s), (unsigned long long *)word_dev);
        hipError_t e = hipGetLastError();
        unsigned long long d = 0;
        // bounded: a kernel that never ran must not hang the caller (about two seconds of polls)
        for (long spins = 0; e == hipSuccess && (d = *word) == 0 && spins < (1L << 31); ++spins) { }
        struct timespec ts;
        clock_gettime(CLOCK_MONOTONIC, &ts);
        const double host_ns = (double)ts.tv_sec * 1e9 + (double)ts.tv_nsec;
        hipError_t e2 = hipStreamSynchronize(native(s));
        if (e != hipSuccess || e2 != hipSuccess || d == 0) {
            hipHostFree((void *)word);
            set_error("gp_device_clock: the probe kernel did not report (%s)", hipGetErrorString(e != hipSuccess ? e : e2));
            return GP_FAIL;
        }
        const double off = host_ns - (double)d * tick;
        if (!have || off < best) { best = off; best_ticks = d; have = true; }
    }
    GP_HIP(hipHostFree((void *)word));
    *tick_ns = tick;
    *offset_ns = best;
    if (ticks) *ticks = best_ticks;
    return GP_SUCC;
}

extern "C" int gp_store_word_async(gp_stream s, int *word_dev, int value) {
    GP_REQUIRE(word_dev != nullptr, "gp_store_word_async: null word");
    hipLaunchKernelGGL(store_word_kernel, dim3(1), dim3(64), 0, native(s), word_dev, value);
    GP_HIP(hipGetLastError());
    return GP_SUCC;
}

extern "C" int gp_report_stop_async(const int *stop_index, unsigned long long *word_dev, unsigned seq, gp_stream s) {
    GP_REQUIRE(word_dev != nullptr && ((uintptr_t)word_dev & 7) == 0, "gp_report_stop_async: an aligned 64-bit word");
    hipLaunchKernelGGL(report_stop_kernel, dim3(1), dim3(64), 0, native(s), stop_index, word_dev, seq);
    GP_HIP(hipGetLastError());
    return GP_SUCC;
}

extern "C" int gp_graph_begin(gp_stream s) {
    GP_REQUIRE(s != nullptr, "graph capture needs an explicit stream");
    GP_HIP(hipStreamBeginCapture(s->s, hipStreamCaptureModeThreadLocal));
    return GP_SUCC;
}
extern "C" int gp_graph_end(gp_stream s, gp_graph *out) {
    GP_REQUIRE(s && out, "null graph out");
    hipGraph_t g;
    GP_HIP(hipStreamEndCapture(s->s, &g));
    hipGraphExec_t x;
    hipError_t e = hipGraphInstantiate(&x, g, nullptr, nullptr, 0);
    if (e != hipSuccess) { hipGraphDestroy(g); set_error("hipGraphInstantiate: %s", hipGetErrorString(e)); return GP_FAIL; }
    *out = new gp_graph_s{g, x};
    return GP_SUCC;
}
extern "C" int gp_graph_launch(gp_graph g, gp_stream s) { GP_REQUIRE(g, "null graph"); GP_HIP(hipGraphLaunch(g->x, native(s))); return GP_SUCC; }
extern "C" int gp_graph_destroy(gp_graph g) {
    if (!g) return GP_SUCC;
    hipGraphExecDestroy(g->x);
    hipGraphDestroy(g->g);
    delete g;
    return GP_SUCC;
}
