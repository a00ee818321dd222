// hip_standin.cpp - the HIP calls and kernel launchers that the host runtime uses, on the CPU, for tests
// of its ordering and error paths. Work on a stream is only queued; it runs when somebody waits for it
// or asks for an event, as late as the program allows. Path launches stop at a gate while it is
// closed. Nothing here traces rays: a path launch steps each stream's engine and counts.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <condition_variable>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <set>
#include <vector>

#include "cortex_rt.h"
#include "crt_kernels.h"
#include "crt_layout.h"
#include "crt_scratch.h"

#define API extern "C" __attribute__((visibility("default")))

namespace {

struct Stream;
struct Event { Stream* s = nullptr; uint64_t recorded = 0, done = 0; };
struct Op { std::function<void()> run; Event* wait = nullptr; Event* record = nullptr; uint64_t gen = 0; bool gated = false; };
struct Stream { std::deque<Op> q; bool busy = false; };
struct Launch { uint64_t mode, requests, paths, most_samples; };

std::mutex g_m;
std::condition_variable g_cv;
std::vector<Stream*> g_streams;   // neither streams nor events are freed: queued work may name them
std::map<void*, size_t> g_mem;
size_t g_allocated = 0, g_limit = 0;
bool g_gate_closed = false;
int g_fail_launch = -1;
uint64_t g_launches = 0, g_elapsed_calls = 0;
std::vector<Launch> g_ran;
std::set<hipStream_t> g_used;   // streams and paths of the launches since a time was asked for
uint64_t g_path_count = 0;
size_t g_overlap = 1;

void progress(Stream* s) {
    if (!s || s->busy) return;
    s->busy = true;
    while (!s->q.empty()) {
        Op& op = s->q.front();
        if (op.wait && op.wait->done < op.gen) {
            progress(op.wait->s);
            if (op.wait->done < op.gen) break;
        }
        if (op.gated && g_gate_closed) break;
        if (op.run) op.run();
        if (op.record) op.record->done = op.gen;
        s->q.pop_front();
    }
    s->busy = false;
}
void wait_for(std::unique_lock<std::mutex>& lk, const std::function<bool()>& done) {
    while (!done()) g_cv.wait(lk);
}
Stream* S(hipStream_t s) { return (Stream*)s; }
Event* E(hipEvent_t e) { return (Event*)e; }
void enqueue(hipStream_t s, std::function<void()> f, bool gated = false) {
    Op op;
    op.run = std::move(f);
    op.gated = gated;
    S(s)->q.push_back(std::move(op));
}
bool launch_fails() { return g_fail_launch >= 0 && g_fail_launch-- == 0; }

}  // namespace

// ------------------------------------------------------------------ what a test sets and reads
API void standin_gate(int closed) { std::lock_guard<std::mutex> g(g_m); g_gate_closed = closed != 0; g_cv.notify_all(); }
API void standin_fail_launch(int n) { std::lock_guard<std::mutex> g(g_m); g_fail_launch = n; }
API void standin_memory_limit(uint64_t bytes) { std::lock_guard<std::mutex> g(g_m); g_limit = bytes; }
API void standin_overlap(int streams) { std::lock_guard<std::mutex> g(g_m); g_overlap = (size_t)streams; }
API uint64_t standin_allocated() { std::lock_guard<std::mutex> g(g_m); return g_allocated; }
API uint64_t standin_launches() { std::lock_guard<std::mutex> g(g_m); return g_launches; }
API uint64_t standin_pending() {
    std::lock_guard<std::mutex> g(g_m);
    uint64_t n = 0;
    for (Stream* s : g_streams) n += s->q.size();
    return n;
}
// mode, requests, paths and most samples a pixel of the k-th path launch that ran; returns their count
API uint64_t standin_ran(uint64_t k, uint64_t out[4]) {
    std::lock_guard<std::mutex> g(g_m);
    if (k < g_ran.size()) { out[0] = g_ran[k].mode; out[1] = g_ran[k].requests; out[2] = g_ran[k].paths; out[3] = g_ran[k].most_samples; }
    return g_ran.size();
}
API void standin_reset() {
    std::lock_guard<std::mutex> g(g_m);
    g_gate_closed = false; g_fail_launch = -1; g_limit = 0; g_launches = 0; g_overlap = 1; g_ran.clear();
    g_cv.notify_all();
}

// ------------------------------------------------------------------ HIP
API hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
API hipError_t hipSetDevice(int) { return hipSuccess; }
API hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) { memset(p, 0, sizeof(*p)); p->multiProcessorCount = 4; return hipSuccess; }
API hipError_t hipMemGetInfo(size_t* f, size_t* t) { *f = *t = (size_t)64 << 30; return hipSuccess; }
API hipError_t hipGetLastError() { return hipSuccess; }
API const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
API hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
    memset(a, 0, sizeof(*a));
    a->type = hipMemoryTypeDevice;
    return hipSuccess;
}
#undef hipMalloc
API hipError_t hipMalloc(void** p, size_t n) {
    std::lock_guard<std::mutex> g(g_m);
    *p = nullptr;
    if (g_limit && g_allocated + n > g_limit) return hipErrorOutOfMemory;
    if (!(*p = calloc(1, n))) return hipErrorOutOfMemory;
    g_mem[*p] = n;
    g_allocated += n;
    return hipSuccess;
}
API hipError_t hipFree(void* p) {
    std::unique_lock<std::mutex> lk(g_m);
    if (!p) return hipSuccess;
    wait_for(lk, []() {
        bool idle = true;
        for (Stream* s : g_streams) { progress(s); idle = idle && s->q.empty(); }
        return idle;
    });
    auto it = g_mem.find(p);
    if (it == g_mem.end()) return hipErrorInvalidValue;
    g_allocated -= it->second;
    g_mem.erase(it);
    free(p);
    return hipSuccess;
}
#undef hipHostMalloc
API hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return (*p = calloc(1, n)) ? hipSuccess : hipErrorOutOfMemory; }
API hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
API hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    std::lock_guard<std::mutex> g(g_m);
    g_streams.push_back(new Stream);
    *s = (hipStream_t)g_streams.back();
    return hipSuccess;
}
API hipError_t hipStreamSynchronize(hipStream_t s) {
    std::unique_lock<std::mutex> lk(g_m);
    wait_for(lk, [s]() { progress(S(s)); return S(s)->q.empty(); });
    return hipSuccess;
}
API hipError_t hipStreamDestroy(hipStream_t s) { return hipStreamSynchronize(s); }
API hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t) new Event; return hipSuccess; }
API hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
API hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
API hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    std::lock_guard<std::mutex> g(g_m);
    Op op;
    op.record = E(e);
    op.gen = ++E(e)->recorded;
    E(e)->s = S(s);
    S(s)->q.push_back(std::move(op));
    return hipSuccess;
}
API hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    std::lock_guard<std::mutex> g(g_m);
    Op op;
    op.wait = E(e);
    op.gen = E(e)->recorded;
    S(s)->q.push_back(std::move(op));
    return hipSuccess;
}
API hipError_t hipEventQuery(hipEvent_t e) {
    std::lock_guard<std::mutex> g(g_m);
    progress(E(e)->s);
    return E(e)->done >= E(e)->recorded ? hipSuccess : hipErrorNotReady;
}
API hipError_t hipEventSynchronize(hipEvent_t e) {
    std::unique_lock<std::mutex> lk(g_m);
    const uint64_t gen = E(e)->recorded;
    wait_for(lk, [e, gen]() { progress(E(e)->s); return E(e)->done >= gen; });
    return hipSuccess;
}
// The time of the path launches since the last question: they overlap on up to g_overlap streams, and
// every measurement is off by up to a hundredth, the later ones the other way than the earlier ones.
API hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    std::lock_guard<std::mutex> g(g_m);
    const size_t n = g_used.size() < g_overlap ? g_used.size() : g_overlap;
    *ms = (float)g_path_count / (float)(n ? n : 1) * (1.0f + 0.0025f * (float)((7u * ++g_elapsed_calls) % 9u) - 0.01f);
    g_used.clear();
    g_path_count = 0;
    return hipSuccess;
}
API hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
    std::lock_guard<std::mutex> g(g_m);
    enqueue(st, [=]() { memcpy(d, s, n); });
    return hipSuccess;
}
API hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t st) {
    std::lock_guard<std::mutex> g(g_m);
    enqueue(st, [=]() { memset(d, v, n); });
    return hipSuccess;
}
// device code is not registered: its host side runs up to the first launch only
API void** __hipRegisterFatBinary(const void*) { static void* handle; return &handle; }
API void __hipUnregisterFatBinary(void**) {}
API void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
API int crt_scratch_setup(int, void** p, size_t* bytes) { *p = nullptr; *bytes = 0; return 0; }

// ------------------------------------------------------------------ kernel launchers
extern "C" {
int crt_k_fill_u32(hipStream_t s, uint32_t* p, uint32_t n, uint32_t v) {
    std::lock_guard<std::mutex> g(g_m);
    enqueue(s, [=]() { for (uint32_t k = 0; k < n; ++k) p[k] = v; });
    return 0;
}
int crt_k_pass_init(hipStream_t s, uint32_t* ctl, uint32_t n) { return crt_k_fill_u32(s, ctl, n, 0u); }
int crt_k_init_request(hipStream_t s, float4* accum, uint32_t* rng, uint32_t W, uint32_t H, uint64_t seed) {
    std::lock_guard<std::mutex> g(g_m);
    enqueue(s, [=]() {
        for (uint32_t k = 0; k < W * H; ++k) { accum[k] = make_float4(0, 0, 0, 0); if (rng) rng[k] = (uint32_t)seed + 7u * k + 1u; }
    });
    return 0;
}
uint32_t crt_k_gstack_entries(void) { return 96; }
uint32_t crt_k_stack_capacity(void) { return 112; }
uint32_t crt_k_paths_waves(uint64_t words) { return (uint32_t)(words / (64u * 104u)); }
int crt_k_paths(hipStream_t s, int mode, int, int, uint32_t, const crt_dev_scene*, const crt_dev_request* reqs, uint32_t nreq,
                uint32_t, uint32_t*, crt_paths, uint32_t, float4*, uint32_t*, uint64_t, crt_dev_counters* counters) {
    std::lock_guard<std::mutex> g(g_m);
    if (launch_fails()) return 1;
    ++g_launches;
    enqueue(s, [=]() {
        Launch l{(uint64_t)mode, nreq, 0, 0};
        for (uint32_t k = 0; k < nreq; ++k) {
            const crt_dev_request& R = reqs[k];
            const uint64_t paths = (uint64_t)R.pix_count * R.sample_count;
            l.paths += paths;
            if (R.sample_count > l.most_samples) l.most_samples = R.sample_count;
            counters->rays += paths;
            g_path_count += paths;
            g_used.insert(s);
            if (R.rays) *R.rays += paths;
            if (mode != CRT_RNG_MINSTD) continue;
            // a pixel's engine and sums go on from where its last sample left them
            float4* acc = (float4*)R.accum;
            for (uint32_t p = R.pix_begin; p < R.pix_begin + R.pix_count; ++p)
                for (uint32_t q = R.sample_begin; q < R.sample_begin + R.sample_count; ++q) {
                    const uint32_t st = (uint32_t)((uint64_t)R.rng_state[p] * 16807u % 2147483647u);
                    R.rng_state[p] = st;
                    acc[p].x += (float)(st & 0xffffu) * 0.37f;
                    acc[p].y = acc[p].y * 0.5f + (float)q;
                    acc[p].w += 1.0f;
                }
        }
        g_ran.push_back(l);
    }, true);
    return 0;
}
int crt_k_resolve(hipStream_t s, const crt_dev_request* reqs, int nreq, uint32_t, const float4*, unsigned long long*) {
    std::lock_guard<std::mutex> g(g_m);
    enqueue(s, [=]() {
        for (int k = 0; k < nreq; ++k) {
            const crt_dev_request& R = reqs[k];
            float4* acc = (float4*)R.accum;
            for (uint32_t p = R.pix_begin; p < R.pix_begin + R.pix_count; ++p)
                for (uint32_t q = R.sample_begin; q < R.sample_begin + R.sample_count; ++q) {
                    acc[p].y = acc[p].y * 0.5f + (float)q;
                    acc[p].w += 1.0f;
                }
        }
    });
    return 0;
}
int crt_k_tonemap(hipStream_t s, const float4* accum, uint32_t n, uint32_t, uint8_t* rgb) {
    std::lock_guard<std::mutex> g(g_m);
    enqueue(s, [=]() {
        for (uint32_t k = 0; k < n; ++k) { rgb[3 * k] = (uint8_t)(uint32_t)accum[k].x; rgb[3 * k + 1] = (uint8_t)(uint32_t)accum[k].y; rgb[3 * k + 2] = (uint8_t)(uint32_t)accum[k].w; }
    });
    return 0;
}
int crt_k_trace_rays(hipStream_t s, int, int, uint32_t, const crt_dev_scene*, const float4* rays, uint32_t n, int, uint32_t* out,
                     uint32_t*, crt_dev_counters*) {
    std::lock_guard<std::mutex> g(g_m);
    if (launch_fails()) return 1;
    enqueue(s, [=]() { for (uint32_t k = 0; k < n; ++k) { out[k] = out[n + k] = ~0u; memcpy(out + 2 * n + k, &rays[2 * k].x, 4); } });
    return 0;
}
int crt_k_report_hits(hipStream_t s, uint32_t, const crt_dev_scene*, const float4*, const uint32_t*, uint32_t n, uint32_t* out) {
    std::lock_guard<std::mutex> g(g_m);
    if (launch_fails()) return 1;
    enqueue(s, [=]() { for (uint32_t k = 0; k < 2 * n; ++k) out[k] = ~0u; });
    return 0;
}
int crt_k_extend(hipStream_t, int, int, int, uint32_t, const crt_dev_scene*, const crt_dev_request*, int32_t, const uint32_t*,
                 const uint32_t*, uint32_t, const float4*, const float4*, const uint2*, float4*, uint32_t*, uint32_t*, uint32_t*,
                 int, uint32_t*, uint32_t, int, const uint32_t*, crt_dev_counters*) {
    std::lock_guard<std::mutex> g(g_m);
    return launch_fails() ? 1 : 0;
}
int crt_k_regen(hipStream_t, int, uint32_t, const crt_dev_request*, int, uint32_t, uint32_t, uint32_t, uint32_t*, uint32_t*,
                const uint32_t*, crt_paths) { return 1; }
int crt_k_shade(hipStream_t, int, int, uint32_t, const crt_dev_scene*, const crt_dev_request*, const uint32_t*, crt_paths, crt_paths,
                uint32_t*, const float4*, const uint32_t*, float4*, uint32_t*, int, int, crt_dev_counters*) { return 1; }
int crt_k_plain(hipStream_t, int, int, int, uint32_t, const crt_dev_scene*, const crt_dev_request*, uint32_t*, crt_dev_counters*) { return 1; }
int crt_k_valu_probe(hipStream_t, int, uint32_t, uint32_t, float*) { return 1; }
}
