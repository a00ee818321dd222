// paths.hip - whole paths in one launch: each wave takes camera paths of one request, follows them to
// their end and gathers the survivors into full waves of its own, so no path state goes through HBM.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cortex_rt.h"
#include "crt_device.h"
#include "crt_kernels.h"
#include "crt_layout.h"

namespace {

// Waves per SIMD the register allocation must allow (96 VGPRs). The 1080p 64-spp frame of the large
// scene takes 21.8 ms at 5, 23.7 at 4 (128 VGPRs, no spills) and 24.8 at 6 (80, spills inside the
// traversal loop); the 2M-triangle room 68.9, 77.0 and 73.8 ms.
constexpr int kWaves = 5;
// Traversal stack: 8 LDS ring entries per lane, so that 20 waves and their queues fit the 160 KB of a
// CU (6.5 KB each; 8.5 KB with 16 entries), then overflow entries in global memory. Together as
// deep as the staged kernels' stack.
constexpr int kLds = 8, kOverflow = 104;
// Camera paths handed to a wave at a time at most, and the smallest group a short launch is cut into:
// see crt_k_paths.
constexpr uint32_t kMaxChunk = 4, kMinGroup = 32;

// State bits of a path beside those of the staged pipeline (depth | bounce << 8 | camera << 16 |
// re-traces << 24): its radiance slot holds what it gathered before its end.
constexpr uint32_t kHasRadiance = 0x20000u;

__device__ __forceinline__ uint32_t lane_rank(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// Follows the paths of one request (ids [0, total): its pixels, each pixel's samples consecutive), or of
// several short ones, to their end in one launch. A workgroup is one wave. Each round the wave holds at most `group` paths,
// one per lane, and traces and shades one segment of each:
//   - lanes whose path ended take a path from the wave's queue in LDS;
//   - when queue and live paths together no longer fill a group, the live ones are put in the queue
//     (it never holds a whole group) and the next `group` ids start at the camera, so camera rays stay
//     in coherent waves of their own and the survivors in full waves of theirs;
//   - ids come in chunks: the first by the wave's number, the next ones from a counter.
// The stages (k_regen, k_extend, k_shade) trace the same waves' worth of rays but carry every path
// through HBM between them: 180 B per ray in the shade stage at 4.5 TB/s, 164 B of state per slot,
// and a launch whose last wave the next one waits for on each bounce. Here a path's state stays in
// registers and LDS, and only its radiance (16 B) is written. What bounds it is the traversal's VALU
// issue. Staged against this, GPU time of one render: 1080p 64 spp large scene 31.5 -> 20.8 ms,
// 2M-triangle room 1024^2 64 spp 81.2 -> 68.5, shapes 640x360 16 spp 4.8 -> 1.25 (latency and tails of
// the 22 launch rounds), box 64^2 16 spp 0.50 -> 0.17; 4,096 instances 4K 1 spp 27.0 -> 26.6.
// MINSTD: an id is a pixel; its samples run one after the other in its lane, each ended path starting
// the next sample, and are added to the accumulation buffer in order (a scene file's 512x388, 49
// samples, depth 100: 61 -> 5.7 ms against one staged pass per sample).
template <int MODE, int TL, bool MERGED>
__global__ __launch_bounds__(64, kWaves) void k_paths(const crt_dev_scene* __restrict__ scenes,
                                                           const crt_dev_request* __restrict__ reqs, uint32_t nreq,
                                                           uint32_t total, uint32_t group, uint32_t chunk,
                                                           uint32_t* __restrict__ next,
                                                           float4* __restrict__ out_rad, uint32_t* __restrict__ gstack,
                                                           crt_dev_counters* __restrict__ counters) {
    constexpr bool STREAM = MODE == CRT_RNG_MINSTD;
    constexpr bool SHAPES = TL != 3;   // shading of shapes and instances
    __shared__ uint32_t s_stack[kLds * 64];
    __shared__ uint32_t s_wait[(STREAM ? 13 : 12) * 64];
    __shared__ uint32_t s_path[6 * 64];
    const uint32_t lane = threadIdx.x;
    bool more = true;
    uint32_t cur = min(blockIdx.x * chunk, total);
    if (MERGED) {
        // one group of ids a wave, none handed out
        more = false;
        cur = blockIdx.x * group;
        const uint32_t base = reqs->path_base;
        uint32_t lo = 0, hi = nreq;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (reqs[mid].path_base - base <= cur) lo = mid; else hi = mid;
        }
        reqs += lo;
        cur -= reqs->path_base - base;
        out_rad += reqs->path_base - base;
        total = STREAM ? reqs->pix_count : reqs->pix_count * reqs->sample_count;
        cur = min(cur, total);
    }
    uint32_t end = min(cur + chunk, total);
    const crt_dev_request& R = *reqs;
    const crt_dev_scene* sc = scenes + R.scene;
    const SceneView S = scene_view(sc);
    const GSlot gst{gstack, (blockIdx.x * 64u + lane) * kOverflow};
    uint64_t cn[5] = {0,0,0,0,0};
    auto count = [&](int k, uint64_t mask) { cn[k] += (uint64_t)__popcll(mask); };
    uint32_t waiting = 0;
    bool live = false;
    V3 o = v3(0.0f, 0.0f, 0.0f), d = o, att = o;
    uint32_t pix = 0, sample = 0, state = 0, ms = 0;
    auto start = [&]() {
        Rng<MODE> g;
        g.dyn = R.rng_mode;
        g.ms = ms;
        if (!STREAM) g.pcg = pcg_keyed(R.seed, ref_pixel_of(R, pix), sample, 0u);
        float tm;
        camera_ray<MODE>(R, pix, sample, g, o, d, tm);
        ms = g.ms;
        state = (R.max_depth & 0xffu) | ST_CAMERA;
        att = v3(1.0f, 1.0f, 1.0f);
    };
    for (;;) {
        const uint64_t lm = __ballot(live);
        const uint32_t n = (uint32_t)__popcll(lm);
        if (n + waiting < group && cur >= end && more) {
            uint32_t b = 0;
            if (lane == 0) b = atomicAdd(next, chunk);
            b = (uint32_t)__builtin_amdgcn_readfirstlane((int)b) + gridDim.x * chunk;
            if (b < total) { cur = b; end = min(b + chunk, total); } else more = false;
        }
        if (n + waiting < group && cur < end) {
            if (live) {
                uint32_t* w = s_wait + waiting + lane_rank(lm);
                w[0] = fbits(o.x); w[64] = fbits(o.y); w[128] = fbits(o.z);
                w[192] = fbits(d.x); w[256] = fbits(d.y); w[320] = fbits(d.z);
                w[384] = fbits(att.x); w[448] = fbits(att.y); w[512] = fbits(att.z);
                w[576] = pix; w[640] = sample; w[704] = state;
                if (STREAM) w[768] = ms;
            }
            waiting += n;
            const uint32_t id = cur + lane;
            live = lane < group && id < end;
            cur += group;
            if (live) {
                const uint32_t sidx = STREAM ? id : id / R.sample_count;
                pix = item_pixel(R, sidx);
                sample = R.sample_begin + (STREAM ? 0u : id - sidx * R.sample_count);
                if (STREAM) ms = ldg(R.rng_state + pix);
                start();
            }
        } else if (waiting) {
            const uint32_t take = min(group > n ? group - n : 0u, waiting);
            const uint32_t r = lane_rank(~lm);
            if (!live && r < take) {
                const uint32_t* w = s_wait + (waiting - 1u - r);
                o = v3(bitsf(w[0]), bitsf(w[64]), bitsf(w[128]));
                d = v3(bitsf(w[192]), bitsf(w[256]), bitsf(w[320]));
                att = v3(bitsf(w[384]), bitsf(w[448]), bitsf(w[512]));
                pix = w[576]; sample = w[640]; state = w[704];
                if (STREAM) ms = w[768];
                live = true;
            }
            waiting -= take;
        }
        __syncthreads();
        const uint64_t am = __ballot(live);
        if (!am) break;
        count(0, am);
        uint32_t pf = 0, lt = 0, ovf = 0, exact = 0;
        if (live) {
            // what the traversal does not need waits in LDS: held in registers across it, the loop spills
            // (24.6 instead of 21.8 ms for the large frame)
            {
                uint32_t* w = s_path + lane;
                w[0] = fbits(att.x); w[64] = fbits(att.y); w[128] = fbits(att.z); w[192] = pix; w[256] = sample; w[320] = state;
                asm volatile("" ::: "memory");
            }
            HitRec h;
            TravCount tc = {0, 0, 0, 0, 0, 0};
            uint32_t xr = 0, xt = 0;
            pf = closest_hit_checked<64, 1, kLds, kOverflow, false, 4, TL>(S, o, d, (state & ST_CAMERA) != 0, s_stack + lane, gst, h,
                                                                         tc, ovf, xr, xt, exact);
            {
                asm volatile("" ::: "memory");
                const uint32_t* w = s_path + lane;
                att = v3(bitsf(w[0]), bitsf(w[64]), bitsf(w[128])); pix = w[192]; sample = w[256]; state = w[320];
            }
            const uint32_t rid = STREAM ? pix - R.pix_begin : (pix - R.pix_begin) * R.sample_count + (sample - R.sample_begin);
            V3 L = v3(0.0f, 0.0f, 0.0f);
            if (state & kHasRadiance) L = v3(ldg(out_rad + rid));
            uint32_t depth = ST_DEPTH(state), bounce = ST_BOUNCE(state);
            const uint32_t retraces = ST_RETRACES(state) + (pf ? 1u : 0u);
            Rng<MODE> g;
            g.ms = ms;
            g.dyn = R.rng_mode;
            const float4 hv = make_float4(h.t, bitsf(h.prim), h.u, h.v);
            const bool keep = shade_hit<MODE, SHAPES>(sc, R, pix, sample, hv, h.inst | pf, o, d, att, L, depth, bounce, g, lt);
            ms = g.ms;
            if (keep) {
                state = (depth & 0xffu) | ((bounce & 0xffu) << 8) | (state & kHasRadiance) | (retraces << 24);
                if (pf & CRT_PASSTHROUGH_WHITE) {
                    state |= kHasRadiance;
                    stg(out_rad + rid, make_float4(L.x, L.y, L.z, 0.0f));
                }
            } else if (STREAM) {
                float4* a = (float4*)R.accum + pix;
                float4 acc = ldg(a);
                acc.x += L.x; acc.y += L.y; acc.z += L.z; acc.w += 1.0f;
                stg(a, acc);
                sample += 1u;
                live = sample < R.sample_begin + R.sample_count;
                if (live) start(); else stg(R.rng_state + pix, ms);
            } else {
                const uint32_t rays = bounce + (h.prim == CRT_MISS ? 1u : 0u) + retraces;
                stg(out_rad + rid, make_float4(L.x, L.y, L.z, (float)rays));
                live = false;
            }
        }
        // counted where the wave has come together again: a ballot inside the branch sees the lanes
        // of one way through it only
        count(1, __ballot(pf != 0u));
        count(2, __ballot(lt != 0u));
        count(3, __ballot(ovf != 0u));
        count(4, __ballot(exact != 0u));
    }
    if (lane == 0) {
        const unsigned long long nrays = cn[0], nretrace = cn[1], nlight = cn[2] * sc->num_lights, novf = cn[3],
                                 nexact = cn[4];
        atomicAdd(&counters->rays, nrays);
        if (nretrace) atomicAdd(&counters->retraces, nretrace);
        if (nlight) atomicAdd(&counters->light_tests, nlight);
        if (novf) atomicAdd(&counters->stack_overflow, novf);
        if (nexact) atomicAdd(&counters->exact, nexact);
        if (R.rays) {
            atomicAdd(R.rays, nrays + nretrace);
            if (novf) atomicOr(R.rays, 1ull << 63);
        }
    }
}

// Waves of one kernel that the device holds at once.
template <typename K> uint32_t resident_waves(K kernel) {
    int nb = 0, dev = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, 64, 0) != hipSuccess || nb <= 0) nb = 1;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus <= 0)
        cus = 256;
    return (uint32_t)nb * (uint32_t)cus;
}

}  // namespace

extern "C" uint32_t crt_k_paths_overflow_entries(void) { return (uint32_t)kOverflow; }

extern "C" int crt_k_paths(hipStream_t s, int rng_mode, int two_level, int shapes, uint32_t max_waves, const crt_dev_scene* scenes,
                           const crt_dev_request* reqs, uint32_t nreq, uint32_t total, uint32_t* next, float4* out_rad,
                           uint32_t* gstack, crt_dev_counters* counters) {
    if (total == 0) return 0;
    if (nreq > 1 && (total > CRT_PATHS_MERGE || total > (uint64_t)max_waves * CRT_PATHS_ALIGN)) return (int)hipErrorInvalidValue;
    auto launch = [&](auto kfn, uint32_t resident) {
        uint32_t waves = resident < max_waves ? resident : max_waves;
        // A launch with fewer paths than lanes is cut into groups of 32, not 64: twice the waves, each
        // done when the longest of half as many rays is (box 64^2 16 spp 0.175 -> 0.165 ms GPU). 16 and
        // 8 cost more waves' worth of instructions than they save (0.21 ms).
        uint32_t group = CRT_PATHS_ALIGN;
        if (group > kMinGroup && (uint64_t)waves * kMinGroup >= total) group = kMinGroup;
        const uint32_t groups = (total + group - 1u) / group;
        if (waves > groups || nreq > 1) waves = groups;
        // Groups per hand-out: large enough that the counter's atomics (about 14 ns each, one after
        // the other across the XCDs) do not bound the launch, small enough that the waves in flight
        // trace neighbouring pixels (large frame at 1, 4, 8, 16, 32 groups: 29.6, 20.8, 21.5, 23.6,
        // 30.5 ms; room 66.3, 67.2, 68.5, 70.9, 74.3), and at least eight hand-outs a wave so that
        // the waves end together.
        uint32_t c = groups / (waves * 8u);
        c = c < 1u ? 1u : (c > kMaxChunk ? kMaxChunk : c);
        hipLaunchKernelGGL(kfn, dim3(waves), dim3(64), 0, s, scenes, reqs, nreq, total, group, nreq > 1 ? group : c * group, next, out_rad, gstack, counters);
    };
#define CRT_PTH(M, T)                                                         \
    {                                                                         \
        static const uint32_t resident = resident_waves(k_paths<M, T, false>); \
        if (nreq > 1) launch(k_paths<M, T, true>, resident);                  \
        else launch(k_paths<M, T, false>, resident);                          \
    }
#define CRT_PTH_T(M)                                                          \
    {                                                                         \
        if (two_level) { if (shapes) CRT_PTH(M, 2) else CRT_PTH(M, 1) }       \
        else { if (shapes) CRT_PTH(M, 0) else CRT_PTH(M, 3) }                 \
    }
    if (rng_mode == CRT_RNG_MINSTD) CRT_PTH_T(CRT_RNG_MINSTD) else CRT_PTH_T(CRT_RNG_PCG)
#undef CRT_PTH_T
#undef CRT_PTH
    return (int)hipGetLastError();
}
