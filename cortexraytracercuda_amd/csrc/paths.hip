// paths.hip - whole paths in one launch: each wave takes camera paths of one request, follows them to
// their end and gathers the survivors into full waves of its own, so no path state goes through HBM.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

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

// Follows the paths of one request (ids [0, total): its pixels, each pixel's samples consecutive) to
// their end in one launch; MERGED, of several short ones (a branch for both in one kernel costs the
// two-level loop 8 %, in registers). A workgroup is one wave. Each round the wave holds at most `group`
// paths, one per lane, and traces and shades one segment of each:
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
// 2M-triangle room 1024^2 64 spp 80.6 -> 67.1, shapes 640x360 16 spp 4.8 -> 1.25 (latency and tails of
// the 22 launch rounds), box 64^2 16 spp 0.50 -> 0.17; 4,096 instances 4K 1 spp 27.0 -> 24.2.
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

// Refilled waves (k_paths_refill). A wave of k_paths waits for its slowest ray: of a room's secondary
// rays 22 % of the lanes work on the average. Here a wave leaves the traversal once kRefill of its lanes
// (or two thirds of those at work) have their hit, shades those and gives them the next ray, while the
// others keep their place in LDS. Leaf lanes wait until 1 / kLeafShare of the wave is at a leaf. Below
// kDrainLive rays, with camera rays left to start, every ray is finished, so that camera rays have the
// wave to themselves; their survivors wait in a queue in global memory, long enough that they leave it in
// full waves, short enough that the launch does not end in waves that empty theirs: a share of the paths
// of a wave, kMinQueue to kMaxQueue (at 25 M paths with kMaxQueue 5.8 ms for the 131,072-node open scene,
// 4.9 so).
// What it costs is the shading of part-filled waves (about 1,500 VALU instructions a time), so it pays
// where traversals are long and launches are: against k_paths on a 2M-triangle room, 1024^2 64 spp,
// 67.1 -> 52.5 ms GPU (200,000 triangles: 59.6 -> 48), the 1080p large frame 20.8 -> 20.2. kRefill 32
// (half of those at work): 53.6; 52 (13 / 16): 54; 64: k_paths's way with this loop, 80.
constexpr uint32_t kRefill = 40, kLeafShare = 4, kDrainLive = 56, kQueueShare = 24, kMinQueue = 128, kMaxQueue = 768;
// Where refilled waves take over: rooms gain from some hundred nodes on, scenes under an open sky, whose
// paths are short, from some ten thousand on with long launches; neither gains with short ones. By nodes, k_paths -> these, 1024^2 36 spp: rooms of 788 nodes 22.2 ->
// 20.6 ms, 19,570: 30.5 -> 26.1, 78,322: 34.2 -> 28.2, the 8-node box 9.7 -> 12.1; open scenes of 8,443:
// 5.0 -> 5.3, 33,066: 5.5 -> 5.7 (1080p 49 spp: 13.0 -> 13.2), 132,139: 6.1 -> 6.2, 526,438: 6.8 -> 6.7. By paths, room of 78,322 and open scene of 132,139 nodes: 4 M 4.46 -> 4.22 and 1.56 -> 1.71, 9 M 9.5 ->
// 8.6 and 2.4 -> 2.5, 16 M 16.1 -> 14.0 and 3.47 -> 3.49.
constexpr uint32_t kRefillNodes = 1u << 14, kRefillPaths = 3u << 21;
// Stack entries of a lane in global memory: the ring's entries have their place there too (as many in
// all as k_paths has with its register entry, 113, and more), three that one node may push beyond, and
// the last one holds the start of a re-traced ray. The state word counts them in 7 bits.
constexpr int kRefillStack = kLds + kOverflow + 8;

// Box tests are accepted up to this multiple of the closest distance so far (the tie window, and the
// box test's own rounding).
#define CRT_CULL (CRT_TIE_HI * CRT_BOX_FAR)

// What a lane keeps in LDS between two runs of the traversal loop, in words of 64 lanes: its ray, the
// closest hit so far, the next node and the stack's counters, and its path.
enum { W_OX, W_OY, W_OZ, W_DX, W_DY, W_DZ, W_T, W_U, W_V, W_PRIM, W_KEY, W_NODE, W_CTL, W_AX, W_AY, W_AZ, W_PIX, W_SMP, W_COUNT
};
// control word: entries on the stack, of them in global memory (7 bits each), flags
constexpr uint32_t kCtlCamera = 1u << 25, kCtlAmb = 1u << 26, kCtlPass = 1u << 27, kCtlWhite = 1u << 28;
// path words: pixel (below 2^28) | radiance flag; sample (below 2^16: both as Job::validate has it) |
// depth left << 16 | pass-through re-traces so far << 24
constexpr uint32_t kPixRadiance = 0x80000000u;

typedef __attribute__((address_space(3))) uint16_t lds_u16;

template <int TL> struct PathTrav {
    static constexpr bool SHAPES = TL == 0;
    V3 o, d, id, on, of;
    uint32_t ox, oy, oz;   // 16 where the hi plane of the axis is the near one
    TriPre tp;
    HitRec best;
    float tmin;
    uint32_t tf;           // bits of the distance beyond which boxes are culled
    int32_t node;
    uint32_t sp, sbase;    // entries on the stack, and how many of them (the oldest) are in global memory, times 256
    uint32_t ring;         // LDS address of this lane's column of the ring of references
    uint32_t kring;        // and of the upper halves of their distances, whose entries lie half as far apart
    glb_u32* over;
    uint32_t goff;
    bool camera, amb, ovf;

    static __device__ __forceinline__ float inv_of(float x) {
        return __builtin_amdgcn_rcpf(fabsf(x) > 1e-30f ? x : copysignf(1e-30f, x));
    }
    __device__ __forceinline__ void set_ray(V3 ro, V3 rd) {
        o = ro; d = rd;
        id = v3(inv_of(d.x), inv_of(d.y), inv_of(d.z));
        const V3 oid = v3(o.x * id.x, o.y * id.y, o.z * id.z);
        const V3 e = v3(fabsf(oid.x) * 2.384185791e-7f, fabsf(oid.y) * 2.384185791e-7f, fabsf(oid.z) * 2.384185791e-7f);
        on = oid + e; of = oid - e;
        ox = id.x < 0.0f ? 16u : 0u;
        oy = id.y < 0.0f ? 16u : 0u;
        oz = id.z < 0.0f ? 16u : 0u;
        tp = tri_pre(d);
    }
    __device__ __forceinline__ void load(const SceneView& S, const uint32_t* w) {
        const V3 wo = v3(bitsf(w[64 * W_OX]), bitsf(w[64 * W_OY]), bitsf(w[64 * W_OZ]));
        const V3 wd = v3(bitsf(w[64 * W_DX]), bitsf(w[64 * W_DY]), bitsf(w[64 * W_DZ]));
        best.t = bitsf(w[64 * W_T]); best.u = bitsf(w[64 * W_U]); best.v = bitsf(w[64 * W_V]);
        best.prim = w[64 * W_PRIM]; best.key = w[64 * W_KEY];
        node = (int32_t)w[64 * W_NODE];
        const uint32_t c = w[64 * W_CTL];
        sp = (c & 0x7fu) << 8; sbase = (c >> 7 & 0x7fu) << 8;
        camera = (c & kCtlCamera) != 0u; amb = false; ovf = false;
        tmin = 0.00001f;
        if (c & kCtlPass) tmin = bitsf(over[goff + (uint32_t)kRefillStack - 1u]);
        set_ray(wo, wd);
        tf = min(fbits(best.t * CRT_CULL), 0x7f7fffffu);
    }
    __device__ __forceinline__ void store(uint32_t* w) const {
        w[64 * W_T] = fbits(best.t); w[64 * W_U] = fbits(best.u); w[64 * W_V] = fbits(best.v);
        w[64 * W_PRIM] = best.prim; w[64 * W_KEY] = best.key;
        w[64 * W_NODE] = (uint32_t)node;
        uint32_t c = (w[64 * W_CTL] & (kCtlCamera | kCtlPass | kCtlWhite)) | (sp >> 8) | (sbase >> 8) << 7 | (amb ? kCtlAmb : 0u);
        w[64 * W_CTL] = c;
    }
    __device__ __forceinline__ uint32_t child_key(float nx, float fx, float ny, float fy, float nz, float fz) const {
        const float nr = fmaxf(fmaxf(fmaf(nx, id.x, -on.x), fmaf(ny, id.y, -on.y)), fmaxf(fmaf(nz, id.z, -on.z), tmin));
        const float fr = fminf(fminf(fmaf(fx, id.x, -of.x), fmaf(fy, id.y, -of.y)), fmaf(fz, id.z, -of.z));
        const int32_t miss = (int32_t)fbits(fmaf(fr, CRT_BOX_FAR, -nr)) >> 31;
        return fbits(nr) | ((uint32_t)miss & 0x7f800000u);
    }
    static __device__ __forceinline__ void order(uint32_t& ka, int32_t& va, uint32_t& kb, int32_t& vb) {
        const bool s = kb < ka;
        const uint32_t lo = min(ka, kb), hi = max(ka, kb);
        ka = lo; kb = hi;
        const int32_t v = s ? vb : va; vb = s ? va : vb; va = v;
    }
    __device__ __forceinline__ void put(uint32_t key, int32_t ref, bool valid) {
        const uint32_t e = (sp & 0x700u) | ring;
        *(lds_u32*)(uintptr_t)e = (uint32_t)ref;
        *(lds_u16*)(uintptr_t)((e >> 1) + kring) = (uint16_t)(key >> 16);
        sp += valid ? 256u : 0u;
    }
    // Room for three entries in the ring: the oldest go to global memory.
    __device__ __forceinline__ void make_room() {
        while (sp + 768u - sbase > 2048u) {
            over[goff + (sbase >> 8)] = *(lds_u32*)(uintptr_t)((sbase & 0x700u) | ring);
            sbase += 256u;
        }
    }
    // Node: box tests, the hit children pushed far to near, on to the nearest; false when none is hit.
    __device__ __forceinline__ bool visit_node(float4 rf, float4 nx, float4 fx, float4 ny, float4 fy, float4 nz, float4 fz) {
        uint32_t k0 = child_key(nx.x, fx.x, ny.x, fy.x, nz.x, fz.x), k1 = child_key(nx.y, fx.y, ny.y, fy.y, nz.y, fz.y),
                 k2 = child_key(nx.z, fx.z, ny.z, fy.z, nz.z, fz.z), k3 = child_key(nx.w, fx.w, ny.w, fy.w, nz.w, fz.w);
        int32_t c0 = (int32_t)fbits(rf.x), c1 = (int32_t)fbits(rf.y), c2 = (int32_t)fbits(rf.z), c3 = (int32_t)fbits(rf.w);
        order(k0, c0, k1, c1); order(k2, c2, k3, c3);
        order(k0, c0, k2, c2); order(k1, c1, k3, c3);
        order(k1, c1, k2, c2);
        if (k0 > tf) return false;
        node = c0;
        if (k1 <= tf) {
            make_room();
            put(k3, c3, k3 <= tf);
            put(k2, c2, k2 <= tf);
            put(k1, c1, true);
            if (sp > (uint32_t)(kRefillStack - 4) * 256u) { ovf = true; sp -= 768u; }
        }
        return true;
    }
    // Leaf, its first record in a0..a3; false when an undecided triangle test ends the query.
    __device__ __forceinline__ bool visit_leaf(const SceneView& S, float4 a0, float4 a1, float4 a2) {
        const uint32_t type = CRT_LEAF_REF_TYPE(node), cnt = CRT_LEAF_REF_COUNT(node), first = CRT_LEAF_REF_FIRST(node);
        if (type == CRT_PRIM_TRI) {
            for (uint32_t k = 0; k < cnt; ++k) {
                if (k) {
                    const uint32_t to = S.tri_off + (first + k) * 48u;
                    a0 = ldg_at(S.nodes, to); a1 = ldg_at(S.nodes, to + 16u); a2 = ldg_at(S.nodes, to + 32u);
                }
                float t, bu, bv;
                if (tri_hit<false>(o, d, tp, a0, a1, a2, tmin, best.t * CRT_TIE_HI, t, bu, bv, amb) && hit_wins(t, fbits(a0.w), best)) {
                    best.t = t; best.u = bu; best.v = bv; best.prim = (CRT_PRIM_TRI << 30) | (first + k);
                    best.key = fbits(a0.w);
                }
            }
            if (amb) return false;
        } else if (type == CRT_PRIM_SPHERE) {
            for (uint32_t k = 0; k < cnt; ++k) {
                if (k) {
                    const uint32_t so = S.sph_off + (first + k) * 32u;
                    a0 = ldg_at(S.nodes, so); a1 = ldg_at(S.nodes, so + 16u);
                }
                const uint32_t key = fbits(a1.x);
                float t;
                if ((fbits(a1.z) & CRT_SF_INVISIBLE) && camera) continue;
                if (sphere_hit(o, d, a0, tmin, best.t * CRT_TIE_HI, t) && hit_wins(t, key, best)) {
                    best.t = t; best.u = 0.0f; best.v = 0.0f; best.prim = (CRT_PRIM_SPHERE << 30) | (first + k);
                    best.key = key;
                }
            }
        } else if (type == CRT_PRIM_QUAD) {
            for (uint32_t k = 0; k < cnt; ++k) {
                float t, qa, qb;
                uint32_t key;
                if (quad_hit<SHAPES>(o, d, S.quad(first + k), tmin, best.t * CRT_TIE_HI, camera, t, qa, qb, key) && hit_wins(t, key, best)) {
                    best.t = t; best.u = qa; best.v = qb; best.prim = (CRT_PRIM_QUAD << 30) | (first + k);
                    best.key = key;
                }
            }
        }
        tf = min(fbits(best.t * CRT_CULL), 0x7f7fffffu);
        return true;
    }
    // Steps the lanes that have a query (`go`) until at most `leave` of them are still going.
    __device__ __forceinline__ void run(const SceneView& S, bool& go, uint32_t leave) {
        for (;;) {
            const uint32_t na = (uint32_t)__popcll(__ballot(go));
            if (na <= leave) break;
            if (!go) continue;
            bool going = true;
            // node lanes and leaf lanes share one set of seven loads (one memory round trip a step)
            const bool isn = node >= 0;
            const uint32_t type = CRT_LEAF_REF_TYPE(node), first = CRT_LEAF_REF_FIRST(node);
            const uint32_t lb = type == CRT_PRIM_TRI ? S.tri_off + first * 48u
                                : (type == CRT_PRIM_SPHERE ? S.sph_off + first * 32u : 0u);
            const uint32_t b0 = isn ? (uint32_t)node << 7 : lb, b1 = b0 + 16u;
            const uint32_t sx = isn ? ox : 0u, sy = isn ? oy : 0u, sz = isn ? oz : 0u;
            const float4 nx = ldg_off<0>(S.nodes, b0 + sx), fx = ldg_off<0>(S.nodes, b1 - sx), ny = ldg_off<32>(S.nodes, b0 + sy),
                         fy = ldg_off<32>(S.nodes, b1 - sy), nz = ldg_off<64>(S.nodes, b0 + sz), fz = ldg_off<64>(S.nodes, b1 - sz),
                         rf = ldg_off<96>(S.nodes, b0);
            __builtin_amdgcn_sched_group_barrier(0x020, 7, 0);   // 0x020: VMEM reads
            const uint32_t nl = (uint32_t)__popcll(__ballot(!isn));
            bool want = false;
            if (isn) want = !visit_node(rf, nx, fx, ny, fy, nz, fz);
            // leaf lanes wait until a share of the wave is at one
            if (nl * kLeafShare >= na) {
                if (!isn) {
                    going = visit_leaf(S, nx, fx, ny);
                    want = going;
                }
            }
            while (want) {
                if (sp == 0u) { going = false; break; }
                sp -= 256u;
                uint32_t key = 0u;
                if (sp < sbase) {
                    sbase = sp;
                    node = (int32_t)over[goff + (sp >> 8)];
                } else {
                    const uint32_t e = (sp & 0x700u) | ring;
                    node = (int32_t)*(lds_u32*)(uintptr_t)e;
                    key = (uint32_t)*(lds_u16*)(uintptr_t)((e >> 1) + kring) << 16;
                }
                want = key > tf;
            }
            go = going;
        }
    }
};


template <int TL>
__global__ __launch_bounds__(64, kWaves) void k_paths_refill(const crt_dev_scene* __restrict__ scenes,
                                                           const crt_dev_request* __restrict__ req, uint32_t total,
                                                           uint32_t group, uint32_t chunk, uint32_t* __restrict__ next,
                                                           crt_paths P, uint32_t qcap,
                                                           float4* __restrict__ out_rad, uint32_t* __restrict__ gstack,
                                                           crt_dev_counters* __restrict__ counters) {
    constexpr int MODE = CRT_RNG_PCG;
    __shared__ __attribute__((aligned(2048))) uint32_t s_stack[kLds * 64];
    __shared__ uint16_t s_key[kLds * 64];
    __shared__ uint32_t s_lane[W_COUNT * 64];
    const uint32_t lane = threadIdx.x;
    const crt_dev_request& R = *req;
    const crt_dev_scene* sc = scenes + R.scene;
    const SceneView S = scene_view(sc);
    const GSlot gst{gstack, (blockIdx.x * 64u + lane) * kRefillStack};
    uint32_t* const w = s_lane + lane;
    float4* const q_o = P.ray_o + (size_t)blockIdx.x * qcap;
    float4* const q_d = P.ray_d + (size_t)blockIdx.x * qcap;
    float4* const q_t = P.thr + (size_t)blockIdx.x * qcap;
    uint64_t nrays = 0, nretrace = 0, novf = 0, nexact = 0, nlight = 0;   // wave totals (scalar)
    uint32_t waiting = 0, cur = min(blockIdx.x * chunk, total), end = min(cur + chunk, total);
    bool more = true;
    enum { IDLE = 0, TRACE = 1, DONE = 2, NEXT = 3 };
    enum { CAMERA = 0, SECOND = 1, DRAIN = 2 };
    uint32_t mode = CAMERA;
    uint32_t ph = IDLE;
    for (int k = 0; k < W_COUNT; ++k) w[64 * k] = 0u;   // idle lanes are loaded and run no step
    auto put_ray = [&](V3 o, V3 d) {
        w[64 * W_OX] = fbits(o.x); w[64 * W_OY] = fbits(o.y); w[64 * W_OZ] = fbits(o.z);
        w[64 * W_DX] = fbits(d.x); w[64 * W_DY] = fbits(d.y); w[64 * W_DZ] = fbits(d.z);
    };
    auto start = [&](uint32_t pix, uint32_t sample) {
        Rng<MODE> g;
        g.dyn = R.rng_mode;
        g.ms = 0u;
        g.pcg = pcg_keyed(R.seed, ref_pixel_of(R, pix), sample, 0u);
        float tm;
        V3 o, d;
        camera_ray<MODE>(R, pix, sample, g, o, d, tm);
        put_ray(o, d);
        w[64 * W_AX] = w[64 * W_AY] = w[64 * W_AZ] = fbits(1.0f);
        w[64 * W_PIX] = pix;
        w[64 * W_SMP] = (sample & 0xffffu) | (R.max_depth & 0xffu) << 16;
        w[64 * W_CTL] = kCtlCamera;
    };
    for (;;) {
        // finished queries: an emitter seen from behind is passed through (re-traced behind it), others
        // are shaded
        if (__ballot(ph == DONE)) {
            uint32_t lt = 0, ex = 0, ov = 0, pf = 0;
            bool counted = false;
            if (ph == DONE) {
                HitRec h;
                h.t = bitsf(w[64 * W_T]); h.u = bitsf(w[64 * W_U]); h.v = bitsf(w[64 * W_V]); h.prim = w[64 * W_PRIM];
                h.inst = CRT_NO_INST;
                const uint32_t c = w[64 * W_CTL];
                V3 o = v3(bitsf(w[64 * W_OX]), bitsf(w[64 * W_OY]), bitsf(w[64 * W_OZ]));
                V3 d = v3(bitsf(w[64 * W_DX]), bitsf(w[64 * W_DY]), bitsf(w[64 * W_DZ]));
                bool again = false;
                if (c & kCtlAmb) {
                    const ExactHit e = exact_hit<64, 1, kLds, kOverflow, 4, TL>(S, o, d, (c & kCtlCamera) != 0u, s_stack + lane, gst);
                    h = e.h;
                    pf = e.pass_flag;
                    ov = e.ovf;
                    ex = 1;
                } else if (c & kCtlPass) {
                    pf = CRT_PASSTHROUGH | ((c & kCtlWhite) ? CRT_PASSTHROUGH_WHITE : 0u);
                } else {
                    const uint32_t p = passes_through(S, h, o, d);
                    if (p) {
                        gstack[gst.off + (uint32_t)kRefillStack - 1u] = fbits(h.t + 0.001f);
                        w[64 * W_CTL] = (c & kCtlCamera) | kCtlPass | ((p & CRT_PASSTHROUGH_WHITE) ? kCtlWhite : 0u);
                        ph = NEXT;
                        again = true;
                    }
                }
                if (!again) {
                    counted = true;
                    V3 att = v3(bitsf(w[64 * W_AX]), bitsf(w[64 * W_AY]), bitsf(w[64 * W_AZ]));
                    const uint32_t pw = w[64 * W_PIX], sw = w[64 * W_SMP], pix = pw & ~kPixRadiance, sample = sw & 0xffffu;
                    uint32_t depth = sw >> 16 & 0xffu, bounce = ((R.max_depth & 0xffu) - depth) & 0xffu;
                    const uint32_t rid = (pix - R.pix_begin) * R.sample_count + (sample - R.sample_begin);
                    V3 L = v3(0.0f, 0.0f, 0.0f);
                    if (pw & kPixRadiance) L = v3(ldg(out_rad + rid));
                    const uint32_t retraces = (sw >> 24) + (pf ? 1u : 0u);
                    Rng<MODE> g;
                    g.ms = 0u;
                    g.dyn = R.rng_mode;
                    const float4 hv = make_float4(h.t, bitsf(h.prim), h.u, h.v);
                    const bool keep = shade_hit<MODE, TL == 0>(sc, R, pix, sample, hv, h.inst | pf, o, d, att, L, depth, bounce, g, lt);
                    if (keep) {
                        put_ray(o, d);
                        w[64 * W_AX] = fbits(att.x); w[64 * W_AY] = fbits(att.y); w[64 * W_AZ] = fbits(att.z);
                        w[64 * W_SMP] = sample | (depth & 0xffu) << 16 | retraces << 24;
                        w[64 * W_CTL] = 0u;
                        if (pf & CRT_PASSTHROUGH_WHITE) {
                            w[64 * W_PIX] = pix | kPixRadiance;
                            stg(out_rad + rid, make_float4(L.x, L.y, L.z, 0.0f));
                        }
                        ph = NEXT;
                    } else {
                        const uint32_t rays = bounce + (h.prim == CRT_MISS ? 1u : 0u) + retraces;
                        stg(out_rad + rid, make_float4(L.x, L.y, L.z, (float)rays));
                        ph = IDLE;
                    }
                }
            }
            // counted where the wave has come together again: a ballot inside the branch sees the lanes
            // of one way through it only
            nrays += (uint64_t)__popcll(__ballot(counted));
            nretrace += (uint64_t)__popcll(__ballot(pf != 0u));
            novf += (uint64_t)__popcll(__ballot(ov != 0u));
            nexact += (uint64_t)__popcll(__ballot(ex != 0u));
            nlight += (uint64_t)__popcll(__ballot(lt != 0u)) * sc->num_lights;
        }
        // the next rays
        const uint64_t mn = __ballot(ph == NEXT);
        const uint32_t nt = (uint32_t)__popcll(__ballot(ph == TRACE));
        uint32_t nn = (uint32_t)__popcll(mn);
        if (mode != SECOND) {
            // survivors of a camera batch and of a drain wait in the queue; re-traces stay
            const bool park = ph == NEXT && !(w[64 * W_CTL] & kCtlPass);
            const uint64_t mp = __ballot(park);
            if (park) {
                const uint32_t k = waiting + lane_rank(mp);
                q_o[k] = make_float4(bitsf(w[64 * W_OX]), bitsf(w[64 * W_OY]), bitsf(w[64 * W_OZ]), bitsf(w[64 * W_PIX]));
                q_d[k] = make_float4(bitsf(w[64 * W_DX]), bitsf(w[64 * W_DY]), bitsf(w[64 * W_DZ]), bitsf(w[64 * W_SMP]));
                q_t[k] = make_float4(bitsf(w[64 * W_AX]), bitsf(w[64 * W_AY]), bitsf(w[64 * W_AZ]), 0.0f);
                ph = IDLE;
            }
            __threadfence_block();   // read by other lanes
            const uint32_t np = (uint32_t)__popcll(mp);
            waiting += np;
            nn -= np;
            if (nt + nn == 0u) mode = CAMERA;
        }
        if (cur >= end && more && mode == CAMERA) {
            uint32_t b = 0;
            if (lane == 0) b = atomicAdd(next, chunk);
            b = (uint32_t)__builtin_amdgcn_readfirstlane((int)b) + gridDim.x * chunk;
            if (b < total) { cur = b; end = min(b + chunk, total); } else more = false;
        }
        if (mode == CAMERA && nt + nn == 0u) {
            if (cur < end && waiting + group <= qcap) {
                const uint32_t id = cur + lane;
                if (lane < group && id < end) {
                    const uint32_t sidx = id / R.sample_count;
                    start(item_pixel(R, sidx), R.sample_begin + id - sidx * R.sample_count);
                    ph = NEXT;
                }
                cur = min(cur + group, end);
            } else {
                mode = SECOND;
            }
        }
        if (mode == SECOND && waiting) {
            const uint64_t mi = __ballot(ph == IDLE);
            const uint32_t live = nt + nn;
            const uint32_t take = min(group > live ? group - live : 0u, waiting);
            const uint32_t r = lane_rank(mi);
            if (ph == IDLE && r < take) {
                const uint32_t k = waiting - 1u - r;
                const float4 a = ldg(q_o + k), b = ldg(q_d + k), c = ldg(q_t + k);
                put_ray(v3(a), v3(b));
                w[64 * W_PIX] = fbits(a.w); w[64 * W_SMP] = fbits(b.w);
                w[64 * W_AX] = fbits(c.x); w[64 * W_AY] = fbits(c.y); w[64 * W_AZ] = fbits(c.z);
                w[64 * W_CTL] = 0u;
                ph = NEXT;
            }
            waiting -= take;
        }
        if (ph == NEXT) {
            w[64 * W_T] = 0x7f7fffffu; w[64 * W_U] = 0u; w[64 * W_V] = 0u; w[64 * W_PRIM] = CRT_MISS; w[64 * W_KEY] = 0u;
            w[64 * W_NODE] = S.root;
            ph = TRACE;
        }
        const uint32_t live = (uint32_t)__popcll(__ballot(ph == TRACE));
        if (!live) {
            if (mode == SECOND && !waiting && cur >= end && !more) break;
            if (mode == SECOND && !waiting) mode = CAMERA;
            continue;
        }
        if (mode == SECOND && !waiting && (cur < end || more) && live < kDrainLive) mode = DRAIN;
        // in a camera batch or a drain every ray is finished; else until kRefill lanes (or two thirds) are
        const uint32_t leave = mode != SECOND ? 0u : live - min(kRefill, (2u * live + 2u) / 3u);
        bool go = ph == TRACE;
        {
            PathTrav<TL> tr;
            tr.ring = (uint32_t)(uintptr_t)(lds_u32*)(s_stack + lane);
            tr.kring = (uint32_t)(uintptr_t)(lds_u16*)(s_key + lane) - (tr.ring >> 1);
            tr.over = (glb_u32*)gst.base;
            tr.goff = gst.off;
            tr.load(S, w);
            tr.run(S, go, leave);
            bool over = false;
            if (ph == TRACE) {
                tr.store(w);
                over = tr.ovf;
                if (!go) ph = DONE;
            }
            novf += (uint64_t)__popcll(__ballot(over));
        }
    }
    if (lane == 0) {
        atomicAdd(&counters->rays, (unsigned long long)nrays);
        if (nretrace) atomicAdd(&counters->retraces, (unsigned long long)nretrace);
        if (nlight) atomicAdd(&counters->light_tests, (unsigned long long)nlight);
        if (novf) atomicAdd(&counters->stack_overflow, (unsigned long long)novf);
        if (nexact) atomicAdd(&counters->exact, (unsigned long long)nexact);
        if (R.rays) {
            atomicAdd(R.rays, (unsigned long long)(nrays + nretrace));
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

static uint32_t waves_of(uint64_t words, int entries) { return (uint32_t)std::min<uint64_t>(words / (64u * (uint32_t)entries), 1u << 20); }

extern "C" uint32_t crt_k_paths_waves(uint64_t gstack_words) { return waves_of(gstack_words, kOverflow); }

extern "C" int crt_k_paths(hipStream_t s, int rng_mode, int two_level, int shapes, uint32_t nodes, const crt_dev_scene* scenes,
                           const crt_dev_request* reqs, uint32_t nreq, uint32_t total, uint32_t* next, crt_paths queue,
                           uint32_t slots, float4* out_rad, uint32_t* gstack, uint64_t gstack_words, crt_dev_counters* counters) {
    const uint32_t max_waves = crt_k_paths_waves(gstack_words);
    if (total == 0) return 0;
    if (nreq > 1 && (total > CRT_PATHS_MERGE || total > (uint64_t)max_waves * CRT_PATHS_ALIGN)) return (int)hipErrorInvalidValue;
    // waves, and ids of a group and of a hand-out, of a launch that may hold `waves`
    struct Shape { uint32_t waves, group, chunk; };
    auto shape = [&](uint32_t waves) {
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
        return Shape{waves, group, nreq > 1 ? group : c * group};
    };
    auto launch = [&](auto kfn, uint32_t resident) {
        const Shape h = shape(std::min(resident, max_waves));
        hipLaunchKernelGGL(kfn, dim3(h.waves), dim3(64), 0, s, scenes, reqs, nreq, total, h.group, h.chunk, next, out_rad, gstack, counters);
    };
    auto refill = [&](auto kfn, uint32_t resident) {
        const Shape h = shape(std::min(resident, waves_of(gstack_words, kRefillStack)));
        const uint32_t q = std::min(slots / h.waves, std::min(kMaxQueue, std::max(kMinQueue, total / (h.waves * kQueueShare)))) & ~63u;
        if (q < kMinQueue) return false;
        hipLaunchKernelGGL(kfn, dim3(h.waves), dim3(64), 0, s, scenes, reqs, total, h.group, h.chunk, next, queue, q, out_rad, gstack, counters);
        return true;
    };
    if (rng_mode == CRT_RNG_PCG && !two_level && nreq == 1 && nodes >= kRefillNodes && total >= kRefillPaths) {
        bool done;
        if (shapes) { static const uint32_t resident = resident_waves(k_paths_refill<0>); done = refill(k_paths_refill<0>, resident); }
        else { static const uint32_t resident = resident_waves(k_paths_refill<3>); done = refill(k_paths_refill<3>, resident); }
        if (done) return (int)hipGetLastError();
    }
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
