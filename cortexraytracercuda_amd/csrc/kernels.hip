// kernels.hip - gfx950 wavefront path-tracing kernels.
//
// One pass of the hot path (core/src/gpu.cu:761-802 per pixel, core/src/cameras/camera.cuh:149-264
// per bounce) is split into stages that run over every live path of every request in the pass:
//   k_regen     camera rays into free path slots   (render kernel sample loop + get_ray)
//   k_extend    BVH traversal, closest hit          (hittable_list/bvh_node/aabb/primitive ::hit)
//   k_shade     emission, scatter, light mixture    (ray_color body, materials, pdfs, textures)
//               + compaction of the survivors (wave ballot, block prefix scan, one atomic per
//               block) into the other state buffer; finished paths write their radiance by path id
// The stages repeat over a fixed pool of path slots until every path of the pass has finished:
// slots freed by one iteration are refilled with new camera paths by the next, so each launch
// works on a full queue instead of the thinning tail of one generation of paths.
//   k_resolve   per-pixel sums in sample order      (pixel_color += ray_color)
//   k_tonemap   NaN->0, /spp, sqrt, clamp, *255.99  (prepare_pixel_color + quantize)
// MFMA is not used: nothing here is a dense contraction. The traversal is bound by node/primitive
// fetches (HBM / L2 / MALL) and VALU; layouts are SoA float4 so every fetch is a dwordx4.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cortex_rt.h"
#include "crt_device.h"
#include "crt_kernels.h"
#include "crt_layout.h"


// ======================================================================================== kernels

// Streaming pass control block (CRT_CTL_* words, crt_kernels.h): two halves alternate between
// iterations. Iteration k reads half k%2 ("in": survivors left by the previous shade stage, next
// path id to generate) and prepares half (k+1)%2 ("out") for its own shade stage. Live paths are
// kept compact: the shade stage writes survivors to the front of the other state buffer and the
// next regeneration appends new camera paths behind them, so every state access is coalesced.
__global__ void k_pass_init(uint32_t* __restrict__ ctl, uint32_t nwords) {
    for (uint32_t i = threadIdx.x; i < nwords; i += blockDim.x) ctl[i] = 0u;
}

// Regeneration: the slots behind the survivors take the next path ids of the (sub-)pass, whose
// ids are [pid0, pid0 + total) (camera rays, in path-id order: pixel-major within each work item,
// the item's samples of one pixel consecutive). ONE: a closed pass of one request (its record is
// wave-uniform: scalar loads, no search).
template <int MODE, bool ONE>
__global__ __launch_bounds__(256) void k_regen(const crt_dev_request* __restrict__ reqs, int nreq, uint32_t pid0,
                                               uint32_t total, uint32_t nslots, uint32_t* __restrict__ ctl_in,
                                               uint32_t* __restrict__ ctl_out, const uint32_t* __restrict__ open_pass,
                                               crt_paths P) {
    // an open pass (serving) grows while it runs: its path count and request count live in device
    // memory, written by the host between iterations
    if (open_pass) { total = open_pass[0]; nreq = (int)open_pass[1]; }
    const uint32_t surv = ctl_in[CRT_CTL_SURV], g0 = ctl_in[CRT_CTL_GEN];
    const uint32_t n_new = min(nslots - surv, total - g0);
    const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x;
    if (tid == 0) {
        ctl_in[CRT_CTL_LIVE] = surv + n_new;
        ctl_in[CRT_CTL_WORK] = 0u;
        ctl_out[CRT_CTL_GEN] = g0 + n_new;
        ctl_out[CRT_CTL_SURV] = 0u;
    }
    for (uint32_t i = tid; i < n_new; i += gridDim.x * blockDim.x) {
        const uint32_t slot = surv + i, pid = pid0 + g0 + i;
        const int r = ONE ? 0 : find_request(reqs, nreq, pid);
        const crt_dev_request& R = reqs[r];
        uint32_t local = pid - R.path_base;
        // pixel-major: the samples of a pixel are consecutive path ids (a wave traces 64 samples of
        // one pixel at high spp: nearly identical camera rays)
        const uint32_t sidx = local / R.sample_count, k = local - sidx * R.sample_count;
        uint32_t pix = item_pixel(R, sidx);
        uint32_t sample = R.sample_begin + k;
        Rng<MODE> g;
        g.dyn = R.rng_mode;
        g.ms = 0u;
        if (g.minstd()) g.ms = ldg(R.rng_state + pix);
        else g.pcg = pcg_keyed(R.seed, ref_pixel_of(R, pix), sample, 0u);
        V3 o, dir;
        float tm;
        camera_ray<MODE>(R, pix, sample, g, o, dir, tm);
        uint32_t state = (R.max_depth & 0xffu) | ST_CAMERA;
        P.ray_o[slot] = make_float4(o.x, o.y, o.z, tm);
        P.ray_d[slot] = make_float4(dir.x, dir.y, dir.z, bitsf(state));
        P.thr[slot] = make_float4(1.0f, 1.0f, 1.0f, bitsf(g.ms));
        P.rad[slot] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        P.ids[slot] = make_uint2(pix, ((uint32_t)r << 16) | (sample & 0xffffu));
    }
}

// Closest-hit stage over the live path queue.
// UNIFORM: every ray of the launch belongs to scene `uniform_scene` (scene pointers stay scalar).
// Minimum resident blocks per CU the register allocation must allow. Blocks are 256 threads, one
// wave on each of a CU's 4 SIMDs, so this is also waves per SIMD. The traversal is latency-bound and
// occupancy pays more than spills outside the traversal loop, not more than spills inside it
// (measured): the single-scene one-level kernel is held to 6 (80 VGPRs, no spill in the loop); the
// multi-scene one-level kernel, whose scene offsets are per-lane values, to 5 (96 VGPRs: at 6 the
// loop spills, and a 64-scene mixed batch and the saturated serving mix run 9-10 % slower);
// two-level kernels to 5 (96 VGPRs: 6 % faster than at 4; at 6 they spill inside the loop and lose
// 17 %). Counting variants are not bounded.
constexpr int extend_min_waves(bool count, bool uniform, bool two_level) {
    return count ? 1 : (two_level ? 5 : (uniform ? 6 : 5));
}

template <int BLOCK, int RS, int LS, int GS, bool COUNT, bool UNIFORM, int WIDTH, int TL>
__global__ __launch_bounds__(BLOCK, extend_min_waves(COUNT, UNIFORM, TL != 0)) void k_extend(const crt_dev_scene* __restrict__ scenes,
                                                  const crt_dev_request* __restrict__ reqs, uint32_t uniform_scene,
                                                  const uint32_t* __restrict__ queue, const uint32_t* __restrict__ count_ptr,
                                                  uint32_t count_direct, const float4* __restrict__ ray_o,
                                                  const float4* __restrict__ ray_d, const uint2* __restrict__ ids,
                                                  float4* __restrict__ hit, uint32_t* __restrict__ hit_inst,
                                                  uint32_t* __restrict__ gstack, uint32_t* __restrict__ zero_counter,
                                                  uint32_t* __restrict__ work_counter, uint32_t chunk_groups,
                                                  crt_dev_counters* __restrict__ counters) {
    __shared__ uint32_t s_stack[LS * BLOCK];
    if (zero_counter && blockIdx.x == 0 && threadIdx.x == 0) *zero_counter = 0u;
    const uint32_t n = count_ptr ? *count_ptr : count_direct;
    const uint32_t gtid = blockIdx.x * BLOCK + threadIdx.x;
    const uint32_t stride = gridDim.x * BLOCK;
    uint32_t* lds_col = s_stack + threadIdx.x;
    const GSlot gst{gstack, gtid * GS};
    TravCount tc = {0, 0, 0, 0, 0, 0};
    uint32_t nrays = 0, nretrace = 0, novf = 0, nexact = 0;
    SceneView SU;
    if (UNIFORM) SU = scene_view(scenes + uniform_scene);
    auto one_ray = [&](uint32_t i) {
        uint32_t slot = queue ? queue[i] : i;
        float4 ro = ray_o[slot], rdv = ray_d[slot];
        uint32_t state = fbits(rdv.w);
        SceneView S;
        if (UNIFORM) S = SU;
        else S = scene_view(scenes + reqs[ids[slot].y >> 16].scene);
        V3 o = v3(ro), d = v3(rdv);
        bool camera = (state & ST_CAMERA) != 0;
        HitRec h;
        const uint32_t pass_flag = closest_hit_checked<BLOCK, RS, LS, GS, COUNT, WIDTH, TL>(
            S, o, d, camera, lds_col, gst, h, tc, novf, nrays, nretrace, nexact);
        hit[slot] = make_float4(h.t, bitsf(h.prim), h.u, h.v);
        hit_inst[slot] = h.inst | pass_flag;
    };
    if (work_counter) {
        // persistent waves (grid sized to the resident waves): each wave takes the next chunk x 64
        // consecutive rays when all its lanes are done, so no wave idles while another still holds
        // a backlog; the fetch and the exit test are wave-uniform
        const uint32_t lane = threadIdx.x & 63u;
        for (;;) {
            uint32_t base = 0;
            if (lane == 0) base = atomicAdd(work_counter, 64u * chunk_groups);
            base = (uint32_t)__shfl((int)base, 0);
            if (base >= n) break;
            const uint32_t wend = min(base + 64u * chunk_groups, n);
            for (uint32_t i = base + lane; i < wend; i += 64u) one_ray(i);
        }
    } else {
        for (uint32_t i = gtid; i < n; i += stride) one_ray(i);
    }
    wave_add(&counters->rays, nrays);
    wave_add(&counters->retraces, nretrace);
    if (COUNT) {
        wave_add(&counters->node_visits, tc.nodes);
        wave_add(&counters->leaf_visits, tc.leaves);
        wave_add(&counters->tri_tests, tc.tris);
        wave_add(&counters->sphere_tests, tc.spheres);
        wave_add(&counters->quad_tests, tc.quads);
        wave_add(&counters->inst_visits, tc.insts);
    }
    wave_add(&counters->stack_overflow, novf);
    wave_add(&counters->exact, nexact);
}

// Closest-hit stage with per-lane refill for the survivors of the last shade stage: every wave owns
// a contiguous share of them, and a lane whose ray is finished takes the wave's next ray instead of
// waiting for the slowest lane of the wave. A refill is made when at least `refill_min` lanes are
// idle (or all are): the idle lanes take the next rays of the share in lane order (mbcnt rank), so
// refilled rays are neighbours of each other and of the rays in flight. Camera rays (behind the
// survivors when `first_camera` is given) keep whole-wave chunks in grid-stride order, whose
// coherence refills would break. Share and chunk pointers are wave-uniform and private: no atomics.
// A wave leaves when its share and chunks are handed out and its lanes are idle; each traversal
// ends (every node is visited at most once per query, at most one re-trace). Pays when rays of one
// wave differ much in length (many primitive tests per ray, little coherence).
// one-level: 6 (80 VGPRs, a few per-ray spills; 2.5 % faster than at 5); two-level: 5 (96 VGPRs,
// 7 % faster on the instanced scene than unbounded at 4; at 6 the loop spills and it takes 1.6x
// as long)
constexpr int extend_pt_min_waves(bool count, bool uniform, bool two_level, int width) {
    return count ? 1 : (two_level ? 5 : 6);
}

template <int BLOCK, int RS, int LS, int GS, bool COUNT, bool UNIFORM, int WIDTH, int TL>
__global__ __launch_bounds__(BLOCK, extend_pt_min_waves(COUNT, UNIFORM, TL != 0, WIDTH)) void k_extend_pt(const crt_dev_scene* __restrict__ scenes,
                                                     const crt_dev_request* __restrict__ reqs, uint32_t uniform_scene,
                                                     const uint32_t* __restrict__ queue,
                                                     const uint32_t* __restrict__ count_ptr, uint32_t count_direct,
                                                     const float4* __restrict__ ray_o, const float4* __restrict__ ray_d,
                                                     const uint2* __restrict__ ids, float4* __restrict__ hit,
                                                     uint32_t* __restrict__ hit_inst, uint32_t* __restrict__ gstack,
                                                     uint32_t* __restrict__ zero_counter, uint32_t refill_min,
                                                     const uint32_t* __restrict__ first_camera,
                                                     crt_dev_counters* __restrict__ counters) {
    __shared__ uint32_t s_stack[LS * BLOCK];
    if (zero_counter && blockIdx.x == 0 && threadIdx.x == 0) *zero_counter = 0u;
    const uint32_t n = count_ptr ? *count_ptr : count_direct;
    const uint32_t cam0 = first_camera ? *first_camera : n;
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t* lds_col = s_stack + threadIdx.x;
    const GSlot gst{gstack, (blockIdx.x * BLOCK + threadIdx.x) * GS};
    TravCount tc = {0, 0, 0, 0, 0, 0};
    uint32_t nrays = 0, nretrace = 0, novf = 0, nexact = 0;
    SceneView S;
    if (UNIFORM) S = scene_view(scenes + uniform_scene);
    Traverser<BLOCK, RS, LS, GS, COUNT, WIDTH, TL, COUNT> tr;
    bool active = false, exhausted = false;
    uint32_t slot = 0, pass_flag = 0;
    // Survivors of the last shade stage, queue [0, nsec): this wave's contiguous share [nxt, wend),
    // idle lanes refilled as soon as refill_min of them are idle. Camera rays, [nsec, n): chunks of
    // 64 consecutive rays in grid-stride order (chunk c of the wave starts at nsec + (wid + c *
    // nwaves) * 64, so neighbouring waves trace neighbouring pixels, as in the grid-stride
    // kernel), a chunk taken when all 64 lanes are idle.
    const uint32_t nwaves = gridDim.x * (BLOCK / 64);
    const uint32_t wid = blockIdx.x * (BLOCK / 64) + (threadIdx.x >> 6);
    const uint32_t nsec = min(cam0, n);
    const uint32_t share = (nsec + nwaves - 1) / nwaves;
    uint32_t nxt = min(wid * share, nsec);
    const uint32_t wend = min(nxt + share, nsec);
    uint32_t cnext = nsec + wid * 64u;
    const uint32_t cstride = nwaves * 64u;
    bool camera_phase = nxt >= wend;
    for (;;) {
        if (!exhausted) {
            uint64_t idle = __ballot(!active);
            uint32_t cnt = (uint32_t)__popcll(idle);
            uint32_t i = 0xffffffffu, lim = 0u;
            if (camera_phase) {
                if (cnt == 64u) {
                    if (cnext >= n) {
                        exhausted = true;
                    } else {
                        i = cnext + lane;
                        lim = n;
                        cnext += cstride;
                    }
                }
            } else if (cnt >= refill_min || cnt == 64u) {
                const uint32_t base = nxt;
                nxt += cnt;
                if (nxt >= wend) camera_phase = true;
                i = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(idle >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)idle, 0u));
                lim = wend;
            }
            if (!active && i < lim) {
                slot = queue ? queue[i] : i;
                float4 ro = ray_o[slot], rdv = ray_d[slot];
                if (!UNIFORM) S = scene_view(scenes + reqs[ids[slot].y >> 16].scene);
                tr.init(S, v3(ro), v3(rdv), 0.00001f, 3.402823466e+38f, (fbits(rdv.w) & ST_CAMERA) != 0, lds_col, gst);
                pass_flag = 0u;
                active = true;
            }
        }
        if (__ballot(active) == 0ull) {
            if (exhausted) break;
            continue;
        }
        if (active && tr.step(S, tc)) {
            const HitRec h = tr.best;
            novf += tr.st.overflow ? 1u : 0u;
            if (!COUNT && h.t < 0.0f) {
                // undecided triangle test: the lane re-traces the query exactly (rare, divergent)
                const ExactHit e = exact_hit<BLOCK, RS, LS, GS, WIDTH, TL>(S, tr.ow, tr.dw, tr.camera, lds_col, gst);
                novf += e.ovf;
                nrays++;
                if (e.pass_flag) nretrace++;
                ++nexact;
                hit[slot] = make_float4(e.h.t, bitsf(e.h.prim), e.h.u, e.h.v);
                hit_inst[slot] = e.h.inst | e.pass_flag;
                active = false;
                continue;
            }
            // an emitter seen from behind: re-trace from t + 0.001 (camera.cuh:179-183)
            const uint32_t again = pass_flag ? 0u : passes_through(S, h, tr.ow, tr.dw);
            if (again) {
                pass_flag = again;
                tr.init(S, tr.ow, tr.dw, h.t + 0.001f, 3.402823466e+38f, tr.camera, lds_col, gst);
            } else {
                nrays++;
                if (pass_flag) nretrace++;
                hit[slot] = make_float4(h.t, bitsf(h.prim), h.u, h.v);
                hit_inst[slot] = h.inst | pass_flag;
                active = false;
            }
        }
    }
    wave_add(&counters->rays, nrays);
    wave_add(&counters->retraces, nretrace);
    if (COUNT) {
        wave_add(&counters->node_visits, tc.nodes);
        wave_add(&counters->leaf_visits, tc.leaves);
        wave_add(&counters->tri_tests, tc.tris);
        wave_add(&counters->sphere_tests, tc.spheres);
        wave_add(&counters->quad_tests, tc.quads);
        wave_add(&counters->inst_visits, tc.insts);
    }
    wave_add(&counters->stack_overflow, novf);
    wave_add(&counters->exact, nexact);
}

// What a query reports of a hit: the global ids its records carry (the caller's numbering), distance
// and coordinates; prim and inst -1 and zeros where nothing is hit. With the host's walk over the hits
// and its id maps, four pageable copies and an allocation for each buffer of the call, 200,000 rays
// took 1.29 ms; with this 0.50, of which the rays' own way to the device is 0.34.
__device__ __forceinline__ void report_hit(const crt_dev_scene* sc, float4 hv, uint32_t iw, uint64_t i, uint64_t n,
                                           uint32_t* __restrict__ out) {
    const uint32_t p = fbits(hv.y), idx = CRT_HIT_INDEX(p), in = iw & CRT_INST_MASK;
    int32_t gid = -1, inst = -1;
    float t = 0.0f, u = 0.0f, v = 0.0f;
    if (p != CRT_MISS) {
        const uint32_t type = CRT_HIT_TYPE(p);
        gid = (int32_t)fbits(type == CRT_PRIM_TRI ? ldg((const float4*)sc->tris + 3 * (size_t)idx).w
                             : type == CRT_PRIM_SPHERE ? ldg((const float4*)sc->spheres + 2 * (size_t)idx + 1).x
                                                       : ldg((const float4*)sc->quads + 5 * (size_t)idx + 3).w);
        if (in != CRT_NO_INST) inst = (int32_t)fbits(ldg((const float4*)sc->insts + 4 * (size_t)in + 3).y);
        t = hv.x; u = hv.z; v = hv.w;
    }
    out[i] = (uint32_t)gid;
    out[n + i] = (uint32_t)inst;
    out[2 * n + i] = fbits(t);
    out[3 * n + 2 * i] = fbits(u);
    out[3 * n + 2 * i + 1] = fbits(v);
}

// Closest hits of caller rays. Bound by the latency of its traversal steps (200,000 rays: 90 us). Every
// ray takes the exact traversal: the float one with an exact re-trace, as in the closest-hit stage,
// measured 97 us, and 1.45 instead of 1.39 ms for 4M rays.
template <int BLOCK, int RS, int LS, int GS, int WIDTH, int TL>
__global__ __launch_bounds__(BLOCK) void k_trace_rays(const crt_dev_scene* __restrict__ sc, const float4* __restrict__ rays,
                                                      uint32_t n, int camera, uint32_t* __restrict__ out,
                                                      uint32_t* __restrict__ gstack, crt_dev_counters* __restrict__ counters) {
    __shared__ uint32_t s_stack[LS * BLOCK];
    const uint32_t gtid = blockIdx.x * BLOCK + threadIdx.x;
    const uint32_t stride = gridDim.x * BLOCK;
    SceneView S = scene_view(sc);
    TravCount tc = {0, 0, 0, 0, 0, 0};
    uint32_t novf = 0;
    for (uint64_t i = gtid; i < n; i += stride) {
        const float4 a = rays[2 * i], b = rays[2 * i + 1];
        HitRec h;
        bool ovf = false;
        trace<BLOCK, RS, LS, GS, false, WIDTH, TL, true>(S, v3(a), v3(b), a.w, b.w, camera != 0, s_stack + threadIdx.x,
                                                                GSlot{gstack, gtid * GS}, h, tc, ovf);
        novf += ovf ? 1u : 0u;
        report_hit(sc, make_float4(h.t, bitsf(h.prim), h.u, h.v), h.inst, i, n, out);
    }
    wave_add(&counters->stack_overflow, novf);
}

// The same report for hits that the closest-hit stage left.
__global__ __launch_bounds__(256) void k_report_hits(const crt_dev_scene* __restrict__ sc, const float4* __restrict__ hit,
                                                     const uint32_t* __restrict__ hit_inst, uint32_t n, uint32_t* __restrict__ out) {
    for (uint64_t i = blockIdx.x * 256u + threadIdx.x; i < n; i += gridDim.x * 256u) report_hit(sc, hit[i], hit_inst[i], i, n, out);
}

// Shade stage. FLAT (no instanced scene and no scene with analytic shapes among the paths) holds the
// kernel to 6 resident workgroups per CU (80 VGPRs, a few spills outside the hot paths), measured
// 2 % faster per frame on single-level scenes, and leaves the shapes' shading out; with instances
// (transforms, textures) the unbounded kernel is faster.
// ONE: the pass holds a single request, so the request record and its scene's pointers are
// wave-uniform (scalar loads once per wave instead of two dependent vector loads per path).
template <int MODE, int BLOCK, bool FLAT, bool ONE>
__global__ __launch_bounds__(BLOCK, FLAT ? 6 : 1) void k_shade(const crt_dev_scene* __restrict__ scenes,
                                                 const crt_dev_request* __restrict__ reqs,
                                                 const uint32_t* __restrict__ count_in, crt_paths Pin, crt_paths Pout,
                                                 uint32_t* __restrict__ count_out, const float4* __restrict__ hit,
                                                 const uint32_t* __restrict__ hit_inst, float4* __restrict__ out_rad,
                                                 uint32_t* __restrict__ live_min, int sort_octant,
                                                 crt_dev_counters* __restrict__ counters) {
    __shared__ uint32_t s_oct[8 * (BLOCK / 64)];
    __shared__ uint32_t s_base;
    __shared__ uint32_t s_min[BLOCK / 64];
    const uint32_t n = *count_in;
    uint32_t min_pid = 0xffffffffu;   // smallest path id among this thread's surviving paths
    const uint32_t stride = gridDim.x * BLOCK;
    uint32_t light_tests = 0;
    // grid-stride loop with a block-uniform trip count so every thread reaches the block scan
    const uint32_t iters = (n + stride - 1) / stride;
    for (uint32_t it = 0; it < iters; ++it) {
        uint32_t i = it * stride + blockIdx.x * BLOCK + threadIdx.x;
        bool keep = false;
        float4 no, nd, nt, nr;
        uint32_t oct = 0;   // direction octant of the next segment
        uint2 idv = make_uint2(0u, 0u);
        if (i < n) {
            float4 hv = hit[i];
            uint32_t iw = hit_inst[i];
            float4 ro = Pin.ray_o[i], rdv = Pin.ray_d[i];
            float4 tv = Pin.thr[i], rv = Pin.rad[i];
            idv = Pin.ids[i];
            uint32_t state = fbits(rdv.w);
            const uint32_t req = ONE ? 0u : (idv.y >> 16);
            const crt_dev_request& R = reqs[req];
            const crt_dev_scene* sc = scenes + R.scene;
            V3 o = v3(ro), d = v3(rdv);
            V3 att = v3(tv), L = v3(rv);
            uint32_t pix = idv.x, sample = idv.y & 0xffffu;
            uint32_t depth = ST_DEPTH(state), bounce = ST_BOUNCE(state);
            // closest-hit queries of this segment beyond the first: the pass-through re-trace
            const uint32_t retraces = ST_RETRACES(state) + ((iw & CRT_PASSTHROUGH) ? 1u : 0u);
            Rng<MODE> g;
            g.ms = fbits(tv.w);
            g.dyn = R.rng_mode;
            keep = shade_hit<MODE, !FLAT>(sc, R, pix, sample, hv, iw, o, d, att, L, depth, bounce, g, light_tests);
            if (keep) {
                min_pid = min(min_pid, R.path_base + (pix - R.pix_begin) * R.sample_count + (sample - R.sample_begin));
                uint32_t ns = (depth & 0xffu) | ((bounce & 0xffu) << 8) | (retraces << 24);
                no = make_float4(o.x, o.y, o.z, ro.w);
                nd = make_float4(d.x, d.y, d.z, bitsf(ns));
                nt = make_float4(att.x, att.y, att.z, bitsf(g.ms));
                nr = make_float4(L.x, L.y, L.z, 0.0f);
                oct = (d.x < 0.0f ? 1u : 0u) | (d.y < 0.0f ? 2u : 0u) | (d.z < 0.0f ? 4u : 0u);
            } else {
                // finished: the radiance goes to the path's id, with the path's closest-hit queries
                // (one per hit, the final miss and every pass-through re-trace) in .w for the
                // per-request ray count
                uint32_t pid = R.path_base + (pix - R.pix_begin) * R.sample_count + (sample - R.sample_begin);
                const uint32_t rays = bounce + (fbits(hv.y) == CRT_MISS ? 1u : 0u) + retraces;
                out_rad[pid] = make_float4(L.x, L.y, L.z, (float)rays);
                if (g.minstd()) stg(R.rng_state + pix, g.ms);
            }
        }
        // survivors go to the front of the other state buffer (grouped by direction octant when
        // sort_octant is set; a launch-uniform choice)
        uint32_t pos = sort_octant ? block_append_sorted<BLOCK>(keep, oct, count_out, s_oct, &s_base)
                                   : block_append<BLOCK>(keep, count_out, s_oct, &s_base);
        if (keep) {
            Pout.ray_o[pos] = no;
            Pout.ray_d[pos] = nd;
            Pout.thr[pos] = nt;
            Pout.rad[pos] = nr;
            Pout.ids[pos] = idv;
        }
    }
    if (live_min) {
        // per block: the smallest live path id after this stage (0xffffffff: none). Every path id
        // below both this minimum over all blocks and the generated count has finished, which is
        // how the serving loop knows a request-table entry is complete (no per-path counters).
        uint32_t m = min_pid;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) m = min(m, (uint32_t)__shfl_xor((int)m, off));
        if ((threadIdx.x & 63u) == 0u) s_min[threadIdx.x >> 6] = m;
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t b = s_min[0];
            for (int w = 1; w < BLOCK / 64; ++w) b = min(b, s_min[w]);
            live_min[blockIdx.x] = b;
        }
    }
    wave_add(&counters->light_tests, light_tests);
}

// One-render-per-launch path tracer, the reference's render kernel design (core/src/gpu.cu:756-801):
// each thread owns pixels, runs their samples in order and follows every path to its end, tracing
// and shading in one kernel. Same estimator, streams and per-pixel float sums as the wavefront
// pipeline, so the images agree; it serves as the plain baseline the batched passes are measured
// against. Grid-stride over the request's pixel range.
template <int MODE, int BLOCK, int RS, int LS, int GS, int WIDTH, int TL>
__global__ __launch_bounds__(BLOCK) void k_plain(const crt_dev_scene* __restrict__ scenes,
                                                 const crt_dev_request* __restrict__ req, uint32_t* __restrict__ gstack,
                                                 crt_dev_counters* __restrict__ counters) {
    __shared__ uint32_t s_stack[LS * BLOCK];
    const crt_dev_request& R = *req;
    const crt_dev_scene* sc = scenes + R.scene;
    const SceneView S = scene_view(sc);
    const uint32_t gtid = blockIdx.x * BLOCK + threadIdx.x;
    const uint32_t stride = gridDim.x * BLOCK;
    uint32_t* lds_col = s_stack + threadIdx.x;
    const GSlot gst{gstack, gtid * GS};
    TravCount tc = {0, 0, 0, 0, 0, 0};
    uint32_t nrays = 0, nretrace = 0, novf = 0, light_tests = 0, nexact = 0;
    float4* accum = (float4*)R.accum;
    for (uint32_t q = gtid; q < R.pix_count; q += stride) {
        uint32_t pix = R.pix_begin + q;
        float4 acc = ldg(accum + pix);
        Rng<MODE> g;
        g.dyn = R.rng_mode;
        g.ms = 0u;
        if (g.minstd()) g.ms = ldg(R.rng_state + pix);
        const uint32_t refp = ref_pixel_of(R, pix);
        for (uint32_t k = 0; k < R.sample_count; ++k) {
            uint32_t sample = R.sample_begin + k;
            if (!g.minstd()) g.pcg = pcg_keyed(R.seed, refp, sample, 0u);
            V3 o, d;
            float tm;
            camera_ray<MODE>(R, pix, sample, g, o, d, tm);
            V3 att = v3(1.0f, 1.0f, 1.0f), L = v3(0.0f, 0.0f, 0.0f);
            uint32_t depth = R.max_depth & 0xffu, bounce = 0u;
            bool camera = true;
            for (;;) {
                HitRec h;
                const uint32_t pf = closest_hit_checked<BLOCK, RS, LS, GS, false, WIDTH, TL>(
                    S, o, d, camera, lds_col, gst, h, tc, novf, nrays, nretrace, nexact);
                camera = false;
                float4 hv = make_float4(h.t, bitsf(h.prim), h.u, h.v);
                if (!shade_hit<MODE, true>(sc, R, pix, sample, hv, h.inst | pf, o, d, att, L, depth, bounce, g, light_tests))
                    break;
            }
            acc.x += L.x; acc.y += L.y; acc.z += L.z;
        }
        acc.w += (float)R.sample_count;
        stg(accum + pix, acc);
        if (g.minstd()) stg(R.rng_state + pix, g.ms);
    }
    wave_add(&counters->rays, nrays);
    wave_add(&counters->retraces, nretrace);
    wave_add(&counters->light_tests, light_tests);
    wave_add(&counters->stack_overflow, novf);
    wave_add(&counters->exact, nexact);
}

// Per-pixel sums in sample order: accum += rad[sample 0] + ... (same float additions as the
// reference's pixel_color += ray_color(...) loop, core/src/gpu.cu:776-790). With `rays` set (one
// request), the paths' closest-hit queries (rad.w) are added to *rays: one atomic per wave.
// A pixel's samples are consecutive in rad, so a block stages 256 pixels x 8 samples at a time
// through LDS: the global loads are whole 128-byte lines (8 lanes per pixel) instead of one
// float4 per lane at a 16*spp-byte stride, and each lane still adds its pixel's samples in order.
constexpr uint32_t kResolveChunk = 8;
__global__ __launch_bounds__(256) void k_resolve(const crt_dev_request* __restrict__ reqs, int nreq,
                                                 const float4* __restrict__ rad, unsigned long long* __restrict__ rays) {
    __shared__ float4 stage[256 * (kResolveChunk + 1)];
    int r = blockIdx.y;
    if (r >= nreq) return;
    const crt_dev_request& R = reqs[r];
    const uint32_t S = R.sample_count;
    uint32_t nr = 0;
    // block-uniform trip counts: every lane reaches each barrier and the wave sum
    const uint32_t stride = gridDim.x * 256u;
    const uint32_t iters = (R.pix_count + stride - 1) / stride;
    for (uint32_t it = 0; it < iters; ++it) {
        const uint32_t q0 = it * stride + blockIdx.x * 256u;
        const uint32_t np = R.pix_count > q0 ? min(256u, R.pix_count - q0) : 0u;
        const uint32_t t = threadIdx.x;
        float4* a = (float4*)R.accum + R.pix_begin + q0 + t;
        float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (t < np) acc = ldg(a);
        const float4* src = rad + R.path_base + q0 * S;
        for (uint32_t k0 = 0; k0 < S; k0 += kResolveChunk) {
            const uint32_t n = min(kResolveChunk, S - k0);
            const uint32_t total = np * n;
            for (uint32_t e = t; e < total; e += 256u) {
                const uint32_t pl = (n == kResolveChunk) ? (e >> 3) : e / n;
                const uint32_t j = e - pl * n;
                stage[pl * (kResolveChunk + 1) + j] = src[pl * S + k0 + j];
            }
            __syncthreads();
            if (t < np) {
                const float4* row = stage + t * (kResolveChunk + 1);
                for (uint32_t j = 0; j < n; ++j) {
                    const float4 v = row[j];
                    acc.x += v.x; acc.y += v.y; acc.z += v.z;
                    nr += (uint32_t)v.w;
                }
            }
            __syncthreads();
        }
        if (t < np) {
            acc.w += (float)S;
            stg(a, acc);
        }
    }
    if (rays) wave_add(rays, nr);
}

// prepare_pixel_color + quantize (core/src/misc/color.cuh:289-309, core/src/gpu.cu:792-799).
__global__ __launch_bounds__(256) void k_tonemap(const float4* __restrict__ accum, uint32_t npix, uint32_t spp,
                                                 uint8_t* __restrict__ rgb) {
    uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npix) return;
    float4 a = accum[p];
    float c[3] = {a.x, a.y, a.z};
    for (int k = 0; k < 3; ++k) {
        float x = c[k];
        x = (x != x) ? 0.0f : x;
        if (spp > 0u) { float scale = 1.0f / (float)spp; x *= scale; }
        x = sqrtf(x);
        float cl = x < 0.0f ? 0.0f : (x > 0.999f ? 0.999f : x);
        rgb[3 * p + k] = (uint8_t)(int)(255.99f * cl);
    }
}

// Start of a request: zero its accumulation buffer and seed the per-pixel minstd engines with
// seed + reference pixel index (core/src/gpu.cu:770), Thrust's seed() rule (s mod m, 0 -> 1).
__global__ __launch_bounds__(256) void k_init_request(float4* __restrict__ accum, uint32_t* __restrict__ rng_state,
                                                      uint32_t W, uint32_t H, uint64_t seed) {
    uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= W * H) return;
    accum[p] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (rng_state) {
        uint32_t jj = p / W, i = p - jj * W;
        uint32_t ref_pixel = (H - 1u - jj) * W + i;
        uint64_t s = (seed + ref_pixel) & 0xffffffffull;
        uint32_t x = (uint32_t)(s % 2147483647ull);
        rng_state[p] = x == 0u ? 1u : x;
    }
}

__global__ void k_fill_u32(uint32_t* __restrict__ p, uint32_t n, uint32_t v) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// VALU issue-rate calibration: each lane runs `iters` rounds of 16 independent dependency chains
// of one instruction (KIND 0: v_fma_f32, 1: v_add_u32, 2: v_mul_f32), 16 wave instructions per
// round and wave, and writes its chains' sum so that none is removed. b and c come from the
// arguments, so nothing folds. KIND 3-7 run the v_fma_f32 rounds on part of each wave: lanes 0-15
// (one 16-lane group), every fourth lane (16 lanes over all four groups), lanes 0-31, lanes 0-62
// and lanes 0-47, which tells how a wave instruction's issue time depends on its active lanes.
// KIND 8 issues the 16 v_fma_f32 of a round with EXEC cleared (saved and restored inside one asm
// block, which touches no memory): what an instruction of a branch that no lane of the wave takes
// costs when the compiler does not jump around it. KIND 9-12 issue other instructions the traversal
// is made of, 16 per round: v_cndmask_b32 (selects of the child sort), v_max_f32 (slab tests),
// v_cmp_lt_f32 (compares into a lane mask) and v_mov_b32; KIND 13 the select in its three-operand
// form with the mask in an SGPR pair instead of VCC. KIND 14 and 15 issue the KIND 8 block with EXEC
// set to lanes 0-15 and to lanes 0-31 inside the asm block (every lane of the wave alive).
template <int KIND>
__global__ __launch_bounds__(256) void k_valu_probe(uint32_t iters, float b, float c, float* __restrict__ out) {
    const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t lane = threadIdx.x & 63u;
    if ((KIND == 3 && lane >= 16u) || (KIND == 4 && (lane & 3u) != 0u) || (KIND == 5 && lane >= 32u) ||
        (KIND == 6 && lane == 63u) || (KIND == 7 && lane >= 48u)) {
        out[tid] = 0.0f;
        return;
    }
    if (KIND >= 9) {
        float a0 = (float)tid * 1e-7f, a1 = a0 + 1.0f, a2 = a0 + 2.0f, a3 = a0 + 3.0f;
        for (uint32_t i = 0; i < iters; ++i) {
            uint64_t m0, m1;
            if (KIND == 9)
                asm volatile(
                    "v_cmp_lt_f32 vcc, %[a0], %[a1]\n\t"
                    "v_cndmask_b32 %[a0], %[a0], %[a1], vcc\n\tv_cndmask_b32 %[a1], %[a1], %[a2], vcc\n\t"
                    "v_cndmask_b32 %[a2], %[a2], %[a3], vcc\n\tv_cndmask_b32 %[a3], %[a3], %[a0], vcc\n\t"
                    "v_cndmask_b32 %[a0], %[a0], %[a1], vcc\n\tv_cndmask_b32 %[a1], %[a1], %[a2], vcc\n\t"
                    "v_cndmask_b32 %[a2], %[a2], %[a3], vcc\n\tv_cndmask_b32 %[a3], %[a3], %[a0], vcc\n\t"
                    "v_cndmask_b32 %[a0], %[a0], %[a1], vcc\n\tv_cndmask_b32 %[a1], %[a1], %[a2], vcc\n\t"
                    "v_cndmask_b32 %[a2], %[a2], %[a3], vcc\n\tv_cndmask_b32 %[a3], %[a3], %[a0], vcc\n\t"
                    "v_cndmask_b32 %[a0], %[a0], %[a1], vcc\n\tv_cndmask_b32 %[a1], %[a1], %[a2], vcc\n\t"
                    "v_cndmask_b32 %[a2], %[a2], %[a3], vcc"
                    : [a0] "+v"(a0), [a1] "+v"(a1), [a2] "+v"(a2), [a3] "+v"(a3) : : "vcc");
            else if (KIND == 10)
                asm volatile(
                    "v_max_f32 %[a0], %[a0], %[a1]\n\tv_max_f32 %[a1], %[a1], %[a2]\n\t"
                    "v_max_f32 %[a2], %[a2], %[a3]\n\tv_max_f32 %[a3], %[a3], %[a0]\n\t"
                    "v_max_f32 %[a0], %[a0], %[a1]\n\tv_max_f32 %[a1], %[a1], %[a2]\n\t"
                    "v_max_f32 %[a2], %[a2], %[a3]\n\tv_max_f32 %[a3], %[a3], %[a0]\n\t"
                    "v_max_f32 %[a0], %[a0], %[a1]\n\tv_max_f32 %[a1], %[a1], %[a2]\n\t"
                    "v_max_f32 %[a2], %[a2], %[a3]\n\tv_max_f32 %[a3], %[a3], %[a0]\n\t"
                    "v_max_f32 %[a0], %[a0], %[a1]\n\tv_max_f32 %[a1], %[a1], %[a2]\n\t"
                    "v_max_f32 %[a2], %[a2], %[a3]\n\tv_max_f32 %[a3], %[a3], %[a0]"
                    : [a0] "+v"(a0), [a1] "+v"(a1), [a2] "+v"(a2), [a3] "+v"(a3));
            else if (KIND == 13)
                asm volatile(
                    "v_cmp_lt_f32 %[m0], %[a0], %[a1]\n\t"
                    "v_cndmask_b32_e64 %[a0], %[a0], %[a1], %[m0]\n\tv_cndmask_b32_e64 %[a1], %[a1], %[a2], %[m0]\n\t"
                    "v_cndmask_b32_e64 %[a2], %[a2], %[a3], %[m0]\n\tv_cndmask_b32_e64 %[a3], %[a3], %[a0], %[m0]\n\t"
                    "v_cndmask_b32_e64 %[a0], %[a0], %[a1], %[m0]\n\tv_cndmask_b32_e64 %[a1], %[a1], %[a2], %[m0]\n\t"
                    "v_cndmask_b32_e64 %[a2], %[a2], %[a3], %[m0]\n\tv_cndmask_b32_e64 %[a3], %[a3], %[a0], %[m0]\n\t"
                    "v_cndmask_b32_e64 %[a0], %[a0], %[a1], %[m0]\n\tv_cndmask_b32_e64 %[a1], %[a1], %[a2], %[m0]\n\t"
                    "v_cndmask_b32_e64 %[a2], %[a2], %[a3], %[m0]\n\tv_cndmask_b32_e64 %[a3], %[a3], %[a0], %[m0]\n\t"
                    "v_cndmask_b32_e64 %[a0], %[a0], %[a1], %[m0]\n\tv_cndmask_b32_e64 %[a1], %[a1], %[a2], %[m0]\n\t"
                    "v_cndmask_b32_e64 %[a2], %[a2], %[a3], %[m0]"
                    : [a0] "+v"(a0), [a1] "+v"(a1), [a2] "+v"(a2), [a3] "+v"(a3), [m0] "=&s"(m0));
            else if (KIND == 11)
                asm volatile(
                    "v_cmp_lt_f32 %[m0], %[a0], %[a1]\n\tv_cmp_lt_f32 %[m1], %[a1], %[a2]\n\t"
                    "v_cmp_lt_f32 %[m0], %[a2], %[a3]\n\tv_cmp_lt_f32 %[m1], %[a3], %[a0]\n\t"
                    "v_cmp_lt_f32 %[m0], %[a0], %[a2]\n\tv_cmp_lt_f32 %[m1], %[a1], %[a3]\n\t"
                    "v_cmp_lt_f32 %[m0], %[a2], %[a0]\n\tv_cmp_lt_f32 %[m1], %[a3], %[a1]\n\t"
                    "v_cmp_lt_f32 %[m0], %[a0], %[a1]\n\tv_cmp_lt_f32 %[m1], %[a1], %[a2]\n\t"
                    "v_cmp_lt_f32 %[m0], %[a2], %[a3]\n\tv_cmp_lt_f32 %[m1], %[a3], %[a0]\n\t"
                    "v_cmp_lt_f32 %[m0], %[a0], %[a2]\n\tv_cmp_lt_f32 %[m1], %[a1], %[a3]\n\t"
                    "v_cmp_lt_f32 %[m0], %[a2], %[a0]\n\tv_cmp_lt_f32 %[m1], %[a3], %[a1]"
                    : [m0] "=&s"(m0), [m1] "=&s"(m1) : [a0] "v"(a0), [a1] "v"(a1), [a2] "v"(a2), [a3] "v"(a3));
            else
                asm volatile(
                    "v_mov_b32 %[a0], %[a1]\n\tv_mov_b32 %[a1], %[a2]\n\tv_mov_b32 %[a2], %[a3]\n\tv_mov_b32 %[a3], %[a0]\n\t"
                    "v_mov_b32 %[a0], %[a1]\n\tv_mov_b32 %[a1], %[a2]\n\tv_mov_b32 %[a2], %[a3]\n\tv_mov_b32 %[a3], %[a0]\n\t"
                    "v_mov_b32 %[a0], %[a1]\n\tv_mov_b32 %[a1], %[a2]\n\tv_mov_b32 %[a2], %[a3]\n\tv_mov_b32 %[a3], %[a0]\n\t"
                    "v_mov_b32 %[a0], %[a1]\n\tv_mov_b32 %[a1], %[a2]\n\tv_mov_b32 %[a2], %[a3]\n\tv_mov_b32 %[a3], %[a0]"
                    : [a0] "+v"(a0), [a1] "+v"(a1), [a2] "+v"(a2), [a3] "+v"(a3));
            if (KIND == 11) a0 += (float)(uint32_t)(m0 ^ m1) * 0.0f;
            (void)m1;
        }
        out[tid] = a0 + a1 + a2 + a3;
        return;
    }
    if (KIND == 14 || KIND == 15) {
        float a0 = (float)tid * 1e-7f, a1 = a0 + 1.0f, a2 = a0 + 2.0f, a3 = a0 + 3.0f;
        const uint64_t em = KIND == 14 ? 0xffffull : 0xffffffffull;
        for (uint32_t i = 0; i < iters; ++i) {
            uint64_t sv;
            asm volatile(
                "s_mov_b64 %[sv], exec\n\t"
                "s_mov_b64 exec, %[em]\n\t"
                "v_fma_f32 %[a0], %[b], %[a0], %[c]\n\tv_fma_f32 %[a1], %[b], %[a1], %[c]\n\t"
                "v_fma_f32 %[a2], %[b], %[a2], %[c]\n\tv_fma_f32 %[a3], %[b], %[a3], %[c]\n\t"
                "v_fma_f32 %[a0], %[b], %[a0], %[c]\n\tv_fma_f32 %[a1], %[b], %[a1], %[c]\n\t"
                "v_fma_f32 %[a2], %[b], %[a2], %[c]\n\tv_fma_f32 %[a3], %[b], %[a3], %[c]\n\t"
                "v_fma_f32 %[a0], %[b], %[a0], %[c]\n\tv_fma_f32 %[a1], %[b], %[a1], %[c]\n\t"
                "v_fma_f32 %[a2], %[b], %[a2], %[c]\n\tv_fma_f32 %[a3], %[b], %[a3], %[c]\n\t"
                "v_fma_f32 %[a0], %[b], %[a0], %[c]\n\tv_fma_f32 %[a1], %[b], %[a1], %[c]\n\t"
                "v_fma_f32 %[a2], %[b], %[a2], %[c]\n\tv_fma_f32 %[a3], %[b], %[a3], %[c]\n\t"
                "s_mov_b64 exec, %[sv]"
                : [a0] "+v"(a0), [a1] "+v"(a1), [a2] "+v"(a2), [a3] "+v"(a3), [sv] "=&s"(sv)
                : [b] "s"(b), [c] "v"(c), [em] "s"(em));
        }
        out[tid] = a0 + a1 + a2 + a3;
        return;
    }
    if (KIND == 8) {
        float a0 = (float)tid * 1e-7f, a1 = a0 + 1.0f, a2 = a0 + 2.0f, a3 = a0 + 3.0f;
        for (uint32_t i = 0; i < iters; ++i) {
            uint64_t sv;
            asm volatile(
                "s_mov_b64 %[sv], exec\n\t"
                "s_mov_b64 exec, 0\n\t"
                "v_fma_f32 %[a0], %[b], %[a0], %[c]\n\tv_fma_f32 %[a1], %[b], %[a1], %[c]\n\t"
                "v_fma_f32 %[a2], %[b], %[a2], %[c]\n\tv_fma_f32 %[a3], %[b], %[a3], %[c]\n\t"
                "v_fma_f32 %[a0], %[b], %[a0], %[c]\n\tv_fma_f32 %[a1], %[b], %[a1], %[c]\n\t"
                "v_fma_f32 %[a2], %[b], %[a2], %[c]\n\tv_fma_f32 %[a3], %[b], %[a3], %[c]\n\t"
                "v_fma_f32 %[a0], %[b], %[a0], %[c]\n\tv_fma_f32 %[a1], %[b], %[a1], %[c]\n\t"
                "v_fma_f32 %[a2], %[b], %[a2], %[c]\n\tv_fma_f32 %[a3], %[b], %[a3], %[c]\n\t"
                "v_fma_f32 %[a0], %[b], %[a0], %[c]\n\tv_fma_f32 %[a1], %[b], %[a1], %[c]\n\t"
                "v_fma_f32 %[a2], %[b], %[a2], %[c]\n\tv_fma_f32 %[a3], %[b], %[a3], %[c]\n\t"
                "s_mov_b64 exec, %[sv]"
                : [a0] "+v"(a0), [a1] "+v"(a1), [a2] "+v"(a2), [a3] "+v"(a3), [sv] "=&s"(sv)
                : [b] "s"(b), [c] "v"(c));
        }
        out[tid] = a0 + a1 + a2 + a3;
        return;
    }
    if (KIND == 1) {
        uint32_t a[16];
        const uint32_t ib = __float_as_uint(b) | 1u;
#pragma unroll
        for (int k = 0; k < 16; ++k) a[k] = tid + (uint32_t)k;
        for (uint32_t i = 0; i < iters; ++i) {
#pragma unroll
            for (int k = 0; k < 16; ++k) a[k] = a[k] + ib;
        }
        uint32_t s = 0;
#pragma unroll
        for (int k = 0; k < 16; ++k) s ^= a[k];
        out[tid] = (float)s;
    } else {
        float a[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) a[k] = (float)(tid + (uint32_t)k) * 1e-7f;
        for (uint32_t i = 0; i < iters; ++i) {
#pragma unroll
            for (int k = 0; k < 16; ++k) a[k] = KIND == 2 ? a[k] * b : __builtin_fmaf(a[k], b, c);
        }
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < 16; ++k) s += a[k];
        out[tid] = s;
    }
}

// ======================================================================================== launchers
#define STK_RS 1
#define STK_LS 16
#define STK_GS 96

extern "C" int crt_k_pass_init(hipStream_t s, uint32_t* ctl, uint32_t nwords) {
    hipLaunchKernelGGL(k_pass_init, dim3(1), dim3(64), 0, s, ctl, nwords);
    return (int)hipGetLastError();
}

extern "C" int crt_k_regen(hipStream_t s, int rng_mode, uint32_t grid, const crt_dev_request* reqs, int nreq,
                           uint32_t pid0, uint32_t total, uint32_t nslots, uint32_t* ctl_in, uint32_t* ctl_out,
                           const uint32_t* open_pass, crt_paths P) {
#define CRT_RG1(M, O)                                                                                                \
    hipLaunchKernelGGL((k_regen<M, O>), dim3(grid), dim3(256), 0, s, reqs, nreq, pid0, total, nslots, ctl_in, ctl_out, \
                       open_pass, P)
#define CRT_RG(M) { if (nreq == 1 && !open_pass) CRT_RG1(M, true); else CRT_RG1(M, false); }
    if (rng_mode == CRT_RNG_MINSTD) CRT_RG(CRT_RNG_MINSTD)
    else if (rng_mode == CRT_RNG_PCG) CRT_RG(CRT_RNG_PCG)
    else CRT_RG(CRT_RNG_DYNAMIC)
#undef CRT_RG
#undef CRT_RG1
    return (int)hipGetLastError();
}

// Resident blocks of one kernel on this device (per-CU occupancy x CUs).
template <typename K> static uint32_t resident_blocks(K kernel, int block) {
    int nb = 0, dev = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, block, 0) != hipSuccess || nb <= 0) nb = 1;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus <= 0)
        cus = 256;
    return (uint32_t)(nb * cus);
}

extern "C" int crt_k_extend(hipStream_t s, int count_mode, int width, int two_level, uint32_t grid,
                            const crt_dev_scene* scenes, const crt_dev_request* reqs, int32_t uniform_scene,
                            const uint32_t* queue, const uint32_t* count_ptr, uint32_t count_direct, const float4* ray_o,
                            const float4* ray_d, const uint2* ids, float4* hit, uint32_t* hit_inst, uint32_t* gstack,
                            uint32_t* zero_counter, int mode, uint32_t* work_counter, uint32_t param, int stack_lds,
                            const uint32_t* first_camera, crt_dev_counters* counters) {
    uint32_t us = uniform_scene >= 0 ? (uint32_t)uniform_scene : 0u;
    if (mode != CRT_EXTEND_WAVE_CHUNK) work_counter = nullptr;
    if (mode == CRT_EXTEND_WAVE_CHUNK && !work_counter) mode = CRT_EXTEND_GRID_STRIDE;
    // grid-stride / wave-chunk kernel with an LDS stack ring of LSV entries per lane
#define CRT_EXT_GS(LSV, C, U, W, T)                                                                                    \
    {                                                                                                                   \
        auto kfn = k_extend<256, STK_RS, LSV, STK_GS, C, U, W, T>;                                                     \
        static uint32_t rb = 0;                                                                                         \
        if (!rb) rb = resident_blocks(kfn, 256);                                                                        \
        uint32_t g = (mode == CRT_EXTEND_WAVE_CHUNK && grid > rb) ? rb : grid;                                          \
        hipLaunchKernelGGL(kfn, dim3(g), dim3(256), 0, s, scenes, reqs, us, queue, count_ptr, count_direct, ray_o,     \
                           ray_d, ids, hit, hit_inst, gstack, zero_counter, work_counter, param ? param : 1u,         \
                           counters);                                                                                   \
    }
    // lane-refill kernel over per-wave shares of the queue (same grid as the grid-stride kernel)
#define CRT_EXT_PT(C, U, W, T)                                                                                         \
    {                                                                                                                   \
        auto kfn = k_extend_pt<256, STK_RS, STK_LS, STK_GS, C, U, W, T>;                                               \
        hipLaunchKernelGGL(kfn, dim3(grid), dim3(256), 0, s, scenes, reqs, us, queue, count_ptr, count_direct, ray_o,  \
                           ray_d, ids, hit, hit_inst, gstack, zero_counter, param ? param : 1u, first_camera,       \
                           counters);                                                                                   \
    }
    // counting variants: one stack depth; timed variants: LDS ring of 8, 16 or 32 entries per lane
#define CRT_EXT_C(U, W, T) \
    if (mode == CRT_EXTEND_PERSISTENT) CRT_EXT_PT(true, U, W, T) else CRT_EXT_GS(STK_LS, true, U, W, T)
#define CRT_EXT_N(U, W, T)                                                     \
    if (mode == CRT_EXTEND_PERSISTENT) CRT_EXT_PT(false, U, W, T)              \
    else if (stack_lds == 8) CRT_EXT_GS(8, false, U, W, T)                     \
    else if (stack_lds == 32) CRT_EXT_GS(32, false, U, W, T)                   \
    else CRT_EXT_GS(STK_LS, false, U, W, T)
#define CRT_EXT_WT(X, U)                                                                     \
    if (width == 2) { if (two_level == 2) { X(U, 2, 2) } else if (two_level) { X(U, 2, 1) } else { X(U, 2, 0) } } \
    else { if (two_level == 2) { X(U, 4, 2) } else if (two_level) { X(U, 4, 1) } else { X(U, 4, 0) } }
    if (count_mode) {
        if (uniform_scene >= 0) { CRT_EXT_WT(CRT_EXT_C, true) } else { CRT_EXT_WT(CRT_EXT_C, false) }
    } else {
        if (uniform_scene >= 0) { CRT_EXT_WT(CRT_EXT_N, true) } else { CRT_EXT_WT(CRT_EXT_N, false) }
    }
#undef CRT_EXT_WT
#undef CRT_EXT_N
#undef CRT_EXT_C
#undef CRT_EXT_PT
#undef CRT_EXT_GS
    return (int)hipGetLastError();
}

extern "C" int crt_k_shade(hipStream_t s, int rng_mode, int full, uint32_t grid, const crt_dev_scene* scenes,
                           const crt_dev_request* reqs, const uint32_t* count_in, crt_paths Pin, crt_paths Pout,
                           uint32_t* count_out, const float4* hit, const uint32_t* hit_inst, float4* out_rad,
                           uint32_t* live_min, int sort_octant, int one_request, crt_dev_counters* counters) {
#define CRT_SH(M, F, O)                                                                                                   \
    hipLaunchKernelGGL((k_shade<M, 256, F, O>), dim3(grid), dim3(256), 0, s, scenes, reqs, count_in, Pin, Pout,         \
                       count_out, hit, hit_inst, out_rad, live_min, sort_octant, counters)
#define CRT_SH_O(M, F) { if (one_request) CRT_SH(M, F, true); else CRT_SH(M, F, false); }
#define CRT_SH_F(M) { if (full) CRT_SH_O(M, false) else CRT_SH_O(M, true) }
    if (rng_mode == CRT_RNG_MINSTD) CRT_SH_F(CRT_RNG_MINSTD)
    else if (rng_mode == CRT_RNG_PCG) CRT_SH_F(CRT_RNG_PCG)
    else CRT_SH_F(CRT_RNG_DYNAMIC)
#undef CRT_SH_F
#undef CRT_SH_O
#undef CRT_SH
    return (int)hipGetLastError();
}

extern "C" int crt_k_trace_rays(hipStream_t s, int width, int two_level, uint32_t grid, const crt_dev_scene* sc,
                                const float4* rays, uint32_t n, int camera, uint32_t* out, uint32_t* gstack,
                                crt_dev_counters* counters) {
#define CRT_TR(W, T)                                                                                              \
    hipLaunchKernelGGL((k_trace_rays<256, STK_RS, STK_LS, STK_GS, W, T>), dim3(grid), dim3(256), 0, s, sc, rays, n, \
                       camera, out, gstack, counters)
    if (width == 2) { if (two_level == 2) CRT_TR(2, 2); else if (two_level) CRT_TR(2, 1); else CRT_TR(2, 0); }
    else { if (two_level == 2) CRT_TR(4, 2); else if (two_level) CRT_TR(4, 1); else CRT_TR(4, 0); }
#undef CRT_TR
    return (int)hipGetLastError();
}

extern "C" int crt_k_report_hits(hipStream_t s, uint32_t grid, const crt_dev_scene* sc, const float4* hit, const uint32_t* hit_inst,
                                 uint32_t n, uint32_t* out) {
    hipLaunchKernelGGL(k_report_hits, dim3(grid), dim3(256), 0, s, sc, hit, hit_inst, n, out);
    return (int)hipGetLastError();
}

extern "C" int crt_k_plain(hipStream_t s, int rng_mode, int width, int two_level, uint32_t grid,
                           const crt_dev_scene* scenes, const crt_dev_request* req, uint32_t* gstack,
                           crt_dev_counters* counters) {
#define CRT_PL(M, W, T)                                                                                          \
    hipLaunchKernelGGL((k_plain<M, 256, STK_RS, STK_LS, STK_GS, W, T>), dim3(grid), dim3(256), 0, s, scenes, req, \
                       gstack, counters)
#define CRT_PL_WT(M)                                                              \
    if (width == 2) { if (two_level == 2) CRT_PL(M, 2, 2); else if (two_level) CRT_PL(M, 2, 1); else CRT_PL(M, 2, 0); } \
    else { if (two_level == 2) CRT_PL(M, 4, 2); else if (two_level) CRT_PL(M, 4, 1); else CRT_PL(M, 4, 0); }
    if (rng_mode == CRT_RNG_MINSTD) { CRT_PL_WT(CRT_RNG_MINSTD) } else { CRT_PL_WT(CRT_RNG_PCG) }
#undef CRT_PL_WT
#undef CRT_PL
    return (int)hipGetLastError();
}

extern "C" int crt_k_resolve(hipStream_t s, const crt_dev_request* reqs, int nreq, uint32_t max_pix, const float4* rad,
                             unsigned long long* rays) {
    if (nreq == 0) return 0;
    uint32_t gx = (max_pix + 255) / 256;
    if (gx > 4096) gx = 4096;
    if (gx == 0) gx = 1;
    hipLaunchKernelGGL(k_resolve, dim3(gx, nreq), dim3(256), 0, s, reqs, nreq, rad, nreq == 1 ? rays : nullptr);
    return (int)hipGetLastError();
}

extern "C" int crt_k_tonemap(hipStream_t s, const float4* accum, uint32_t npix, uint32_t spp, uint8_t* rgb) {
    if (npix == 0) return 0;
    hipLaunchKernelGGL(k_tonemap, dim3((npix + 255) / 256), dim3(256), 0, s, accum, npix, spp, rgb);
    return (int)hipGetLastError();
}

extern "C" int crt_k_init_request(hipStream_t s, float4* accum, uint32_t* rng_state, uint32_t W, uint32_t H, uint64_t seed) {
    uint32_t n = W * H;
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_init_request, dim3((n + 255) / 256), dim3(256), 0, s, accum, rng_state, W, H, seed);
    return (int)hipGetLastError();
}

extern "C" int crt_k_fill_u32(hipStream_t s, uint32_t* p, uint32_t n, uint32_t v) {
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_fill_u32, dim3((n + 255) / 256), dim3(256), 0, s, p, n, v);
    return (int)hipGetLastError();
}

extern "C" int crt_k_valu_probe(hipStream_t s, int kind, uint32_t blocks, uint32_t iters, float* out) {
    if (kind == 0) hipLaunchKernelGGL(k_valu_probe<0>, dim3(blocks), dim3(256), 0, s, iters, 0.999f, 1e-6f, out);
    else if (kind == 1) hipLaunchKernelGGL(k_valu_probe<1>, dim3(blocks), dim3(256), 0, s, iters, 0.999f, 1e-6f, out);
    else if (kind == 2) hipLaunchKernelGGL(k_valu_probe<2>, dim3(blocks), dim3(256), 0, s, iters, 0.999f, 1e-6f, out);
    else if (kind == 3) hipLaunchKernelGGL(k_valu_probe<3>, dim3(blocks), dim3(256), 0, s, iters, 0.999f, 1e-6f, out);
    else if (kind == 4) hipLaunchKernelGGL(k_valu_probe<4>, dim3(blocks), dim3(256), 0, s, iters, 0.999f, 1e-6f, out);
    else if (kind == 5) hipLaunchKernelGGL(k_valu_probe<5>, dim3(blocks), dim3(256), 0, s, iters, 0.999f, 1e-6f, out);
    else if (kind == 6) hipLaunchKernelGGL(k_valu_probe<6>, dim3(blocks), dim3(256), 0, s, iters, 0.999f, 1e-6f, out);
    else if (kind == 7) hipLaunchKernelGGL(k_valu_probe<7>, dim3(blocks), dim3(256), 0, s, iters, 0.999f, 1e-6f, out);
    else if (kind == 8) hipLaunchKernelGGL(k_valu_probe<8>, dim3(blocks), dim3(256), 0, s, iters, 0.999f, 1e-6f, out);
    else if (kind == 9) hipLaunchKernelGGL(k_valu_probe<9>, dim3(blocks), dim3(256), 0, s, iters, 0.999f, 1e-6f, out);
    else if (kind == 10) hipLaunchKernelGGL(k_valu_probe<10>, dim3(blocks), dim3(256), 0, s, iters, 0.999f, 1e-6f, out);
    else if (kind == 11) hipLaunchKernelGGL(k_valu_probe<11>, dim3(blocks), dim3(256), 0, s, iters, 0.999f, 1e-6f, out);
    else if (kind == 12) hipLaunchKernelGGL(k_valu_probe<12>, dim3(blocks), dim3(256), 0, s, iters, 0.999f, 1e-6f, out);
    else if (kind == 13) hipLaunchKernelGGL(k_valu_probe<13>, dim3(blocks), dim3(256), 0, s, iters, 0.999f, 1e-6f, out);
    else if (kind == 14) hipLaunchKernelGGL(k_valu_probe<14>, dim3(blocks), dim3(256), 0, s, iters, 0.999f, 1e-6f, out);
    else hipLaunchKernelGGL(k_valu_probe<15>, dim3(blocks), dim3(256), 0, s, iters, 0.999f, 1e-6f, out);
    return (int)hipGetLastError();
}

extern "C" uint32_t crt_k_stack_capacity(void) { return STK_RS + STK_LS + STK_GS; }
extern "C" uint32_t crt_k_gstack_entries(void) { return STK_GS; }
