// Wavefront form of the plain path tracer (gfx950).
//
// The reference integrator (intergrators/PathTracingIntegrator.cuh:38-104 with estimateDirect,
// IntegratorHelper.cuh:51-125) is cut at its three ray casts:
//   extend   closest hit of every live path ray                     (persistent)
//   shade    (by default in material order within chunks of the queue) emission, BSDF, light sample + MIS-BSDF
//            sample (NEE set-up), continuation, roulette; appends one shadow ray and one MIS ray per path at
//            most; first completes the paths that ended at the bounce before
//   shadow   any hit of the shadow rays                             (persistent, in extend's launch)
//   mis      whether an MIS-BSDF ray reaches its light              (persistent, in extend's launch)
//   finalize L += beta * ((Ld_light + Ld_bsdf) / p_pick), the reference's order of additions, for the paths that
//            ended at the last bounce
// Each path's arithmetic is that of whole paths (paths.hip), so the image does not depend on queue order or form.
// Every count lives in device memory and is reset by kernels, so the bounce loop of a pass is
// captured once in a hipGraph and replayed.
#include <algorithm>

#include "path_order.h"
#include "pt_device.h"

namespace lts {

namespace {

constexpr int kShadeBlock = 256;

// Training paths of the radiance cache: in scene 0, every trainStride-th (sample, pixel) pair of
// the pass in sample-major, row-major order from trainOffset, so that the set and its slot order
// do not depend on the order in which the pass walks its pixels (tileRows); the slot, or -1.
LTS_D int train_slot(const WfParams& P, const WfSceneSlot& sl, int scene, int pixel, int sample) {
    if (P.trainSlots > 0 && scene == 0) {
        const long c = (long)(sample - sl.s0) * ((long)sl.width * sl.height) + pixel;
        if (c >= P.trainOffset) {
            const long d = c - P.trainOffset;
            if (d % P.trainStride == 0 && d / P.trainStride < P.trainSlots) return (int)(d / P.trainStride);
        }
    }
    return -1;
}

// The camera rays of the pass. The path records are not written here: at bounce 0 every field
// follows from the path index, and the first shading builds them.
__global__ __launch_bounds__(256) void k_wf_generate(const SceneView* __restrict__ scenes, const WfParams* __restrict__ prm,
                                                     const WfSceneSlot* __restrict__ slots, WfRay* __restrict__ rays,
                                                     int32_t* __restrict__ counts, WfTrainRec* __restrict__ tRec) {
    const WfParams P = *prm;
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i == 0) counts[0] = (int)P.nPaths;  // bounce 0 has every path of the pass, in order (no queue)
    for (long k = i; k < P.nPaths; k += (long)gridDim.x * 256) {
        int sc, pixel, sample;
        path_origin(P, slots, k, sc, pixel, sample);
        const SceneView& sv = scenes[sc];
        const WfSceneSlot& sl = slots[sc];
        const int px = pixel % sv.cam.width, py = pixel / sv.cam.width;
        const Ray cr = camera_ray(sv, camera_sample(sv, px, py, sample, sl.spp, sl.stratified, sl.seed));
        const int ts = train_slot(P, sl, sc, pixel, sample);
        if (ts >= 0)
            for (int b = 0; b < P.maxBounce; b++) tRec[(size_t)ts * kWfMaxBounce + b].valid = 0;
        WfRay r;
        r.o[0] = cr.o.x; r.o[1] = cr.o.y; r.o[2] = cr.o.z;
        r.d[0] = cr.d.x; r.d[1] = cr.d.y; r.d[2] = cr.d.z;
        r.scene = sc; r.pad = 0;
        rays[k] = r;
    }
}

// Rank of each lane among the lanes of its wave holding the same bin (bin < 0: none), offset by
// the running count h[bin], which grows by the number of such lanes (one LDS atomic per bin).
LTS_D int wave_bin_rank(int bin, int32_t* h) {
    const int lane = threadIdx.x & 63;
    const uint64_t below = lane ? ~0ull >> (64 - lane) : 0ull;
    int slot = 0;
    uint64_t todo = __ballot(bin >= 0);
    while (todo) {
        const int leader = __ffsll((unsigned long long)todo) - 1;
        const int b = __shfl(bin, leader);
        const uint64_t peers = __ballot(bin == b);
        int base = 0;
        if (lane == leader) base = atomicAdd(&h[b], (int)__popcll(peers));
        base = __shfl(base, leader);
        if (bin == b) slot = base + (int)__popcll(peers & below);
        todo &= ~peers;
    }
    return slot;
}

LTS_D float clamp01(float x) { return fminf(fmaxf(x, 0.0f), 1.0f); }

// The cache's 16-float record of a shading point (layout in include/lts.h, lts_nrc_config).
LTS_D void nrc_raw_record(const SurfacePoint& si, const Bsdf& bsdf, const WfSceneSlot& sl, float* __restrict__ o) {
    const V3 wo = si.wo, n = faceTowards(si.sn, si.wo);
    const bool glossy = bsdf.kind == 4;
    float4 r0, r1, r2, r3;
    r0.x = clamp01((si.p.x - sl.boxMin[0]) * sl.boxInv[0]);
    r0.y = clamp01((si.p.y - sl.boxMin[1]) * sl.boxInv[1]);
    r0.z = clamp01((si.p.z - sl.boxMin[2]) * sl.boxInv[2]);
    r0.w = acosf(fminf(fmaxf(wo.z, -1.0f), 1.0f)) * INV_PI_F;
    r1.x = atan2f(wo.y, wo.x) * (0.5f * INV_PI_F) + 0.5f;
    r1.y = acosf(fminf(fmaxf(n.z, -1.0f), 1.0f)) * INV_PI_F;
    r1.z = atan2f(n.y, n.x) * (0.5f * INV_PI_F) + 0.5f;
    r1.w = glossy ? fminf(bsdf.alpha, 1.0f) : 1.0f;
    r2.x = glossy ? 0.0f : bsdf.R.r;
    r2.y = glossy ? 0.0f : bsdf.R.g;
    r2.z = glossy ? 0.0f : bsdf.R.b;
    r2.w = glossy ? bsdf.R.r : 0.0f;
    r3.x = glossy ? bsdf.R.g : 0.0f;
    r3.y = glossy ? bsdf.R.b : 0.0f;
    r3.z = r3.w = 0.0f;
    float4* q = reinterpret_cast<float4*>(o);
    q[0] = r0; q[1] = r1; q[2] = r2; q[3] = r3;
}

// The traced light sample of a path that ended with one in flight completes its radiance (a continuing
// path takes its sample at the start of the next bounce's shading).
LTS_D void finalize_path(const WfParams& P, const WfSceneSlot* slots, const WfPath* paths, const WfNee* nee, int pi) {
    const WfPath p = paths[pi];
    const WfNee ne = nee[pi];
    Spec L = spec(p.L[0], p.L[1], p.L[2]);
    Spec Ld = spec(ne.p1[0], ne.p1[1], ne.p1[2]) + spec(ne.p2[0], ne.p2[1], ne.p2[2]);
    L = L + spec(ne.nb[0], ne.nb[1], ne.nb[2]) * (Ld / ne.lpdf);
    const WfSceneSlot& sl = slots[path_scene(P, slots, pi)];
    const int sample = (int)(p.sampleFlags >> kWfFlagBits);
    float* o = sl.sampleL + 3 * ((size_t)(sample - sl.s0) * sl.width * sl.height + p.pixel);
    o[0] = L.r; o[1] = L.g; o[2] = L.b;
}

// One shading kernel per (integrator, first bounce or not), so that each carries only its own code
// and registers: the radiance cache's records, and the camera-ray differentials of bounce 0. It first
// completes the paths that ended at the previous bounce (prevDone).
//
// Material order. A block takes chunks of up to kSortChunk paths from the bounce's work counter and
// orders each by the material bin the trace filed (bins; null: queue order) in LDS, so that most waves
// shade one material. A chunk is 64-path pieces at equal strides over the queue: every chunk holds
// about the pass's mix of materials and costs about the same (chunks of neighbouring paths are all
// sky or all marble, and the last ones kept the launch waiting: 23.5 ms instead of 20.8 for the
// shading of a 64-spp 1920x1080 frame of the 1M-triangle displaced sphere), and the waves of the
// resident blocks work on neighbouring pieces. That frame with chunks of 256/512/1024/2048/4096
// paths: 58.0/53.0/51.8/51.7/52.1 ms; a count, scan and scatter of the whole queue before the
// shading: 54.5 ms. Small launches halve the chunk until every resident block has kChunksPerBlock
// (a 256x256 4-spp frame: 2.38 ms with 1 chunk a block, 2.29 with 2, 2.26 with 4).
constexpr int kSortChunk = 1024, kChunksPerBlock = 4;
constexpr int kShadeGrid = 3 * 256;  // the workgroups resident at once: 3 of 4 waves on each of 256 CUs

// queue position of item x of chunk c
__device__ __forceinline__ int chunk_item(int x, int c, int chunks) { return ((x >> 6) * chunks + c) * 64 + (x & 63); }

constexpr int kSortItemsPerThread = kSortChunk / kShadeBlock;

template <bool kCached, bool kFirst>
__global__ __launch_bounds__(kShadeBlock, 3) void k_wf_shade(const SceneView* __restrict__ scenes, const WfParams* __restrict__ prm,
                                                          const WfSceneSlot* __restrict__ slots, int bounce,
                                                          WfPath* __restrict__ paths, WfRay* __restrict__ rays,
                                                          const WfHit* __restrict__ hits, WfNee* __restrict__ nee,
                                                          const int32_t* __restrict__ queue, const int32_t* __restrict__ count,
                                                          const uint8_t* __restrict__ bins,
                                                          const int32_t* __restrict__ prevDone, const int32_t* __restrict__ prevDoneCount,
                                                          int32_t* __restrict__ work,
                                                          int32_t* __restrict__ nextQueue, int32_t* __restrict__ nextCount,
                                                          WfLightRay* __restrict__ shadows, int32_t* __restrict__ shadowCount,
                                                          WfLightRay* __restrict__ misRays, int32_t* __restrict__ misCount,
                                                          float* __restrict__ qRaw, NrcQuery* __restrict__ qMeta,
                                                          int32_t* __restrict__ qCount,
                                                          WfTrainRec* __restrict__ tRec, float* __restrict__ tRaw,
                                                          int32_t* __restrict__ doneQueue, int32_t* __restrict__ doneCount,
                                                          int32_t* __restrict__ shadowQueue, int32_t* __restrict__ misQueue) {
    const int n = *count;
    const int maxBounce = prm->maxBounce, rrStart = prm->rrStart, queryBounce = prm->queryBounce;
    constexpr bool cached = kCached;
    __shared__ NoiseTables perm;  // every scene view points at its context's one permutation
    __shared__ int32_t appendLds[2][5 * (kShadeBlock / 64) + 5];
    // a query's raw record (4 float4) and its NrcQuery (3 float4), held by the thread that makes it
    // until the round's append gives the query its compact slot
    constexpr int kStage = 7;
    __shared__ float4 qStage[kCached ? kShadeBlock * kStage : 1];
    __shared__ int32_t nextChunk;
    __shared__ int32_t order[kSortChunk], binCount[kWfMaxMatBins], binBase[kWfMaxMatBins];
    noise_tables(perm, scenes[0].perm, threadIdx.x, kShadeBlock);
    if (!kFirst) {
        const int nDone = *prevDoneCount;
        const WfParams P = *prm;
        for (int k = blockIdx.x * kShadeBlock + threadIdx.x; k < nDone; k += gridDim.x * kShadeBlock)
            finalize_path(P, slots, paths, nee, prevDone[k]);
    }
    int per = kSortChunk;  // paths of a chunk
    while (per > kShadeBlock && (long)per * gridDim.x * kChunksPerBlock > n) per >>= 1;
    const int chunks = (n + per - 1) / per;
    __syncthreads();
    int turn = 0;
    while (true) {
        if (threadIdx.x == 0) nextChunk = atomicAdd(work, 1);
        __syncthreads();  // also: the previous chunk's order has been read
        const int c = __builtin_amdgcn_readfirstlane(nextChunk);
        if (c >= chunks) break;
        int m = 0;
        if (bins) {
            // counting sort of the chunk: ranks within each bin, then the bins' starts
            int pis[kSortItemsPerThread], slots_[kSortItemsPerThread], bin[kSortItemsPerThread];
            if (threadIdx.x < kWfMaxMatBins) binCount[threadIdx.x] = 0;
            __syncthreads();
#pragma unroll
            for (int j = 0; j < kSortItemsPerThread; j++) {
                const int x = j * kShadeBlock + threadIdx.x;
                const int k = chunk_item(x, c, chunks);
                pis[j] = x < per && k < n ? (kFirst ? k : queue[k]) : -1;
                bin[j] = pis[j] >= 0 ? (int)bins[pis[j]] : -1;
                slots_[j] = wave_bin_rank(bin[j], binCount);
            }
            __syncthreads();
            if (threadIdx.x < kWfMaxMatBins) {
                const int c = binCount[threadIdx.x];
                int x = c;
#pragma unroll
                for (int o = 1; o < kWfMaxMatBins; o <<= 1) {
                    const int y = __shfl_up(x, o);
                    if ((int)threadIdx.x >= o) x += y;
                }
                binBase[threadIdx.x] = x - c;
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < kSortItemsPerThread; j++)
                if (pis[j] >= 0) order[binBase[bin[j]] + slots_[j]] = pis[j];
            __syncthreads();
            m = binBase[kWfMaxMatBins - 1] + binCount[kWfMaxMatBins - 1];
        }
        for (int sub = 0; sub < (bins ? m : per); sub += kShadeBlock, turn++) {
            const int x = sub + threadIdx.x;
            const int k = chunk_item(x, c, chunks);
            const bool active = bins ? x < m : k < n;
            const int pi = !active ? 0 : bins ? order[x] : kFirst ? k : queue[k];
            bool wantShadow = false, wantMis = false, wantNext = false, wantQuery = false, wantDone = false;
            if (active) {
                const WfParams P = *prm;
                WfPath p;
                int scene, pixel, sample, pflags;
                if (kFirst) {
                    // bounce 0: the path record follows from the path index
                    p.beta[0] = p.beta[1] = p.beta[2] = 1.0f;
                    p.L[0] = p.L[1] = p.L[2] = 0.0f;
                    path_origin(P, slots, pi, scene, pixel, sample);
                    pflags = kWfAlive;
                } else {
                    p = paths[pi];
                    scene = path_scene(P, slots, pi);
                    pixel = p.pixel;
                    sample = (int)(p.sampleFlags >> kWfFlagBits);
                    pflags = (int)(p.sampleFlags & ((1u << kWfFlagBits) - 1));
                }
                const WfHit hh = hits[pi];
                const SceneView& sv = scenes[scene];
                const WfSceneSlot& sl = slots[scene];
                const int trainSlot = cached ? train_slot(P, sl, scene, pixel, sample) : -1;
                Ray r;
                CameraSample cam;
                if (kFirst) {
                    // the camera ray, drawn again as the generate kernel drew it (a path that escapes has no
                    // need of it)
                    if (hh.leaf >= 0) {
                        cam = camera_sample(sv, pixel % sv.cam.width, pixel / sv.cam.width, sample, sl.spp, sl.stratified, sl.seed);
                        r = camera_ray(sv, cam);
                    }
                } else {
                    const WfRay rr = rays[pi];
                    r.o = v3(rr.o[0], rr.o[1], rr.o[2]);
                    r.d = v3(rr.d[0], rr.d[1], rr.d[2]);
                }
                r.tMax = INFINITY;
                Spec L = spec(p.L[0], p.L[1], p.L[2]), beta = spec(p.beta[0], p.beta[1], p.beta[2]);
                if (!kFirst) {
                    // the light sample of the previous vertex, traced since: added before anything of
                    // this vertex, as the reference's loop adds it before the next intersection
                    const WfNee pn = nee[pi];
                    if (pn.used) {
                        Spec Ld = spec(pn.p1[0], pn.p1[1], pn.p1[2]) + spec(pn.p2[0], pn.p2[1], pn.p2[2]);
                        L = L + spec(pn.nb[0], pn.nb[1], pn.nb[2]) * (Ld / pn.lpdf);
                    }
                }
                const bool specularBounce = (pflags & kWfSpecular) != 0;
                WfNee ne;
                ne.used = 0;
                ne.p1[0] = ne.p1[1] = ne.p1[2] = 0.0f;
                ne.p2[0] = ne.p2[1] = ne.p2[2] = 0.0f;
                bool alive = true;
                if (kFirst || specularBounce) add_emission(sv, hh.leaf, r, hh.u, hh.v, hh.invDet, beta, L);
                if (hh.leaf < 0) {
                    alive = false;
                } else {
                    SurfacePoint si = make_surface(sv, hh.leaf, r, hh.u, hh.v, hh.invDet);
                    if (kFirst) camera_footprint(sv, si, cam, sl.spp, r, hh.invDet);
                    Bsdf bsdf = make_bsdf(sv, si, perm);
                    const int slot = (sample - sl.s0) * sl.width * sl.height + pixel;  // sample index of the path
                    if (cached && (bsdf.kind == 0 || bsdf.kind == 1 || bsdf.kind == 4)) {
                        if (trainSlot >= 0) {
                            // training vertex: radiance so far and throughput, for the suffix target
                            const size_t r = (size_t)trainSlot * kWfMaxBounce + bounce;
                            nrc_raw_record(si, bsdf, sl, tRaw + 16 * r);
                            WfTrainRec tr;
                            tr.Lb[0] = L.r; tr.Lb[1] = L.g; tr.Lb[2] = L.b;
                            tr.beta[0] = beta.r; tr.beta[1] = beta.g; tr.beta[2] = beta.b;
                            tr.a[0] = bsdf.R.r; tr.a[1] = bsdf.R.g; tr.a[2] = bsdf.R.b;
                            tr.slot = slot; tr.valid = 1; tr.pad = 0;
                            tRec[r] = tr;
                        } else if (bounce >= queryBounce) {
                            // the cache stands for all radiance scattered here
                            nrc_raw_record(si, bsdf, sl, reinterpret_cast<float*>(&qStage[kStage * threadIdx.x]));
                            NrcQuery q;
                            q.beta[0] = beta.r; q.beta[1] = beta.g; q.beta[2] = beta.b;
                            q.a[0] = bsdf.R.r; q.a[1] = bsdf.R.g; q.a[2] = bsdf.R.b;
                            q.L[0] = q.L[1] = q.L[2] = 0.0f;  // set where the path ends, below
                            q.slot = slot; q.pad[0] = q.pad[1] = 0;
                            *reinterpret_cast<NrcQuery*>(&qStage[kStage * threadIdx.x + 4]) = q;
                            wantQuery = true;
                            alive = false;
                        }
                    }
                    Sampler smp;
                    smp.seed = sl.seed; smp.pixel = (uint32_t)pixel; smp.sample = (uint32_t)sample;
                    float u0[4], u1[4];
                    smp.block(1 + 2 * bounce, u0);
                    smp.block(2 + 2 * bounce, u1);
                    if (!wantQuery && sv.nLights > 0) {
                        float lpdf;
                        const int li = sample_light(sv, u0[0], &lpdf);
                        ne.used = 1;
                        ne.nb[0] = beta.r; ne.nb[1] = beta.g; ne.nb[2] = beta.b;
                        ne.lpdf = lpdf;
                        // the records are per path; the queues below list the paths
                        auto record = [&](V3 o, V3 d, Spec c, float tMax, int tieLeaf) {
                            WfLightRay q;
                            q.o[0] = o.x; q.o[1] = o.y; q.o[2] = o.z;
                            q.d[0] = d.x; q.d[1] = d.y; q.d[2] = d.z;
                            q.scene = scene; q.tieLeaf = tieLeaf; q.tMax = tMax;
                            q.c[0] = c.r; q.c[1] = c.g; q.c[2] = c.b;
                            return q;
                        };
                        light_rays(sv, si, bsdf, li, u0, u1, specularBounce,
                                   [&](V3 o, V3 d, Spec c) { shadows[pi] = record(o, d, c, 1 - SHADOW_EPS, -1); wantShadow = true; },
                                   [&](V3 o, V3 d, float tMax, int tieLeaf, Spec c) { misRays[pi] = record(o, d, c, tMax, tieLeaf); wantMis = true; });
                    }
                    // continuation (PathTracingIntegrator.cuh:79-103)
                    V3 wo = -r.d, wi;
                    float pdf;
                    int flags = 0;
                    Spec f = wantQuery ? spec(0.0f) : bsdf.sampleF(wo, &wi, v2(u1[1], u1[2]), &pdf, B_ALL, &flags);
                    if (wantQuery || isBlack(f) || pdf == 0) {
                        alive = false;
                    } else {
                        pflags = (flags & B_SPEC) ? (pflags | kWfSpecular) : (pflags & ~kWfSpecular);
                        beta = beta * (f * absDot(wi, si.sn) / pdf);
                        Ray nr = spawn_ray(si, wi);
                        WfRay o;
                        o.o[0] = nr.o.x; o.o[1] = nr.o.y; o.o[2] = nr.o.z;
                        o.d[0] = wi.x; o.d[1] = wi.y; o.d[2] = wi.z;
                        o.scene = scene; o.pad = 0;
                        rays[pi] = o;
                        if (bounce >= rrStart) {
                            float q = fmaxf(0.05f, 1 - lum(beta));
                            if (u1[3] < q) alive = false;
                            else beta = beta / (1 - q);
                        }
                    }
                }
                p.L[0] = L.r; p.L[1] = L.g; p.L[2] = L.b;
                p.beta[0] = beta.r; p.beta[1] = beta.g; p.beta[2] = beta.b;
                if (!alive) pflags &= ~kWfAlive;
                p.pixel = pixel;
                p.sampleFlags = ((uint32_t)sample << kWfFlagBits) | (uint32_t)pflags;
                wantNext = alive && bounce + 1 < maxBounce;
                // the records are read again only by the next shading or by finalize
                if (wantNext || ne.used) {
                    paths[pi] = p;
                    nee[pi] = ne;
                }
                if (!wantNext) {
                    // the path ends here: its sample is final now, or once its light sample is traced
                    if (ne.used) {
                        wantDone = true;
                    } else if (cached && wantQuery) {
                        // the sample is written by inference: L plus the cache's estimate
                        NrcQuery* q = reinterpret_cast<NrcQuery*>(&qStage[kStage * threadIdx.x + 4]);
                        q->L[0] = L.r; q->L[1] = L.g; q->L[2] = L.b;
                    } else {
                        float* o = sl.sampleL + 3 * ((size_t)(sample - sl.s0) * sl.width * sl.height + pixel);
                        o[0] = L.r; o[1] = L.g; o[2] = L.b;
                    }
                }
            }
            // The round's appends, aggregated per block: each wave files its counts in LDS, one lane per
            // queue reserves the block's range with a single device atomic (one per wave on a handful of
            // shared counters serialised), and every lane writes at its offset. The buffers alternate
            // between rounds so that one barrier pair per round suffices.
            constexpr int kQueues = 5, kWaves = kShadeBlock / 64;
            const bool want[kQueues] = {wantShadow, wantMis, wantNext, wantDone, cached && wantQuery};
            int32_t* const counter[kQueues] = {shadowCount, misCount, nextCount, doneCount, qCount};
            int32_t* const lds = appendLds[turn & 1];
            const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
            const uint64_t below = lane ? ~0ull >> (64 - lane) : 0ull;
            uint64_t mask[kQueues];
#pragma unroll
            for (int q = 0; q < kQueues; q++) {
                mask[q] = __ballot(want[q]);
                if (lane == 0) lds[q * kWaves + wave] = (int)__popcll(mask[q]);
            }
            __syncthreads();
            if (threadIdx.x < kQueues && (threadIdx.x < 4 || cached)) {
                const int q = threadIdx.x;
                int run = 0;
                for (int w = 0; w < kWaves; w++) { const int c = lds[q * kWaves + w]; lds[q * kWaves + w] = run; run += c; }
                lds[kQueues * kWaves + q] = run ? atomicAdd(counter[q], run) : 0;
            }
            __syncthreads();
            int32_t* const out[kQueues - 1] = {shadowQueue, misQueue, nextQueue, doneQueue};
#pragma unroll
            for (int q = 0; q < kQueues - 1; q++)
                if (want[q]) out[q][lds[kQueues * kWaves + q] + lds[q * kWaves + wave] + (int)__popcll(mask[q] & below)] = pi;
            if (cached && want[4]) {
                // queries are stored compactly in append order, so inference reads them in sequence
                const size_t at = (size_t)(lds[kQueues * kWaves + 4] + lds[4 * kWaves + wave] + (int)__popcll(mask[4] & below));
                float4* r = reinterpret_cast<float4*>(qRaw + 16 * at);
#pragma unroll
                for (int j = 0; j < 4; j++) r[j] = qStage[kStage * threadIdx.x + j];
                float4* m = reinterpret_cast<float4*>(qMeta + at);
#pragma unroll
                for (int j = 0; j < 3; j++) m[j] = qStage[kStage * threadIdx.x + 4 + j];
            }
        }
    }
}

// Builds the training batch from this pass's training records in record order, so the batch and
// the step that follows are deterministic: (1) each block counts the valid records of its 2048,
// (2) one block turns the counts into block offsets, (3) each block writes its records at its
// offset plus an in-block prefix. A record contributes its raw encoding input and the suffix target
// (L_final - Lb) / beta / a per channel (0 where beta or a is 0).
constexpr int kCollectPerThread = 8;
constexpr int kCollectBlock = 256;
constexpr int kCollectPerBlock = kCollectPerThread * kCollectBlock;

LTS_D size_t train_record(int i, int maxBounce) { return (size_t)(i / maxBounce) * kWfMaxBounce + (i % maxBounce); }

// Block-wide exclusive prefix of v (256 threads); total receives the block sum.
LTS_D int block_prefix(int v, int* sh, int& total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int x = v;
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) sh[wave] = x;
    __syncthreads();
    int waveBase = 0;
    for (int w = 0; w < wave; w++) waveBase += sh[w];
    total = sh[0] + sh[1] + sh[2] + sh[3];
    __syncthreads();
    return waveBase + x - v;
}

// Whether the records i0 + 256 j + thread of a block are valid, one bit for each j. Neighbouring threads read
// neighbouring records (eight consecutive ones each made the scatter take 69 us instead of 44, of 8
// bounces of 262144 paths).
LTS_D int valid_records(const WfTrainRec* __restrict__ tRec, int i0, int nRec, int maxBounce) {
    int bits = 0;
#pragma unroll
    for (int j = 0; j < kCollectPerThread; j++) {
        const int i = i0 + j * kCollectBlock + threadIdx.x;
        if (i < nRec && tRec[train_record(i, maxBounce)].valid) bits |= 1 << j;
    }
    return bits;
}

__global__ __launch_bounds__(kCollectBlock) void k_wf_nrc_count(const WfParams* __restrict__ prm, const WfTrainRec* __restrict__ tRec,
                                                                int32_t* __restrict__ blockCount) {
    __shared__ int sh[4];
    const int maxBounce = prm->maxBounce, nRec = prm->trainSlots * maxBounce;
    int total;
    block_prefix(__popc(valid_records(tRec, blockIdx.x * kCollectPerBlock, nRec, maxBounce)), sh, total);
    if (threadIdx.x == 0) blockCount[blockIdx.x] = total;
}

// One wave, 64 blocks at a time (one after the other by a single thread: 94 us for 1024 blocks).
__global__ __launch_bounds__(64) void k_wf_nrc_scan(int32_t* __restrict__ blockCount, int nBlocks, int cap,
                                                    NrcState* __restrict__ state) {
    const int lane = threadIdx.x;
    int run = 0;
    for (int b = 0; b < nBlocks; b += 64) {
        const int c = b + lane < nBlocks ? blockCount[b + lane] : 0;
        int x = c;
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(x, o);
            if (lane >= o) x += y;
        }
        if (b + lane < nBlocks) blockCount[b + lane] = run + x - c;
        run += __shfl(x, 63);
    }
    if (lane == 0) state->nTotal = min(run, cap);
}

__global__ __launch_bounds__(kCollectBlock) void k_wf_nrc_scatter(const WfParams* __restrict__ prm, const WfTrainRec* __restrict__ tRec,
                                                                  const float* __restrict__ tRaw, const float* __restrict__ sampleBase,
                                                                  const int32_t* __restrict__ blockBase, int batchCap,
                                                                  float* __restrict__ outRaw, float* __restrict__ outTarget) {
    constexpr int kWaves = kCollectBlock / 64;
    __shared__ int count[kCollectPerThread * kWaves];
    const int maxBounce = prm->maxBounce, nRec = prm->trainSlots * maxBounce;
    const int i0 = blockIdx.x * kCollectPerBlock, wave = threadIdx.x >> 6;
    const int bits = valid_records(tRec, i0, nRec, maxBounce);
#pragma unroll
    for (int j = 0; j < kCollectPerThread; j++) {
        const unsigned long long m = __ballot(bits >> j & 1);
        if ((threadIdx.x & 63) == 0) count[j * kWaves + wave] = (int)__popcll(m);
    }
    __syncthreads();
    int base = blockBase[blockIdx.x];  // of the records before those of this j and wave
    for (int j = 0, k = 0; j < kCollectPerThread; j++) {
        for (; k < j * kWaves + wave; k++) base += count[k];
        const bool valid = bits >> j & 1;
        const int pos = base + lanes_below(__ballot(valid));
        if (!valid || pos >= batchCap) continue;
        const size_t r = train_record(i0 + j * kCollectBlock + threadIdx.x, maxBounce);
        const WfTrainRec t = tRec[r];
        const float* Lf = sampleBase + 3 * (size_t)t.slot;
        for (int ch = 0; ch < 3; ch++) {
            const float suffix = t.beta[ch] > 0.0f ? (Lf[ch] - t.Lb[ch]) / t.beta[ch] : 0.0f;
            outTarget[3 * (size_t)pos + ch] = t.a[ch] > 0.0f ? suffix / t.a[ch] : 0.0f;
        }
        const float4* src = reinterpret_cast<const float4*>(tRaw + 16 * r);
        float4* dst = reinterpret_cast<float4*>(outRaw + 16 * (size_t)pos);
        dst[0] = src[0]; dst[1] = src[1]; dst[2] = src[2]; dst[3] = src[3];
    }
}

// One persistent launch traces every ray that is ready: the path rays of the next bounce (queue
// `ext`), then the shadow rays and the MIS rays of the bounce just shaded. The three sets do not
// depend on each other, so one work counter over their concatenation balances long rays against
// short ones and leaves one tail per bounce instead of three. Counts may be null (empty set).
//
// A wave's rays differ in length by a factor of ten, so a wave that traced 64 rays to their ends ran its
// steps with 26 % of its lanes. Instead a lane whose ray has ended takes the next one as soon as half of
// the wave's lanes are free (refilling at a quarter measured the same, at three quarters 8 % slower), and
// the lanes that hold a triangle wait until they are half as many as those that hold a node
// (kGateRatio; measured before rays were shared: 29.5 ms of tracing per 64-spp frame of the 1M-triangle
// displaced sphere at 1920x1080, 30.5 at a ratio of 1, 29.8 at 3, 31.1 at 6 and 38.0 without waiting; 43 ms
// before both). Once no rays are left, a wave's free lanes help the others (ray_share). The lanes carry
// rays of any kind.
// The launch asks for 6 waves per SIMD (80 VGPRs): 25.1 ms for that frame, 27.3 at 7 waves (72 VGPRs, spilling
// in the loop), 26.9 at 5.
// kCount: the counting instantiation, which also adds every lane's render-node fetches and
// triangle tests per ray kind (path, shadow, MIS) to traceCounts[0..5] (nodes, tests per kind).
constexpr int kTraceWaves = 6;  // per SIMD
constexpr int kMinWidth = 4;    // fewest lanes of a wave that carry rays
// Workgroups of BS threads that the 1024 SIMDs hold at once: a grid above that leaves late workgroups.
constexpr int resident_blocks(int bs) { return kTraceWaves * 65536 / bs; }

// Rays that a wave takes at a time: its width, and up to 256 where every wave still has some 8 turns (tracing
// of that frame: 27.2 ms with up to 256, 28.6 with 64, 28.1 with 1024).
LTS_D int trace_chunk(int n, int waves, int width) {
    int c = width;
    while (c < 256 && (long)c * waves * 8 < n) c <<= 1;
    return c;
}

template <int BS, bool kCount>
__global__ __launch_bounds__(BS, kTraceWaves) void k_wf_trace(const SceneView* __restrict__ scenes, const WfRay* __restrict__ rays, WfHit* __restrict__ hits,
                                                 const int32_t* __restrict__ ext, const int32_t* __restrict__ extCount,
                                                 uint8_t* __restrict__ bins, int nBins, const WfLightRay* __restrict__ shadows, const int32_t* __restrict__ shadowCount,
                                                 const WfLightRay* __restrict__ misRays, const int32_t* __restrict__ misCount,
                                                 const int32_t* __restrict__ shadowQueue, const int32_t* __restrict__ misQueue,
                                                 WfNee* __restrict__ nee, int32_t* __restrict__ work,
                                                 unsigned long long* __restrict__ traceCounts) {
    __shared__ int stk[kShortStack * BS];
    const TraceStack ts = lds_stack(stk, threadIdx.x, BS);
    const int nE = extCount ? *extCount : 0;
    const int nS = shadowCount ? *shadowCount : 0;
    const int nM = misCount ? *misCount : 0;
    const int n = nE + nS + nM;
    // lanes of a wave that carry rays: 64, or fewer in a small launch so that every wave gets some (a step
    // takes as long as the slowest of its lanes, and a wave with few lanes alternates less between node
    // and triangle steps: 1.61 against 1.74 ms of tracing for one sample of an 853x479 frame)
    const int waves = (int)gridDim.x * (BS / 64);
    int width = 64;
    while (width > kMinWidth && (long)width * waves > 2L * n) width >>= 1;
    const int spare = 64 - width, refill = spare + width / 2;
    WorkDeal<int> q = work_deal(n, trace_chunk(n, waves, width));
    unsigned long long tally[6] = {0, 0, 0, 0, 0, 0};
    int spill[kStack - kShortStack];
    __shared__ uint8_t marks[BS];
    uint8_t* const mark = marks + (threadIdx.x & ~63);
    const int lane = threadIdx.x & 63;
    TraceRay t;
    ray_none(t, lane);
    int path = 0, wait = 0;
    auto finish = [&]() {
        if (t.kind == kRayClosest) {
            WfHit o;
            o.leaf = t.best; o.u = t.u; o.v = t.v; o.invDet = t.invDet;
            hits[path] = o;
            if (bins) bins[path] = (uint8_t)(t.best < 0 ? nBins - 1 : (t.mat < nBins - 1 ? t.mat : nBins - 2));
        } else if (!t.mat) {
            const bool shadow = t.kind == kRayShadow;
            const float* c = (shadow ? shadows : misRays)[path].c;
            float* p = shadow ? nee[path].p1 : nee[path].p2;
            p[0] = c[0]; p[1] = c[1]; p[2] = c[2];
        }
        t.kind = kRayNone;
    };
    for (;;) {
        const unsigned long long idle = __ballot(t.l.cur == kTraceDone);
        if (q.open && (idle == ~0ull || __popcll(idle) >= refill)) {
            if (t.l.cur == kTraceDone && t.kind >= 0) finish();
            if (q.next >= q.end) {
                work_next(q, BS / 64, resident_blocks(BS), work);
                if (!q.open) continue;
            }
            const int rank = lanes_below(idle), k = q.next + rank;
            const int give = min((int)__popcll(idle) - spare, q.end - q.next);
            if (t.l.cur == kTraceDone && rank < give) {
                const float4* src;
                int kind;
                if (k < nE) {
                    kind = kRayClosest;
                    path = ext ? ext[k] : k;  // bounce 0 has no queue
                    src = reinterpret_cast<const float4*>(rays + path);
                } else if (k < nE + nS) {
                    kind = kRayShadow;
                    path = shadowQueue[k - nE];
                    src = reinterpret_cast<const float4*>(shadows + path);
                } else {
                    kind = kRayMis;
                    path = misQueue[k - nE - nS];
                    src = reinterpret_cast<const float4*>(misRays + path);
                }
                const float4 a = src[0], b = src[1];
                const SceneView& sv = scenes[__float_as_int(b.z)];
                const bool closest = kind == kRayClosest;
                ray_begin(t, kind, v3(a.x, a.y, a.z), v3(a.w, b.x, b.y), closest ? INFINITY : src[2].w,
                          closest ? -1 : __float_as_int(b.w), sv.recs, sv.root, ts);
            }
            q.next += give;
            continue;
        }
        if (!q.open && idle == ~0ull) {
            ray_settle(t, lane);
            if (t.kind >= 0) finish();
            break;
        }
        if (!kCount && !q.open && __popcll(idle) >= kShareIdle && --wait < 0) {
            wait = kShareSteps;
            ray_settle(t, lane);
            const bool held = ray_held(t, lane, mark), free = t.l.cur == kTraceDone && !held;
            if (free && t.kind >= 0) finish();
            ray_share(t, free, lane, ts);
        }
        ray_step<kCount>(t, ts, spill, tally);
    }
    if constexpr (kCount) {
        for (int q = 0; q < 6; q++) atomicAdd(&traceCounts[q], tally[q]);
    }
}

// Completes the paths that ended at the last bounce with a light sample in flight.
__global__ __launch_bounds__(256) void k_wf_finalize(const WfParams* __restrict__ prm, const WfSceneSlot* __restrict__ slots,
                                                     const WfPath* __restrict__ paths, const WfNee* __restrict__ nee,
                                                     const int32_t* __restrict__ done, const int32_t* __restrict__ count) {
    const int n = *count;
    const WfParams P = *prm;
    for (int k = blockIdx.x * 256 + threadIdx.x; k < n; k += gridDim.x * 256) finalize_path(P, slots, paths, nee, done[k]);
}

// Passes with max_bounce == 0 produce black samples.
__global__ __launch_bounds__(256) void k_wf_zero(const WfParams* __restrict__ prm, const WfSceneSlot* __restrict__ slots) {
    const WfParams P = *prm;
    for (long k = (long)blockIdx.x * 256 + threadIdx.x; k < P.nPaths; k += (long)gridDim.x * 256) {
        int s = 0;
        while (s + 1 < P.nScenes && k >= slots[s + 1].pathBase) s++;
        const WfSceneSlot& sl = slots[s];
        sl.sampleL[3 * (k - sl.pathBase) + 0] = 0.0f;
        sl.sampleL[3 * (k - sl.pathBase) + 1] = 0.0f;
        sl.sampleL[3 * (k - sl.pathBase) + 2] = 0.0f;
    }
}

__global__ void k_wf_fill(int32_t* p, int n, int32_t v) {
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) p[i] = v;
}

}  // namespace

int wf_trace_grid(int traceBlock, int persistentBlocks) { return std::min(persistentBlocks, resident_blocks(traceBlock)); }

hipError_t wf_enqueue_pass(const WfBuffers& b, const WfTuning& t, int maxBounce, const NrcBuffers* nrc, hipStream_t s,
                           const WfProfile* prof, unsigned long long* traceCounts) {
    auto mark = [&](int i) {
        if (prof) (void)hipEventRecord(prof->ev[i], s);
    };
    const int gridAll = t.sweepBlocks;
    const int ncounts = kWfBounceBase + kWfCountsPerBounce * (maxBounce + 1);
    k_wf_fill<<<(ncounts + 255) / 256, 256, 0, s>>>(b.counts, ncounts, 0);
    if (maxBounce <= 0) {
        k_wf_zero<<<gridAll, 256, 0, s>>>(b.params, b.slots);
        return hipGetLastError();
    }
    const bool cached = nrc != nullptr;
    int32_t* qCount = b.counts + kWfGlobalBase;
    int32_t* const bounce0 = b.counts + kWfBounceBase;
    k_wf_generate<<<gridAll, 256, 0, s>>>(b.scenes, b.params, b.slots, b.rays, bounce0, b.tRec);
    uint8_t* const bins = t.sortMaterials ? b.bins : nullptr;
    // traces the path rays of `bounce` (queue q, count cnt[0]) and the shadow and MIS rays of the
    // bounce before it (counts prev[1], prev[2]), with the work counters of `bounce`
    auto trace = [&](int bounce, const int32_t* extCount, const int32_t* shadowCount, const int32_t* misCount) {
        const int32_t* ext = bounce > 0 ? b.queue[bounce & 1] : nullptr;
        int32_t* work = bounce0 + kWfCountsPerBounce * bounce + kWfWorkBase;
        auto launch = [&](auto kernel, int bs) {
            kernel<<<wf_trace_grid(bs, t.persistentBlocks), bs, 0, s>>>(b.scenes, b.rays, b.hits, ext, extCount, bins, b.matBins, b.shadows, shadowCount,
                                                     b.mis, misCount, b.shadowQ, b.misQ, b.nee, work, traceCounts);
        };
        const bool counting = traceCounts != nullptr;
        switch (t.traceBlock) {
            case 64: launch(counting ? k_wf_trace<64, true> : k_wf_trace<64, false>, 64); break;
            case 128: launch(counting ? k_wf_trace<128, true> : k_wf_trace<128, false>, 128); break;
            default: launch(counting ? k_wf_trace<256, true> : k_wf_trace<256, false>, 256); break;
        }
    };
    mark(8 * kWfMaxBounce + 3);
    trace(0, bounce0, nullptr, nullptr);
    for (int bounce = 0; bounce < maxBounce; bounce++) {
        const int q = bounce & 1;
        int32_t* cnt = bounce0 + kWfCountsPerBounce * bounce;
        int32_t* nxt = cnt + kWfCountsPerBounce;
        mark(8 * bounce + 0);
        {
            auto shade = cached ? (bounce == 0 ? k_wf_shade<true, true> : k_wf_shade<true, false>)
                                : (bounce == 0 ? k_wf_shade<false, true> : k_wf_shade<false, false>);
            shade<<<kShadeGrid, kShadeBlock, 0, s>>>(b.scenes, b.params, b.slots, bounce, b.paths, b.rays, b.hits, b.nee, b.queue[q], cnt,
                                                  bins, b.done[q ^ 1], cnt - kWfCountsPerBounce + 3, cnt + kWfShadeWork, b.queue[q ^ 1], nxt, b.shadows,
                                                  cnt + 1, b.mis, cnt + 2, cached ? b.qRaw : nullptr, b.qMeta, qCount, b.tRec, b.tRaw,
                                                  b.done[q], cnt + 3, b.shadowQ, b.misQ);
        }
        mark(8 * bounce + 1);
        // the next bounce's path rays (none after the last bounce) with this bounce's shadow and MIS rays
        trace(bounce + 1, nxt, cnt + 1, cnt + 2);
        mark(8 * bounce + 2);
        if (bounce + 1 == maxBounce) k_wf_finalize<<<gridAll, 256, 0, s>>>(b.params, b.slots, b.paths, b.nee, b.done[q], cnt + 3);
        mark(8 * bounce + 3);
    }
    if (cached) {
        mark(8 * kWfMaxBounce + 0);
        hipError_t e = nrc_infer_queries(*nrc, b.qRaw, b.qMeta, qCount, (int)b.cap, b.sampleBase, s);
        if (e != hipSuccess) return e;
        mark(8 * kWfMaxBounce + 1);
        const int nb = (b.trainCap * maxBounce + kCollectPerBlock - 1) / kCollectPerBlock;
        if (nb > 0) {
            k_wf_nrc_count<<<nb, kCollectBlock, 0, s>>>(b.params, b.tRec, b.tCount);
            const int cap = nrc->batchCap * nrc->chunks;
            k_wf_nrc_scan<<<1, 64, 0, s>>>(b.tCount, nb, cap, nrc->state);
            k_wf_nrc_scatter<<<nb, kCollectBlock, 0, s>>>(b.params, b.tRec, b.tRaw, b.sampleBase, b.tCount, cap,
                                                          nrc->trainRaw, nrc->trainTarget);
        }
        if ((e = nrc_train(*nrc, s, nrc->steps)) != hipSuccess) return e;  // batches cycle when steps > batches
        mark(8 * kWfMaxBounce + 2);
    }
    return hipGetLastError();
}

}  // namespace lts

namespace lts {

template <typename T>
static hipError_t wf_alloc(T** p, size_t count) {
    return hipMalloc((void**)p, (count ? count : 1) * sizeof(T));
}

hipError_t wf_reserve(WfBuffers& b, size_t cap, int maxScenes) {
    if (cap <= b.cap && maxScenes <= b.maxScenes) return hipSuccess;
    wf_release(b);
    hipError_t e = hipSuccess;
#define WTRY(x) do { e = (x); if (e != hipSuccess) { wf_release(b); return e; } } while (0)
    WTRY(wf_alloc(&b.scenes, maxScenes));
    WTRY(wf_alloc(&b.params, 1));
    WTRY(wf_alloc(&b.slots, maxScenes));
    WTRY(wf_alloc(&b.paths, cap));
    WTRY(wf_alloc(&b.rays, cap));
    WTRY(wf_alloc(&b.hits, cap));
    WTRY(wf_alloc(&b.nee, cap));
    WTRY(wf_alloc(&b.queue[0], cap));
    WTRY(wf_alloc(&b.queue[1], cap));
    WTRY(wf_alloc(&b.done[0], cap));
    WTRY(wf_alloc(&b.done[1], cap));
    WTRY(wf_alloc(&b.shadowQ, cap));
    WTRY(wf_alloc(&b.misQ, cap));
    WTRY(wf_alloc(&b.bins, cap));
    WTRY(wf_alloc(&b.shadows, cap));
    WTRY(wf_alloc(&b.mis, cap));
    WTRY(wf_alloc(&b.counts, (size_t)kWfBounceBase + kWfCountsPerBounce * (kWfMaxBounce + 1)));
#undef WTRY
    b.cap = cap;
    b.maxScenes = maxScenes;
    b.gen = next_buffer_generation();
    return hipSuccess;
}

hipError_t wf_reserve_cache(WfBuffers& b, size_t cap, int trainCap) {
    if (cap <= b.cacheCap && trainCap <= b.trainCap) return hipSuccess;
    void* ps[] = {b.qRaw, b.qMeta, b.tRec, b.tRaw, b.tCount};
    for (void* p : ps)
        if (p) (void)hipFree(p);
    b.qRaw = nullptr; b.qMeta = nullptr; b.tRec = nullptr; b.tRaw = nullptr; b.tCount = nullptr;
    b.cacheCap = 0; b.trainCap = 0;
    hipError_t e = hipSuccess;
#define CTRY(x) do { e = (x); if (e != hipSuccess) return e; } while (0)
    CTRY(wf_alloc(&b.qRaw, cap * kNrcRaw));
    CTRY(wf_alloc(&b.qMeta, cap));
    CTRY(wf_alloc(&b.tRec, (size_t)trainCap * kWfMaxBounce));
    CTRY(wf_alloc(&b.tRaw, (size_t)trainCap * kWfMaxBounce * kNrcRaw));
    CTRY(wf_alloc(&b.tCount, ((size_t)trainCap * kWfMaxBounce + kCollectPerBlock - 1) / kCollectPerBlock));
#undef CTRY
    b.cacheCap = cap;
    b.trainCap = trainCap;
    b.cacheGen = next_buffer_generation();
    return hipSuccess;
}

void wf_release(WfBuffers& b) {
    void* cs[] = {b.qRaw, b.qMeta, b.tRec, b.tRaw, b.tCount};
    for (void* p : cs)
        if (p) (void)hipFree(p);
    void* ps[] = {b.scenes, b.params, b.slots, b.paths, b.rays, b.hits, b.nee, b.queue[0], b.queue[1], b.done[0], b.done[1], b.shadowQ, b.misQ, b.bins, b.shadows, b.mis, b.counts};
    for (void* p : ps)
        if (p) (void)hipFree(p);
    b = WfBuffers();
}

}  // namespace lts
