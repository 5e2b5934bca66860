// Whole paths in one launch (gfx950): the form for small passes.
//
// Each lane carries one path through the reference integrator (intergrators/PathTracingIntegrator.cuh:26-109
// with estimateDirect, IntegratorHelper.cuh:51-125) as a sequence of rays: the path's ray, and after its hit
// is shaded the shadow ray, the MIS-BSDF ray and the next path ray. A lane whose path has ended takes the
// next one. The arithmetic of a path is the wavefront's, so the image does not depend on the form.
//
// What bounds it: the latency of the longest paths, and vector instructions with 27 % of the lanes at work over
// an 853x479 sample (986 us) and 35 % over a 256x256 16-spp Cornell frame (1.74 ms), at 3 waves per SIMD (168
// VGPRs of shading code). The wavefront keeps 57 % of them in tracing and sorts its shading by material, and pays
// some 100 us for each of its launches; a lane here goes on as soon as its own ray has ended.
#include "path_order.h"
#include "pt_device.h"

namespace lts {

namespace {

// 3 waves per SIMD: 5.44 ms for an 8-spp 1280x720 frame of a 360k-triangle displaced sphere, 5.64 at 4 and
// 6.98 at 5 (spilling), 6.58 at 2. One path per thread, the whole wave waiting for its longest ray at each
// vertex, at 5 waves: 5.83.
constexpr int kPathWaves = 3;
constexpr int kPathMinWidth = 4;  // fewest lanes of a wave that carry paths, see trace_width
// Shading and dealing wait until the lanes that need them are half as many as those with a ray to trace (that
// frame: 5.44 ms when they have to be as many, 5.33 at two thirds, 5.26 at a half and at a third); a path's
// next ray begins once half as many lanes are between two rays as trace (5.39 and 5.61 at as many and at a
// quarter).
constexpr int kPathTurn = 2, kPathNext = 2;
// A wave whose lanes have traced for kPathLong steps without a turn, with kPathIdle lanes or more without a
// path, shares its rays (one sample of that frame: 1.88 -> 1.27 ms).
constexpr int kPathLong = 16, kPathIdle = 48;

// Path k of a pass -> (pixel, sample), or false past the last pixel. The samples of 64 neighbouring pixels
// follow each other.
LTS_D bool film_path(const SceneView& sv, const RenderLaunch& rl, long k, int& pixel, int& sample) {
    const long g = k >> 6;
    const int n = rl.s1 - rl.s0, j = (int)(g / n) * 64 + (int)(k & 63);
    sample = rl.s0 + (int)(g % n);
    if (j >= sv.cam.width * sv.cam.height) return false;
    pixel = band_pixel(j, sv.cam.width, sv.cam.height, kPathRows);
    return true;
}

LTS_D float* film_sample_out(const SceneView& sv, const RenderLaunch& rl, int pixel, int sample) {
    return rl.sampleL + 3 * ((size_t)(sample - rl.s0) * sv.cam.width * sv.cam.height + pixel);
}

// what a path still has to do after its current ray
enum PathTodo { kTodoShadow = 1, kTodoMis = 2, kTodoNext = 4, kTodoLight = 8, kTodoSpecular = 16 };
constexpr int kTodoBounce = 5;  // shift of the bounce

// words of a path's state that wait in private memory while its rays are traced
enum PathWord {
    kWordL = 0, kWordBeta = 3, kWordNb = 6, kWordLpdf = 9, kWordLd = 10, kWordMisC = 13, kWordRay = 16, kWordShadow = 22, kWordMis = 28,
    kWordPixel = 36, kWordSample, kPathWords
};

// work: the dealing's counters, 0 at the start; other: those of the next launch, cleared here.
// kCount: adds every lane's render-node fetches and triangle tests per kind of ray to rl.counters[0..5].
template <bool kCount>
__global__ __launch_bounds__(256, kPathWaves) void k_paths(SceneView sv, RenderLaunch rl, int32_t* __restrict__ work,
                                                           int32_t* __restrict__ other) {
    __shared__ int stk[kShortStack * 256];
    __shared__ NoiseTables perm;
    if (blockIdx.x == 0 && threadIdx.x < kPathWork) other[threadIdx.x] = 0;
    noise_tables(perm, sv.perm, threadIdx.x, 256);
    __syncthreads();
    const TraceStack ts = lds_stack(stk, threadIdx.x, 256);
    const long n = (long)((sv.cam.width * sv.cam.height + 63) / 64) * 64 * (rl.s1 - rl.s0);
    const int waves = (int)gridDim.x * 4;
    int width = 64;
    while (width > kPathMinWidth && (long)width * waves > 2L * n) width >>= 1;
    const bool carrier = (int)(threadIdx.x & 63) < width;
    WorkDeal<long> q = work_deal(n, width);
    unsigned long long tally[6] = {0, 0, 0, 0, 0, 0};
    // deep stack entries, then the path's words
    int store[kStack - kShortStack + kPathWords];
    int* const state = store + (kStack - kShortStack);
    auto put = [&](int i, float v) { state[i] = __float_as_int(v); };
    auto get = [&](int i) { return __int_as_float(state[i]); };
    auto put3 = [&](int i, V3 v) { put(i, v.x); put(i + 1, v.y); put(i + 2, v.z); };
    auto get3 = [&](int i) { return v3(get(i), get(i + 1), get(i + 2)); };
    auto putS = [&](int i, Spec v) { put(i, v.r); put(i + 1, v.g); put(i + 2, v.b); };
    auto getS = [&](int i) { return spec(get(i), get(i + 1), get(i + 2)); };

    const int lane = threadIdx.x & 63;
    // t.kind is the kind of ray that the lane's path waits for
    TraceRay t;
    ray_none(t, lane);
    int todo = 0;
    for (;;) {
        const bool dry = !q.open;
        const bool ended = t.l.cur == kTraceDone;
        const bool hit = ended && t.kind == kRayClosest;
        const int nRun = (int)__popcll(__ballot(t.kind != kRayNone && !hit));
        const unsigned long long atHit = __ballot(hit);
        const unsigned long long empty = dry ? 0 : __ballot(carrier && ended && t.kind == kRayNone);
        const bool turn = kPathTurn * (int)(__popcll(atHit) + __popcll(empty)) >= nRun;
        bool advance = ended && t.kind > kRayClosest;
        if (turn && atHit) {
            if (hit) {
                const int pixel = state[kWordPixel], sample = state[kWordSample];
                const int bounce = todo >> kTodoBounce;
                const bool specularBounce = (todo & kTodoSpecular) != 0;
                Ray r;
                r.o = t.l.o; r.d = t.d; r.tMax = INFINITY;
                Spec L = getS(kWordL), beta = getS(kWordBeta);
                todo = (bounce + 1) << kTodoBounce;
                if (bounce == 0 || specularBounce) {
                    add_emission(sv, t.best, r, t.u, t.v, t.invDet, beta, L);
                    putS(kWordL, L);
                }
                if (t.best >= 0) {
                    SurfacePoint si = make_surface(sv, t.best, r, t.u, t.v, t.invDet);
                    if (bounce == 0 && sv.mats[sv.shade[si.leaf].mat].footprint) {
                        const int px = pixel % sv.cam.width, py = pixel / sv.cam.width;
                        camera_footprint(sv, si, camera_sample(sv, px, py, sample, rl.spp, rl.stratified, rl.seed),
                                         rl.spp, r, t.invDet);
                    }
                    Bsdf bsdf = make_bsdf(sv, si, perm);
                    Sampler smp;
                    smp.seed = rl.seed; smp.pixel = (uint32_t)pixel; smp.sample = (uint32_t)sample;
                    float u0[4], u1[4];
                    smp.block(1 + 2 * bounce, u0);
                    smp.block(2 + 2 * bounce, u1);
                    if (sv.nLights > 0) {
                        float lpdf;
                        const int li = sample_light(sv, u0[0], &lpdf);
                        todo |= kTodoLight;
                        putS(kWordNb, beta);
                        put(kWordLpdf, lpdf);
                        putS(kWordLd, spec(0.0f));
                        light_rays(sv, si, bsdf, li, u0, u1, specularBounce,
                                   [&](V3 o, V3 dir, Spec c) {
                                       todo |= kTodoShadow;
                                       put3(kWordShadow, o); put3(kWordShadow + 3, dir);
                                       putS(kWordLd, c);
                                   },
                                   [&](V3 o, V3 dir, float tMax, int tieLeaf, Spec c) {
                                       todo |= kTodoMis;
                                       put3(kWordMis, o); put3(kWordMis + 3, dir); put(kWordMis + 6, tMax); state[kWordMis + 7] = tieLeaf;
                                       putS(kWordMisC, c);
                                   });
                    }
                    // continuation (PathTracingIntegrator.cuh:79-103)
                    V3 wo = -r.d, wi;
                    float pdf;
                    int flags = 0;
                    Spec f = bsdf.sampleF(wo, &wi, v2(u1[1], u1[2]), &pdf, B_ALL, &flags);
                    if (!(isBlack(f) || pdf == 0)) {
                        if (flags & B_SPEC) todo |= kTodoSpecular;
                        beta = beta * (f * absDot(wi, si.sn) / pdf);
                        Ray nr = spawn_ray(si, wi);
                        bool alive = true;
                        if (bounce >= rl.rrStart) {
                            float q = fmaxf(0.05f, 1 - lum(beta));
                            if (u1[3] < q) alive = false;
                            else beta = beta / (1 - q);
                        }
                        if (alive && bounce + 1 < rl.maxBounce) {
                            todo |= kTodoNext;
                            putS(kWordBeta, beta);
                            put3(kWordRay, nr.o); put3(kWordRay + 3, wi);
                        }
                    }
                }
                advance = true;
            }
        }
        if (__ballot(advance)) {
            if (advance) {
                if (t.kind == kRayShadow) {
                    if (t.mat) putS(kWordLd, spec(0.0f));
                } else if (t.kind == kRayMis && !t.mat) {
                    putS(kWordLd, getS(kWordLd) + getS(kWordMisC));
                }
                int from = -1, kind = kRayNone, tie = -1;
                float tMax = INFINITY;
                if (todo & kTodoShadow) {
                    todo &= ~kTodoShadow;
                    kind = kRayShadow;
                    from = kWordShadow;
                    tMax = 1 - SHADOW_EPS;
                } else if (todo & kTodoMis) {
                    todo &= ~kTodoMis;
                    kind = kRayMis;
                    from = kWordMis;
                    tMax = get(kWordMis + 6); tie = state[kWordMis + 7];
                } else {
                    Spec L = getS(kWordL);
                    if (todo & kTodoLight) {
                        L = L + getS(kWordNb) * (getS(kWordLd) / get(kWordLpdf));
                        putS(kWordL, L);
                    }
                    if (todo & kTodoNext) {
                        kind = kRayClosest;
                        from = kWordRay;
                    } else {
                        float* o = film_sample_out(sv, rl, state[kWordPixel], state[kWordSample]);
                        o[0] = L.r; o[1] = L.g; o[2] = L.b;
                        t.kind = kRayNone;
                    }
                }
                if (from >= 0) {
                    ray_begin(t, kind, get3(from), get3(from + 3), tMax, tie, sv.recs, sv.root, ts);
                }
            }
        }
        if (turn && !dry) {
            const unsigned long long idle = __ballot(carrier && t.kind == kRayNone);
            if (idle) {
                if (q.next >= q.end) work_next(q, 4, kPathWaves * 256, work);
                const int rank = lanes_below(idle);
                const int give = (int)min((long)__popcll(idle), q.end - q.next);
                if (carrier && t.kind == kRayNone && rank < give) {
                    int pixel, sample;
                    if (!film_path(sv, rl, q.next + rank, pixel, sample)) {
                        // past the last pixel
                    } else if (rl.maxBounce <= 0) {
                        float* o = film_sample_out(sv, rl, pixel, sample);
                        o[0] = o[1] = o[2] = 0.0f;
                    } else {
                        const int px = pixel % sv.cam.width, py = pixel / sv.cam.width;
                        const Ray r = camera_ray(sv, camera_sample(sv, px, py, sample, rl.spp, rl.stratified, rl.seed));
                        state[kWordPixel] = pixel; state[kWordSample] = sample;
                        putS(kWordL, spec(0.0f));
                        putS(kWordBeta, spec(1.0f));
                        todo = 0;
                        ray_begin(t, kRayClosest, r.o, r.d, INFINITY, -1, sv.recs, sv.root, ts);
                    }
                }
                q.next += give;
                continue;
            }
        }
        if (!__ballot(t.kind != kRayNone)) break;
        int steps = 0;
        const int nIdle = dry ? 0 : (int)__popcll(__ballot(carrier && t.kind == kRayNone));
        for (;;) {
            const bool done = t.l.cur == kTraceDone;
            const int active = (int)__popcll(__ballot(!done));
            const int light = (int)__popcll(__ballot(done && t.kind > kRayClosest));
            const int atHit = (int)__popcll(__ballot(done && t.kind == kRayClosest));
            if (active == 0 || kPathNext * light >= active || kPathTurn * (atHit + nIdle) >= active + light) break;
            if (!kCount && ++steps > kPathLong && 64 - active - light - atHit >= kPathIdle) {
                ray_finish_shared(t, ts, store);
                break;
            }
            ray_step<kCount>(t, ts, store, tally);
        }
    }
    if constexpr (kCount) {
        for (int q = 0; q < 6; q++)
            if (tally[q]) atomicAdd(&rl.counters[q], tally[q]);
    }
}

}  // namespace

hipError_t launch_paths(const SceneView& sv, const RenderLaunch& rl, int32_t* work, int32_t* other, hipStream_t stream) {
    constexpr int grid = 256 * kPathWaves;  // the workgroups resident at once
    if (rl.counters) k_paths<true><<<grid, 256, 0, stream>>>(sv, rl, work, other);
    else k_paths<false><<<grid, 256, 0, stream>>>(sv, rl, work, other);
    return hipGetLastError();
}

}  // namespace lts
