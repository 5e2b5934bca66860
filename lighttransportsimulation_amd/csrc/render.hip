// Film and query kernels (gfx950): the deterministic film gather (rendering/Camera.cu:192-218 without
// atomics, then getRender, Camera.cu:256-289), caller-given rays, and small fills and copies.
#include "pt_device.h"
#include "lts_internal.h"

namespace lts {

namespace {

__global__ __launch_bounds__(256) void k_rec_materials(const ShadeTri* __restrict__ shade, int n, TraceRec* __restrict__ recs, int nRecs) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= nRecs) return;
    const uint32_t leaf = recs[k].w[11];
    if (leaf < (uint32_t)n) recs[k].w[10] = (uint32_t)shade[leaf].mat;
}

// Pixel (x, y) gathers, for each sample in order and each owner pixel (ox, oy) with ox in
// x-2..x+1 and oy in y-2..y+1 (row major), the owner's filtered contribution when its addSample
// footprint [ceil(p - 1), floor(p + 1) + 1) covers (x, y). A film position p = owner + f with f in
// (0, 1) covers owner..owner+1; f = 1 adds owner+2; and p rounding down to the owner itself (f
// below half an ulp of the owner coordinate, possible from 1024 pixels on) adds owner-1, which is
// why the window reaches one owner past the pixel. A 16x16 block stages, per sample, the film
// positions and radiance of the 19x19 owners its pixels read in LDS, so each owner's film position
// is drawn once per block instead of once per covered pixel; the sums keep their order.
__global__ __launch_bounds__(256) void k_film_gather(SceneView sv, RenderLaunch rl) {
    constexpr int T = 16, R = T + 3;
    __shared__ float own[R * R][5];  // film position x, y and radiance r, g, b of each owner
    const int W = sv.cam.width, H = sv.cam.height;
    const int x0 = blockIdx.x * T, y0 = blockIdx.y * T;
    const int x = x0 + (threadIdx.x & 15), y = y0 + (threadIdx.x >> 4);
    const bool inside = x < W && y < H;
    float4 acc = inside ? reinterpret_cast<float4*>(rl.film)[(size_t)y * W + x] : make_float4(0.f, 0.f, 0.f, 0.f);
    Spec rgb = spec(acc.x, acc.y, acc.z);
    float wsum = acc.w;
    for (int s = rl.s0; s < rl.s1; s++) {
        __syncthreads();  // the previous sample's owners have been read
        for (int e = threadIdx.x; e < R * R; e += 256) {
            const int ox = x0 - 2 + e % R, oy = y0 - 2 + e / R;
            if (ox < 0 || oy < 0 || ox >= W || oy >= H) continue;
            Sampler smp;
            smp.seed = rl.seed; smp.pixel = (uint32_t)(oy * W + ox); smp.sample = (uint32_t)s;
            float d[4];
            smp.block(0, d);
            const V2 pf = film_sample(ox, oy, s, rl.spp, rl.stratified, d);
            const float* l = rl.sampleL + 3 * ((size_t)(s - rl.s0) * W * H + (size_t)oy * W + ox);
            own[e][0] = pf.x; own[e][1] = pf.y;
            own[e][2] = l[0]; own[e][3] = l[1]; own[e][4] = l[2];
        }
        __syncthreads();
        if (!inside) continue;
        for (int oy = y - 2; oy <= y + 1; oy++) {
            if (oy < 0 || oy >= H) continue;
            for (int ox = x - 2; ox <= x + 1; ox++) {
                if (ox < 0 || ox >= W) continue;
                const float* o = own[(oy - y0 + 2) * R + (ox - x0 + 2)];
                const V2 pf = v2(o[0], o[1]);
                int p0x = max((int)ceilf(pf.x - 1.0f), 0), p0y = max((int)ceilf(pf.y - 1.0f), 0);
                int p1x = min((int)floorf(pf.x + 1.0f) + 1, W), p1y = min((int)floorf(pf.y + 1.0f) + 1, H);
                if (x < p0x || x >= p1x || y < p0y || y >= p1y) continue;
                float dx = fabsf((x - pf.x - 0.5f) * 1.0f * 16);
                float dy = fabsf((y - pf.y - 0.5f) * 1.0f * 16);
                int ix = (int)fminf((float)(int)floorf(dx), 15.0f);
                int iy = (int)fminf((float)(int)floorf(dy), 15.0f);
                float w = sv.filter[iy * 16 + ix];
                rgb = rgb + spec(o[2], o[3], o[4]) * w;
                wsum += w;
            }
        }
    }
    if (inside) reinterpret_cast<float4*>(rl.film)[(size_t)y * W + x] = make_float4(rgb.r, rgb.g, rgb.b, wsum);
}

__global__ void k_film_clear(float4* film, int npix) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i < npix) film[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

__global__ void k_get_render(const float4* film, float* rgb, int W, int H) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= W * H) return;
    int j = i / W, c = i % W;
    float4 p = film[(size_t)(H - 1 - j) * W + c];
    float inv = 1 / p.w;
    rgb[3 * (size_t)i] = fmaxf(0.0f, p.x * inv);
    rgb[3 * (size_t)i + 1] = fmaxf(0.0f, p.y * inv);
    rgb[3 * (size_t)i + 2] = fmaxf(0.0f, p.z * inv);
}

}  // namespace

hipError_t launch_film_gather(const SceneView& sv, const RenderLaunch& rl, hipStream_t stream) {
    const int W = sv.cam.width, H = sv.cam.height;
    dim3 grid((W + 15) / 16, (H + 15) / 16);
    k_film_gather<<<grid, 256, 0, stream>>>(sv, rl);
    return hipGetLastError();
}

hipError_t launch_rec_materials(const ShadeTri* shade, int n, TraceRec* recs, int nRecs, hipStream_t s) {
    if (nRecs < 1) return hipSuccess;
    k_rec_materials<<<(nRecs + 255) / 256, 256, 0, s>>>(shade, n, recs, nRecs);
    return hipGetLastError();
}

// Closest hits of caller-given rays by the renderer's own traversal, one thread per ray; a miss gives prim -1.
// 500000 rays at a 90k-triangle torus: 180 us with every lane waiting for its wave's longest ray, 162 with
// trace_wave (201 without the bound on waves: 130 VGPRs), with 40 % of the lanes at work.
__global__ __launch_bounds__(256, 6) void k_trace_rays(SceneView sv, const float* __restrict__ origins, const float* __restrict__ dirs,
                                                    int stride, int n, int32_t* __restrict__ prim, float* __restrict__ tOut) {
    __shared__ int lds[4][kWaveTraceWords];
    const int i = blockIdx.x * 256 + threadIdx.x;
    RayQuery q;
    q.kind = kRayNone;
    if (i < n) {
        const float* o = origins + (size_t)stride * i;
        const float* d = dirs + (size_t)stride * i;
        q.kind = kRayClosest;
        q.o = v3(o[0], o[1], o[2]);
        q.d = v3(d[0], d[1], d[2]);
        q.tMax = INFINITY;
    }
    const RayAnswer h = trace_wave(sv, q, lds[threadIdx.x >> 6]);
    if (i >= n) return;
    int p = -1;
    if (h.leaf >= 0) {
        V3 p0, p1, p2;
        load_tri(sv.tris, h.leaf, p0, p1, p2, p);
    }
    prim[i] = p;
    tOut[i] = h.leaf >= 0 ? h.t : INFINITY;
}

hipError_t launch_trace_rays(const SceneView& sv, const float* origins, const float* dirs, int stride, int n, int32_t* prim,
                             float* t, hipStream_t stream) {
    if (n < 1) return hipSuccess;
    k_trace_rays<<<(n + 255) / 256, 256, 0, stream>>>(sv, origins, dirs, stride, n, prim, t);
    return hipGetLastError();
}

hipError_t launch_film_clear(float* film, int npix, hipStream_t stream) {
    k_film_clear<<<(npix + 255) / 256, 256, 0, stream>>>(reinterpret_cast<float4*>(film), npix);
    return hipGetLastError();
}

hipError_t launch_get_render(const SceneView& sv, const float* film, float* rgb, hipStream_t stream) {
    const int W = sv.cam.width, H = sv.cam.height;
    k_get_render<<<(W * H + 255) / 256, 256, 0, stream>>>(reinterpret_cast<const float4*>(film), rgb, W, H);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_copy(float4* __restrict__ dst, const float4* __restrict__ src, size_t n4) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (size_t)gridDim.x * 256) dst[i] = src[i];
}

hipError_t launch_copy(void* dst, const void* src, size_t bytes, hipStream_t stream) {
    size_t n4 = bytes / 16;
    k_copy<<<2048, 256, 0, stream>>>(reinterpret_cast<float4*>(dst), reinterpret_cast<const float4*>(src), n4);
    return hipGetLastError();
}



}  // namespace lts
