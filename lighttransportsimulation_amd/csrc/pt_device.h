// Path-tracer device routines shared by the whole-path, wavefront and bidirectional kernels.
// Each routine restates a reference routine (tierChampion/LightTransportSimulation/src) with
// the same fp32 evaluation order; see lts_device.h for the arithmetic conventions.
#pragma once
#include "lts_device.h"
#include "lts_scene.h"

namespace lts {

struct Ray {
    V3 o, d;
    float tMax;
};

struct SurfacePoint {
    V3 p, pError, wo, n;
    V2 uv;
    V3 dpdu, dpdv;
    V3 sn, sdpdu;
    V3 dpdx, dpdy;
    float dudx, dvdx, dudy, dvdy;  // uv differentials (primary hits; read by filtered textures)
    int leaf;  // BVH leaf of the triangle, which indexes its ShadeTri record
};

// The scene's arrays live in device (global) memory. Kernels that read a SceneView from memory see
// its pointers as generic ones, whose flat loads also count against the LDS wait counter (so a wait
// for a traversal-stack read waits for node loads too); the traversal's loads go through global
// pointers instead.
typedef float GlobalF4 __attribute__((ext_vector_type(4)));
typedef unsigned GlobalU4 __attribute__((ext_vector_type(4)));
LTS_D GlobalF4 load_global_f4(const void* p, int i) { return ((const __attribute__((address_space(1))) GlobalF4*)p)[i]; }
LTS_D GlobalU4 load_global_u4(const void* p, int i) { return ((const __attribute__((address_space(1))) GlobalU4*)p)[i]; }
LTS_D float word_f(unsigned w) { return __uint_as_float(w); }

LTS_D void load_tri(const TriLeaf* __restrict__ tris, int k, V3& p0, V3& p1, V3& p2, int& prim) {
    const GlobalF4 a = load_global_f4(tris + k, 0), b = load_global_f4(tris + k, 1), c = load_global_f4(tris + k, 2);
    p0 = v3(a.x, a.y, a.z);
    p1 = v3(a.w, b.x, b.y);
    p2 = v3(b.z, b.w, c.x);
    prim = __float_as_int(c.y);
}

// The reference's triangle tests take 1.0 / det in double and compare float barycentrics with the
// double 1 -/+ SHADOW_EPS. Both have exact float forms: a double quotient of float operands rounded
// to float is the correctly rounded float quotient (53 >= 2 * 24 + 2 bits: the double rounding is
// innocuous), which the IEEE float division gives; and for a float x, (double)x > c holds exactly
// when x exceeds the largest float not above c, the two constants below.
constexpr float kOneMinusEpsF = 0x1.fff2e4p-1f;  // largest float <= 1.0 - (double)SHADOW_EPS
constexpr float kOnePlusEpsF = 0x1.00068cp+0f;   // largest float <= 1.0 + (double)SHADOW_EPS

// Triangle::intersect hit test (shapes/Triangle.cu:94-128) without its distance test: true when
// the ray meets the triangle inside the barycentric margins [SHADOW_EPS, limit], at distance t of either
// sign. Triangle::simpleIntersect (shapes/Triangle.cu:50-84) is the same test with p1 and p2 exchanged
// and limit 1 + SHADOW_EPS.
LTS_D bool tri_mt(V3 p0, V3 p1, V3 p2, const Ray& r, float limit, float& t, float& u, float& v, float& invDetOut) {
    V3 edge1 = p1 - p0, edge2 = p2 - p0;
    V3 pVec = cross(r.d, edge2);
    float det = dot(edge1, pVec);
    if (det == 0) return false;
    float invDet = 1.0f / det;
    V3 tVec = r.o - p0;
    u = invDet * dot(tVec, pVec);
    if (u < SHADOW_EPS || u > limit) return false;
    V3 qVec = cross(tVec, edge1);
    v = invDet * dot(r.d, qVec);
    if (v < SHADOW_EPS || u + v > limit) return false;
    t = invDet * dot(edge2, qVec);
    invDetOut = invDet;
    return true;
}

// Triangle::intersect hit test (shapes/Triangle.cu:94-128): t in (0, tMax).
LTS_D bool tri_hit(V3 p0, V3 p1, V3 p2, const Ray& r, float& t, float& u, float& v, float& invDetOut) {
    return tri_mt(p0, p1, p2, r, kOneMinusEpsF, t, u, v, invDetOut) && t > 0 && t < r.tMax;
}

// Bounds3::simpleIntersect (geometry/Bound.cuh:200-227); also returns the entry distance.
LTS_D bool box_hit(const float* mn, const float* mx, const Ray& r, V3 inv, int nx, int ny, int nz, float& tEnter) {
    const float g3 = 1 + 2 * gammaN(3);
    float tMin = ((nx ? mx[0] : mn[0]) - r.o.x) * inv.x;
    float tMax = ((nx ? mn[0] : mx[0]) - r.o.x) * inv.x;
    float tyMin = ((ny ? mx[1] : mn[1]) - r.o.y) * inv.y;
    float tyMax = ((ny ? mn[1] : mx[1]) - r.o.y) * inv.y;
    tMax *= g3;
    tyMax *= g3;
    if (tMin > tyMax || tyMin > tMax) return false;
    if (tyMin > tMin) tMin = tyMin;
    if (tyMax < tMax) tMax = tyMax;
    float tzMin = ((nz ? mx[2] : mn[2]) - r.o.z) * inv.z;
    float tzMax = ((nz ? mn[2] : mx[2]) - r.o.z) * inv.z;
    tzMax *= g3;
    if (tMin > tzMax || tzMin > tMax) return false;
    if (tzMin > tMin) tMin = tzMin;
    if (tzMax < tMax) tMax = tzMax;
    tEnter = tMin;
    return (tMin < r.tMax) && (tMax > 0);
}

// The reference's leaf-box test for a shadow ray (its inverse direction, BVH.cuh:336, and the
// triangle's bounds).
LTS_D bool leaf_box_passes(V3 p0, V3 p1, V3 p2, const Ray& r) {
    const V3 inv = v3(1.0f / r.d.x, 1.0f / r.d.y, 1.0f / r.d.z);
    const float mn[3] = {fminf(fminf(p0.x, p1.x), p2.x), fminf(fminf(p0.y, p1.y), p2.y), fminf(fminf(p0.z, p1.z), p2.z)};
    const float mx[3] = {fmaxf(fmaxf(p0.x, p1.x), p2.x), fmaxf(fmaxf(p0.y, p1.y), p2.y), fmaxf(fmaxf(p0.z, p1.z), p2.z)};
    float tEnter;
    return box_hit(mn, mx, r, inv, inv.x < 0, inv.y < 0, inv.z < 0, tEnter);
}

constexpr int kStack = kTraceStack;
// Stack entries kept in LDS (the first is the end marker); deeper entries go to private memory. 22
// entries of a 256-lane block (22528 B) plus the 256 B of ray_held's marks let 7 trace blocks (7
// waves per SIMD) share a CU's 160 KB of LDS.
constexpr int kShortStack = 22;
constexpr int kTraceDone = -1;  // bottom of the stack: the traversal has ended

// Traversal stack of one lane: entries [0, kShortStack) in LDS (entry e at lds[e * stride], so the
// lanes of a wave touch consecutive words), deeper entries in a private array that only deep
// traversals reach. A private 64-entry array alone is scratch memory, and its traffic dominated
// the traversal kernels.
struct TraceStack {
    int* lds;
    int stride;
};

// LDS stack of thread `tid` in a block-wide array __shared__ int[kShortStack * blockSize].
LTS_D TraceStack lds_stack(int* shared, int tid, int blockSize) { return TraceStack{shared + tid, blockSize}; }

// 1 / d by v_rcp_f32 (within 1 ulp) with its magnitude held to 2^100, for the node test only: a
// zero direction component gives slab distances that are hugely negative or positive, never NaN.
LTS_D float slab_inverse(float d) { return __builtin_amdgcn_fmed3f(__builtin_amdgcn_rcpf(d), -0x1p100f, 0x1p100f); }

// The traversal of one lane. A ray's slab constants, then the stack (entry e in LDS below kShortStack,
// else in `spill`) and the record to visit next.
struct TraceLane {
    V3 o, inv;
    bool nx, ny, nz;
    int cur, sp;
};

// Whether a ray has an infinite or NaN component: it then passes no triangle test.
LTS_D bool ray_degenerate(V3 o, V3 d) { return !(0 * o.x + 0 * o.y + 0 * o.z + 0 * d.x + 0 * d.y + 0 * d.z == 0); }

LTS_D void trace_begin(TraceLane& l, V3 o, V3 d, int root, TraceStack ts) {
    l.o = o;
    l.inv = v3(slab_inverse(d.x), slab_inverse(d.y), slab_inverse(d.z));
    l.nx = l.inv.x < 0; l.ny = l.inv.y < 0; l.nz = l.inv.z < 0;
    ts.lds[0] = kTraceDone;
    l.sp = 1;
    l.cur = ray_degenerate(o, d) ? kTraceDone : root;
}

LTS_D void trace_pop(TraceLane& l, TraceStack ts, const int* spill) {
    --l.sp;
    if (__builtin_expect(__any(l.sp >= kShortStack), 0)) l.cur = l.sp < kShortStack ? ts.lds[l.sp * ts.stride] : spill[l.sp - kShortStack];
    else l.cur = ts.lds[l.sp * ts.stride];
}

// One node of the 4-wide render tree (BVH::intersect / BVH::simpleIntersect, acceleration/BVH.cuh:331-398):
// tests the boxes of its children, goes on to the nearest one hit and stacks the others. Every triangle
// whose box the ray passes before its current tMax is reached, so the closest hit is the reference
// traversal's in any order of visits (ray_step settles equal distances).
//
// A child's planes are origin + q * 2^e with 8-bit q, and the builder encloses the child's box between
// the exact planes (quantize_node). Their slab distances come as one fused multiply-add each,
// t = q * (2^e inv) + (origin - o) inv: 2^e inv is exact, so a distance is off by the rounding of
// origin - o and of its product, at most 2.01 u |B| with B = (origin - o) inv, by the final rounding
// (1 u) and by the reciprocal's 2 u, a factor common to the axis. Near distances take B - 4u|B| and far
// ones B + 4u|B|, the far minimum is scaled by 1 + 2 gamma(4) > 1 + 6u, and tBox exceeds tMax by 2^-20
// of it: the test passes every box that exact arithmetic passes, boxes entered exactly at tMax included
// (a tie there may go to a lower leaf). A zero direction component (inv = +-2^100) passes exactly the
// slabs that hold the origin, but for a flat one at the node's minimum with the ray in its plane, whose
// triangles the ray is parallel to (det = 0).
constexpr float kTieScale = 1 + 0x1p-20f;

LTS_D void trace_node(TraceLane& l, const TraceRec* recs, float tMax, TraceStack ts, int* spill) {
    const void* rec = reinterpret_cast<const char*>(recs) + ((size_t)(unsigned)l.cur << 4);
    const GlobalU4 hd = load_global_u4(rec, 0), lo = load_global_u4(rec, 1), hi = load_global_u4(rec, 2);
    const float ax = __builtin_amdgcn_ldexpf(l.inv.x, (int)(int8_t)(hd.w & 0xffu));
    const float ay = __builtin_amdgcn_ldexpf(l.inv.y, (int)(int8_t)((hd.w >> 8) & 0xffu));
    const float az = __builtin_amdgcn_ldexpf(l.inv.z, (int)(int8_t)((hd.w >> 16) & 0xffu));
    const int count = (int)((hd.w >> 24) & 7u);
    const float bx = (word_f(hd.x) - l.o.x) * l.inv.x, by = (word_f(hd.y) - l.o.y) * l.inv.y, bz = (word_f(hd.z) - l.o.z) * l.inv.z;
    constexpr float k4u = 0x1p-22f;
    const float bxn = __builtin_fmaf(fabsf(bx), -k4u, bx), bxf = __builtin_fmaf(fabsf(bx), k4u, bx);
    const float byn = __builtin_fmaf(fabsf(by), -k4u, by), byf = __builtin_fmaf(fabsf(by), k4u, by);
    const float bzn = __builtin_fmaf(fabsf(bz), -k4u, bz), bzf = __builtin_fmaf(fabsf(bz), k4u, bz);
    // lo = (qlo x, qlo y, qlo z, qhi x), hi = (qhi y, qhi z, first child, -1); byte k belongs to child k
    const unsigned nearX = l.nx ? lo.w : lo.x, farX = l.nx ? lo.x : lo.w;
    const unsigned nearY = l.ny ? hi.x : lo.y, farY = l.ny ? lo.y : hi.x;
    const unsigned nearZ = l.nz ? hi.y : lo.z, farZ = l.nz ? lo.z : hi.y;
    const float g4 = 1 + 2 * gammaN(4), tBox = tMax * kTieScale;
    float t[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const unsigned s = 8 * k;
        const float tn = fmaxf(fmaxf(__builtin_fmaf((float)((nearX >> s) & 0xffu), ax, bxn),
                                     __builtin_fmaf((float)((nearY >> s) & 0xffu), ay, byn)),
                               __builtin_fmaf((float)((nearZ >> s) & 0xffu), az, bzn));
        const float tf = fminf(fminf(__builtin_fmaf((float)((farX >> s) & 0xffu), ax, bxf),
                                     __builtin_fmaf((float)((farY >> s) & 0xffu), ay, byf)),
                               __builtin_fmaf((float)((farZ >> s) & 0xffu), az, bzf));
        const float enter = fmaxf(tn, 0.0f), leave = fminf(tf * g4, tBox);
        t[k] = enter <= leave && (k < 2 || k < count) ? enter : INFINITY;  // a node has two children at least
    }
    // the nearest child next, the other three stacked with the nearer pair's loser on top
    const unsigned first = hi.z, leafBit = 0x80000000u;
    const int c0 = (int)(first | (hd.w & leafBit)), c1 = (int)((first + kRecUnits) | ((hd.w << 1) & leafBit)),
              c2 = (int)((first + 2 * kRecUnits) | ((hd.w << 2) & leafBit)),
              c3 = (int)((first + 3 * kRecUnits) | ((hd.w << 3) & leafBit));
    const bool sa = t[1] < t[0], sb = t[3] < t[2];
    const float ta = fminf(t[0], t[1]), tb = fminf(t[2], t[3]), ua = fmaxf(t[0], t[1]), ub = fmaxf(t[2], t[3]);
    const int ca = sa ? c1 : c0, da = sa ? c0 : c1, cb = sb ? c3 : c2, db = sb ? c2 : c3;
    const bool sw = tb < ta;
    const float tw = fminf(ta, tb), tl = fmaxf(ta, tb);
    const int cw = sw ? cb : ca, cl = sw ? ca : cb;
    if (__builtin_expect(__any(l.sp > kShortStack - 3), 0)) {
        const float pt[3] = {ua, ub, tl};
        const int pc[3] = {da, db, cl};
        for (int k = 0; k < 3; k++) {
            if (pt[k] < INFINITY) {
                if (l.sp < kShortStack) ts.lds[l.sp * ts.stride] = pc[k];
                else spill[l.sp - kShortStack] = pc[k];
                l.sp++;
            }
        }
    } else {
        // written whether or not the box was hit: an entry above the top is never read
        ts.lds[l.sp * ts.stride] = da;
        l.sp += ua < INFINITY;
        ts.lds[l.sp * ts.stride] = db;
        l.sp += ub < INFINITY;
        ts.lds[l.sp * ts.stride] = cl;
        l.sp += tl < INFINITY;
    }
    if (tw < INFINITY) l.cur = cw;
    else trace_pop(l, ts, spill);
}

// The triangle record at the lane's current entry.
struct TraceTri {
    V3 p0, p1, p2;
    int mat, leaf;
};
LTS_D TraceTri trace_triangle(const TraceLane& l, const TraceRec* recs) {
    const void* rec = reinterpret_cast<const char*>(recs) + ((size_t)((unsigned)l.cur & 0x7fffffffu) << 4);
    const GlobalU4 a = load_global_u4(rec, 0), b = load_global_u4(rec, 1), c = load_global_u4(rec, 2);
    TraceTri t;
    t.p0 = v3(word_f(a.x), word_f(a.y), word_f(a.z));
    t.p1 = v3(word_f(a.w), word_f(b.x), word_f(b.y));
    t.p2 = v3(word_f(b.z), word_f(b.w), word_f(c.x));
    t.mat = (int)c.z;
    t.leaf = (int)c.w;
    return t;
}

// ---------------------------------------------------------------- a wave of independent rays
// What a ray asks: the closest hit, whether a shadow ray is blocked (Triangle::simpleIntersect within the
// leaf's box), whether an MIS-BSDF ray is (any triangle that would win the closest hit against `best` at tMax).
enum RayKind { kRayNone = -1, kRayClosest, kRayShadow, kRayMis };

// One lane's ray of a wave whose lanes carry rays of any kind.
struct TraceRay {
    TraceLane l;
    const TraceRec* recs;
    V3 d;
    float tMax, u, v, invDet;  // the closest hit so far
    int best;                  // its leaf (-1: none); an MIS ray's tie leaf
    int mat;                   // its material; 1 for a light ray that is blocked
    int kind;
    int base;                  // stack index of the end marker
    int owner;                 // lane whose ray this is: its own, or the lane it helps
};

LTS_D void ray_none(TraceRay& t, int lane) {
    t.l.cur = kTraceDone; t.l.sp = 1; t.l.o = t.l.inv = t.d = v3(0, 0, 0);
    t.l.nx = t.l.ny = t.l.nz = false;
    t.recs = nullptr;
    t.tMax = t.u = t.v = t.invDet = 0;
    t.best = -1; t.mat = 0; t.kind = kRayNone; t.base = 0; t.owner = lane;
}

LTS_D void ray_begin(TraceRay& t, int kind, V3 o, V3 d, float tMax, int best, const TraceRec* recs, int root, TraceStack ts) {
    t.kind = kind;
    t.recs = recs;
    t.d = d;
    t.tMax = tMax;
    t.best = best;
    t.mat = 0;
    t.u = t.v = t.invDet = 0;
    t.base = 0;
    trace_begin(t.l, o, d, root, ts);
}

// One step of the wave: the node step for the lanes that hold a node, or the triangle step (fp64 cross
// products) for those that hold a triangle once they are half as many (kGateRatio). The records were checked
// when the scene was loaded (k_check_recs): children lie in range and after their node, so each traversal ends,
// and no accepted tree needs more than kStack entries.
//
// A triangle becomes the closest hit when it is nearer, or exactly as near with a lower leaf index.
// BVH::intersect (BVH.cuh:365-398) keeps the first triangle it meets at the closest distance, and its
// depth-first, left-first walk meets the leaves in index order, so of several triangles at exactly that distance
// the lowest leaf wins; this rule gives the same winner in any visiting order. A shadow ray's triangle test
// (Triangle::simpleIntersect, shapes/Triangle.cu:50-84) is the closest-hit test with the triangle's second and
// third corners exchanged and wider margins: it accepts points up to SHADOW_EPS outside the triangle's edges,
// and the reference reaches a triangle only through its leaf's box test (BVH.cuh:343-348: the leaf node's
// bounds, the primitive's own bounds). The render tree's quantized boxes are wider than that leaf box, so a
// triangle the enlarged test accepts is also put to the leaf-box test. (The closest-hit test accepts only points
// inside the triangle shrunk by SHADOW_EPS, which lie inside its bounds.)
constexpr int kGateRatio = 2;

template <bool kCount>
LTS_D void ray_step(TraceRay& t, TraceStack ts, int* spill, unsigned long long* tally) {
    const bool leafStep = t.l.cur < 0 && t.l.cur != kTraceDone;
    const unsigned long long waiting = __ballot(leafStep), walking = __ballot(t.l.cur >= 0);
    if (walking != 0 && kGateRatio * __popcll(waiting) < __popcll(walking)) {
        if (t.l.cur >= 0) {
            if (kCount) tally[0] += t.kind == kRayClosest, tally[2] += t.kind == kRayShadow, tally[4] += t.kind == kRayMis;
            trace_node(t.l, t.recs, t.tMax, ts, spill);
        }
    } else if (leafStep) {
        if (kCount) tally[1] += t.kind == kRayClosest, tally[3] += t.kind == kRayShadow, tally[5] += t.kind == kRayMis;
        const TraceTri tr = trace_triangle(t.l, t.recs);
        Ray r;
        r.o = t.l.o; r.d = t.d; r.tMax = t.tMax;
        const bool shadow = t.kind == kRayShadow;
        const V3 p1 = shadow ? tr.p2 : tr.p1, p2 = shadow ? tr.p1 : tr.p2;
        const float limit = shadow ? kOnePlusEpsF : kOneMinusEpsF;
        float h, u, v, id;
        bool over = false;
        if (tri_mt(tr.p0, p1, p2, r, limit, h, u, v, id) && h > 0 && (h < t.tMax || (h == t.tMax && !shadow && tr.leaf < t.best))) {
            if (t.kind == kRayClosest) {
                t.tMax = h;
                t.best = tr.leaf; t.mat = tr.mat; t.u = u; t.v = v; t.invDet = id;
            } else if (!shadow || leaf_box_passes(tr.p0, tr.p1, tr.p2, r)) {
                t.mat = 1;
                over = true;
            }
        }
        if (over) t.l.cur = kTraceDone;
        else trace_pop(t.l, ts, spill);
    }
}

// Sharing of a wave's last rays. A launch waits for its longest rays (a ray past the pole of a million-
// triangle sphere takes 2382 steps, the average path ray 13), and each step is a chain of dependent
// instructions and loads that no other lane's work hides by then. So once no rays are left to deal and
// at least kShareIdle lanes of the wave are free, every kShareSteps steps each lane that has stacked
// entries hands the one at the bottom of its stack, its largest subtree, to a free lane, which traverses
// it as a helper with the same ray. A ray's answer does not depend on the order of its visits, nor on who
// makes them: the helper keeps the closest hit of its part, which its owner takes if it is nearer, or
// equally near with a lower leaf. Longest trace launch of one sample of a 1280x720 frame of a 360k-triangle
// displaced sphere: 888 -> 266 us; all tracing of a 64-spp 1920x1080 frame of the 1M-triangle one: 27.5 ->
// 25.1 ms. Sharing from 32 free lanes on, or every 8 steps, measures the same.
constexpr int kShareIdle = 16, kShareSteps = 4;

LTS_D int lane_int(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
LTS_D float lane_float(float v, int lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane)); }
LTS_D int pull_int(int v, int lane) { return __builtin_amdgcn_ds_bpermute(4 * lane, v); }
LTS_D float pull_float(float v, int lane) { return __int_as_float(__builtin_amdgcn_ds_bpermute(4 * lane, __float_as_int(v))); }
LTS_D int lanes_below(unsigned long long m) {
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
}

// Gives the results of the helpers that have ended to their owners and frees them. Run by all lanes.
LTS_D void ray_settle(TraceRay& t, int lane) {
    unsigned long long m = __ballot(t.owner != lane && t.l.cur == kTraceDone);
    while (m) {
        const int h = __ffsll(m) - 1;
        m &= m - 1;
        const int owner = lane_int(t.owner, h), best = lane_int(t.best, h), mat = lane_int(t.mat, h);
        const float tMax = lane_float(t.tMax, h), u = lane_float(t.u, h), v = lane_float(t.v, h), id = lane_float(t.invDet, h);
        if (lane == owner) {
            if (t.kind != kRayClosest) {
                if (mat) { t.mat = 1; t.l.cur = kTraceDone; }
            } else if (tMax < t.tMax || (tMax == t.tMax && best < t.best)) {
                t.tMax = tMax; t.best = best; t.mat = mat; t.u = u; t.v = v; t.invDet = id;
            }
        }
        if (lane == h) { t.owner = lane; t.kind = kRayNone; }
    }
}

// Whether helpers are at work on the lane's own ray. mark: 64 bytes of the wave. Run by all lanes, after
// ray_settle.
LTS_D bool ray_held(const TraceRay& t, int lane, volatile uint8_t* mark) {
    mark[lane] = 0;
    __builtin_amdgcn_wave_barrier();
    if (t.owner != lane) mark[t.owner] = 1;
    __builtin_amdgcn_wave_barrier();
    return mark[lane] != 0;
}

// Hands stacked entries to free lanes; helpers take their owner's closest hit so far as their bound, and
// stop once their owner's light ray is blocked. Run by all lanes.
LTS_D void ray_share(TraceRay& t, bool free, int lane, TraceStack ts) {
    const float ownerT = pull_float(t.tMax, t.owner);
    const int ownerBest = pull_int(t.best, t.owner), ownerMat = pull_int(t.mat, t.owner);
    if (t.owner != lane) {
        if (t.kind != kRayClosest) {
            if (ownerMat) { t.l.cur = kTraceDone; t.mat = 1; }
        } else if (ownerT < t.tMax || (ownerT == t.tMax && ownerBest < t.best)) {
            t.tMax = ownerT; t.best = ownerBest;
        }
    }
    const bool gives = t.l.cur != kTraceDone && t.base + 1 < t.l.sp && t.base + 1 < kShortStack;
    const unsigned long long givers = __ballot(gives), takers = __ballot(free);
    const int pairs = min((int)__popcll(givers), (int)__popcll(takers));
    if (pairs > 0) {
        int entry = kTraceDone;
        const int rank = lanes_below(givers), nGivers = (int)__popcll(givers);
        if (gives) entry = ts.lds[(t.base + 1) * ts.stride];
        // lane r of `giver` holds the r-th giving lane
        const int giver = __builtin_amdgcn_ds_permute(4 * (gives ? rank : nGivers + lane - rank), lane);
        const int turn = lanes_below(takers);
        const bool takes = free && turn < pairs;
        const int from = pull_int(giver, turn);
        const int src = takes ? from : lane;
        TraceRay g;
        g.l.o = v3(pull_float(t.l.o.x, src), pull_float(t.l.o.y, src), pull_float(t.l.o.z, src));
        g.l.inv = v3(pull_float(t.l.inv.x, src), pull_float(t.l.inv.y, src), pull_float(t.l.inv.z, src));
        g.d = v3(pull_float(t.d.x, src), pull_float(t.d.y, src), pull_float(t.d.z, src));
        const uint64_t recs = (uint64_t)t.recs;
        const uint32_t lo = (uint32_t)pull_int((int)(uint32_t)recs, src), hi = (uint32_t)pull_int((int)(uint32_t)(recs >> 32), src);
        g.tMax = pull_float(t.tMax, src);
        g.best = pull_int(t.best, src); g.kind = pull_int(t.kind, src); g.owner = pull_int(t.owner, src);
        // a helper's own hit may pass to its owner by way of the lane it hands an entry to
        g.u = pull_float(t.u, src); g.v = pull_float(t.v, src); g.invDet = pull_float(t.invDet, src);
        g.mat = pull_int(t.mat, src);
        const int first = pull_int(entry, src);
        if (gives && rank < pairs) ts.lds[++t.base * ts.stride] = kTraceDone;
        if (takes) {
            t.l.o = g.l.o; t.l.inv = g.l.inv; t.d = g.d;
            t.l.nx = t.l.inv.x < 0; t.l.ny = t.l.inv.y < 0; t.l.nz = t.l.inv.z < 0;
            t.recs = reinterpret_cast<const TraceRec*>((uint64_t)lo | (uint64_t)hi << 32);
            t.tMax = g.tMax; t.best = g.best; t.kind = g.kind; t.owner = g.owner;
            t.u = g.u; t.v = g.v; t.invDet = g.invDet; t.mat = g.mat;
            t.base = 0;
            ts.lds[0] = kTraceDone;
            t.l.sp = 1;
            t.l.cur = first;
        }
    }
}

// Traces the wave's rays to their ends, sharing them among the lanes without one (kind kRayNone), which are
// without one again afterwards. Run by all lanes. A function of its own, with the stack's LDS address as a
// number (a generic pointer would make every access to it a flat one): inlined, its registers took the trace
// loop's.
__attribute__((noinline)) static __device__ void ray_finish_shared(TraceRay* ray, unsigned ldsAddress, int stride, int* spill) {
    const int lane = threadIdx.x & 63;
    const TraceStack ts{(int*)(__attribute__((address_space(3))) int*)ldsAddress, stride};
    TraceRay t = *ray;
    int wait = 0;
    while (__ballot(t.l.cur != kTraceDone)) {
        if (--wait < 0) {
            wait = kShareSteps;
            ray_settle(t, lane);
            ray_share(t, t.kind == kRayNone, lane, ts);
        }
        ray_step<false>(t, ts, spill, nullptr);
    }
    ray_settle(t, lane);
    *ray = t;
}
LTS_D void ray_finish_shared(TraceRay& t, TraceStack ts, int* spill) {
    TraceRay c = t;
    ray_finish_shared(&c, (unsigned)(uintptr_t)(__attribute__((address_space(3))) int*)ts.lds, ts.stride, spill);
    t = c;
}

// A lane's ray for trace_wave, and its answer: the closest hit (leaf -1: none), or whether a light ray is blocked.
struct RayQuery {
    int kind;  // kRayNone: the lane has no ray
    V3 o, d;
    float tMax;
};
struct RayAnswer {
    int leaf;
    float t, u, v, invDet;
    bool blocked;
};

// Traces one ray of every lane of the wave, all lanes taking part (BVH::intersect, BVH::simpleIntersect,
// acceleration/BVH.cuh:331-398): lanes whose ray has ended, or that have none, help the others. A function of
// its own, so that its registers are not the caller's. ldsAddress: the wave's kWaveTraceWords words.
constexpr int kWaveTraceWords = 64 * kShortStack + 16;
__attribute__((noinline)) static __device__ void trace_wave(const TraceRec* recs, int root, const RayQuery* query, RayAnswer* answer,
                                                            unsigned ldsAddress) {
    const int lane = threadIdx.x & 63;
    int* const lds = (int*)(__attribute__((address_space(3))) int*)ldsAddress;
    const TraceStack ts{lds + lane, 64};
    volatile uint8_t* const mark = reinterpret_cast<volatile uint8_t*>(lds + 64 * kShortStack);
    int spill[kStack - kShortStack];
    TraceRay t;
    ray_none(t, lane);
    if (query->kind != kRayNone) ray_begin(t, query->kind, query->o, query->d, query->tMax, -1, recs, root, ts);
    RayAnswer a;
    a.leaf = -1; a.t = a.u = a.v = a.invDet = 0; a.blocked = false;
    int wait = 0;
    for (;;) {
        const unsigned long long idle = __ballot(t.l.cur == kTraceDone);
        if (idle == ~0ull || (__popcll(idle) >= kShareIdle && --wait < 0)) {
            wait = kShareSteps;
            ray_settle(t, lane);
            const bool held = ray_held(t, lane, mark), free = t.l.cur == kTraceDone && !held;
            if (free && t.kind != kRayNone) {
                a.leaf = t.best; a.t = t.tMax; a.u = t.u; a.v = t.v; a.invDet = t.invDet;
                a.blocked = t.mat != 0;
                t.kind = kRayNone;
            }
            if (idle == ~0ull) break;
            ray_share(t, free, lane, ts);
        }
        ray_step<false>(t, ts, spill, nullptr);
    }
    *answer = a;
}
LTS_D RayAnswer trace_wave(const SceneView& sv, const RayQuery& query, int* lds) {
    RayQuery q = query;
    RayAnswer a;
    trace_wave(sv.recs, sv.root, &q, &a, (unsigned)(uintptr_t)(__attribute__((address_space(3))) int*)lds);
    return a;
}

// Triangle::intersect interaction part + SurfaceInteraction constructor / setShaddingGeometry
// (shapes/Triangle.cu:130-200, geometry/Interaction.cuh:85-116)
LTS_D SurfacePoint make_surface(const SceneView& sv, int leaf, const Ray& r, float u, float v, float invDet) {
    V3 p0, p1, p2; int prim;
    load_tri(sv.tris, leaf, p0, p1, p2, prim);
    const ShadeTri& st = sv.shade[leaf];
    V3 edge1 = p1 - p0, edge2 = p2 - p0;
    float w = 1 - u - v;
    V2 uv0 = v2(st.uv[0], st.uv[1]), uv1 = v2(st.uv[2], st.uv[3]), uv2 = v2(st.uv[4], st.uv[5]);
    V2 duv02 = uv0 - uv2, duv12 = uv1 - uv2;
    V3 dp02 = p0 - p2, dp12 = p1 - p2;
    float determinant = duv02.x * duv12.y - duv02.y * duv12.x;
    V3 dpdu, dpdv;
    if (determinant == 0) coordinateSystem(normalize(cross(edge2, edge1)), &dpdu, &dpdv);
    else {
        dpdu = (dp02 * duv12.y - dp12 * duv02.y) * invDet;
        dpdv = (dp02 * -duv12.x + dp12 * duv02.x) * invDet;
    }
    float xs = fabsf(w * p0.x) + fabsf(u * p1.x) + fabsf(v * p2.x);
    float ys = fabsf(w * p0.y) + fabsf(u * p1.y) + fabsf(v * p2.y);
    float zs = fabsf(w * p0.z) + fabsf(u * p1.z) + fabsf(v * p2.z);
    SurfacePoint s;
    s.pError = v3(xs, ys, zs) * gammaN(7);
    s.p = p0 * w + p1 * u + p2 * v;
    s.uv = uv0 * w + uv1 * u + uv2 * v;
    s.wo = -r.d;
    s.dpdu = dpdu;
    s.n = normalize(cross(dpdu, dpdv));
    s.sn = s.n;
    s.sdpdu = dpdu;
    s.leaf = leaf;
    s.dpdx = s.dpdy = v3(0, 0, 0);
    s.dpdv = dpdv;
    s.dudx = s.dvdx = s.dudy = s.dvdy = 0.0f;
    if (st.hasN) {
        V3 n0 = v3(st.n[0], st.n[1], st.n[2]), n1 = v3(st.n[3], st.n[4], st.n[5]), n2 = v3(st.n[6], st.n[7], st.n[8]);
        V3 ns = normalize(n0 * w + n1 * u + n2 * v);
        V3 tg = s.dpdu;
        V3 bt = cross(ns, tg);
        if (lengthSq(bt) > 0.0f) { bt = normalize(bt); tg = cross(bt, ns); }
        else coordinateSystem(ns, &tg, &bt);
        s.sn = normalize(cross(tg, bt));
        s.n = faceTowards(s.n, s.sn);
        s.sdpdu = tg;
        s.n = faceTowards(s.n, s.sn);
    }
    return s;
}

LTS_D Ray spawn_ray(const SurfacePoint& it, V3 d) {
    Ray r;
    r.o = offsetRayOrigin(it.p, it.pError, it.n, d);
    r.d = d;
    r.tMax = INFINITY;
    return r;
}

// ---------------------------------------------------------------- sampling (sampling/Sampling.cuh)
LTS_D V2 uniform_disk(V2 u) {
    float r = sqrtf(u.x);
    float theta = 2 * PI_F * u.y;
    float sn, cs;
    f_sincos(theta, sn, cs);
    return v2(r * cs, r * sn);
}
LTS_D V3 cosine_hemisphere(V2 u) {
    V2 d = uniform_disk(u);
    float z = sqrtf(fmaxf(0.0f, 1 - d.x * d.x - d.y * d.y));
    return v3(d.x, d.y, z);
}
LTS_D V3 uniform_hemisphere(V2 u) {
    float z = u.x;
    float r = sqrtf(fmaxf(0.0f, 1.0f - z * z));
    float phi = 2 * PI_F * u.y;
    float sn, cs;
    f_sincos(phi, sn, cs);
    return v3(r * cs, r * sn, z);
}
LTS_D float power_heuristic(float fPdf, float gPdf) {
    float f = 1 * fPdf, g = 1 * gPdf;
    return (f * f) / (f * f + g * g);
}

// ---------------------------------------------------------------- BxDFs (materials/models/*.cuh)
enum { B_REFL = 1, B_TRANS = 2, B_DIFF = 4, B_GLOSSY = 8, B_SPEC = 16, B_ALL = 31 };

LTS_D float cosT(V3 w) { return w.z; }
LTS_D float absCosT(V3 w) { return fabsf(w.z); }
LTS_D float cos2T(V3 w) { return w.z * w.z; }
LTS_D float sin2T(V3 w) { return fmaxf(1 - cos2T(w), 0.0f); }
LTS_D float sinT(V3 w) { return sqrtf(sin2T(w)); }
LTS_D float tanT(V3 w) { return sinT(w) / cosT(w); }
LTS_D float tan2T(V3 w) { return sin2T(w) / cos2T(w); }
LTS_D float cosPhi(V3 w) { float s = sinT(w); return clampf(w.x / s, -1, 1); }  // BxDF.cuh:144-147
LTS_D float sinPhi(V3 w) { float s = sinT(w); return clampf(w.y / s, -1, 1); }
LTS_D float cos2Phi(V3 w) { return cosPhi(w) * cosPhi(w); }
LTS_D float sin2Phi(V3 w) { return sinPhi(w) * sinPhi(w); }
LTS_D bool sameHemi(V3 a, V3 b) { return a.z * b.z > 0; }

// fresnelReflectionDielectric (BxDF.cuh:16-37), including its clamp(cos, 1, -1)
LTS_D float fr_dielectric(float cosThetaI, float etaI, float etaT) {
    cosThetaI = clampf(cosThetaI, 1, -1);
    bool entering = cosThetaI > 0.0f;
    if (!entering) { float tmp = etaI; etaI = etaT; etaT = tmp; cosThetaI = fabsf(cosThetaI); }
    float sinThetaI = sqrtf(fmaxf(0.0f, 1 - cosThetaI * cosThetaI));
    float sinThetaT = etaI / etaT * sinThetaI;
    if (sinThetaT >= 1) return 1;
    float cosThetaT = sqrtf(fmaxf(0.0f, 1 - sinThetaT * sinThetaT));
    float rpar = ((etaT * cosThetaI) - (etaI * cosThetaT)) / ((etaT * cosThetaI) + (etaI * cosThetaT));
    float rperp = ((etaI * cosThetaI) - (etaT * cosThetaT)) / ((etaI * cosThetaI) + (etaT * cosThetaT));
    return (rpar * rpar + rperp * rperp) / 2;
}
LTS_D bool refract_dir(V3 wi, V3 n, float eta, V3* wt) {
    float cosThetaI = dot(n, wi);
    float sin2ThetaI = fmaxf(0.0f, 1.0f - cosThetaI * cosThetaI);
    float sin2ThetaT = eta * eta * sin2ThetaI;
    if (sin2ThetaT >= 1) return false;
    float cosThetaT = sqrtf(1 - sin2ThetaT);
    *wt = -wi * eta + n * (eta * cosThetaI - cosThetaT);
    return true;
}

// Trowbridge-Reitz distribution (Microfacet.cuh:124-181)
LTS_D float tr_lambda(V3 w, float ax, float ay) {
    float absTan = fabsf(tanT(w));
    if (isinf(absTan)) return 0.0f;
    float alpha = sqrtf(cos2Phi(w) * ax * ax + sin2Phi(w) * ay * ay);
    float a2t2 = (alpha * absTan) * (alpha * absTan);
    return (-1 + sqrtf(1.0f + a2t2)) / 2;
}
LTS_D float tr_D(V3 wh, float ax, float ay) {
    float tan2 = tan2T(wh);
    if (isinf(tan2)) return 0;
    const float cos4 = cos2T(wh) * cos2T(wh);
    float e = (cos2Phi(wh) / (ax * ax) + sin2Phi(wh) / (ay * ay)) * tan2;
    return 1 / (PI_F * ax * ay * cos4 * (1 + e) * (1 + e));
}
LTS_D float tr_G1(V3 w, float ax, float ay) { return 1 / (1 + tr_lambda(w, ax, ay)); }
LTS_D float tr_G(V3 wo, V3 wi, float ax, float ay) { return 1 / (1 + tr_lambda(wo, ax, ay) + tr_lambda(wi, ax, ay)); }
LTS_D float tr_pdf(V3 wo, V3 wh, float ax, float ay) { return tr_D(wh, ax, ay) * tr_G1(wo, ax, ay) * absDot(wo, wh) / absCosT(wo); }

// TrowbridgeReitzSample11 / TrowbridgeReitzSample (Microfacet.cuh:53-121)
LTS_D void tr_sample11(float cosTheta, float U1, float U2, float* sx, float* sy) {
    if ((double)cosTheta > .9999) {
        float r = sqrtf(U1 / (1 - U1));
        float phi = (float)(6.28318530718 * (double)U2);
        float sn, cs;
        f_sincos(phi, sn, cs);
        *sx = r * cs;
        *sy = r * sn;
        return;
    }
    float sinTheta = sqrtf(fmaxf(0.0f, 1.0f - cosTheta * cosTheta));
    float tanTheta = sinTheta / cosTheta;
    float a = 1 / tanTheta;
    float G1 = 2 / (1 + sqrtf(1.f + 1.f / (a * a)));
    float A = 2 * U1 / G1 - 1;
    float tmp = 1.f / (A * A - 1.f);
    if ((double)tmp > 1e10) tmp = (float)1e10;
    float B = tanTheta;
    float D = sqrtf(fmaxf(float(B * B * tmp * tmp - (A * A - B * B) * tmp), 0.0f));
    float sx1 = B * tmp - D, sx2 = B * tmp + D;
    *sx = (A < 0 || sx2 > 1.f / tanTheta) ? sx1 : sx2;
    float S;
    if (U2 > 0.5f) { S = 1.f; U2 = 2.f * (U2 - .5f); }
    else { S = -1.f; U2 = 2.f * (.5f - U2); }
    float z = (U2 * (U2 * (U2 * 0.27385f - 0.73369f) + 0.46341f)) /
              (U2 * (U2 * (U2 * 0.093073f + 0.309420f) - 1.000000f) + 0.597999f);
    *sy = S * z * sqrtf(1.f + *sx * *sx);
}
LTS_D V3 tr_sample(V3 wi, float ax, float ay, float U1, float U2) {
    V3 ws = normalize(v3(ax * wi.x, ay * wi.y, wi.z));
    float sx, sy;
    tr_sample11(cosT(ws), U1, U2, &sx, &sy);
    float tmp = cosPhi(ws) * sx - sinPhi(ws) * sy;
    sy = sinPhi(ws) * sx + cosPhi(ws) * sy;
    sx = tmp;
    sx = ax * sx;
    sy = ay * sy;
    return normalize(v3(-sx, -sy, (float)1.));
}

// The BSDF of one hit: at most one BxDF (Material.cuh:31-130 and the microfacet mirror extension).
struct Bsdf {
    V3 ns, ng, ss, ts;
    int kind;   // -1 none, 0 Lambert, 1 OrenNayar, 2 SpecularReflection, 3 FresnelSpecular, 4 MicrofacetReflection
    int type;
    Spec R, T;
    float A, B, eta, alpha;

    LTS_D V3 toLocal(V3 v) const { return v3(dot(v, ss), dot(v, ts), dot(v, ns)); }
    LTS_D V3 toWorld(V3 v) const {
        return v3(ss.x * v.x + ts.x * v.y + ns.x * v.z, ss.y * v.x + ts.y * v.y + ns.y * v.z, ss.z * v.x + ts.z * v.y + ns.z * v.z);
    }
    LTS_D bool matches(int flags) const { return kind >= 0 && (type & flags) == type; }

    LTS_D Spec fLocal(V3 wo, V3 wi) const {
        if (kind == 0) return R * INV_PI_F;
        if (kind == 1) {
            float sinThetaO = sinT(wo), sinThetaI = sinT(wi);
            float maxCos = 0.0f;
            if ((double)sinThetaI > 1e-4 && (double)sinThetaO > 1e-4) {
                float sinPhiO = sinPhi(wo), cosPhiO = cosPhi(wo);
                float sinPhiI = sinPhi(wi), cosPhiI = cosPhi(wi);
                float dCos = cosPhiI * cosPhiO + sinPhiI * sinPhiO;
                maxCos = fmaxf(0.0f, dCos);
            }
            float sinAlpha, tanBeta;
            if (absCosT(wi) > absCosT(wo)) { sinAlpha = sinThetaO; tanBeta = sinThetaI / absCosT(wi); }
            else { sinAlpha = sinThetaI; tanBeta = sinThetaO / absCosT(wo); }
            return R * INV_PI_F * (A + B * maxCos * sinAlpha * tanBeta);
        }
        if (kind == 4) {
            float cosThetaO = absCosT(wo), cosThetaI = absCosT(wi);
            V3 wh = wi + wo;
            if (cosThetaI == 0 || cosThetaO == 0) return spec(0.0f);
            if (wh.x == 0.0f && wh.y == 0.0f && wh.z == 0.0f) return spec(0.0f);
            wh = normalize(wh);
            Spec F = spec(1.0f);
            return R * tr_D(wh, alpha, alpha) * tr_G(wo, wi, alpha, alpha) * F / (4 * cosThetaI * cosThetaO);
        }
        return spec(0.0f);
    }
    LTS_D float pdfLocal(V3 wo, V3 wi) const {
        if (kind == 0 || kind == 1) return sameHemi(wo, wi) ? absCosT(wi) * INV_PI_F : 0;
        if (kind == 4) {
            if (!sameHemi(wo, wi)) return 0;
            V3 wh = normalize(wo + wi);
            return tr_pdf(wo, wh, alpha, alpha) / (4 * dot(wo, wh));
        }
        return 0.0f;
    }
    // BSDF::f (BSDF.cuh:60-72)
    LTS_D Spec f(V3 woW, V3 wiW, int flags) const {
        V3 wi = toLocal(wiW), wo = toLocal(woW);
        bool reflect = dot(wiW, ng) * dot(woW, ng) > 0;
        Spec r = spec(0.0f);
        if (matches(flags) && ((reflect && (type & B_REFL)) || (!reflect && (type & B_TRANS)))) r = r + fLocal(wo, wi);
        return r;
    }
    // BSDF::Pdf (BSDF.cuh:129-144)
    LTS_D float pdf(V3 woW, V3 wiW, int flags) const {
        if (kind < 0) return 0.0f;
        V3 wo = toLocal(woW), wi = toLocal(wiW);
        if (wo.z == 0) return 0.0f;
        float p = 0.0f;
        int m = 0;
        if (matches(flags)) { m++; p = p + pdfLocal(wo, wi); }
        return m > 0 ? p / m : 0.0f;
    }
    // BSDF::sampleF (BSDF.cuh:74-127) with one component
    LTS_D Spec sampleF(V3 woW, V3* wiW, V2 u, float* pdfOut, int flags, int* sampledType) const {
        if (!matches(flags)) { *pdfOut = 0; return spec(0.0f); }
        V3 wo = toLocal(woW), wi;
        *pdfOut = 0;
        *sampledType = type;
        Spec f = spec(0.0f);
        switch (kind) {
            case 0: case 1:
                wi = cosine_hemisphere(u);
                if (wo.z < 0) wi.z *= -1;
                *pdfOut = pdfLocal(wo, wi);
                f = fLocal(wo, wi);
                break;
            case 2:
                wi = v3(-wo.x, -wo.y, wo.z);
                *pdfOut = 1.0f;
                f = (spec(1.0f) * R) / absCosT(wi);
                break;
            case 3: {
                float F = fr_dielectric(cosT(wo), 1.0f, eta);
                if (u.x < F) {
                    wi = v3(-wo.x, -wo.y, -wo.z);
                    *sampledType = B_SPEC | B_REFL;
                    *pdfOut = F;
                    f = F * R / absCosT(wi);
                } else {
                    bool entering = cosT(wo) > 0;
                    float etaI = entering ? 1.0f : eta, etaT = entering ? eta : 1.0f;
                    if (!refract_dir(wo, faceTowards(v3(0, 0, 1), wo), etaI / etaT, &wi)) return spec(0.0f);
                    Spec ft = T * (1 - F);
                    ft = ft * ((etaI * etaI) / (etaT * etaT));
                    *sampledType = B_SPEC | B_TRANS;
                    *pdfOut = 1.0f - F;
                    f = ft / absCosT(wi);
                }
                break;
            }
            case 4: {
                if (wo.z == 0) return spec(0.0f);
                bool flip = wo.z < 0;
                V3 wh = tr_sample(flip ? -wo : wo, alpha, alpha, u.x, u.y);
                if (flip) wh = -wh;
                if (dot(wo, wh) < 0) return spec(0.0f);
                wi = -wo + wh * (2 * dot(wo, wh));
                if (!sameHemi(wo, wi)) return spec(0.0f);
                *pdfOut = tr_pdf(wo, wh, alpha, alpha) / (4 * dot(wo, wh));
                f = fLocal(wo, wi);
                break;
            }
        }
        if (*pdfOut == 0) return spec(0.0f);
        *wiW = toWorld(wi);
        return f;
    }
};

// ---------------------------------------------------------------- textures (Procedural.cuh)
LTS_D float noise_weight(float t) { float t3 = t * t * t; float t4 = t3 * t; return 6 * t4 * t - 15 * t4 + 10 * t3; }
LTS_D float smooth_step(float mn, float mx, float val) {
    float v = clampf((val - mn) / (mx - mn), 0, 1);
    return v * v * (-2 * v + 3);
}
// The noise's tables in LDS: the permutation, whose three chained lookups a kernel's lanes make eight
// times per noise value, and for each entry the gradient its last lookup selects (x, y, z in {-1, 0, 1}
// as fp16 pairs): the reference's choice of two coordinates and their signs (Procedural.cuh grad) as a
// dot product of three mixed-precision fused operations, exact but for the one rounding of the sum of
// its two nonzero terms, as the reference's addition rounds.
struct NoiseTables {
    int perm[512];
    uint2 grad[512];
};
LTS_D void noise_tables(NoiseTables& t, const int* __restrict__ perm, int tid, int threads) {
    for (int i = tid; i < 512; i += threads) {
        const int w = perm[i], h = w & 15;
        const unsigned one = 0x3c00u, su = (h & 1) ? 0x8000u : 0u, sv = (h & 2) ? 0x8000u : 0u;
        const bool ux = h < 8 || h == 12 || h == 13, vy = h < 4 || h == 12 || h == 13;
        const unsigned gx = ux ? one | su : 0u, gy = (ux ? 0u : one | su) | (vy ? one | sv : 0u), gz = vy ? 0u : one | sv;
        t.perm[i] = w;
        t.grad[i] = make_uint2(gx | (gy << 16), gz);
    }
}
LTS_D float grad(const NoiseTables& t, int i, float dx, float dy, float dz) {
    typedef _Float16 Half2 __attribute__((ext_vector_type(2)));
    const uint2 g = t.grad[i];
    const Half2 xy = __builtin_bit_cast(Half2, g.x), z = __builtin_bit_cast(Half2, g.y);
    return __builtin_fmaf((float)xy.x, dx, __builtin_fmaf((float)xy.y, dy, __builtin_fmaf((float)z.x, dz, 0.0f)));
}
LTS_D float perlin(const NoiseTables& t, V3 p) {
    int ix = (int)floorf(p.x), iy = (int)floorf(p.y), iz = (int)floorf(p.z);
    float dx = p.x - ix, dy = p.y - iy, dz = p.z - iz;
    ix &= 255; iy &= 255; iz &= 255;
    const int p0 = t.perm[ix] + iy, p1 = t.perm[ix + 1] + iy;
    const int p00 = t.perm[p0] + iz, p01 = t.perm[p0 + 1] + iz, p10 = t.perm[p1] + iz, p11 = t.perm[p1 + 1] + iz;
    float w000 = grad(t, p00, dx, dy, dz);
    float w100 = grad(t, p10, dx - 1, dy, dz);
    float w010 = grad(t, p01, dx, dy - 1, dz);
    float w001 = grad(t, p00 + 1, dx, dy, dz - 1);
    float w110 = grad(t, p11, dx - 1, dy - 1, dz);
    float w011 = grad(t, p01 + 1, dx, dy - 1, dz - 1);
    float w101 = grad(t, p10 + 1, dx - 1, dy, dz - 1);
    float w111 = grad(t, p11 + 1, dx - 1, dy - 1, dz - 1);
    float wx = noise_weight(dx), wy = noise_weight(dy), wz = noise_weight(dz);
    float x00 = lerpf(wx, w000, w100), x10 = lerpf(wx, w010, w110);
    float x01 = lerpf(wx, w001, w101), x11 = lerpf(wx, w011, w111);
    float y0 = lerpf(wy, x00, x10), y1 = lerpf(wy, x01, x11);
    return lerpf(wz, y0, y1);
}
// Octaves of a footprint: clamp(-1 - log2(len2) / 2, 0, maxOct). At or below 2^(-2 maxOct - 2) (every
// hit after the first bounce, which has no footprint, and most first ones) it is maxOct: rounding is
// monotone, so the rounded logarithm is at most -2 maxOct - 2.
LTS_D float noise_octaves(V3 dpdx, V3 dpdy, int maxOct) {
    float len2 = fmaxf(lengthSq(dpdx), lengthSq(dpdy));
    if (maxOct >= 0 && len2 <= __builtin_amdgcn_ldexpf(1.0f, -2 * maxOct - 2)) return (float)maxOct;
    return clampf(-1 - 0.5f * f_log2(len2), 0, (float)maxOct);
}
// fbm (turb false) or turbulence over n = noise_octaves octaves: the whole ones, then the fraction, with
// one copy of the noise code for all of them (every inlined copy is 1.5 KB of instructions, and the
// shading kernels once held thirty). The fraction is skipped where its weight is 0 (a whole number of
// octaves): one noise value in seven at six octaves.
LTS_D float noise_sum(const NoiseTables& T, V3 p, float n, float omega, int maxOct, bool turb) {
    const int nInt = (int)floorf(n);
    const float part = smooth_step(0.3f, 0.7f, n - nInt);
    const int count = nInt + (part != 0);
    float sum = 0, lambda = 1, o = 1;
#pragma unroll 1
    for (int i = 0; i < count; i++) {
        float v = perlin(T, p * lambda);
        if (turb) v = fabsf(v);
        if (i < nInt) {
            sum += o * v;
            lambda *= 1.99f;
            o *= omega;
        } else {
            sum += turb ? o * lerpf(part, 0.2f, v) : o * part * v;
        }
    }
    if (turb) {
        if (part == 0) sum += o * 0.2f;
#pragma unroll 1
        for (int i = nInt; i < maxOct; i++) { sum += o * 0.2f; o *= omega; }
    }
    return sum;
}
// MarbleTexture's colour at m = p.y + variation * fbm
LTS_D Spec marble_colour(float m) {
    // MarbleTexture colours (Procedural.cuh:278-282); the zero row stands in for the read past the
    // table at t == 1, where its weight is exactly 0
    const float C[10][3] = {{.58f, .58f, .6f}, {.58f, .58f, .6f}, {.58f, .58f, .6f}, {.5f, .5f, .5f},
                            {.6f, .59f, .58f}, {.58f, .58f, .6f}, {.58f, .58f, .6f}, {.2f, .2f, .33f},
                            {.58f, .58f, .6f}, {0, 0, 0}};
    float t = 0.5f + 0.5f * f_sin(m);
    int first = (int)floorf(t * 6.0f);
    first = first < 0 ? 0 : (first > 6 ? 6 : first);  // t is in [0, 1]; the clamp only fences NaN
    t = (t * 6.0f - first);
    Spec c0 = spec(C[first][0], C[first][1], C[first][2]);
    Spec c1 = spec(C[first + 1][0], C[first + 1][1], C[first + 1][2]);
    Spec c2 = spec(C[first + 2][0], C[first + 2][1], C[first + 2][2]);
    Spec c3 = spec(C[first + 3][0], C[first + 3][1], C[first + 3][2]);
    Spec s0 = (1.0f - t) * c0 + t * c1;
    Spec s1 = (1.0f - t) * c1 + t * c2;
    Spec s2 = (1.0f - t) * c2 + t * c3;
    s0 = (1.0f - t) * s0 + t * s1;
    s1 = (1.0f - t) * s1 + t * s2;
    return 1.5f * ((1.0f - t) * s0 + t * s1);
}

// Mipmap texel / triangle / lookUp (materials/textures/Mipmap.cuh:14-72)
LTS_D Spec mip_texel(const SceneView& sv, const MipDesc& m, int s, int t, int l) {
    const MipLevelDesc& L = m.lv[l];
    if (m.filtered) {
        // row-major texels; repeat wraps to [0, res), clamp clamps, black is zero outside
        if (m.wrap == 0) { s = ((s % L.ures) + L.ures) % L.ures; t = ((t % L.vres) + L.vres) % L.vres; }
        else if (m.wrap == 2) { s = min(max(s, 0), L.ures - 1); t = min(max(t, 0), L.vres - 1); }
        else if (s < 0 || s >= L.ures || t < 0 || t >= L.vres) return spec(0.0f);
        const float* px = sv.mipData + 3 * (L.offset + (long long)t * L.ures + s);
        return spec(px[0], px[1], px[2]);
    }
    if (m.wrap == 0) { s = (int)fmodf((float)s, (float)L.ures); t = (int)fmodf((float)t, (float)L.vres); }
    else if (m.wrap == 2) { s = (int)clampf((float)s, 0, (float)(L.ures - 1)); t = (int)clampf((float)t, 0, (float)(L.vres - 1)); }
    else if (s < 0 || s >= L.ures || t < 0 || t >= L.vres) return spec(0.0f);
    if (s < 0 || t < 0 || s >= L.ures || t >= L.vres) return spec(0.0f);
    long long slot = L.offset + 16LL * ((long long)L.ublocks * (t >> 2) + (s >> 2)) + 4LL * (t >> 2) + (s & 3);
    const float* px = sv.mipData + 3 * slot;
    return spec(px[0], px[1], px[2]);
}
LTS_D Spec mip_triangle(const SceneView& sv, const MipDesc& m, int l, V2 st) {
    l = (int)clampf((float)l, 0, (float)(m.levels - 1));
    float s = st.x * m.lv[l].ures - 0.5f;
    float t = st.y * m.lv[l].vres - 0.5f;
    int s0 = (int)floorf(s), t0 = (int)floorf(t);
    float ds = s - s0, dt = t - t0;
    return (1 - ds) * (1 - dt) * mip_texel(sv, m, s0, t0, l) + (1 - ds) * dt * mip_texel(sv, m, s0, t0 + 1, l) +
           ds * (1 - dt) * mip_texel(sv, m, s0 + 1, t0, l) + ds * dt * mip_texel(sv, m, s0 + 1, t0 + 1, l);
}
// The reference's fixed width 0.01 gives a precomputed level; the filtered pipeline takes the
// width of the lookup and reads the top level correctly (the reference swaps texel's arguments
// there: texel (levels - 1, 0) of level 0).
LTS_D Spec mip_lookup(const SceneView& sv, const MipDesc& m, V2 st, float width) {
    float levels = m.filtered ? (float)(m.levels - 1) + f_log2(fmaxf(width, (float)1e-8)) : m.lookupLevel;
    if (levels < 0) return mip_triangle(sv, m, 0, st);
    if (levels >= m.levels - 1) return m.filtered ? mip_texel(sv, m, 0, 0, m.levels - 1) : mip_texel(sv, m, m.levels - 1, 0, 0);
    int iLevel = (int)floorf(levels);
    float delta = levels - iLevel;
    return lerpS(delta, mip_triangle(sv, m, iLevel, st), mip_triangle(sv, m, iLevel + 1, st));
}

LTS_D Spec eval_tex(const SceneView& sv, int ti, const SurfacePoint& s, const NoiseTables& noise) {
    const TexDesc& X = sv.texs[ti];
    if (X.type == TEX_CONST) return spec(X.c[0], X.c[1], X.c[2]);
    if (X.type == TEX_IMAGE) {
        // filtered pipeline: PBRT's isotropic width 2 max(|ds/dx|, |dt/dx|, |ds/dy|, |dt/dy|) of
        // UVMapping2D (st = uv, Mapping.cuh:19-37); the reference's lookup ignores it
        const float width = 2 * fmaxf(fmaxf(fabsf(s.dudx), fabsf(s.dvdx)), fmaxf(fabsf(s.dudy), fabsf(s.dvdy)));
        return mip_lookup(sv, sv.mips[X.img], v2(1 * s.uv.x + 0, 1 * s.uv.y + 0), width);
    }
    const bool marble = X.type == TEX_MARBLE;
    if (!marble && X.type != TEX_FBM && X.type != TEX_WRINKLED) return spec(0.0f);
    V3 p = identityMap(s.p), dx = identityMap(s.dpdx), dy = identityMap(s.dpdy);
    if (marble) { p = p * X.scale; dx = dx * X.scale; dy = dy * X.scale; }
    const float v = noise_sum(noise, p, noise_octaves(dx, dy, X.octaves), X.omega, X.octaves, X.type == TEX_WRINKLED);
    return marble ? marble_colour(p.y + X.variation * v) : spec(v);
}

// Material::computeScatteringFunctions (materials/Material.cuh:31-130)
LTS_D Bsdf make_bsdf(const SceneView& sv, const SurfacePoint& s, const NoiseTables& noise) {
    Bsdf b;
    b.ns = s.sn; b.ng = s.n;
    b.ss = normalize(s.sdpdu);
    b.ts = cross(b.ns, b.ss);
    b.kind = -1; b.type = 0;
    b.R = b.T = spec(0.0f);
    b.A = b.B = b.eta = b.alpha = 0;
    const MatDesc& M = sv.mats[sv.shade[s.leaf].mat];
    Spec r = spec(0.0f), t = spec(0.0f);
#pragma unroll 1
    for (int k = 0; k < (M.type == MAT_GLASS ? 2 : 1); k++) {  // one copy of the texture code
        t = eval_tex(sv, k ? M.tex1 : M.tex0, s, noise);
        if (k == 0) r = t;
    }
    if (isBlack(r) && (M.type != MAT_GLASS || isBlack(t))) return b;
    b.R = r;
    switch (M.type) {
        case MAT_MATTE: b.type = B_REFL | B_DIFF; b.kind = M.extra == 0 ? 0 : 1; b.A = M.onA; b.B = M.onB; break;
        case MAT_GLASS: b.kind = 3; b.type = B_REFL | B_TRANS | B_SPEC; b.T = t; b.eta = M.extra; break;
        case MAT_MIRROR: b.kind = 2; b.type = B_REFL | B_SPEC; break;
        case MAT_MICROFACET: b.kind = 4; b.type = B_REFL | B_GLOSSY; b.alpha = M.alpha; break;
    }
    return b;
}

// ---------------------------------------------------------------- lights (lights/Light.cu)
struct LightPoint { V3 p, n, pError; };

LTS_D LightPoint tri_sample(const SceneView& sv, const LightDesc& L, V2 u) {
    float t = sqrtf(u.x);
    V2 b = v2(1 - t, u.y * t);
    V3 p0, p1, p2; int prim;
    load_tri(sv.tris, L.leaf, p0, p1, p2, prim);
    const ShadeTri& st = sv.shade[L.leaf];
    LightPoint lp;
    lp.p = p0 * b.x + p1 * b.y + p2 * (1 - b.x - b.y);
    if (st.hasN)
        lp.n = normalize(v3(st.n[0], st.n[1], st.n[2]) * b.x + v3(st.n[3], st.n[4], st.n[5]) * b.y +
                         v3(st.n[6], st.n[7], st.n[8]) * (1 - b.x - b.y));
    else
        lp.n = normalize(cross(p1 - p0, p2 - p0));
    V3 pAbs = vabs(p0 * b.x) + vabs(p1 * b.y) + vabs(p2 * (1 - b.x - b.y));
    lp.pError = pAbs * gammaN(6);
    return lp;
}

// Where a ray r spawned from `it` meets the triangle of area light L: the distance, whether it meets
// the emitting side, and Triangle::Pdf(it, r.d) (shapes/Triangle.cu:211-225). False for a miss.
struct LightHit {
    float t, pdf;
    bool front;
};
LTS_D bool light_hit(const SceneView& sv, const LightDesc& L, const SurfacePoint& it, const Ray& r, LightHit& h) {
    V3 p0, p1, p2; int prim;
    load_tri(sv.tris, L.leaf, p0, p1, p2, prim);
    float t, u, v, id;
    h.pdf = 0;
    if (!tri_hit(p0, p1, p2, r, t, u, v, id)) return false;
    SurfacePoint is = make_surface(sv, L.leaf, r, u, v, id);
    h.t = t;
    h.front = dot(is.n, -r.d) > 0.f;
    h.pdf = lengthSq(it.p - is.p) / (absDot(is.n, -r.d) * L.area);
    return true;
}

LTS_D float inf_pdf(V3 wi) {
    float sinTheta = f_sin_acos(clampf(wi.z, -1.0f, 1.0f));
    return (0.5f * INV_PI_F) / (2 * PI_F * PI_F * sinTheta);
}

LTS_D Spec light_le(const LightDesc& L) { return spec(L.le[0], L.le[1], L.le[2]); }

LTS_D Spec sample_li(const SceneView& sv, const LightDesc& L, const SurfacePoint& it, V2 u, V3* wi, float* pdf, LightPoint* target) {
    if (L.kind == 0) {
        LightPoint ps = tri_sample(sv, L, u);
        *wi = normalize(ps.p - it.p);
        LightHit lh;
        light_hit(sv, L, it, spawn_ray(it, *wi), lh);
        *pdf = lh.pdf;
        *target = ps;
        return dot(ps.n, -*wi) > 0.f ? light_le(L) : spec(0.0f);
    }
    V3 w = uniform_hemisphere(u);
    V3 ref = v3(0, 1, 0), a, b;
    coordinateSystem(ref, &a, &b);
    w = a * w.x + b * w.y + ref * w.z;
    V3 pL = v3(L.center[0], L.center[1], L.center[2]) + w * L.radius;
    *wi = normalize(pL - it.p);
    *pdf = inf_pdf(*wi);
    target->p = pL; target->n = v3(0, 0, 0); target->pError = v3(0, 0, 0);
    return light_le(L);
}

// Distribution1D::sampleDiscrete with the reference's search length (Sampling.cuh:155-188)
LTS_D int sample_light(const SceneView& sv, float u, float* pdf) {
    int size = sv.nLights, off;
    if (size == 1) off = 0;
    else {
        int first = 0, len = size;
        while (len > 0) {
            int half = len >> 1, middle = first + half;
            if (sv.lcdf[middle] <= u) { first = middle + 1; len -= half + 1; }
            else len = half;
        }
        off = (int)clampf((float)(first - 1), 0, (float)(size - 2));
    }
    *pdf = sv.lfunc[off] / (sv.funcInt * size);
    return off;
}

// The MIS-BSDF ray r = spawn_ray(si, wi) toward light li (IntegratorHelper.cuh:96-122): false when it
// contributes nothing whatever lies in its way; else the weight of its contribution, and the any-hit
// traversal that is left to do. The reference finds the closest hit and asks whether it is the light's
// triangle seen from its emitting side, or for the infinite light whether the ray escapes. A ray that
// misses the light's triangle, or meets its back, never contributes. A ray that meets its front at t
// reaches it unless some triangle would win the closest hit against it (nearer, or at exactly t with a
// lower leaf index, ray_step), which an any-hit traversal bounded at tMax = t with tieLeaf
// answers; the same t, u, v and 1/det come out of the triangle test whatever tMax is.
LTS_D bool mis_ray(const SceneView& sv, const LightDesc& L, int li, const SurfacePoint& si, const Ray& r, bool sampledSpecular,
                   float scatteringPdf, float& weight, float& tMax, int& tieLeaf) {
    weight = 1;
    tMax = INFINITY;
    tieLeaf = -1;
    if (L.kind == 0) {
        LightHit lh;
        const bool hit = light_hit(sv, L, si, r, lh);
        if (!sampledSpecular) {
            if (lh.pdf == 0) return false;
            weight = power_heuristic(scatteringPdf, lh.pdf);
        }
        if (!hit || !lh.front || sv.shade[L.leaf].light != li) return false;
        tMax = lh.t;
        tieLeaf = L.leaf;
    } else if (!sampledSpecular) {
        const float lightPdf = inf_pdf(r.d);
        if (lightPdf == 0) return false;
        weight = power_heuristic(scatteringPdf, lightPdf);
    }
    return true;
}

// Radiance that a path sees of a light directly, at its first vertex and after specular ones: emission
// of the hit's front (leaf >= 0), or of the infinite lights where the ray escapes.
LTS_D void add_emission(const SceneView& sv, int leaf, const Ray& r, float u, float v, float invDet, Spec beta, Spec& L) {
    if (leaf >= 0) {
        const int l = sv.shade[leaf].light;
        // the geometric normal decides emission; it needs the full interaction
        if (l >= 0) {
            SurfacePoint e = make_surface(sv, leaf, r, u, v, invDet);
            Spec le = dot(e.n, -r.d) > 0.f ? light_le(sv.lights[l]) : spec(0.0f);
            L = L + beta * le;
        } else {
            L = L + beta * spec(0.0f);
        }
    } else {
        for (int l = 0; l < sv.nLights; l++) L = L + beta * (sv.lights[l].kind == 1 ? light_le(sv.lights[l]) : spec(0.0f));
    }
}

// estimateDirect (intergrators/IntegratorHelper.cuh:51-125) up to its two ray casts. shadow(o, d, c) takes
// the shadow ray of the light sample with the contribution it carries when nothing blocks it before
// 1 - SHADOW_EPS, then mis(o, d, tMax, tieLeaf, c) the MIS-BSDF ray (see mis_ray); neither is called for a
// sample that contributes nothing. u0, u1: the vertex's sampler blocks.
template <class Shadow, class Mis>
LTS_D void light_rays(const SceneView& sv, const SurfacePoint& si, const Bsdf& bsdf, int li, const float* u0, const float* u1,
                      bool specular, Shadow shadow, Mis mis) {
    const LightDesc& Lt = sv.lights[li];
    const int flags = specular ? B_ALL : (B_ALL & ~B_SPEC);
    // light sample with MIS (IntegratorHelper.cuh:76-95)
    V3 wi;
    float lightPdf = 0.0f, scatteringPdf = 0.0f;
    LightPoint vis;
    Spec Li = sample_li(sv, Lt, si, v2(u0[1], u0[2]), &wi, &lightPdf, &vis);
    if (lightPdf > 0 && !isBlack(Li)) {
        Spec f = bsdf.f(si.wo, wi, flags) * absDot(wi, si.sn);
        scatteringPdf = bsdf.pdf(si.wo, wi, flags);
        if (!isBlack(f)) {
            float weight = power_heuristic(lightPdf, scatteringPdf);
            Spec c = f * Li * weight / lightPdf;
            V3 origin = offsetRayOrigin(si.p, si.pError, si.n, vis.p - si.p);
            V3 target = offsetRayOrigin(vis.p, vis.pError, vis.n, origin - vis.p);
            shadow(origin, target - origin, c);
        }
    }
    // BSDF sample with MIS (IntegratorHelper.cuh:96-122)
    int sampledType = 0;
    Spec f2 = bsdf.sampleF(si.wo, &wi, v2(u0[3], u1[0]), &scatteringPdf, flags, &sampledType);
    f2 = f2 * absDot(wi, si.sn);
    const bool sampledSpecular = (sampledType & B_SPEC) != 0;
    const Spec Li2 = light_le(Lt);
    if (!isBlack(f2) && scatteringPdf > 0 && !isBlack(Li2)) {
        const Ray mr = spawn_ray(si, wi);
        float weight, tMax;
        int tieLeaf;
        if (mis_ray(sv, Lt, li, si, mr, sampledSpecular, scatteringPdf, weight, tMax, tieLeaf))
            mis(mr.o, wi, tMax, tieLeaf, f2 * Li2 * spec(1.0f) * weight / scatteringPdf);
    }
}

// Film sample position of (pixel, sample): dims 0-1, stratified per Sampler::stratifiedSample
// (sampling/Sampler.cuh:49-64) when requested.
LTS_D V2 film_sample(int px, int py, int sample, int spp, int stratified, const float d0[4]) {
    V2 film = v2(d0[0], d0[1]);
    if (stratified) {
        int strata = (int)floorf(sqrtf((float)spp));
        if (sample - 1 < strata * strata) {
            float inv = (float)1 / strata;
            film = v2(film.x * inv, film.y * inv);
            film = film + v2((sample % strata) / (float)strata, (sample / strata) / (float)strata);
        }
    }
    return v2((float)(px + film.x), (float)(py + film.y));
}

// ---------------------------------------------------------------- camera (rendering/Camera.cu:51-81)
struct CamRays {
    V3 rxO, rxD, ryO, ryD;  // the differential rays
};

LTS_D void camera_ray(const CameraDesc& c, V2 pf, V2 lens, V3* o, V3* d) {
    V3 cu = v3(c.u[0], c.u[1], c.u[2]), cv = v3(c.v[0], c.v[1], c.v[2]);
    V3 co = v3(c.o[0], c.o[1], c.o[2]);
    V3 offset = (cu * lens.x + cv * lens.y) * c.lensRadius;
    V2 pr = v2(pf.x / (c.width - 1), pf.y / (c.height - 1));
    *o = co + offset;
    *d = normalize(v3(c.llc[0], c.llc[1], c.llc[2]) + v3(c.right[0], c.right[1], c.right[2]) * pr.x +
                   v3(c.up[0], c.up[1], c.up[2]) * pr.y - co - offset);
}

// Film position and lens sample of one (pixel, sample): dims 0-1 and 2-3. A pinhole (lens radius 0,
// the only camera the scene files describe) has no use for the lens sample.
struct CameraSample {
    V2 film, lens;
};
LTS_D CameraSample camera_sample(const SceneView& sv, int px, int py, int sample, int spp, int stratified, uint32_t seed) {
    Sampler smp;
    smp.seed = seed;
    smp.pixel = (uint32_t)(py * sv.cam.width + px);
    smp.sample = (uint32_t)sample;
    float d[4];
    smp.block(0, d);
    CameraSample cs;
    cs.film = film_sample(px, py, sample, spp, stratified, d);
    cs.lens = v2(0, 0);
    if (sv.cam.lensRadius != 0) cs.lens = uniform_disk(v2(d[2], d[3]));
    return cs;
}
LTS_D Ray camera_ray(const SceneView& sv, const CameraSample& cs) {
    Ray r;
    camera_ray(sv.cam, cs.film, cs.lens, &r.o, &r.d);
    r.tMax = INFINITY;
    return r;
}

// generateDifferentialRay + Ray::scaleDifferentials(rsqrt(spp)) (Camera.cu:67-81, Ray.cuh:35-40): the
// differential rays of the camera ray (o, d) of a sample.
LTS_D CamRays camera_differentials(const CameraDesc& c, const CameraSample& cs, int spp, V3 o, V3 d) {
    CamRays cr;
    camera_ray(c, cs.film + v2(1, 0), cs.lens, &cr.rxO, &cr.rxD);
    camera_ray(c, cs.film + v2(0, 1), cs.lens, &cr.ryO, &cr.ryD);
    float sc = quake((float)spp);
    cr.rxO = o + (cr.rxO - o) * sc;
    cr.ryO = o + (cr.ryO - o) * sc;
    cr.rxD = d + (cr.rxD - d) * sc;
    cr.ryD = d + (cr.ryD - d) * sc;
    return cr;
}

// invDet * determinant of a hit: Triangle::intersect scales dpdu and dpdv by the ray's invDet where
// the uv parametrisation's 1 / determinant belongs (Triangle.cu:147-149), so the interaction's dpdu,
// dpdv are k times the true derivatives (k = 1 when the uv determinant is 0 and dpdu, dpdv come
// from coordinateSystem). The shading frame only uses their directions; uv differentials need k.
LTS_D float uv_derivative_scale(const SceneView& sv, int leaf, float invDet) {
    const ShadeTri& st = sv.shade[leaf];
    V2 uv0 = v2(st.uv[0], st.uv[1]), uv1 = v2(st.uv[2], st.uv[3]), uv2 = v2(st.uv[4], st.uv[5]);
    V2 duv02 = uv0 - uv2, duv12 = uv1 - uv2;
    float determinant = duv02.x * duv12.y - duv02.y * duv12.x;
    return determinant == 0 ? 1.0f : invDet * determinant;
}

// SurfaceInteraction::computeDifferentials (Interaction.cuh:118-160). The uv differentials, read
// only by the filtered texture pipeline, are those of the true uv parametrisation: solved against
// the interaction's dpdu, dpdv (k times too long, see uv_derivative_scale) and multiplied by k.
LTS_D void differentials(SurfacePoint& s, const CamRays& cr, float k) {
    float d = -dot(s.n, s.p);
    float tx = (-dot(s.n, cr.rxO) - d) / dot(s.n, cr.rxD);
    V3 px = cr.rxO + cr.rxD * tx;
    float ty = (-dot(s.n, cr.ryO) - d) / dot(s.n, cr.ryD);
    V3 py = cr.ryO + cr.ryD * ty;
    s.dpdx = px - s.p;
    s.dpdy = py - s.p;
    // du/dx, dv/dx, du/dy, dv/dy on the two axes other than the normal's dominant one
    // (Interaction.cuh:134-153, solveLinearSystem2x2 GeneralHelper.cuh:127-134)
    int d0, d1;
    if (fabsf(s.n.x) > fabsf(s.n.y) && fabsf(s.n.x) > fabsf(s.n.z)) { d0 = 1; d1 = 2; }
    else if (fabsf(s.n.y) > fabsf(s.n.z)) { d0 = 0; d1 = 2; }
    else { d0 = 0; d1 = 1; }
    auto c = [](V3 v, int k) { return k == 0 ? v.x : k == 1 ? v.y : v.z; };
    const float a00 = c(s.dpdu, d0), a01 = c(s.dpdv, d0), a10 = c(s.dpdu, d1), a11 = c(s.dpdv, d1);
    auto solve = [&](float b0, float b1, float& x0, float& x1) {
        const float det = a00 * a11 - a01 * a10;
        if (fabsf(det) < 1e-10f) { x0 = x1 = 0.0f; return; }
        x0 = (a11 * b0 - a01 * b1) / det;
        x1 = (a00 * b1 - a10 * b0) / det;
        if (isnan(x0) || isnan(x1)) x0 = x1 = 0.0f;
    };
    solve(c(px, d0) - c(s.p, d0), c(px, d1) - c(s.p, d1), s.dudx, s.dvdx);
    solve(c(py, d0) - c(s.p, d0), c(py, d1) - c(s.p, d1), s.dudy, s.dvdy);
    s.dudx *= k; s.dvdx *= k; s.dudy *= k; s.dvdy *= k;
}

// The footprint of a camera hit, for the materials whose textures read it (procedural and filtered
// image textures).
LTS_D void camera_footprint(const SceneView& sv, SurfacePoint& si, const CameraSample& cs, int spp, const Ray& r, float invDet) {
    if (sv.mats[sv.shade[si.leaf].mat].footprint)
        differentials(si, camera_differentials(sv.cam, cs, spp, r.o, r.d), uv_derivative_scale(sv, si.leaf, invDet));
}

}  // namespace lts
