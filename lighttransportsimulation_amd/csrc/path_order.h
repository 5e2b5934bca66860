// The order in which the paths of a pass walk its scenes, samples and pixels, and the dealing of a launch's
// items to its waves.
#pragma once

#include "lts_device.h"
#include "lts_internal.h"

namespace lts {

// Pixel of the j-th path of a sample: the image is cut into bands of T rows and each band is walked
// column by column, so 64 consecutive paths (one wave) cover a T x 64/T tile and their rays stay
// close (T = 8: an 8x8 tile; T = 1: scanline order). The last band holds the remaining rows.
LTS_D int band_pixel(int j, int W, int H, int T) {
    const int band = j / (T * W);
    const int rows = min(T, H - T * band);
    const int jj = j - band * T * W;
    return (T * band + jj % rows) * W + jj / rows;
}

// Scene of path i of the pass: the last slot whose path range starts at or before i.
LTS_D int path_scene(const WfParams& P, const WfSceneSlot* slots, long i) {
    int lo = 0, hi = P.nScenes - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (slots[mid].pathBase <= i) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Path i of the pass -> (scene, pixel, sample).
LTS_D void path_origin(const WfParams& P, const WfSceneSlot* slots, long i, int& scene, int& pixel, int& sample) {
    const int s = path_scene(P, slots, i);
    const WfSceneSlot& sl = slots[s];
    const long local = i - sl.pathBase;
    const long npix = (long)sl.width * sl.height;
    scene = s;
    sample = sl.s0 + (int)(local / npix);
    pixel = band_pixel((int)(local % npix), sl.width, sl.height, P.tileRows);
}

// Deals the items 0..n of a persistent launch to its waves. The items are cut into one segment per XCD
// (workgroups are dealt to the 8 XCDs round robin), so that neighbouring items meet one L2; a wave takes
// chunks of its XCD's segment, then of the others. A wave's first chunk is its own; the next ones come from
// the segment's counter in `work` (cleared before the launch). The counters are shared by all XCDs, and an
// atomic on one takes the longer the more waves wait for it (some 15 ns each): with a first chunk from the
// counters too, and a failed try at each of the 8 segments before a wave ended, the 7 trace launches of one
// sample of an 853x479 frame took 1.65 ms instead of 0.84. So a wave reads all counters at once before it
// tries another segment.
// T: int, or long where the items may be more than an int counts. All fields are the same in every lane.
template <class T>
struct WorkDeal {
    T n, next, end;  // next..end: the items that the wave holds
    int chunk;
    int open;        // segments that may have chunks left, the wave's own in bit 0; bit kWfWorkSegments: the
                     // wave's first chunk is still to come; 0: no items are left
};

template <class T>
LTS_D WorkDeal<T> work_deal(T n, int chunk) {
    return WorkDeal<T>{n, 0, 0, chunk, (2 << kWfWorkSegments) - 1};
}

// The wave's next chunk, once it has handed out the last one. waves: waves per workgroup; resident: the
// workgroups that run from the start (only they have first chunks). Run by all lanes.
template <class T>
LTS_D void work_next(WorkDeal<T>& q, int waves, int resident, int32_t* work) {
    const int lane = threadIdx.x & 63;
    const int own = blockIdx.x % kWfWorkSegments;
    const T segLen = ((q.n + kWfWorkSegments - 1) / kWfWorkSegments + 63) / 64 * 64;
    // the first item, in its segment, of the c-th chunk that is nobody's first one
    auto start = [&](int s, int c) { return (T)(((min((int)gridDim.x, resident) - s + kWfWorkSegments - 1) / kWfWorkSegments) * waves + c) * q.chunk; };
    auto take = [&](int s, T at) {
        q.next = s * segLen + at;
        // a segment's last chunk ends with it: what lies behind is another wave's
        q.end = at < segLen ? min(q.next + min((T)q.chunk, segLen - at), q.n) : q.next;
        return q.next < q.end;
    };
    if (q.open >> kWfWorkSegments) {
        q.open &= (1 << kWfWorkSegments) - 1;
        const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        if ((int)blockIdx.x < resident && take(own, (T)((blockIdx.x / kWfWorkSegments) * waves + wave) * q.chunk)) return;
    }
    bool peeked = false;
    while (q.open) {
        const int k = __ffs(q.open) - 1, s = (own + k) % kWfWorkSegments;
        if (k > 0 && !peeked) {
            peeked = true;
            bool left = false;
            const int t = (own + lane) % kWfWorkSegments;
            if (lane < kWfWorkSegments && (q.open >> lane & 1) && start(t, 0) < segLen) {
                const T at = start(t, __hip_atomic_load(&work[kWfWorkStride * t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                left = at < segLen && t * segLen + at < q.n;
            }
            q.open = (int)__ballot(left);
            continue;
        }
        if (start(s, 0) < segLen) {
            int c = 0;
            if (lane == 0) c = atomicAdd(&work[kWfWorkStride * s], 1);
            if (take(s, start(s, __builtin_amdgcn_readfirstlane(c)))) return;
        }
        q.open &= ~(1 << k);
    }
    q.next = q.end = 0;
}

}  // namespace lts
