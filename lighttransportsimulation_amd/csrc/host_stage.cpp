// Copies between device memory and a caller's pageable memory, through a pinned ring.
//
// The runtime's own copies of pageable memory take 125 us for 256 KiB, 503 us for 1 MiB, 352 us for 5 MiB
// and 1594 us for 25 MiB to the host: staged chunk by chunk without overlap, or pinned for the one copy.
// Here a transfer runs while the calling thread copies the one before: 25, 59, 216 and 987 us. A transfer
// takes 18 us and 1 us for each 53 KB, a memcpy 1 us for each 25 KB, so chunks of 1 MiB hide most of one
// behind the other (25 MiB with chunks of 256 KiB: 1911 us, 512 KiB: 1180 us, 2 MiB: 987 us); up to 7 helper
// threads made 3 to 30 % of difference, less than their start costs below 8 MiB, and are left out.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "lts_internal.h"

namespace lts {

namespace {

constexpr size_t kChunk = (size_t)1 << 20, kMinChunk = (size_t)1 << 18;

// two chunks at least where that is worth a transfer of its own
size_t chunk_bytes(size_t bytes) { return std::min(kChunk, std::max(kMinChunk, (bytes / 2 + 4095) / 4096 * 4096)); }

}  // namespace

hipError_t stage_create(HostStage& st) {
    hipError_t e = hipHostMalloc((void**)&st.mem, kStageSlots * kChunk, hipHostMallocDefault);
    for (hipEvent_t& ev : st.ev)
        if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    return e;
}

void stage_destroy(HostStage& st) {
    for (hipEvent_t ev : st.ev)
        if (ev) (void)hipEventDestroy(ev);
    if (st.mem) (void)hipHostFree(st.mem);
    st = HostStage{};
}

void stage_touch(void* dst, size_t bytes) {
    volatile char* p = static_cast<volatile char*>(dst);
    for (size_t i = 0; i < bytes; i += 4096) p[i] = p[i];
    if (bytes) p[bytes - 1] = p[bytes - 1];
}

hipError_t stage_to_host(HostStage& st, void* dst, const void* src, size_t bytes, hipStream_t s) {
    const size_t chunk = chunk_bytes(bytes), n = (bytes + chunk - 1) / chunk;
    auto issue = [&](size_t i) {
        const size_t at = i * chunk, slot = i % kStageSlots;
        const hipError_t e = hipMemcpyAsync(st.mem + slot * kChunk, (const char*)src + at, std::min(chunk, bytes - at), hipMemcpyDeviceToHost, s);
        return e == hipSuccess ? hipEventRecord(st.ev[slot], s) : e;
    };
    hipError_t e = hipSuccess;
    for (size_t i = 0; e == hipSuccess && i < std::min<size_t>(n, kStageSlots); i++) e = issue(i);
    for (size_t i = 0; e == hipSuccess && i < n; i++) {
        const size_t at = i * chunk, slot = i % kStageSlots;
        if ((e = hipEventSynchronize(st.ev[slot])) != hipSuccess) break;
        std::memcpy((char*)dst + at, st.mem + slot * kChunk, std::min(chunk, bytes - at));
        if (i + kStageSlots < n) e = issue(i + kStageSlots);
    }
    return e;
}

hipError_t stage_to_device(HostStage& st, void* dst, const void* src, size_t bytes, hipStream_t s) {
    const size_t chunk = chunk_bytes(bytes), n = (bytes + chunk - 1) / chunk;
    hipError_t e = hipSuccess;
    for (size_t i = 0; e == hipSuccess && i < n; i++) {
        const size_t at = i * chunk, slot = i % kStageSlots, m = std::min(chunk, bytes - at);
        // the slot's last transfer, of this copy or an earlier one
        if ((e = hipEventSynchronize(st.ev[slot])) != hipSuccess) break;
        std::memcpy(st.mem + slot * kChunk, (const char*)src + at, m);
        e = hipMemcpyAsync((char*)dst + at, st.mem + slot * kChunk, m, hipMemcpyHostToDevice, s);
        if (e == hipSuccess) e = hipEventRecord(st.ev[slot], s);
    }
    return e;
}

}  // namespace lts
