// Host transfers through pinned chunks. The runtime copies pageable memory through one staging buffer on the calling
// thread: 26 GB/s up and 10 GB/s down (into fresh pages) at 235 MB. Here a few threads copy chunks between the caller's
// memory and pinned slots while the copies of the slots before are on the bus: 36 GB/s both ways. Four threads of two
// 2 MiB slots: 1 MiB slots take 18 % longer; the pinned memory costs 0.4 ms once.
#include <algorithm>
#include <cstring>
#include <exception>
#include <thread>

#include "stage.hpp"

namespace sr {

// on the stream's device, which need not be the calling thread's current one
bool HostStage::ready(hipStream_t s) {
    if (buf) return true;
    if (refused) return false;
    const int n = STAGE_THREADS * STAGE_SLOTS;
    int current = 0;
    bool ok = hipGetDevice(&current) == hipSuccess && hipStreamGetDevice(s, &device) == hipSuccess &&
              hipSetDevice(device) == hipSuccess;
    ok = ok && hipHostMalloc(&buf, (size_t)STAGE_CHUNK * n) == hipSuccess;
    for (int i = 0; ok && i < n; i++) ok = hipEventCreateWithFlags(&ev[i], hipEventDisableTiming) == hipSuccess;
    (void)hipSetDevice(current);
    if (!ok) {
        (void)hipGetLastError();
        release();
        refused = true;
    }
    return ok;
}

void HostStage::release() {
    for (auto &e : ev) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    if (buf) (void)hipHostFree(buf);
    buf = nullptr;
}

// whether the runtime would have to stage p itself: pinned (or device) memory goes over the bus in one copy of its own (an
// upload of 2048^2 4.6 ms, a readback 4.3; through the slots 6.3 each)
static bool pageable(const void *p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return true;
}

#define STAGE_TRY(call)                                                                                                \
    do {                                                                                                               \
        const hipError_t e_ = (call);                                                                                  \
        if (e_ != hipSuccess) return e_;                                                                               \
    } while (0)

// Thread k's chunks are k, k + threads, ...; its slots are its own, and a slot's event is its last copy's.
hipError_t HostStage::chunks_up(int k, int threads, char *dev, const char *host, size_t bytes, hipStream_t s) {
    int turn = 0;
    for (size_t at = (size_t)k * STAGE_CHUNK; at < bytes; at += (size_t)threads * STAGE_CHUNK, turn ^= 1) {
        const int i = k * STAGE_SLOTS + turn;
        char *slot = buf + (size_t)i * STAGE_CHUNK;
        const size_t len = std::min<size_t>(STAGE_CHUNK, bytes - at);
        STAGE_TRY(hipEventSynchronize(ev[i]));
        std::memcpy(slot, host + at, len);
        STAGE_TRY(hipMemcpyAsync(dev + at, slot, len, hipMemcpyHostToDevice, s));
        STAGE_TRY(hipEventRecord(ev[i], s));
    }
    return hipSuccess;
}

hipError_t HostStage::chunks_down(int k, int threads, const char *dev, char *host, size_t bytes, hipStream_t s) {
    const size_t step = (size_t)threads * STAGE_CHUNK;
    auto fetch = [&](size_t at, int i) -> hipError_t {
        STAGE_TRY(hipMemcpyAsync(buf + (size_t)i * STAGE_CHUNK, dev + at, std::min<size_t>(STAGE_CHUNK, bytes - at),
                                 hipMemcpyDeviceToHost, s));
        return hipEventRecord(ev[i], s);
    };
    int turn = 0;
    size_t at = (size_t)k * STAGE_CHUNK;
    if (at < bytes) STAGE_TRY(fetch(at, k * STAGE_SLOTS));
    for (; at < bytes; at += step, turn ^= 1) {
        const int i = k * STAGE_SLOTS + turn;
        if (at + step < bytes) STAGE_TRY(fetch(at + step, k * STAGE_SLOTS + (turn ^ 1)));
        STAGE_TRY(hipEventSynchronize(ev[i]));
        std::memcpy(host + at, buf + (size_t)i * STAGE_CHUNK, std::min<size_t>(STAGE_CHUNK, bytes - at));
    }
    return hipSuccess;
}

// part(k, threads) on up to STAGE_THREADS threads, this one among them; a thread that cannot be started (none to be had,
// or no memory for one) leaves its share to this one
template <class F> int HostStage::spread(size_t bytes, hipStream_t s, F part) {
    const int threads = (int)std::min<size_t>(STAGE_THREADS, (bytes + STAGE_CHUNK - 1) / STAGE_CHUNK);
    hipError_t err[STAGE_THREADS] = {};
    std::thread th[STAGE_THREADS];
    for (int k = 1; k < threads; k++) {
        try {
            th[k] = std::thread([&, k] {
                err[k] = hipSetDevice(device);
                if (err[k] == hipSuccess) err[k] = part(k, threads);
            });
        } catch (const std::exception &) {
        }
    }
    err[0] = part(0, threads);
    for (int k = 1; k < threads; k++)
        if (th[k].joinable())
            th[k].join();
        else
            err[k] = part(k, threads);
    for (int k = 0; k < threads; k++)
        if (err[k] != hipSuccess) (void)hipStreamSynchronize(s);  // no copy goes on in a slot that the next call takes
    for (int k = 0; k < threads; k++) SR_HIP(err[k]);
    return SR_OK;
}

int HostStage::to_device(void *dst, const void *src, size_t bytes, hipStream_t s) {
    if (bytes < STAGE_LEAST_UP || !pageable(src) || !ready(s)) {
        SR_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s));
        return SR_OK;
    }
    return spread(bytes, s, [&](int k, int threads) {
        return chunks_up(k, threads, (char *)dst, (const char *)src, bytes, s);
    });
}

int HostStage::to_host(void *dst, const void *src, size_t bytes, hipStream_t s) {
    if (bytes < STAGE_LEAST_DOWN || !pageable(dst) || !ready(s)) {
        SR_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s));
        SR_HIP(hipStreamSynchronize(s));
        return SR_OK;
    }
    return spread(bytes, s, [&](int k, int threads) {
        return chunks_down(k, threads, (const char *)src, (char *)dst, bytes, s);
    });
}

} // namespace sr
