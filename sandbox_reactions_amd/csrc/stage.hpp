// Host transfers through pinned chunks: large planes between a caller's pageable memory and the device.
#pragma once
#include "common.hpp"

namespace sr {

#define STAGE_THREADS 4
#define STAGE_SLOTS 2               // per thread: one is copied by the host while the other is on the bus
#define STAGE_CHUNK (2u << 20)      // bytes of one slot
// Transfers below these stay with the runtime's own copy. Up, by the runtime against the slots: 0.49 / 0.52 ms at 14.7 MB,
// 0.73 / 0.72 at 22.9, 1.10 / 0.97 at 33.0, 8.5 / 6.3 at 235. Down: 0.29 / 0.26 at 3.7 (within its spread), 0.57 / 0.36 at
// 8.6, 1.39 / 0.68 at 22.9, 13.5 / 5.9 at 235.
#define STAGE_LEAST_UP (24u << 20)
#define STAGE_LEAST_DOWN (8u << 20)

// Not for concurrent use (a world's transfers are its caller's, one at a time, all on one device's streams). The pinned
// memory and the events are kept from the first large transfer until release().
class HostStage {
  public:
    // Queued on s: pageable memory may be changed when it returns (pinned memory once s's work is done), the device's copy
    // is ordered on s
    int to_device(void *dst, const void *src, size_t bytes, hipStream_t s);
    // Done when it returns (s's work before it too)
    int to_host(void *dst, const void *src, size_t bytes, hipStream_t s);
    // After s's work is done
    void release();

  private:
    bool ready(hipStream_t s);
    hipError_t chunks_up(int k, int threads, char *dev, const char *host, size_t bytes, hipStream_t s);
    hipError_t chunks_down(int k, int threads, const char *dev, char *host, size_t bytes, hipStream_t s);
    template <class F> int spread(size_t bytes, hipStream_t s, F part);
    char *buf = nullptr;
    int device = 0;  // the stream's, where the events are
    hipEvent_t ev[STAGE_THREADS * STAGE_SLOTS] = {};
    bool refused = false;  // no pinned memory to be had: the runtime's own copies
};

} // namespace sr
