// The planes' transfers (csrc/stage.hip) over the stand-in runtime. stage CASE: exits 0 when the case holds.
#include "fake_hip.hpp"

#include <cstdio>
#include <new>
#include <vector>

#include "../../sandbox_reactions_amd/csrc/stage.hpp"

using namespace sr;

// allocations that fail while a thread is started
static thread_local bool starting = false;
static bool no_threads = false;
void *operator new(size_t n) {
    if (starting) throw std::bad_alloc();
    if (void *p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

// both ways through one world's stage at sizes below, at and past the line, ending inside a chunk
static bool round_trips(char *a, size_t most, hipStream_t s) {
    HostStage stage;
    std::vector<char> dev(most);
    bool ok = stage.to_host(a, dev.data(), STAGE_LEAST_DOWN, s) == SR_OK;  // the slots are made with it
    fake::copies = 0;
    for (size_t n : {(size_t)1000, (size_t)STAGE_LEAST_DOWN - 1, (size_t)STAGE_LEAST_DOWN, (size_t)STAGE_LEAST_UP - 1,
                     (size_t)STAGE_LEAST_UP + 4321, most}) {
        for (size_t i = 0; i < n; i++) a[i] = (char)(i * 2654435761u >> 24);
        starting = no_threads;
        ok &= stage.to_device(dev.data(), a, n, s) == SR_OK;
        starting = false;
        std::memset(a, 0, n);
        starting = no_threads;
        ok &= stage.to_host(a, dev.data(), n, s) == SR_OK;
        starting = false;
        for (size_t i = 0; i < n; i++) ok &= a[i] == (char)(i * 2654435761u >> 24);
    }
    stage.release();
    return ok;
}

int main(int, char **argv) {
    const std::string name = argv[1];
    const size_t most = (size_t)40 << 20;
    hipStream_t s;
    (void)hipStreamCreateWithFlags(&s, 0);
    bool ok = false;
    if (name == "pageable") {
        std::vector<char> a(most);
        ok = round_trips(a.data(), most, s) && fake::largest_copy == STAGE_LEAST_UP - 1;  // 24 MiB up
    } else if (name == "pinned") {  // in one copy
        void *a = nullptr;
        (void)hipHostMalloc(&a, most);
        ok = round_trips((char *)a, most, s) && fake::copies == 12 && fake::largest_copy == most;
    } else if (name == "threads") {  // none to be had: the caller's own
        std::vector<char> a(most);
        no_threads = true;
        ok = round_trips(a.data(), most, s);
    } else if (name == "device") {  // the stream's is not the caller's current one
        std::vector<char> a(most);
        (void)hipSetDevice(1);
        ok = round_trips(a.data(), most, s) && fake::device == 1;
    }
    std::printf("%s %s\n", name.c_str(), ok ? "holds" : "does not hold");
    return !ok;
}
