// sr_upload and sr_readback with a copy that fails, over the stand-in runtime: the error comes back and no device memory of
// the call is left behind. Below and above the staging slots' lines, at each of the first copies.
#include "fake_hip.hpp"

#include <cstdio>
#include <vector>

#include "../../include/sr_hip.h"

int main() {
    int bad = 0, calls = 0;
    for (int side : {64, 768}) {
        sr_physics ph;
        sr_physics_defaults(&ph);
        sr_switches sw = {};
        sw.hydro = 1;
        sr_world *w = nullptr;
        if (sr_world_create(side, side, &ph, &sw, nullptr, &w) != SR_OK) return 2;
        std::vector<float> planes((size_t)14 * side * side, 1.0f);
        for (int at = -1; at < 4; at++)
            for (bool up : {true, false}) {
                const int live = fake::async_live;
                fake::copies = 0;
                fake::fail_at = at;
                const int code = up ? sr_upload(w, planes.data(), planes.size()) : sr_readback(w, planes.data(), planes.size());
                const bool failed = fake::copies > at && at >= 0;
                fake::fail_at = -1;
                calls++;
                if (code != (failed ? SR_ERR_DEVICE : SR_OK) || fake::async_live != live) {
                    std::printf("side %d, %s, copy %d: code %d, %d buffers left\n", side, up ? "up" : "down", at, code,
                                fake::async_live - live);
                    bad++;
                }
            }
        sr_destroy(w);
    }
    std::printf("%d of %d calls wrong\n", bad, calls);
    return bad != 0;
}
