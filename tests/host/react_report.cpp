// sr_read_react over the stand-in runtime: what comes over the bus for the report does not grow with the world.
#include "fake_hip.hpp"

#include <cstdio>
#include <vector>

#include "../../include/sr_hip.h"

int main() {
    size_t most[2] = {0, 0};
    for (int k = 0; k < 2; k++) {
        const int side = k ? 1024 : 64;
        sr_physics ph;
        sr_physics_defaults(&ph);
        sr_switches sw = {};
        sr_world *w = nullptr;
        if (sr_world_create(side, side, &ph, &sw, nullptr, &w) != SR_OK) return 2;
        sr_react_params p = {};
        p.n_records = SR_REACT_RECORDS;
        p.nfe = -1;
        p.burn_dx = p.burn_dt = 0.1;
        for (auto &c : p.rec) {
            c.n_in = 4;
            c.n_out = 1;
            c.out_species[0] = 5;
            c.out_share[0] = 1.0;
            for (int i = 0; i < 4; i++) c.in_species[i] = i, c.in_share[i] = 0.25, c.in_order[i] = 1.0;
        }
        sr_react_report r;
        if (sr_set_reactions(w, &p) != SR_OK || sr_react_apply(w, 0.1) != SR_OK) return 2;
        fake::largest_copy = 0;
        if (sr_read_react(w, &r) != SR_OK) return 2;
        most[k] = fake::largest_copy;
        sr_destroy(w);
    }
    std::printf("%zu bytes for 64^2, %zu for 1024^2\n", most[0], most[1]);
    return most[1] > 4096;
}
