// The P6 launch of worlds with different records: a kernel's limit of dynamic LDS is the process's, so no world may lower
// it below what another world's launch takes.
#include "fake_hip.hpp"

#include <cstdio>

#include "../../sandbox_reactions_amd/csrc/common.hpp"
#include "../../sandbox_reactions_amd/csrc/react.hpp"

using namespace sr;

int main() {
    int bad = 0;
    std::map<const void *, int> before;
    fake::launched = [&](const void *k, dim3, dim3 block, size_t lds) {
        const int limit = fake::attribute[k];
        std::printf("%u threads, %zu bytes, limit %d\n", block.x, lds, limit);
        bad += (int)lds > limit || limit < before[k];
        before[k] = limit;
    };
    sr_physics ph = {};
    // one input each, then three: 256 threads; four inputs: 64
    for (int turn = 0; turn < 2; turn++)
        for (int inputs : {3, 1, 4, 2})
            for (int records : {2, 16, 5}) {
                static ReactDev D;
                sr_react_params p = {};
                p.n_records = records;
                p.nfe = -1;
                p.burn_dx = p.burn_dt = 0.1;
                for (int r = 0; r < records; r++) {
                    p.rec[r].n_in = inputs;
                    p.rec[r].n_out = 1;
                    p.rec[r].out_species[0] = 5;
                    p.rec[r].out_share[0] = 1.0;
                    for (int k = 0; k < inputs; k++) {
                        p.rec[r].in_species[k] = k;
                        p.rec[r].in_share[k] = 1.0 / inputs;
                        p.rec[r].in_order[k] = 1.0;
                    }
                }
                if (react_check(&p) != SR_OK) return 2;
                react_build(&p, ph, &D);
                const ReactLaunch plan = react_plan(D);
                if (react_prepare(plan) != SR_OK) return 2;
                if (react_launch(&D, plan, HydroState{}, 1000, 0.1, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr,
                                 nullptr, nullptr) != SR_OK)
                    return 2;
            }
    return bad != 0;
}
