// P6 burning: what the pass reads besides the state, and the shape of its linear system. Plain C++, so that the system's
// solve (react_solve.hpp) is also built by a CPU compiler with its checks of indexes.
#pragma once
#include "../../include/sr_hip.h"

namespace sr {

#define REACT_NS 10
#define REACT_TABLE 256
#define REACT_COLD 512  // the cold energy's nodes
#define REACT_ITEMS (SR_REACT_RECORDS * 4 * 8)  // a record's inputs times the species it changes, at most

// Everything the pass reads besides the state, in device memory: the records and constants as given, each record's
// nu (outputs' shares minus inputs'), its ln f table, Sigma_vac, T_floor and the cold energy's tables in FP64 (the
// electrons' and the neutrons' ln u at the nodes, a pair's flag 0 when it is off; ln x_min and the node spacing in
// ln x), so that T = mu (e - eps_cold) carries no f32 rounding into the rates
struct ReactDev {
    sr_react_params P;
    double nu[SR_REACT_RECORDS][REACT_NS];
    double ln_f[SR_REACT_RECORDS][REACT_TABLE];
    double sigma_vac, t_floor;
    double cold_lnu[2][REACT_COLD];
    int cold_pair[2];
    double cold_ln_min, cold_step;
    // The linear system's shape, built on the host from the records. Entry e is a record's derivative by one of its inputs
    // (the records in order, N_Fe left out, ent0[r] the first of record r). The matrix's items in row order, a position's
    // together, its last flagged: entry e times nu. Row i: bits 0..9 the columns that have items, bits
    // 16..25 the columns j < i that can be nonzero when the row is eliminated without exchanges.
    struct Item {
        double nu;
        int e, last;
    };
    int entries, items, ent0[SR_REACT_RECORDS + 1], slots, slot[SR_REACT_RECORDS];  // slot: a record's but N_Fe's
    unsigned row[REACT_NS];
    Item item[REACT_ITEMS];
    // f's tables: record r reads table f_of[r] (records of the same law share one), tables in all
    int f_of[SR_REACT_RECORDS], tables;
};

// nu, and the linear system's entries, items and elimination pattern, from out->P (the rest of *out zeroed)
inline void react_shape(ReactDev *out) {
    const sr_react_params &p = out->P;
    for (int r = 0; r < p.n_records; r++) {
        const sr_react_record &c = p.rec[r];
        for (int k = 0; k < c.n_out; k++) out->nu[r][c.out_species[k]] += c.out_share[k];
        for (int k = 0; k < c.n_in; k++) out->nu[r][c.in_species[k]] -= c.in_share[k];
    }
    for (int r = 0; r < p.n_records; r++) {
        out->ent0[r] = out->entries;
        out->slot[r] = out->slots;
        if (r == p.nfe) continue;
        out->entries += p.rec[r].n_in;
        out->slots++;
    }
    out->ent0[p.n_records] = out->entries;
    unsigned reach[REACT_NS];  // the columns a row can hold a value in
    for (int i = 0; i < REACT_NS; i++) {
        reach[i] = 1u << i;
        for (int j = 0; j < REACT_NS; j++) {
            const int first = out->items;
            for (int r = 0; r < p.n_records; r++) {
                if (r == p.nfe || out->nu[r][i] == 0.0) continue;
                for (int k = 0; k < p.rec[r].n_in; k++)
                    if (p.rec[r].in_species[k] == j)
                        out->item[out->items++] = {out->nu[r][i], out->ent0[r] + k, 0};
            }
            if (out->items == first) continue;
            out->item[out->items - 1].last = 1;
            out->row[i] |= 1u << j;
            reach[i] |= 1u << j;
        }
        for (int j = 0; j < i; j++)
            if (reach[i] >> j & 1) reach[i] |= reach[j] >> j << j;
        out->row[i] |= (reach[i] & ((1u << i) - 1)) << 16;
    }
}

} // namespace sr
