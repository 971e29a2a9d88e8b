// P6 burning: the records and constants on the device, the pass's per-cell kernel.
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/sr_hip.h"
#include "cold.hpp"
#include "hydro.hpp"

namespace sr {

#define REACT_NS 10
#define REACT_TABLE 256
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
    double cold_lnu[2][COLD_POINTS];
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
    // f's tables: record r reads table f_of[r] (records of the same law share one), tables in all; ln T_thr per record
    int f_of[SR_REACT_RECORDS], tables;
    double ln_thr[SR_REACT_RECORDS];
};

// the host's checks of the records and the device copy's build (tables in FP64 on the host) for the world's physics
int react_check(const sr_react_params *p);
void react_build(const sr_react_params *p, const sr_physics &ph, ReactDev *out);

// P6 over dt (dt < 0: the step's dt, scal[0]) on the world's state; per cell the energy booked per group (7 n), the
// neutrino loss and S_nu (n each); per block partials: sums (substeps, retried, unfinished, nuclear x 7, lost) into
// psum[11][nb], maxima (max sub-steps, max dX, max dT/T, latch) into pmax[4][nb]
constexpr int REACT_SUMS = 11, REACT_MAXES = 4;
// how to launch the pass for the parameters: threads and LDS bytes per block, whether the linear system holds the neutrons
struct ReactLaunch {
    int nt, lds;
    bool neutrons;
    int blocks(size_t n) const { return (int)((n + nt - 1) / nt); }
};
constexpr int REACT_NT_LEAST = 64;
ReactLaunch react_plan(const ReactDev &h);
int react_launch(const ReactDev *D, const ReactLaunch &plan, const HydroState &st, int n, double dt, const double *scal,
                 double *nuclear, double *lost, double *snu, double *psum, double *pmax, int *nblocks, hipStream_t s);

} // namespace sr
