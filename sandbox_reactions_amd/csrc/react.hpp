// P6 burning: the records and constants on the device, the pass's per-cell kernel.
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/sr_hip.h"
#include "cold.hpp"
#include "hydro.hpp"
#include "react_dev.hpp"

namespace sr {

static_assert(REACT_COLD == COLD_POINTS, "the cold energy's nodes");

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
// once before a plan's first launch
int react_prepare(const ReactLaunch &plan);
int react_launch(const ReactDev *D, const ReactLaunch &plan, const HydroState &st, int n, double dt, const double *scal,
                 double *nuclear, double *lost, double *snu, double *psum, double *pmax, int *nblocks, hipStream_t s);
// the partials of nb blocks into out: the REACT_SUMS sums, then the REACT_MAXES maxima
int react_report(const double *psum, const double *pmax, int nb, double *out, hipStream_t s);

} // namespace sr
