// P6 burning: the rates' temperature factor (crates/sr-physics/src/rates.rs:44-118) and the sub-step's linear system,
// (I - h J) dX = h S (reference/react.rs:515-560). Compiled for the device by react.hip; plain C++, so a CPU compiler builds
// it too.
#pragma once
#include <cmath>

#include "react_dev.hpp"

#ifdef __HIPCC__
#define REACT_HD __host__ __device__
#else
#define REACT_HD
#endif

namespace sr {

// The tables and the threads' private arrays in LDS: the cold pairs' ln u, f's tables, then per thread a value by species
// (x while the rates are formed, dX after a solve), omega by record and the derivatives by entry. A species or record
// index is the wave's own but not the compiler's, so such an array in registers would go to scratch memory (as the whole
// pass's did: 587 us a pass at 512^2). What still goes there: 109 spilled registers (up to 153 with the neutrons) and the
// arrays of the rare forms (the pivoted system, N_Fe's closed form), 1456 to 1552 bytes a lane. A thread's element k lies NT
// values from its element k - 1: no bank conflicts. NT = 256 threads share the tables, so that two blocks (two waves a SIMD) fit a CU; with so many
// inputs that they would not (the shipped records: 78 KB), 64.
struct Lds {
    const double *cold, *ln_f;
    double *v, *omega, *grad;  // the thread's own: element k at [k * NT]
};

// ln of one Gamow-shaped term and f's direct form (rates.rs:44-53), on either side
REACT_HD inline double term_ln(double t_k, double nu, double w, double t) {
    const double u = log(t / t_k);
    return log(w) - 2.0 / 3.0 * u - (3.0 * nu + 2.0) * expm1(-u / 3.0);
}

REACT_HD inline double f_sum(const sr_react_record &r, double t) {
    double s = 0.0;
    for (int k = 0; k < r.n_terms; k++) s += exp(term_ln(r.t_k[k], r.nu[k], r.w[k], t));
    return s;
}

// f(T) through the table (rates.rs:98-118): 0 below T_thr, the direct sum past the table's span (and for a T that is no
// number, which stays none)
REACT_HD inline double temp_factor(const ReactDev &D, const Lds &M, int r, double t) {
    const sr_react_record &c = D.P.rec[r];
    if (c.n_terms == 0) return 1.0;
    if (t < c.t_thr) return 0.0;
    const double step = log(2.5) / (double)(REACT_TABLE - 1);
    const double pos = log(t / c.t_thr) / step;
    if (!(pos < (double)(REACT_TABLE - 1))) return f_sum(c, t);
    const int i = (int)floor(pos);
    const double frac = pos - (double)i;
    const double *ln_f = M.ln_f + D.f_of[r] * REACT_TABLE;
    return exp(ln_f[i] + frac * (ln_f[i + 1] - ln_f[i]));
}

// (I - h J) dX = h S, Gaussian elimination with partial pivoting, the last of equal pivots (react.rs:515-560): the form
// for a system that needs a row exchange, its matrix in scratch memory
template <int NT>
REACT_HD __attribute__((noinline)) void solve_pivoted(const ReactDev &D, const Lds &M, const double *s, double h,
                                                      double *dx) {
    double a[REACT_NS][REACT_NS + 1];
    int q = 0;
    for (int i = 0; i < REACT_NS; i++) {
        for (int j = 0; j < REACT_NS; j++) {
            a[i][j] = i == j ? 1.0 : 0.0;
            if (D.row[i] >> j & 1) do {
                    a[i][j] -= h * D.item[q].nu * M.grad[D.item[q].e * NT];
                } while (!D.item[q++].last);
        }
        a[i][REACT_NS] = h * s[i];
    }
    for (int col = 0; col < REACT_NS; col++) {
        int piv = col;
        for (int p = col + 1; p < REACT_NS; p++)
            if (fabs(a[p][col]) >= fabs(a[piv][col])) piv = p;
        if (piv != col)
            for (int j = 0; j <= REACT_NS; j++) {
                const double t = a[col][j];
                a[col][j] = a[piv][j];
                a[piv][j] = t;
            }
        const double d = a[col][col];
        if (d == 0.0) continue;
        for (int row = col + 1; row < REACT_NS; row++) {
            const double f = a[row][col] / d;
            if (f != 0.0)
                for (int j = col; j <= REACT_NS; j++) a[row][j] -= f * a[col][j];
        }
    }
    for (int i = REACT_NS - 1; i >= 0; i--) {
        double v = a[i][REACT_NS];
        for (int j = i + 1; j < REACT_NS; j++) v -= a[i][j] * dx[j];
        dx[i] = a[i][i] == 0.0 ? 0.0 : v / a[i][i];
    }
}

// The same system by rows in registers: each row is built and reduced by the rows above it (the columns it can hold a
// value in, bits 16..25 of D.row), the same operations in the same order on every element as by columns. Where the pivoted form would
// exchange rows (an element at least as large as its pivot) the pivoted form solves the system instead; the consumed
// species' diagonal 1 + h sum of its losses exceeds what any product's row holds, so no physical system is. NA: the
// species to solve for (9 where the last, the neutrons, has no items, as with N_Fe in closed form: dX = 0).
template <int NA, int NT>
REACT_HD inline void solve(const ReactDev &D, const Lds &M, const double (&s)[REACT_NS], double h,
                           double (&dx)[REACT_NS]) {
    double u[NA][NA];
    bool exchange = false;
    int q = 0;
#pragma unroll
    for (int i = 0; i < NA; i++) {
        double b = h * s[i];
        const unsigned shape = D.row[i];
#pragma unroll
        for (int j = 0; j < NA; j++) {
            u[i][j] = i == j ? 1.0 : 0.0;
            if (shape >> j & 1) do {
                    u[i][j] -= h * D.item[q].nu * M.grad[D.item[q].e * NT];
                } while (!D.item[q++].last);
        }
#pragma unroll
        for (int col = 0; col < i; col++) {
            if (!(shape >> (16 + col) & 1)) continue;
            const double d = u[col][col];
            exchange |= fabs(u[i][col]) >= fabs(d);
            const double f = u[i][col] / d;
#pragma unroll
            for (int j = col + 1; j < NA; j++) u[i][j] -= f * u[col][j];
            b -= f * dx[col];
        }
        dx[i] = b;
    }
#pragma unroll
    for (int i = NA - 1; i >= 0; i--) {
        double v = dx[i];
#pragma unroll
        for (int j = i + 1; j < NA; j++) v -= u[i][j] * dx[j];
        exchange |= u[i][i] == 0.0;
        dx[i] = v / u[i][i];
    }
#pragma unroll
    for (int i = NA; i < REACT_NS; i++) dx[i] = 0.0;
    if (exchange) {
        double sv[REACT_NS], dv[REACT_NS];
        for (int i = 0; i < REACT_NS; i++) sv[i] = s[i];
        solve_pivoted<NT>(D, M, sv, h, dv);
#pragma unroll
        for (int i = 0; i < REACT_NS; i++) dx[i] = dv[i];
    }
}

} // namespace sr
