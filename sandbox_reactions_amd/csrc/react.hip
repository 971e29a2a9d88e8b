// P6 burning on the GPU (crates/sr-physics/src/reference/react.rs; the rate law crates/sr-physics/src/rates.rs): one
// thread per cell in FP64, each cell burning alone over the pass's dt. N_Fe first in closed form, then the other
// enabled records sub-cycled by linearised backward Euler, (I - hJ) dX = h S, each sub-step sized by burn_dx on the
// fractions and burn_dt on T, checked, halved until it holds; the heat of the mass each sub-step moved into the energy
// and the record's group; the burn clock slowing a sub-step whose heating passes eps_th c_s / K_burn; the neutrino loss
// eps_nu h with the cooling on; with T pinned the energy follows the final composition at T0. A cell below Sigma_vac is
// not touched and a cell no record converts is left bit for bit. The state's fractions and energy are the world's f32
// planes, Sigma its FP64 plane; the cold energy is read from FP64 tables; every expression and sum order is the
// oracle's, so the cells differ from it only by the device's f64 elementary functions and the f32 planes.
#include <cfloat>
#include <cmath>
#include <cstring>

#include "common.hpp"
#include "react.hpp"
#include "react_solve.hpp"

namespace sr {

#define NS REACT_NS
#define NR SR_REACT_RECORDS
#define NG SR_REACT_GROUPS
#define ID_N 9
#define X_N_STAR 0.5

__constant__ double r_z[NS] = {1, 2, 6, 8, 10, 12, 14, 16, 26, 0};
__constant__ double r_a[NS] = {1, 4, 12, 16, 20, 24, 28, 32, 56, 1};
// (Z + 1) / A and Z / A per species
__constant__ double r_zp1_a[NS] = {2.0, 3.0 / 4.0, 7.0 / 12.0, 9.0 / 16.0, 11.0 / 20.0, 13.0 / 24.0, 15.0 / 28.0,
                                   17.0 / 32.0, 27.0 / 56.0, 1.0};
__constant__ double r_z_a[NS] = {1.0, 0.5, 0.5, 0.5, 0.5, 0.5, 0.5, 0.5, 26.0 / 56.0, 0.0};

int react_check(const sr_react_params *p) {
    if (!p) return SR_OK;
    if (p->n_records < 0 || p->n_records > NR) return SR_ERR_ARGUMENT;
    if (p->nfe < -1 || p->nfe >= p->n_records) return SR_ERR_ARGUMENT;
    if (!(p->burn_dx > 0.0) || !(p->burn_dt > 0.0) || !(p->burn_k >= 0.0)) return SR_ERR_ARGUMENT;
    if (p->neutrinos && !(p->t_nu > 0.0)) return SR_ERR_ARGUMENT;
    for (int r = 0; r < p->n_records; r++) {
        const sr_react_record &c = p->rec[r];
        if (c.n_in < 1 || c.n_in > 4 || c.n_out < 0 || c.n_out > 4 || c.group < 0 || c.group >= NG) return SR_ERR_ARGUMENT;
        if (c.n_terms < 0 || c.n_terms > 4 || (c.n_terms > 0 && !(c.t_thr > 0.0))) return SR_ERR_ARGUMENT;
        for (int k = 0; k < c.n_terms; k++)
            if (!(c.t_k[k] > 0.0) || !(c.w[k] > 0.0)) return SR_ERR_ARGUMENT;
        for (int k = 0; k < c.n_in; k++)
            if (c.in_species[k] < 0 || c.in_species[k] >= NS || !(c.in_order[k] > 0.0)) return SR_ERR_ARGUMENT;
        for (int k = 0; k < c.n_out; k++)
            if (c.out_species[k] < 0 || c.out_species[k] >= NS) return SR_ERR_ARGUMENT;
        if (c.gated && !(c.sigma_g > 0.0)) return SR_ERR_ARGUMENT;
    }
    if (p->nfe >= 0) {  // the closed form's shape (react.rs:205-212)
        const sr_react_record &c = p->rec[p->nfe];
        if (c.n_terms != 0 || c.n_in != 1 || c.n_out != 1 || c.in_order[0] != 1.0 || !c.gated || c.gate_p != 1.0 ||
            c.out_species[0] != ID_N)
            return SR_ERR_ARGUMENT;
    }
    return SR_OK;
}

void react_build(const sr_react_params *p, const sr_physics &ph, ReactDev *out) {
    std::memset(out, 0, sizeof *out);
    out->P = *p;
    for (int r = 0; r < p->n_records; r++) {
        const sr_react_record &c = p->rec[r];
        // rates.rs:62-71: log-spaced nodes from T_thr over the span; a record of the same law as an earlier one reads its
        out->f_of[r] = -1;
        if (c.n_terms == 0) continue;
        for (int q = 0; q < r && out->f_of[r] < 0; q++) {
            const sr_react_record &o = p->rec[q];
            bool same = o.n_terms == c.n_terms && o.t_thr == c.t_thr;
            for (int k = 0; same && k < c.n_terms; k++)
                same = o.t_k[k] == c.t_k[k] && o.nu[k] == c.nu[k] && o.w[k] == c.w[k];
            if (same) out->f_of[r] = out->f_of[q];
        }
        if (out->f_of[r] >= 0) continue;
        out->f_of[r] = out->tables++;
        for (int i = 0; i < REACT_TABLE; i++)
            out->ln_f[out->f_of[r]][i] =
                std::log(f_sum(c, c.t_thr * std::exp(std::log(2.5) * (double)i / (double)(REACT_TABLE - 1))));
    }
    react_shape(out);
    out->sigma_vac = ph.sigma_vac;
    out->t_floor = ph.t_floor;
    const double k[2][2] = {{ph.k1e, ph.k2e}, {ph.k1n, ph.k2n}};
    for (int q = 0; q < 2; q++) {
        out->cold_pair[q] = k[q][0] > 0.0 && k[q][1] > 0.0;
        if (out->cold_pair[q]) cold_table(k[q][0], k[q][1], out->cold_lnu[q]);
    }
    out->cold_ln_min = std::log(1e-8);
    out->cold_step = (std::log(1e8) - std::log(1e-8)) / (COLD_POINTS - 1);
}

// -------------------------------------------------------------------------------------------------- the device side

// 1/mu and Y_e (registry.rs:146-154): sums of X (Z + 1) / A and X Z / A in species order
__device__ inline void comp(const double *x, double *mu, double *y_e) {
    double im = 0.0, ye = 0.0;
#pragma unroll
    for (int s = 0; s < NS; s++) {
        im += x[s] * r_zp1_a[s];
        ye += x[s] * r_z_a[s];
    }
    *mu = 1.0 / im;
    *y_e = ye;
}

// u(x) of one pair from its FP64 table: linear in (ln x, ln u), the K1 x^2 power law below the first node
__device__ inline double cold_u_d(const ReactDev &D, const double *lnu, double x) {
    if (x <= 0.0) return 0.0;
    const double pos = (log(x) - D.cold_ln_min) / D.cold_step;
    if (pos < 0.0) return exp(lnu[0]) * (x / 1e-8) * (x / 1e-8);
    int i = (int)floor(pos);
    if (i > COLD_POINTS - 2) i = COLD_POINTS - 2;
    const double frac = pos - (double)i;
    return exp(lnu[i] + frac * (lnu[i + 1] - lnu[i]));
}

__device__ inline double eps_cold_d(const ReactDev &D, const Lds &M, double sigma, double y_e, double x_n) {
    double u = 0.0;
    if (D.cold_pair[0]) u += cold_u_d(D, M.cold, y_e * sigma);
    if (D.cold_pair[1]) u += cold_u_d(D, M.cold + COLD_POINTS, x_n * sigma);
    return u / sigma;
}

// x^n for the whole orders 0..3 by products, pow() otherwise
__device__ __forceinline__ double ipow(double x, double n) {
    if (n == 1.0) return x;
    if (n == 2.0) return x * x;
    if (n == 3.0) return x * x * x;
    if (n == 0.0) return 1.0;
    return pow(x, n);
}

// the gate g(Y_e Sigma) (rates.rs:119-125)
__device__ inline double gate(const sr_react_record &c, double sigma, double y_e) {
    if (!c.gated) return 1.0;
    const double yes = y_e * sigma;
    return yes > c.sigma_g ? pow(yes / c.sigma_g - 1.0, c.gate_p) : 0.0;
}

// N_Fe over dt in closed form (react.rs:470-513)
__device__ double nfe_exact(const ReactDev &D, double sigma, double *x, double dt) {
    const sr_react_record &c = D.P.rec[D.P.nfe];
    const int fe = c.in_species[0], n = c.out_species[0];
    const double y_fe = r_z_a[fe];
    const double b = c.sigma_g / sigma;
    double others[NS], mu, a_y;
    for (int s = 0; s < NS; s++) others[s] = x[s];
    others[fe] = 0.0;
    comp(others, &mu, &a_y);
    const double cc = b - a_y;
    const double v = y_fe * x[fe];
    const double u = v - cc;
    if (!(u > 0.0 && v > 0.0) || dt <= 0.0) return 0.0;
    const double k = c.a_coef * ipow(sigma, c.a_sigma) / b;
    const double w = cc >= 0.0 ? u : v, s = cc >= 0.0 ? cc : -cc;
    const double ks = k * s * dt;
    const double phi = ks > 0.0 ? -expm1(-ks) / s : k * dt;
    const double dy = u * v * phi / (1.0 + w * phi);
    double dm = fmin(dy / y_fe, x[fe]);
    const double left = w * exp(-ks) / (1.0 + w * phi);
    if (left <= 4.0 * DBL_EPSILON * b) {
        if (cc >= 0.0) {
            x[fe] -= dm;
            x[n] += dm;
            double nudge = DBL_EPSILON * x[fe];
            for (int it = 0; it < 16; it++) {
                double m2, y_e;
                comp(x, &m2, &y_e);
                if (y_e * sigma <= c.sigma_g || x[fe] == 0.0) break;
                const double more = fmin(fmax((y_e * sigma - c.sigma_g) / (sigma * y_fe), nudge), x[fe]);
                x[fe] -= more;
                x[n] += more;
                dm += more;
                nudge *= 2.0;
            }
            return dm;
        }
        dm = x[fe];
    }
    x[fe] -= dm;
    x[n] += dm;
    return dm;
}

struct CellOut {
    double de, lost, booked[NG], pinned_e;
    int nfe, pinned, unfinished, changed;
    double substeps, retried, max_dx, max_dt_rel;
};

// one cell over dt (react.rs:272-449), its fractions in x; the composition, the cold energy and T of a state are formed
// once, with the sub-step that reaches it
template <int NA, int NT>
__device__ inline void burn(const ReactDev &D, const Lds &M, double sigma, double (&x)[NS], double e_tot, double dt,
                            CellOut &cell) {
    const sr_react_params &P = D.P;
    const int nr = P.n_records, pin = P.pin_temperature;
    cell.de = cell.lost = cell.pinned_e = cell.substeps = cell.retried = cell.max_dx = cell.max_dt_rel = 0.0;
#pragma unroll
    for (int g = 0; g < NG; g++) cell.booked[g] = 0.0;
    cell.nfe = cell.pinned = cell.unfinished = cell.changed = 0;
    double mu, y_e;
    comp(x, &mu, &y_e);
    double t = mu * fmax(e_tot - eps_cold_d(D, M, sigma, y_e, x[ID_N]), D.t_floor / mu);
    const double t0 = t;
    if (P.nfe >= 0) {
        // N_Fe's rate at the start (no temperature law: f = 1)
        const sr_react_record &c = P.rec[P.nfe];
        const double g = gate(c, sigma, y_e);
        double x_in = 0.0;
#pragma unroll
        for (int s = 0; s < NS; s++)
            if (s == c.in_species[0]) x_in = x[s];
        const double w_nfe = g > 0.0 ? c.a_coef * ipow(sigma, c.a_sigma) * x_in * g : 0.0;
        cell.nfe = w_nfe > 0.0;
        if (cell.nfe) {
            double xn[NS];
            for (int s = 0; s < NS; s++) xn[s] = x[s];
            const double dm = nfe_exact(D, sigma, xn, dt);
            const double heat = c.q * dm;
            if (!pin) e_tot += heat;
            cell.de += heat;
#pragma unroll
            for (int q = 0; q < NG; q++)
                if (q == c.group) cell.booked[q] += heat;
            cell.changed |= dm > 0.0;
#pragma unroll
            for (int s = 0; s < NS; s++) x[s] = xn[s];
            comp(x, &mu, &y_e);
            if (!pin) t = mu * fmax(e_tot - eps_cold_d(D, M, sigma, y_e, x[ID_N]), D.t_floor / mu);
        }
    }
    double t_done = 0.0, h_try = HUGE_VAL;
    unsigned long long attempts = 0;
    while (t_done < dt) {
        double t_rem = dt - t_done;
        double s[NS], qdot = 0.0;
#pragma unroll
        for (int i = 0; i < NS; i++) {
            s[i] = 0.0;
            M.v[i * NT] = x[i];
        }
        double enu = P.neutrinos && t >= P.t_nu ? P.a_nu * pow(t / P.t_nu, P.m_nu) : 0.0;
        int any = 0, f_last = -1;
        double f_val = 1.0;
        for (int r = 0; r < nr; r++) {
            if (r == P.nfe) continue;
            const sr_react_record &c = P.rec[r];
            // omega at X and, for each input j, at X with X_j = 1 (whose factor 1^n is exactly 1): f, g and A Sigma^a
            // once (f kept for a next record of the same law), each input's power once, the products in their order
            if (c.n_terms == 0 || D.f_of[r] != f_last) f_val = temp_factor(D, M, r, t);
            f_last = D.f_of[r];
            const double f = f_val, g = gate(c, sigma, y_e);
            const double ap = c.a_coef * ipow(sigma, c.a_sigma);
            const int n_in = c.n_in;
            double xk[4], pw[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                xk[k] = k < n_in ? M.v[c.in_species[k] * NT] : 1.0;
                pw[k] = k < n_in ? ipow(xk[k], c.in_order[k]) : 1.0;
            }
            double orders = 1.0;
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (k < n_in) orders *= pw[k];
            const double w = ap * orders * f * g;
            M.omega[D.slot[r] * NT] = w;
            cell.nfe |= c.latch && w > 0.0;
            double *grad = M.grad + D.ent0[r] * NT;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                if (k >= n_in) break;
                const int j = c.in_species[k];
                const double n = c.in_order[k];
                double oj = 1.0;
#pragma unroll
                for (int q = 0; q < 4; q++)
                    if (q < n_in) oj *= c.in_species[q] == j ? 1.0 : pw[q];
                grad[k * NT] = n * ipow(xk[k], n - 1.0) * (ap * oj * f * g);
            }
#pragma unroll
            for (int i = 0; i < NS; i++) s[i] += D.nu[r][i] * w;
            qdot += c.q * w;
            any |= w != 0.0;
        }
        if (enu == 0.0 && !any) break;
        double k = 1.0;  // the burn clock (react.rs:451-462)
        if (!pin && P.burn_k > 0.0) {
            const double eps_th = t / mu;
            const double q_max = eps_th * sqrt(2.0 * eps_th) / P.burn_k;
            if (qdot > q_max) k = qdot / q_max;
        }
        if (k != 1.0) {
            t_rem = t_rem / k;
            enu = enu * k;
        }
        double s_max = 0.0;
#pragma unroll
        for (int i = 0; i < NS; i++) s_max = fmax(s_max, fabs(s[i]));
        double h = t_rem;
        if (s_max > 0.0) h = fmin(h, P.burn_dx / s_max);
        if (!pin) {
            double dinv_mu = 0.0;
#pragma unroll
            for (int i = 0; i < NS; i++) dinv_mu += s[i] * r_zp1_a[i];
            const double dt_dt = mu * (qdot - enu) - t * mu * dinv_mu;
            if (dt_dt != 0.0) h = fmin(h, P.burn_dt * t / fabs(dt_dt));
        }
        h = fmin(h, h_try);
        for (;;) {
            attempts++;
            if (attempts > 1000000ull) {
                cell.unfinished = 1;
                break;
            }
            const int last = h >= t_rem;
            const double h_use = fmin(h, t_rem);
            double dx[NS];
            solve<NA, NT>(D, M, s, h_use, dx);
            double worst = 0.0;
            int negative = 0;
#pragma unroll
            for (int i = 0; i < NS; i++) {
                M.v[i * NT] = dx[i];
                worst = fmax(worst, fabs(dx[i]));
                dx[i] += x[i];  // the new fractions from here
                if (dx[i] < -1e-12) negative = 1;
            }
            double de = 0.0, by_group[NG];
#pragma unroll
            for (int g = 0; g < NG; g++) by_group[g] = 0.0;
            for (int r = 0; r < nr; r++) {
                if (r == P.nfe) continue;
                const sr_react_record &c = P.rec[r];
                double lin = 0.0;
                for (int q = 0; q < c.n_in; q++)
                    lin += M.grad[(D.ent0[r] + q) * NT] * M.v[c.in_species[q] * NT];
                const double e = c.q * (h_use * (M.omega[D.slot[r] * NT] + lin));
                de += e;
#pragma unroll
                for (int g = 0; g < NG; g++)
                    if (g == c.group) by_group[g] += e;
            }
            const double lost = enu * h_use;
            double sum = 0.0;
#pragma unroll
            for (int i = 0; i < NS; i++) {
                dx[i] = fmax(dx[i], 0.0);
                sum += dx[i];
            }
#pragma unroll
            for (int i = 0; i < NS; i++) dx[i] /= sum;
            double mu_new, y_e_new, e_new = e_tot, t_new = t0;
            comp(dx, &mu_new, &y_e_new);
            if (!pin) {
                e_new = e_tot + de - lost;
                t_new = mu_new * fmax(e_new - eps_cold_d(D, M, sigma, y_e_new, dx[ID_N]), D.t_floor / mu_new);
            }
            const double dt_rel = pin ? 0.0 : fabs(t_new - t) / t;
            const int bad = worst > P.burn_dx * (1.0 + 1e-12) || dt_rel > P.burn_dt * (1.0 + 1e-12) || negative;
            if (bad && h_use > 1e-14 * dt) {
                h = 0.5 * h_use;
                cell.retried += 1.0;
                continue;
            }
#pragma unroll
            for (int i = 0; i < NS; i++) x[i] = dx[i];
            e_tot = e_new;
            mu = mu_new;
            y_e = y_e_new;
            t = t_new;
            cell.de += de - lost;
            cell.lost += lost;
#pragma unroll
            for (int g = 0; g < NG; g++) cell.booked[g] += by_group[g];
            cell.substeps += 1.0;
            cell.changed = 1;
            cell.max_dx = fmax(cell.max_dx, worst);
            cell.max_dt_rel = fmax(cell.max_dt_rel, dt_rel);
            t_done = last ? dt : (k == 1.0 ? t_done + h_use : t_done + h_use * k);
            h_try = fmax(2.0 * h_use, DBL_MIN);
            break;
        }
        if (cell.unfinished) break;
    }
    if (pin && cell.changed) {
        cell.pinned = 1;
        cell.pinned_e = t0 / mu + eps_cold_d(D, M, sigma, y_e, x[ID_N]);
    }
}

// one thread per cell (a sum carried over more would hold 30 registers through the solve)
template <int NA, int NT>
__global__ void __launch_bounds__(NT, 2) k_react(const ReactDev *__restrict__ Dp, HydroState st, int n, double dt_arg,
                                                      const double *__restrict__ scal, double *__restrict__ nuclear,
                                                      double *__restrict__ lost, double *__restrict__ snu, double *psum,
                                                      double *pmax) {
    extern __shared__ double mem[];
    const ReactDev &D = *Dp;
    const int nt = D.tables * REACT_TABLE, i = blockIdx.x * NT + threadIdx.x;
    for (int k = threadIdx.x; k < 2 * COLD_POINTS; k += NT) mem[k] = (&D.cold_lnu[0][0])[k];
    for (int k = threadIdx.x; k < nt; k += NT) mem[2 * COLD_POINTS + k] = (&D.ln_f[0][0])[k];
    __syncthreads();
    Lds M;
    M.cold = mem;
    M.ln_f = mem + 2 * COLD_POINTS;
    M.v = mem + 2 * COLD_POINTS + nt + threadIdx.x;
    M.omega = M.v + NS * NT;
    M.grad = M.omega + D.slots * NT;
    const double dt = dt_arg >= 0.0 ? dt_arg : scal[0];
    double vs[REACT_SUMS], vm[REACT_MAXES];
    for (int k = 0; k < REACT_SUMS; k++) vs[k] = 0.0;
    for (int k = 0; k < REACT_MAXES; k++) vm[k] = 0.0;
    if (i < n) {
        const double sigma = st.sigma[i];
        double x[NS];
#pragma unroll
        for (int s = 0; s < NS; s++) x[s] = (double)st.x[(size_t)s * n + i];
        CellOut c{};
        if (!(sigma < D.sigma_vac)) {
            const double mx = st.mx[i], my = st.my[i];
            const double kinetic = 0.5 * (mx * mx + my * my) / (sigma * sigma);
            burn<NA, NT>(D, M, sigma, x, st.e[i] / sigma - kinetic, dt, c);
            vs[0] = c.substeps;
            vs[1] = c.retried;
            vs[2] = (double)c.unfinished;
            vm[0] = c.substeps;
            vm[1] = c.max_dx;
            vm[2] = c.max_dt_rel;
            vm[3] = (double)c.nfe;
            if (c.changed) {
#pragma unroll
                for (int s = 0; s < NS; s++) st.x[(size_t)s * n + i] = (float)x[s];
                st.e[i] = (float)(c.pinned ? sigma * (c.pinned_e + kinetic) : st.e[i] + sigma * c.de);
            }
        }
        // booked as the cell changed, zero elsewhere
        const double on = c.changed ? sigma : 0.0;
#pragma unroll
        for (int g = 0; g < NG; g++) nuclear[(size_t)g * n + i] = vs[3 + g] = on * c.booked[g];
        lost[i] = vs[3 + NG] = on * c.lost;
        snu[i] = c.changed && x[ID_N] >= X_N_STAR && dt > 0.0 ? sigma * c.lost / dt : 0.0;
    }
    block_partials<REACT_SUMS>(vs, psum, gridDim.x);
    block_partials<REACT_MAXES, 1>(vm, pmax, gridDim.x);
}

// The report's sums and maxima over the blocks, a block each, in a fixed order. On the host, over one block's worth of
// partials per 64 or 256 cells, reading the report took 236 us at 2048^2.
__global__ void __launch_bounds__(256) k_react_report(const double *psum, const double *pmax, int nb, double *out) {
    const int k = blockIdx.x;
    if (k < REACT_SUMS) {
        const double s = sum_partials(psum + (size_t)k * nb, nb);
        if (threadIdx.x == 0) out[k] = s;
    } else {
        double m[1] = {0.0};
        for (int i = threadIdx.x; i < nb; i += 256) m[0] = fmax(m[0], pmax[(size_t)(k - REACT_SUMS) * nb + i]);
        block_partials<1, 1>(m, out, 1, k);
    }
}

int react_report(const double *psum, const double *pmax, int nb, double *out, hipStream_t s) {
    hipLaunchKernelGGL(k_react_report, dim3(REACT_SUMS + REACT_MAXES), dim3(256), 0, s, psum, pmax, nb, out);
    SR_HIP(hipGetLastError());
    return SR_OK;
}

// whether the records' system leaves the neutrons out
static bool react_neutrons(const ReactDev &h) {
    unsigned any = h.row[ID_N];
    for (int i = 0; i < NS; i++) any |= h.row[i] >> ID_N & 1;
    for (int r = 0; r < h.P.n_records; r++)
        if (r != h.P.nfe) any |= h.nu[r][ID_N] != 0.0;
    return any != 0;
}

#define REACT_LDS (78 * 1024)  // a block of 256 threads: two blocks, each with 2 KB of partial sums, fill a CU's 160 KB
static int react_lds(int nt, int tables, int slots, int entries) {
    return (int)sizeof(double) * (2 * COLD_POINTS + tables * REACT_TABLE + nt * (NS + slots + entries));
}

ReactLaunch react_plan(const ReactDev &h) {
    const bool fits = react_lds(256, h.tables, h.slots, h.entries) <= REACT_LDS;
    const int nt = fits ? 256 : REACT_NT_LEAST;
    return {nt, react_lds(nt, h.tables, h.slots, h.entries), react_neutrons(h)};
}

static auto react_kernel(const ReactLaunch &plan) {
    return plan.nt == 256 ? (plan.neutrons ? k_react<NS, 256> : k_react<NS - 1, 256>)
                          : (plan.neutrons ? k_react<NS, REACT_NT_LEAST> : k_react<NS - 1, REACT_NT_LEAST>);
}

int react_prepare(const ReactLaunch &plan) {
    // a kernel's limit is the process's, not the world's: always the most that any records take (87 KB with 64 threads)
    const int most = plan.nt == 256 ? REACT_LDS : react_lds(plan.nt, NR, NR, 4 * NR);
    SR_HIP(hipFuncSetAttribute((const void *)react_kernel(plan), hipFuncAttributeMaxDynamicSharedMemorySize, most));
    return SR_OK;
}

int react_launch(const ReactDev *D, const ReactLaunch &plan, const HydroState &st, int n, double dt, const double *scal,
                 double *nuclear, double *lost, double *snu, double *psum, double *pmax, int *nblocks, hipStream_t s) {
    const int nb = plan.blocks(n);
    auto kernel = react_kernel(plan);
    hipLaunchKernelGGL(kernel, dim3(nb), dim3(plan.nt), plan.lds, s, D, st, n, dt, scal, nuclear, lost, snu, psum, pmax);
    if (nblocks) *nblocks = nb;
    SR_HIP(hipGetLastError());
    return SR_OK;
}

} // namespace sr
