// P6's temperature factor and linear system on the CPU. The system: random records, derivatives and steps through solve<9> (no neutrons) and
// solve<10>, against Gaussian elimination with partial pivoting in long double. Prints the largest error of a system's dX
// over its largest element, and how many systems needed a row exchange.
#include <cstdio>
#include <cstring>
#include <random>

#include "../../sandbox_reactions_amd/csrc/react_solve.hpp"

using namespace sr;

static std::mt19937_64 rng(7);
static double uniform(double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); }
static int pick(int n) { return (int)(rng() % n); }

static void reference(const ReactDev &D, const double *grad, const double *s, double h, long double *dx) {
    long double a[REACT_NS][REACT_NS + 1] = {};
    for (int i = 0; i < REACT_NS; i++) {
        a[i][i] = 1.0L;
        a[i][REACT_NS] = (long double)h * s[i];
        for (int r = 0; r < D.P.n_records; r++) {
            if (r == D.P.nfe) continue;
            for (int k = 0; k < D.P.rec[r].n_in; k++)
                a[i][D.P.rec[r].in_species[k]] -= (long double)h * D.nu[r][i] * grad[D.ent0[r] + k];
        }
    }
    for (int c = 0; c < REACT_NS; c++) {
        int p = c;
        for (int i = c + 1; i < REACT_NS; i++)
            if (fabsl(a[i][c]) > fabsl(a[p][c])) p = i;
        for (int j = 0; j <= REACT_NS; j++) std::swap(a[c][j], a[p][j]);
        for (int i = c + 1; i < REACT_NS; i++) {
            const long double f = a[i][c] / a[c][c];
            for (int j = c; j <= REACT_NS; j++) a[i][j] -= f * a[c][j];
        }
    }
    for (int i = REACT_NS - 1; i >= 0; i--) {
        long double v = a[i][REACT_NS];
        for (int j = i + 1; j < REACT_NS; j++) v -= a[i][j] * dx[j];
        dx[i] = v / a[i][i];
    }
}

template <int NA> static void run(int systems) {
    double worst = 0.0;
    for (int n = 0; n < systems; n++) {
        static ReactDev D;
        std::memset(&D, 0, sizeof D);
        D.P.n_records = 1 + pick(SR_REACT_RECORDS);
        D.P.nfe = NA < REACT_NS && pick(2) ? pick(D.P.n_records) : -1;
        for (int r = 0; r < D.P.n_records; r++) {
            sr_react_record &c = D.P.rec[r];
            const int ns = r == D.P.nfe ? REACT_NS : NA;
            c.n_in = 1 + pick(3);
            c.n_out = 1 + pick(3);
            for (int k = 0; k < c.n_in; k++) c.in_species[k] = pick(ns), c.in_share[k] = 1.0 / c.n_in;
            for (int k = 0; k < c.n_out; k++) c.out_species[k] = pick(ns), c.out_share[k] = 1.0 / c.n_out;
        }
        react_shape(&D);
        double grad[4 * SR_REACT_RECORDS], s[REACT_NS] = {}, dx[REACT_NS];
        for (double &g : grad) g = pick(4) ? std::exp(uniform(-3.0, 3.0)) : 0.0;
        for (int i = 0; i < NA; i++) s[i] = uniform(-1.0, 1.0);
        const double h = std::exp(uniform(-4.0, 1.0));
        const Lds M = {nullptr, nullptr, nullptr, nullptr, grad};
        solve<NA, 1>(D, M, s, h, dx);
        long double ref[REACT_NS], most = 0.0L, err = 0.0L;
        reference(D, grad, s, h, ref);
        for (int i = 0; i < REACT_NS; i++) {
            most = std::max(most, fabsl(ref[i]));
            err = std::max(err, fabsl(ref[i] - dx[i]));
        }
        worst = std::max(worst, (double)(err / most));
    }
    std::printf("%d %.3e\n", NA, worst);
}

// f(T) from just above T_thr to past the table's span against the same interpolation in long double, and T that is no
// number. Prints the largest relative error.
static void factor() {
    double worst = 0.0;
    for (int n = 0; n < 20000; n++) {
        static ReactDev D;
        std::memset(&D, 0, sizeof D);
        sr_react_record &c = D.P.rec[0];
        c.n_terms = 1;
        c.t_thr = std::exp(uniform(-20.0, 20.0));
        c.t_k[0] = 100.0 * c.t_thr;
        c.nu[0] = uniform(1.0, 8.0);
        c.w[0] = 1.0;
        double ln_f[REACT_TABLE];
        for (int i = 0; i < REACT_TABLE; i++)
            ln_f[i] = std::log(f_sum(c, c.t_thr * std::exp(std::log(2.5) * i / (REACT_TABLE - 1))));
        const Lds M = {nullptr, ln_f, nullptr, nullptr, nullptr};
        const double t = c.t_thr * (n % 2 ? uniform(1.0, 2.49) : 1.0 + std::exp(uniform(-30.0, 0.0)));
        const long double pos = logl((long double)t / c.t_thr) / (logl(2.5L) / (REACT_TABLE - 1));
        const int i = (int)floorl(pos);
        const long double ref = expl(ln_f[i] + (pos - i) * ((long double)ln_f[i + 1] - ln_f[i]));
        worst = std::max(worst, (double)fabsl(temp_factor(D, M, 0, t) / ref - 1.0L));
        if (!std::isnan(temp_factor(D, M, 0, NAN)) || temp_factor(D, M, 0, 0.999 * c.t_thr) != 0.0) worst = NAN;
    }
    std::printf("factor %.3e\n", worst);
}

int main() {
    factor();
    run<REACT_NS - 1>(4000);
    run<REACT_NS>(4000);
}
