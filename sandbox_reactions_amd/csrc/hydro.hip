// P4: unsplit MUSCL-Hancock hydro with the MC limiter and HLL fluxes (Davis speeds), 14 channels, gravity's
// half-step source with the face work, the radiation force with its share cap, and FP64 mass.
//
// The scheme is the reference's (crates/sr-physics/src/reference/hydro.rs, module doc :1-96; GPU
// crates/sr-engine/shaders/hydro.wgsl:910-1153); the kernel layout is this library's own:
//   * one 320-thread block (five wave64s) per 16x16 tile: 256 threads own the tile's cells and 64 its one-cell
//     ring (the face neighbours), so every predicted face state the tile's fluxes read is made once in the block;
//   * primitives of the tile and a two-cell halo (ghosts by the edge rules) are staged in LDS as structure of
//     arrays; the slots' predicted low faces go to LDS and every HLL flux and gravity face work is made once, by the
//     slot whose high face it is, and read back by the cell on the other side (so the flux differences telescope);
//   * the ten species are not carried through the main pass: their mass-weighted mean 1/mu is linear in the
//     fractions and rides along as a pseudo-species, and each species' face value and flux is made in a short loop
//     after the main fluxes, the species' shared limiter factor kept in registers; a species that the staged cells
//     hold none of is left out of both;
//   * Sigma is stored and updated in FP64 (flux differences of FP32 fluxes summed in FP64), so the total mass is
//     conserved to FP64 round-off; the other channels are FP32.
// Two modes share the code: MID writes Sigma_mid = (Sigma^n + Sigma^{n+1}) / 2 from the mass fluxes
// (hydro.rs:817-836) for the half-step gravity solve; UPDATE writes the next state.
#include <algorithm>
#include <cfloat>
#include <cmath>

#include "common.hpp"
#include "hydro.hpp"

namespace sr {

#define T 16
#define HALO 2
#define PW (T + 2 * HALO) // 20
#define NPRIM (PW * PW)   // 400
#define NSLOT (T * T + 4 * T) // 320
#define NS 10
#define HOT_FACE 2.0f

// (Z + 1) / A per species, assets/elements.json order: H He C O Ne Mg Si S Fe n (registry.rs:146-154)
__constant__ float c_imu[NS] = {2.0f, 0.75f, 7.0f / 12.0f, 9.0f / 16.0f, 11.0f / 20.0f,
                                13.0f / 24.0f, 15.0f / 28.0f, 17.0f / 32.0f, 27.0f / 56.0f, 1.0f};

__device__ __forceinline__ unsigned long long wave_most(unsigned long long v) {
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long other = __shfl_xor(v, o, 64);
        v = other > v ? other : v;
    }
    return v;
}

struct Prim {
    float s, u, v, p, im;
    float ye, xn;  // Y_e and X_n, read only with the cold pressure on
};

__device__ __forceinline__ float mc(float l, float c, float r) {
    const float a = c - l, b = r - c;
    if (a * b <= 0.0f) return 0.0f;
    const float m = fminf(fminf(fabsf(0.5f * (a + b)), 2.0f * fabsf(a)), 2.0f * fabsf(b));
    return copysignf(m, a);
}

__device__ __forceinline__ float eps_floor(const HydroParams &P, float im) { return P.t_floor_g * im; }

__device__ __forceinline__ float sound(const HydroParams &P, float s, float p) {
    return sqrtf(fmaxf(__fdividef(P.gamma * p, s), 0.0f));
}

// E of a primitive state (hydro.rs:444-459 with gamma): eps = max((Pi - Pi_cold) / ((gamma-1) Sigma), floor),
// E = Sigma (eps + eps_cold) + kinetic
template <bool COLD> __device__ __forceinline__ float cons_e(const HydroParams &P, const Prim &q) {
    const float pc = COLD ? pi_cold(P.cold, q.s, q.ye, q.xn) : 0.0f;
    const float eps = fmaxf(__fdividef(q.p - pc, P.gm1 * q.s), eps_floor(P, q.im));
    const float ec = COLD ? eps_cold(P.cold, q.s, q.ye, q.xn) : 0.0f;
    return q.s * (eps + ec) + 0.5f * q.s * (q.u * q.u + q.v * q.v);
}

// primitives of a conserved (s, mx, my, E, s*im, s*Y_e, s*X_n); false when not a state (hydro.rs:462-479)
template <bool COLD>
__device__ __forceinline__ bool prim_of(const HydroParams &P, float s, float mx, float my, float e, float sim,
                                        float sye, float sxn, Prim &o) {
    if (!(s > 0.0f) || !isfinite(s) || !isfinite(mx) || !isfinite(my) || !isfinite(e) || !isfinite(sim))
        return false;
    const float is = 1.0f / s;
    const float im = sim * is, u = mx * is, v = my * is, ye = sye * is, xn = sxn * is;
    const float raw = e * is - 0.5f * (u * u + v * v) - (COLD ? eps_cold(P.cold, s, ye, xn) : 0.0f);
    if (!(raw > 0.0f)) return false;
    const float eps = fmaxf(raw, eps_floor(P, im));
    o.s = s;
    o.u = u;
    o.v = v;
    o.p = P.gm1 * s * eps + (COLD ? pi_cold(P.cold, s, ye, xn) : 0.0f);
    o.im = im;
    o.ye = ye;
    o.xn = xn;
    return true;
}

// normal flux of (Sigma, mx, my, E) through a face normal to dir of a state with energy e
__device__ __forceinline__ void flux4(const Prim &q, float e, int dir, float f[4]) {
    const float un = dir ? q.v : q.u, ut = dir ? q.u : q.v;
    const float m = q.s * un;
    f[0] = m;
    f[1 + dir] = m * un + q.p;
    f[2 - dir] = m * ut;
    f[3] = (e + q.p) * un;
}

// HLL between face states l and r (hydro.rs:516-540); returns the 4 fluxes, and whether the left side is upwind
__device__ __forceinline__ bool hll(const HydroParams &P, const Prim &l, float el, const Prim &r, float er, int dir,
                                    float f[4]) {
    const float unl = dir ? l.v : l.u, unr = dir ? r.v : r.u;
    const float cl = sound(P, l.s, l.p), cr = sound(P, r.s, r.p);
    const float sl = fminf(unl - cl, unr - cr), sr = fmaxf(unl + cl, unr + cr);
    float fl[4], fr[4];
    flux4(l, el, dir, fl);
    flux4(r, er, dir, fr);
    if (sl >= 0.0f) {
        for (int k = 0; k < 4; k++) f[k] = fl[k];
    } else if (sr <= 0.0f) {
        for (int k = 0; k < 4; k++) f[k] = fr[k];
    } else {
        const float ul[4] = {l.s, l.s * l.u, l.s * l.v, el}, ur[4] = {r.s, r.s * r.u, r.s * r.v, er};
        const float inv = 1.0f / (sr - sl);
        for (int k = 0; k < 4; k++) f[k] = (sr * fl[k] - sl * fr[k] + sl * sr * (ur[k] - ul[k])) * inv;
    }
    return f[0] > 0.0f;
}

// gravity's source at one face (hydro.rs:1048-1067); d = (phi_low - phi_high) / dx
__device__ inline void face_work(float q, float sl, float sh, float pl, float ph, float d, float dt, float out[3]) {
    const float a = fmaxf(sl, 0.0f), b = fmaxf(sh, 0.0f);
    const float w = a + b > 0.0f ? a / (a + b) : 0.5f;
    const float extra = dt * (q - 0.5f * (pl + ph)) * d;
    float c = 0.0f, kick = 0.0f, el = 0.0f, eh = 0.0f;
    if (extra < 0.0f && a > 0.0f && b > 0.0f) {
        const float ul = pl / a, uh = ph / b, du = ul - uh, inv = 1.0f / a + 1.0f / b;
        c = fminf(-extra, 0.25f * du * du / inv);
        if (c > 0.0f) {
            const float disc = sqrtf(fmaxf(du * du - 2.0f * inv * c, 0.0f));
            const float sg = signbit(du) ? -1.0f : 1.0f;
            kick = -2.0f * c / (du + sg * disc);
            el = ul * kick + 0.5f * kick * kick / a;
            eh = -uh * kick + 0.5f * kick * kick / b;
        }
    }
    const float rest = extra + c;
    out[0] = kick;
    out[1] = 0.5f * dt * pl * d + w * rest + el;
    out[2] = 0.5f * dt * ph * d + (1.0f - w) * rest + eh;
}

// slot index of a local tile position (x, y in -1..T), -1 for the corners
__device__ __forceinline__ int slot_of(int x, int y) {
    if (x >= 0 && x < T && y >= 0 && y < T) return y * T + x;
    if (x == -1 && y >= 0 && y < T) return T * T + y;
    if (x == T && y >= 0 && y < T) return T * T + T + y;
    if (y == -1 && x >= 0 && x < T) return T * T + 2 * T + x;
    if (y == T && x >= 0 && x < T) return T * T + 3 * T + x;
    return -1;
}

__device__ __forceinline__ void slot_pos(int t, int &x, int &y) {
    if (t < T * T) {
        x = t % T;
        y = t / T;
    } else if (t < T * T + T) {
        x = -1;
        y = t - T * T;
    } else if (t < T * T + 2 * T) {
        x = T;
        y = t - T * T - T;
    } else if (t < T * T + 3 * T) {
        x = t - T * T - 2 * T;
        y = -1;
    } else {
        x = t - T * T - 3 * T;
        y = T;
    }
}

// The block's LDS. MULTI: the composition is staged (without it 1/mu is one number and no species is updated, so the
// half step reads none). `f` holds, one after the other: the slots' predicted low faces (five fields, two axes) with
// the half-step states; the high faces' fluxes, kicks and works; the species' low faces and fluxes; the partial sums.
template <int MODE, bool COLD, bool MULTI> struct Lds {
    static constexpr int NF = MODE == HYDRO_MID ? 10 : 13;
    float s[NPRIM], u[NPRIM], v[NPRIM], p[NPRIM], im[MULTI ? NPRIM : 1];
    float ye[COLD ? NPRIM : 1];  // Y_e, with the cold pressure on
    float x[MULTI ? NS : 1][MULTI ? NPRIM : 1];
    alignas(8) float f[NF][NSLOT];
    unsigned present[NSLOT / 64];
};

// What bounds it: vector instructions (2048^2, one species: the half step 98 us and its ALUs always busy, the update
// 383 us and half busy, where the planes' traffic alone takes about 45 and 105 us). So every face's flux, work and
// species fluxes are made once, by the slot on its low side, which holds its own side's state in registers and reads
// only the other side's from LDS; and a species of which neither the tile nor its halo holds any is left out of the
// limiter and of the species' loop (its fluxes are zeros). Before, with each face made on both sides and all species in
// the loop, the two took 313 and 732 us; with all ten species and the cold pressure at 512^2 29 + 74 us now, 49 + 104
// before. 41 KB of LDS and 96 registers: four blocks to a CU (loading the update's inputs ahead of the fluxes spilled
// and cost 20 %). With the sinks two registers spill (12 bytes a lane; 20 steps of 512^2 with four sinks 5.2 ms, 6.1 before);
// with the cold pressure it is 42 KB and 97 registers, three blocks (20 steps 4.6 ms, 5.7 before).
template <int MODE, bool COLD, bool SINKS = false, bool MULTI = true>
__global__ void __launch_bounds__(NSLOT, 5) k_hydro(HydroParams P, HydroState in, HydroState out,
                                                 const double *__restrict__ scal, const float *__restrict__ gx,
                                                 const float *__restrict__ gy, const float *__restrict__ sigma_mid,
                                                 const float *__restrict__ phi_mid, const float *__restrict__ rfx,
                                                 const float *__restrict__ rfy, float *__restrict__ sigma_mid_out,
                                                 float *__restrict__ pushmag, double *__restrict__ escaped,
                                                 HydroPartials part, SinkPlanes SP) {
    __shared__ Lds<MODE, COLD, MULTI> L;
    const int w = P.w, h = P.h;
    const int tile = xcd_tile();
    const int bx = (tile % gridDim.x) * T, by = (tile / gridDim.x) * T;
    const int tid = threadIdx.x;
    const double dt = scal[0];
    const float dtf = (float)dt, half = 0.5f * dtf, hdx = half * P.inv_dx;
    const double dtdx = dt * (double)P.inv_dx;
    const bool grav = gx != nullptr;
    const size_t n = (size_t)w * h;

    // ---- phase 0: primitives of the tile and a two-cell halo, ghosts by the edge rules (hydro.rs:673-710)
    unsigned present = 0u;  // the species that the lanes' cells hold
    for (int t = tid; t < NPRIM; t += NSLOT) {
        const int lx = t % PW, ly = t / PW;
        int gxi = bx + lx - HALO, gyi = by + ly - HALO;
        bool fx = false, fy = false;
        if (gxi < 0 || gxi >= w) {
            fx = true;
            gxi = P.edge == 0 ? (gxi < 0 ? -gxi - 1 : 2 * w - 1 - gxi) : (gxi < 0 ? 0 : w - 1);
            gxi = min(max(gxi, 0), w - 1);
        }
        if (gyi < 0 || gyi >= h) {
            fy = true;
            gyi = P.edge == 0 ? (gyi < 0 ? -gyi - 1 : 2 * h - 1 - gyi) : (gyi < 0 ? 0 : h - 1);
            gyi = min(max(gyi, 0), h - 1);
        }
        const size_t i = (size_t)gyi * w + gxi;
        float xs[NS];
        float im = 0.0f, ye = 0.0f;
        if constexpr (MULTI)
            for (int s = 0; s < NS; s++) {
                xs[s] = in.x[s * n + i];
                im += xs[s] * c_imu[s];
                if (COLD) ye += xs[s] * c_ye[s];
                if (xs[s] != 0.0f) present |= 1u << s;
            }
        if (P.fixed_imu > 0.0f) im = P.fixed_imu;
        const double sig = in.sigma[i];
        Prim q;
        if (sig < (double)P.sigma_vac) {
            q.s = P.sigma_floor;
            q.u = q.v = 0.0f;
            q.p = P.gm1 * P.sigma_floor * eps_floor(P, im) +
                  (COLD ? pi_cold(P.cold, P.sigma_floor, ye, xs[NS - 1]) : 0.0f);
        } else {
            const float s = (float)sig, is = 1.0f / s;
            const float u = in.mx[i] * is, v = in.my[i] * is;
            const float raw = in.e[i] * is - 0.5f * (u * u + v * v) -
                              (COLD ? eps_cold(P.cold, s, ye, xs[NS - 1]) : 0.0f);
            const float eps = fmaxf(raw, eps_floor(P, im));
            q.s = s;
            q.u = u;
            q.v = v;
            q.p = P.gm1 * s * eps + (COLD ? pi_cold(P.cold, s, ye, xs[NS - 1]) : 0.0f);
        }
        if (P.edge == 0) {
            if (fx) q.u = -q.u;
            if (fy) q.v = -q.v;
        } else {
            const bool hx = gxi == w - 1 && bx + lx - HALO >= w, hy = gyi == h - 1 && by + ly - HALO >= h;
            if (fx) q.u = hx ? fmaxf(q.u, 0.0f) : fminf(q.u, 0.0f);
            if (fy) q.v = hy ? fmaxf(q.v, 0.0f) : fminf(q.v, 0.0f);
        }
        L.s[t] = q.s;
        L.u[t] = q.u;
        L.v[t] = q.v;
        L.p[t] = q.p;
        if (COLD) L.ye[t] = ye;
        if constexpr (MULTI) {
            L.im[t] = im;
            for (int s = 0; s < NS; s++) L.x[s][t] = xs[s];
        }
    }
    if constexpr (MULTI) {
        for (int o = 32; o > 0; o >>= 1) present |= __shfl_xor(present, o, 64);
        if ((tid & 63) == 0) L.present[tid >> 6] = present;
    }
    __syncthreads();
    if constexpr (MULTI) {
        present = 0u;
        for (int k = 0; k < NSLOT / 64; k++) present |= L.present[k];
        present = __builtin_amdgcn_readfirstlane(present);
    }
    auto imu_at = [&](int i) { return MULTI ? L.im[i] : P.fixed_imu; };
    auto xn_at = [&](int i) { return COLD ? L.x[NS - 1][i] : 0.0f; };

    // ---- phase 1: every slot's slopes and Hancock predictor (hydro.rs:587-614)
    int sx_, sy_;
    slot_pos(tid, sx_, sy_);
    const int lc = (sy_ + HALO) * PW + sx_ + HALO;
    const int cgx = min(max(bx + sx_, 0), w - 1), cgy = min(max(by + sy_, 0), h - 1);
    float gcx = 0.0f, gcy = 0.0f;
    if (grav) {
        gcx = gx[(size_t)cgy * w + cgx];
        gcy = gy[(size_t)cgy * w + cgx];
    }
    float theta[2];            // the species' shared limiter factor per axis
    float fs_w[4], f0_w[4];    // reconstructed faces' Sigma and mass flux
    float is_e[4];             // the evolved faces' 1 / Sigma (0 when the unevolved face is kept)
    Prim hf[2];                // the high faces' predicted states
    float hf_e[2];
    float m0, m1, m2;          // the half-step state
    {
        const Prim c = {L.s[lc], L.u[lc], L.v[lc], L.p[lc], imu_at(lc), COLD ? L.ye[lc] : 0.0f, xn_at(lc)};
        Prim wf[4];
        for (int ax = 0; ax < 2; ax++) {
            const int off = ax ? PW : 1;
            const int il = lc - off, ir = lc + off;
            const Prim l = {L.s[il], L.u[il], L.v[il], L.p[il], imu_at(il), COLD ? L.ye[il] : 0.0f, xn_at(il)};
            const Prim r = {L.s[ir], L.u[ir], L.v[ir], L.p[ir], imu_at(ir), COLD ? L.ye[ir] : 0.0f, xn_at(ir)};
            float ss = mc(l.s, c.s, r.s), su = mc(l.u, c.u, r.u), sv = mc(l.v, c.v, r.v), sp = mc(l.p, c.p, r.p);
            float th = 1.0f;
            if constexpr (MULTI)
                for (unsigned todo = present; todo; todo &= todo - 1u) {
                    const int s = __builtin_ctz(todo);
                    const float xl = L.x[s][il], xc = L.x[s][lc], xr = L.x[s][ir];
                    const float central = 0.5f * (xr - xl);
                    if (central != 0.0f) th = fminf(th, __fdividef(mc(xl, xc, xr), central));
                }
            theta[ax] = th;
            // 1/mu, Y_e and X_n are linear in the fractions: their faces take the species' shared slope
            const float sim = th * 0.5f * (r.im - l.im);
            const float sye = COLD ? th * 0.5f * (r.ye - l.ye) : 0.0f, sxn = COLD ? th * 0.5f * (r.xn - l.xn) : 0.0f;
            const float hottest = fmaxf(fmaxf(__fdividef(l.p, l.s), __fdividef(c.p, c.s)), __fdividef(r.p, r.s));
            bool hot = false;
            for (int k = 0; k < 2; k++) {
                const float f = k ? 0.5f : -0.5f;
                const float pi = c.p + f * sp, bound = HOT_FACE * hottest * (c.s + f * ss);
                if (!(pi <= bound)) hot = true;
            }
            if (hot) {
                ss = 0.0f;
                sp = 0.0f;
            }
            for (int k = 0; k < 2; k++) {
                const float f = k ? 0.5f : -0.5f;
                Prim &q = wf[2 * ax + k];
                q.s = c.s + f * ss;
                q.u = c.u + f * su;
                q.v = c.v + f * sv;
                q.p = c.p + f * sp;
                q.im = c.im + f * sim;
                q.ye = c.ye + f * sye;
                q.xn = c.xn + f * sxn;
            }
        }
        float ue[4], fl[4][4];
        for (int k = 0; k < 4; k++) {
            ue[k] = cons_e<COLD>(P, wf[k]);
            flux4(wf[k], ue[k], k >> 1, fl[k]);
            fs_w[k] = wf[k].s;
            f0_w[k] = fl[k][0];
        }
        float delta[7];
        for (int c4 = 0; c4 < 4; c4++) delta[c4] = hdx * ((fl[0][c4] - fl[1][c4]) + (fl[2][c4] - fl[3][c4]));
        delta[4] = hdx * ((fl[0][0] * wf[0].im - fl[1][0] * wf[1].im) + (fl[2][0] * wf[2].im - fl[3][0] * wf[3].im));
        delta[5] = COLD ? hdx * ((fl[0][0] * wf[0].ye - fl[1][0] * wf[1].ye) +
                                 (fl[2][0] * wf[2].ye - fl[3][0] * wf[3].ye))
                        : 0.0f;
        delta[6] = COLD ? hdx * ((fl[0][0] * wf[0].xn - fl[1][0] * wf[1].xn) +
                                 (fl[2][0] * wf[2].xn - fl[3][0] * wf[3].xn))
                        : 0.0f;
        m0 = c.s + delta[0], m1 = c.s * c.u + delta[1], m2 = c.s * c.v + delta[2];
        if (grav) {
            m1 += half * c.s * gcx;
            m2 += half * c.s * gcy;
        }
        if constexpr (MODE == HYDRO_UPDATE) {
            L.f[10][tid] = m0;
            L.f[11][tid] = m1;
            L.f[12][tid] = m2;
        }
        for (int k = 0; k < 4; k++) {
            const Prim &q = wf[k];
            float d1 = delta[1], d2 = delta[2], d3 = delta[3];
            if (grav) {
                d1 += half * q.s * gcx;
                d2 += half * q.s * gcy;
                d3 += half * q.s * ((q.u + 0.5f * half * gcx) * gcx + (q.v + 0.5f * half * gcy) * gcy);
            }
            const float s0 = q.s + delta[0], mx = q.s * q.u + d1, my = q.s * q.v + d2, e = ue[k] + d3;
            const float sim = q.s * q.im + delta[4], sye = q.s * q.ye + delta[5], sxn = q.s * q.xn + delta[6];
            Prim o;
            float oe;
            if (prim_of<COLD>(P, s0, mx, my, e, sim, sye, sxn, o)) {
                oe = e;
                is_e[k] = 1.0f / s0;
            } else {
                o = q;
                oe = ue[k];
                is_e[k] = 0.0f;
            }
            const int ax = k >> 1;
            if (k & 1) {
                hf[ax] = o;
                hf_e[ax] = oe;
            } else {
                L.f[5 * ax][tid] = o.s;
                L.f[5 * ax + 1][tid] = o.u;
                L.f[5 * ax + 2][tid] = o.v;
                L.f[5 * ax + 3][tid] = o.p;
                if constexpr (MODE == HYDRO_UPDATE) L.f[5 * ax + 4][tid] = oe;
            }
        }
    }
    __syncthreads();

    // ---- phase 2: the fluxes through the slots' high faces (hydro.rs:744-778, boundary :569-582): a cell's two, the
    // left ring's x faces and the upper ring's y faces; the others' are not read
    const bool own = tid < T * T;
    const int gxc = bx + sx_, gyc = by + sy_;
    const bool live = own && gxc < w && gyc < h;
    const int up_x = own ? (sx_ + 1 < T ? tid + 1 : T * T + T + sy_) : min(max(sy_, 0), T - 1) * T;  // (x + 1, y)
    const int up_y = own ? (sy_ + 1 < T ? tid + T : T * T + 3 * T + sx_) : min(max(sx_, 0), T - 1);  // (x, y + 1)
    float F[4][4];  // fluxes of faces x-, x+, y-, y+ along +x / +y
    bool upl[2];    // whether the high faces' low side is upwind
    bool wallf[2];  // a wall face (bounce, or leave with inflow): no species flux
    float kick_f[4], work_l[2], work_h[4];  // gravity's source at the faces: kick, and the low and high sides' work
    const int rw = w + 2;
    const float *pr = nullptr, *ps = nullptr;
    float phi_c = 0.0f;
    if constexpr (MODE == HYDRO_UPDATE)
        if (grav) {
            const size_t at = (size_t)(min(gyc, h - 1) + 1) * rw + min(gxc, w - 1) + 1;
            pr = phi_mid + at;
            phi_c = pr[0];
            // phi_mid as the faces' work reads it: the gas's with the sinks' potential
            if constexpr (SINKS) {
                ps = SP.ps + at;
                phi_c += ps[0];
            }
        }
    for (int ax = 0; ax < 2; ax++) {
        const int k = 2 * ax + 1, hs = ax ? up_y : up_x;
        const Prim lp = hf[ax];
        const Prim hp = {L.f[5 * ax][hs], L.f[5 * ax + 1][hs], L.f[5 * ax + 2][hs], L.f[5 * ax + 3][hs], 0.0f};
        const float he = MODE == HYDRO_UPDATE ? L.f[5 * ax + 4][hs] : 0.0f;
        const int at = ax ? gyc : gxc, last = (ax ? h : w) - 1;
        const bool low = at < 0, edge = low || at == last;
        wallf[ax] = edge && P.edge == 0;
        upl[ax] = true;
        if (!wallf[ax]) {
            upl[ax] = hll(P, lp, hf_e[ax], hp, he, ax, F[k]);
            wallf[ax] = edge && (low ? F[k][0] > 0.0f : F[k][0] < 0.0f);
        }
        if (wallf[ax]) {
            for (int c4 = 0; c4 < 4; c4++) F[k][c4] = 0.0f;
            F[k][1 + ax] = low ? hp.p : lp.p; // the own face's pressure
        }
        if constexpr (MODE == HYDRO_UPDATE)
            if (grav) {
                // the world's edge does no work (the cell's own values on both sides)
                const float mh = L.f[10][hs], ph = L.f[11 + ax][hs], ml = m0, pl = ax ? m2 : m1;
                float pn = pr[ax ? rw : 1];
                if constexpr (SINKS) pn += ps[ax ? rw : 1];
                const float d = edge ? 0.0f : (phi_c - pn) * P.inv_dx;
                float o[3];
                face_work(F[k][0], low ? mh : ml, edge && !low ? ml : mh, low ? ph : pl, edge && !low ? pl : ph, d, dtf,
                          o);
                kick_f[k] = o[0];
                work_l[ax] = o[1];
                work_h[k] = o[2];
            }
    }
    __syncthreads();
    for (int ax = 0; ax < 2; ax++) {
        const int k = 2 * ax + 1;
        L.f[6 * ax][tid] = F[k][0];
        if constexpr (MODE == HYDRO_UPDATE) {
            for (int c4 = 1; c4 < 4; c4++) L.f[6 * ax + c4][tid] = F[k][c4];
            if (grav) {
                L.f[6 * ax + 4][tid] = kick_f[k];
                L.f[6 * ax + 5][tid] = work_h[k];
            }
        }
    }
    __syncthreads();
    const int dn_x = own ? (sx_ > 0 ? tid - 1 : T * T + sy_) : 0;          // (x - 1, y)
    const int dn_y = own ? (sy_ > 0 ? tid - T : T * T + 2 * T + sx_) : 0;  // (x, y - 1)
    for (int ax = 0; ax < 2; ax++) {
        const int k = 2 * ax, ls = ax ? dn_y : dn_x;
        F[k][0] = L.f[6 * ax][ls];
        if constexpr (MODE == HYDRO_UPDATE) {
            for (int c4 = 1; c4 < 4; c4++) F[k][c4] = L.f[6 * ax + c4][ls];
            if (grav) {
                kick_f[k] = L.f[6 * ax + 4][ls];
                work_h[k] = L.f[6 * ax + 5][ls];
            }
        }
    }
    const size_t ci = (size_t)min(gyc, h - 1) * w + min(gxc, w - 1);
    const double sig0 = live ? in.sigma[ci] : 0.0;
    bool empty = false;
    if (live) {
        auto vac = [&](int x, int y) { return in.sigma[(size_t)y * w + x] < (double)P.sigma_vac; };
        empty = vac(gxc, gyc) && (gxc == 0 || vac(gxc - 1, gyc)) && (gxc + 1 == w || vac(gxc + 1, gyc)) &&
                (gyc == 0 || vac(gxc, gyc - 1)) && (gyc + 1 == h || vac(gxc, gyc + 1));
    }
    const bool vacuum = sig0 < (double)P.sigma_vac;
    const double start = vacuum ? (double)P.sigma_floor : sig0;
    const double divm = ((double)F[1][0] - (double)F[0][0]) + ((double)F[3][0] - (double)F[2][0]);

    if (MODE == HYDRO_MID) {
        if (live) {
            double s = empty ? 0.0 : 0.5 * (sig0 + (start - dtdx * divm));
            sigma_mid_out[ci] = s >= (double)P.sigma_vac ? (float)s : 0.0f;
        }
        return;
    } else {

    // ---- phase 3: the update (hydro.rs:864-984)
    double kick_net[2] = {0.0, 0.0}, push_net[3] = {0.0, 0.0, 0.0};
    unsigned long long dkey = 0ull;
    double u0 = start;
    float u1 = 0.f, u2 = 0.f, u3 = 0.f;
    if (live && !empty) {
        if (vacuum) {
            const Prim fq = {L.s[lc], L.u[lc], L.v[lc], L.p[lc], L.im[lc], COLD ? L.ye[lc] : 0.0f, xn_at(lc)};
            u1 = 0.0f;
            u2 = 0.0f;
            u3 = cons_e<COLD>(P, fq);
        } else {
            u1 = in.mx[ci];
            u2 = in.my[ci];
            u3 = in.e[ci];
        }
        u0 -= dtdx * divm;
        const float dtdxf = (float)dtdx;
        u1 -= dtdxf * ((F[1][1] - F[0][1]) + (F[3][1] - F[2][1]));
        u2 -= dtdxf * ((F[1][2] - F[0][2]) + (F[3][2] - F[2][2]));
        u3 -= dtdxf * ((F[1][3] - F[0][3]) + (F[3][3] - F[2][3]));
        if (grav) {
            const float src = sigma_mid[ci];
            const float gmx = -(pr[1] - pr[-1]) * 0.5f * P.inv_dx, gmy = -(pr[rw] - pr[-rw]) * 0.5f * P.inv_dx;
            float kick[2] = {dtf * src * gmx, dtf * src * gmy};
            // the net kick taken back is the gas's own field's; the sinks' pull is the sinks' to book
            kick_net[0] = (double)kick[0];
            kick_net[1] = (double)kick[1];
            if constexpr (SINKS) {
                kick[0] += dtf * src * SP.gsx[ci];
                kick[1] += dtf * src * SP.gsy[ci];
            }
            if (src > 0.0f) dkey = ((unsigned long long)__float_as_uint(src) << 32) | (0xffffffffu - (unsigned)ci);
            kick[0] += kick_f[1] - kick_f[0];
            kick[1] += kick_f[3] - kick_f[2];
            u1 += kick[0];
            u2 += kick[1];
            u3 += work_l[0] + work_h[0] + work_l[1] + work_h[2];
        }
        if (rfx) {
            // the radiation force from the previous step's flux, capped by the heat above the floor
            float ax = 0.0f, ay = 0.0f;
            if (!vacuum) {
                float im = L.im[lc];
                float kap = P.kappa0 * (1.0f + L.x[0][lc]);
                if (P.opacity == 1 || P.kappa_dust != 0.0f) {
                    const float s = (float)sig0, mx = in.mx[ci], my = in.my[ci];
                    const float raw = in.e[ci] / s - 0.5f * (mx * mx + my * my) / (s * s) -
                                      (COLD ? eps_cold(P.cold, s, L.ye[lc], L.x[NS - 1][lc]) : 0.0f);
                    const float t = P.gm1 * fmaxf(raw, eps_floor(P, im)) / im;
                    if (P.opacity == 1) {
                        kap = P.kappa0 * s * powf(t, -3.5f);
                    } else if (t < P.t_dust) {
                        const float zm = 1.0f - L.x[0][lc] - L.x[1][lc] - L.x[9][lc];
                        kap += P.kappa_dust * zm;
                    }
                }
                const float ks = kap * (float)sig0 / P.c_sb;
                ax = ks * rfx[ci];
                ay = ks * rfy[ci];
            }
            const float d0 = dtf * ax, d1 = dtf * ay, d2 = d0 * d0 + d1 * d1;
            float share = 1.0f;
            if (d2 != 0.0f) {
                const float s = (float)u0;
                // the cell's composition before the update, as for 1/mu
                const float raw = u3 / s - 0.5f * (u1 * u1 + u2 * u2) / (s * s) -
                                  (COLD ? eps_cold(P.cold, s, L.ye[lc], L.x[NS - 1][lc]) : 0.0f);
                const float a = s * (raw - eps_floor(P, L.im[lc]));
                if (!(a > 0.0f)) {
                    share = 0.0f;
                } else {
                    const float q = u1 * d0 + u2 * d1;
                    const float disc = sqrtf(q * q + 2.0f * s * a * d2);
                    share = fminf(q >= 0.0f ? 2.0f * s * a / (q + disc) : (disc - q) / d2, 1.0f);
                }
            }
            const float p0 = share * d0, p1 = share * d1;
            u1 += p0;
            u2 += p1;
            const float pm = sqrtf(p0 * p0 + p1 * p1);
            pushmag[ci] = pm;
            push_net[0] = p0;
            push_net[1] = p1;
            push_net[2] = pm;
        }
        // escaped through the world's edge (hydro.rs:954-976): dt/dx f, signed, per boundary-face slot
        {
            const int nf = 2 * (w + h);
            const int slots[4] = {gyc, h + gyc, 2 * h + gxc, 2 * h + w + gxc};
            const bool edges[4] = {gxc == 0, gxc + 1 == w, gyc == 0, gyc + 1 == h};
            for (int k = 0; k < 4; k++)
                if (edges[k]) {
                    const double sg = (k & 1) ? 1.0 : -1.0;
                    for (int c4 = 0; c4 < 4; c4++) escaped[(size_t)c4 * nf + slots[k]] += sg * dtdx * F[k][c4];
                    escaped[(size_t)3 * nf + slots[k]] += sg * dtdx * (double)F[k][0] * (double)phi_c;
                }
        }
    }
    if (live) {
        if (empty) {
            out.sigma[ci] = sig0;
            out.mx[ci] = in.mx[ci];
            out.my[ci] = in.my[ci];
            out.e[ci] = in.e[ci];
        } else {
            out.sigma[ci] = u0;
            out.mx[ci] = u1;
            out.my[ci] = u2;
            out.e[ci] = u3;
        }
    }

    const double inv_u0 = u0 != 0.0 ? 1.0 / u0 : 0.0;
    // ---- phase 4: the species that are here, one at a time (flux = mass flux x the upwind face's fraction): fields 0
    // and 1 of L.f hold its low faces, 2 and 3 its high faces' fluxes
    const int nf = 2 * (w + h);
    const int slots[4] = {gyc, h + gyc, 2 * h + gxc, 2 * h + w + gxc};
    const bool edges[4] = {gxc == 0, gxc + 1 == w, gyc == 0, gyc + 1 == h};
    __syncthreads(); // the fluxes' fields are reused
    for (unsigned todo = present; todo; todo &= todo - 1u) {
        const int s = __builtin_ctz(todo);
        const float *xp = L.x[s];
        const float xc = xp[lc];  // the cell's own fraction, staged in phase 0
        const int offs[2] = {1, PW};
        float xf[4], f[2];
        for (int ax = 0; ax < 2; ax++) {
            const float central = 0.5f * (xp[lc + offs[ax]] - xp[lc - offs[ax]]);
            xf[2 * ax] = xc - 0.5f * theta[ax] * central;
            xf[2 * ax + 1] = xc + 0.5f * theta[ax] * central;
        }
        const float ds = hdx * ((f0_w[0] * xf[0] - f0_w[1] * xf[1]) + (f0_w[2] * xf[2] - f0_w[3] * xf[3]));
        for (int k = 0; k < 4; k++) {
            const float v = is_e[k] != 0.0f ? (fs_w[k] * xf[k] + ds) * is_e[k] : xf[k];
            if (k & 1)
                f[k >> 1] = v;
            else
                L.f[k >> 1][tid] = v;
        }
        __syncthreads();
        for (int ax = 0; ax < 2; ax++) {
            const float hx = L.f[ax][ax ? up_y : up_x];
            f[ax] = wallf[ax] ? 0.0f : F[2 * ax + 1][0] * (upl[ax] ? f[ax] : hx);
            L.f[2 + ax][tid] = f[ax];
        }
        __syncthreads();
        if (live) {
            const float fsx[4] = {L.f[2][dn_x], f[0], L.f[3][dn_y], f[1]};
            const double um = start * (double)xc - dtdx * (((double)fsx[1] - fsx[0]) + ((double)fsx[3] - fsx[2]));
            out.x[(size_t)s * n + ci] = empty ? xc : (float)(um * inv_u0);
            if (!empty)
                for (int k = 0; k < 4; k++)
                    if (edges[k])
                        escaped[(size_t)(4 + s) * nf + slots[k]] += ((k & 1) ? 1.0 : -1.0) * dtdx * fsx[k];
        }
    }
    // the species that are not: no fluxes, unless the gas's are not numbers (those spread to every species)
    if (live) {
        const float none = empty ? 0.0f : (float)(0.0 * (start - dtdx * divm) * inv_u0);
        for (unsigned todo = ~present & ((1u << NS) - 1u); todo; todo &= todo - 1u) {
            const int s = __builtin_ctz(todo);
            out.x[(size_t)s * n + ci] = none;
            if (!empty)
                for (int k = 0; k < 4; k++)
                    if (edges[k] && !isfinite(F[k][0])) escaped[(size_t)(4 + s) * nf + slots[k]] += 0.0 * F[k][0];
        }
    }

    // ---- block partials of gravity's net kick, the densest free cell and the radiation force's net push
    if (grav || rfx) {
        const int lane = tid & 63, wid = tid >> 6;
        double v[5] = {kick_net[0], kick_net[1], push_net[0], push_net[1], push_net[2]};
        for (int k = 0; k < 5; k++)
            if (k < 2 ? grav : rfx != nullptr) v[k] = wave_sum(v[k]);
        const unsigned long long kk = wave_most(dkey);
        double(*red)[5] = (double(*)[5])L.f[0];
        unsigned long long *redk = (unsigned long long *)L.f[1];
        __syncthreads();
        if (lane == 0) {
            for (int k = 0; k < 5; k++) red[wid][k] = v[k];
            redk[wid] = kk;
        }
        __syncthreads();
        if (tid == 0) {
            double acc[5] = {0, 0, 0, 0, 0};
            unsigned long long best = 0ull;
            for (int wv = 0; wv < NSLOT / 64; wv++) {
                for (int k = 0; k < 5; k++) acc[k] += red[wv][k];
                best = redk[wv] > best ? redk[wv] : best;
            }
            const int b = tile;  // partials in tile order
            for (int k = 0; k < 5; k++) part.sums[(size_t)b * 5 + k] = acc[k];
            part.keys[b] = best;
        }
    }
    }
}

// The take-backs (hydro.rs:986-1001): the radiation force's net push from every pushed cell in proportion to its
// push, gravity's net kick from the densest free cell. Up to TAKE_ROWS blocks reduce the tiles' partials, each to one
// row (five sums and the key), in a fixed order (2048^2's 16384 tiles: 4.6 us, by one block alone 31); every
// block of the take-back adds the rows up itself. Without radiation one cell is changed and one block is launched.
__global__ void __launch_bounds__(256) k_hydro_reduce(HydroPartials part, int nblocks, double *__restrict__ rows) {
    __shared__ double sh[4][5];
    __shared__ unsigned long long shk[4];
    double acc[5] = {0, 0, 0, 0, 0};
    unsigned long long best = 0ull;
    for (int b = blockIdx.x * 256 + threadIdx.x; b < nblocks; b += gridDim.x * 256) {
        for (int k = 0; k < 5; k++) acc[k] += part.sums[(size_t)b * 5 + k];
        best = part.keys[b] > best ? part.keys[b] : best;
    }
    for (int k = 0; k < 5; k++) acc[k] = wave_sum(acc[k]);
    best = wave_most(best);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) {
        for (int k = 0; k < 5; k++) sh[wid][k] = acc[k];
        shk[wid] = best;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double *row = rows + (size_t)blockIdx.x * 6;
        for (int k = 0; k < 5; k++) row[k] = sh[0][k] + sh[1][k] + sh[2][k] + sh[3][k];
        for (int wv = 1; wv < 4; wv++) best = shk[wv] > best ? shk[wv] : best;
        row[5] = __longlong_as_double((long long)best);
    }
}

__global__ void __launch_bounds__(256) k_hydro_takeback(HydroState st, const float *__restrict__ pushmag,
                                                        const double *__restrict__ rows, int nrows, int n,
                                                        int radiation) {
    __shared__ double tb[5];
    __shared__ unsigned long long key;
    if (threadIdx.x < 64) {
        const double *row = rows + (size_t)threadIdx.x * 6;
        const bool has = (int)threadIdx.x < nrows;
        for (int k = 0; k < 5; k++) {
            const double v = wave_sum(has ? row[k] : 0.0);
            if (threadIdx.x == 0) tb[k] = v;
        }
        const unsigned long long best = wave_most(has ? (unsigned long long)__double_as_longlong(row[5]) : 0ull);
        if (threadIdx.x == 0) key = best;
    }
    __syncthreads();
    const int densest = key ? (int)(0xffffffffu - (unsigned)(key & 0xffffffffu)) : -1;
    int i = blockIdx.x * 256 + threadIdx.x;
    if (!radiation) {
        i = threadIdx.x == 0 ? densest : -1;
        if (i < 0) return;
    }
    if (i >= n) return;
    const float m = radiation && tb[4] > 0.0 ? pushmag[i] : 0.0f;
    if (m == 0.0f && i != densest) return;
    float mx = st.mx[i], my = st.my[i];
    if (m != 0.0f) {
        mx -= (float)((double)m * tb[2] / tb[4]);
        my -= (float)((double)m * tb[3] / tb[4]);
    }
    if (i == densest) {
        mx -= (float)tb[0];
        my -= (float)tb[1];
    }
    st.mx[i] = mx;
    st.my[i] = my;
}

// ------------------------------------------------------------------------------------------------------------ host

int hydro_launch(int mode, const HydroParams &P, const HydroState &in, const HydroState &out, const double *scal,
                 const float *gx, const float *gy, const float *sigma_mid, const float *phi_mid, const float *rfx,
                 const float *rfy, float *sigma_mid_out, float *pushmag, double *escaped, const HydroPartials &part,
                 hipStream_t s, const SinkPlanes *sinks) {
    dim3 grid((P.w + T - 1) / T, (P.h + T - 1) / T);
    const SinkPlanes sp = sinks ? *sinks : SinkPlanes{nullptr, nullptr, nullptr};
    const bool with_sinks = mode == HYDRO_UPDATE && sp.ps && phi_mid;
    // the cold pressure's variant only where a pair is on, the sinks' only with sinks: the plain gas keeps the kernel
    // without them
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(NSLOT), 0, s, P, in, out, scal, gx, gy, sigma_mid, phi_mid, rfx, rfy,
                           sigma_mid_out, pushmag, escaped, part, sp);
    };
    if (mode == HYDRO_MID)
        // one 1/mu and no cold pressure: the half step needs no composition
        P.cold.on            ? go(k_hydro<HYDRO_MID, true>)
        : P.fixed_imu > 0.0f ? go(k_hydro<HYDRO_MID, false, false, false>)
                             : go(k_hydro<HYDRO_MID, false>);
    else if (with_sinks)
        P.cold.on ? go(k_hydro<HYDRO_UPDATE, true, true>) : go(k_hydro<HYDRO_UPDATE, false, true>);
    else
        P.cold.on ? go(k_hydro<HYDRO_UPDATE, true>) : go(k_hydro<HYDRO_UPDATE, false>);
    SR_HIP(hipGetLastError());
    return SR_OK;
}

int hydro_takeback(const HydroParams &P, const HydroState &st, const float *pushmag, const HydroPartials &part,
                   double *rows, bool radiation, hipStream_t s) {
    const int nb = hydro_blocks(P.w, P.h), nrows = std::min(TAKE_ROWS, (nb + 255) / 256);
    hipLaunchKernelGGL(k_hydro_reduce, dim3(nrows), dim3(256), 0, s, part, nb, rows);
    const int n = P.w * P.h;
    hipLaunchKernelGGL(k_hydro_takeback, dim3(radiation ? (n + 255) / 256 : 1), dim3(256), 0, s, st, pushmag, rows,
                       nrows, n, radiation ? 1 : 0);
    SR_HIP(hipGetLastError());
    return SR_OK;
}

int hydro_blocks(int w, int h) { return ((w + T - 1) / T) * ((h + T - 1) / T); }

} // namespace sr
