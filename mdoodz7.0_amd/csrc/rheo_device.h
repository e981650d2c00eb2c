// Device restatement of ViscosityConcise (RheologyDensity.c:385-1080) for
// constant, power-law, diffusion, grain-boundary-sliding and Peierls creep,
// Maxwell elasticity and Drucker-Prager (plast = 1) phases, shared by the
// grid update and the tangent (Newton) coefficients.
#pragma once
#include <cmath>

#include "mdg_internal.h"

namespace rheo {

struct rheo_ctl {
    int    step, elastic, average, nph;
    double dt, R, zeroC, min_eta, max_eta, eta_tol, Tiimin, scale_E, scale_eta, T_peierls, d_min;
};

// One phase as the kernels read it: the caller's record and the factors of
// its laws that no node changes, worked out once per call on the host (the
// kernels took four of their pow per node and phase for them).
struct rheo_phase {
    mdg_phase_prop m;
    double A_pwl, f_pwl, A_lin, f_lin, A_gbs, f_gbs;   // A^(-1/n), f^(-r/n)
    double sin_fric, cos_fric, sin_dil;
    int    k_pwl, k_lin;      // the stress exponent where it is 1, 2 or 3, else 0
    int    p_free, pad;       // no law's prefactor depends on the pressure
};
inline rheo_phase make_phase(const mdg_phase_prop &m) {
    auto k = [](double n) { return n == 1.0 ? 1 : (n == 2.0 ? 2 : (n == 3.0 ? 3 : 0)); };
    rheo_phase r{};
    r.m = m;
    r.A_pwl = std::pow(m.A_pwl, -1.0 / m.n_pwl);
    r.f_pwl = std::pow(m.f_pwl, -m.r_pwl / m.n_pwl);
    r.A_lin = std::pow(m.A_lin, -1.0 / m.n_lin);
    r.f_lin = std::pow(m.f_lin, -m.r_lin / m.n_lin);
    r.A_gbs = std::pow(m.A_gbs, -1.0 / m.n_gbs);
    r.f_gbs = std::pow(m.f_gbs, -m.r_gbs / m.n_gbs);
    r.sin_fric = std::sin(m.fric);
    r.cos_fric = std::cos(m.fric);
    r.sin_dil = std::sin(m.dil);
    r.k_pwl = k(m.n_pwl);
    r.k_lin = k(m.n_lin);
    r.p_free = (!m.pwlv || m.V_pwl == 0.0) && (!m.linv || m.V_lin == 0.0) && (!m.gbsv || m.V_gbs == 0.0);
    return r;
}

// Control flow in the evaluation is the wave's: a branch or loop is entered by
// all lanes when one of them needs it, and the lanes that do not keep their
// values through selects (`on`: the node has the phase; `run`: its iteration
// goes on).  A branch per lane is not safe here.  hipcc 7.2 keeps a test that
// is the same for all lanes (whether the phase has a law) as a mask of the
// lanes active where it is first compared.  With a break per lane in local_ve
// that was inside the loop, the tangent's evaluations at perturbed states read
// the mask again, and where the base state's longest lanes had finished there
// the others took a law that the phase does not have (a viscosity of zero).
// Made by all lanes, a compare leaves no partial mask.

// The library's pow as a call: with its dozen copies inlined k_tangent_grid<true>
// has 11500 instructions, past the 64 KB instruction cache, and 118 spilled
// scalars; as calls 4500 and 60.
__device__ __noinline__ double pow_call(double x, double y) { return pow(x, y); }
// x^n with k the small whole value of n, or 0: products in place of the
// library's pow (about 20 instructions instead of 200, within 1.5 ulp).
__device__ __forceinline__ double pow_k(double x, double n, int k) {
    if (k == 0) return pow_call(x, n);
    double p = x;
    if (k > 1) p *= x;
    if (k > 2) p *= x;
    return p;
}
// x^e where e may be zero (laws without that factor): exactly 1, as pow gives
__device__ __forceinline__ double pow_or_1(double x, double e) { return e == 0.0 ? 1.0 : pow_call(x, e); }
// exp(e) where e is zero (no melt): exactly 1, as exp gives
__device__ __forceinline__ double exp_or_1(double e) { return __any(e != 0.0) ? exp(e) : 1.0; }

// The creep laws active at one (node, phase) and their coefficients, which
// depend on temperature, pressure, grain size and melt but not on the strain
// rate: strain rate C T^n of each viscous law at deviatoric stress invariant T.
struct creep_laws {
    bool   elastic, constant, dislocation, peierls, diffusion, gbs;
    int    k_pwl, k_lin;
    double eta_el, eta_cst, C_pwl, n_pwl, C_exp, nST, C_lin, n_lin, dm_lin;
    double B_pwl, B_lin, B_gbs, B_exp;
};

// LocalIterationViscoElastic (RheologyDensity.c:152-197): Newton iterations on
// eta_ve so that E = el*T/(2 eta_el) + sum of the viscous strain rates,
// T = 2 eta_ve E.  The grain-boundary-sliding term of the reference is
// C_gbs T^n_gbs with C_gbs never set (zero), so it is absent here.  Returns
// false when the reference would exit (20 iterations, res > tol).
__device__ __forceinline__ bool local_ve(const creep_laws &L, bool on, double Eii, double &eta, double &Eii_pwl,
                                         double &Eii_exp, double &Eii_lin) {
    constexpr double tol = 1.0e-11, stop = tol / 100;
    double res = 0.0;
    bool run = on;
    for (int it = 0; it < 20; it++) {
        const double Tii = 2.0 * eta * Eii;
        const double e_cst = L.constant ? Tii / 2.0 / L.eta_cst : 0.0;
        const double e_pwl = L.dislocation ? L.C_pwl * pow_k(Tii, L.n_pwl, L.k_pwl) : 0.0;
        const double t_exp = __any(L.peierls) ? L.C_exp * pow_call(Tii, L.nST) : 0.0;
        const double e_exp = L.peierls ? t_exp : 0.0;
        const double e_lin = L.diffusion ? L.C_lin * pow_k(Tii, L.n_lin, L.k_lin) * L.dm_lin : 0.0;
        Eii_pwl = run ? e_pwl : Eii_pwl;
        Eii_exp = run ? e_exp : Eii_exp;
        Eii_lin = run ? e_lin : Eii_lin;
        const double r = Eii - (L.elastic ? 1.0 : 0.0) * Tii / (2.0 * L.eta_el) - (e_pwl + e_exp + e_lin + e_cst);
        res = fabs(r / Eii);
        run = run && !(res < stop);
        if (!__any(run)) break;
        double dfdeta = 0.0;
        if (L.elastic) dfdeta += -Eii / L.eta_el;
        const double d_exp = __any(L.peierls) ? dfdeta + -e_exp * L.nST / eta : 0.0;
        dfdeta = L.peierls ? d_exp : dfdeta;
        if (L.diffusion) dfdeta += -e_lin * L.n_lin / eta;
        if (L.dislocation) dfdeta += -e_pwl * L.n_pwl / eta;
        if (L.constant) dfdeta += -Eii / L.eta_cst;
        const double next = eta - r / dfdeta;
        eta = run ? next : eta;
    }
    return !run || !(res > tol);
}

// Failure codes of viscosity_concise, or-ed into the caller's flag.
constexpr int FAIL_LOCAL_ITER = 1;     // local iterations failed (reference exits, :174-177)
constexpr int FAIL_GRAIN_SIZE = 2;     // d < d_min with m_lin > 0 (reference exits, :506-509)

// The strain-rate independent part of ViscosityConcise (RheologyDensity.c:
// 457-523) for one (node, phase).  EXT = false compiles the diffusion,
// GBS and Peierls laws and the power law's d, f, phi factors out (the
// caller launches it when no phase uses them: the factors are then exactly
// 1 and the laws absent, so the results are the same bits), which keeps
// the register count, and the occupancy, of the constant + power-law case.
template <bool EXT>
__device__ __forceinline__ creep_laws laws_at(const rheo_phase &ph, const rheo_ctl &md, bool on, double G, double T, double P,
                                              double d, double phi, double pref_mult, int &fail) {
    const mdg_phase_prop &m = ph.m;
    creep_laws L = {};
    const double dt = (md.step == 0) ? 1e100 : md.dt;
    L.elastic = md.elastic != 0 && md.step != 0;                       // :483
    L.constant = m.cstv != 0;
    L.dislocation = m.pwlv != 0;
    L.peierls = EXT && m.expv != 0 && T < md.T_peierls;               // :474, before the T floor
    L.diffusion = EXT && m.linv != 0;
    L.gbs = EXT && m.gbsv != 0;
    L.eta_el = (L.elastic ? G : 1e1) * dt;                            // :493
    L.eta_cst = L.constant ? m.eta0 : 0.0;
    L.k_pwl = ph.k_pwl;
    L.k_lin = ph.k_lin;
    L.n_pwl = m.n_pwl;
    L.n_lin = m.n_lin;
    T = T < md.zeroC ? md.zeroC : T;
    if (L.dislocation) {                                               // :501-504
        L.B_pwl = m.pref_pwl * pref_mult * m.F_pwl * ph.A_pwl * exp((m.Q_pwl + P * m.V_pwl) / md.R / m.n_pwl / T);
        if (EXT)
            L.B_pwl = L.B_pwl * pow_or_1(d, m.m_pwl / m.n_pwl) * ph.f_pwl * exp_or_1(-m.a_pwl * phi / m.n_pwl);
        L.C_pwl = L.k_pwl ? 1.0 / pow_k(2.0 * L.B_pwl, m.n_pwl, L.k_pwl) : pow_call(2.0 * L.B_pwl, -m.n_pwl);
    }
    L.dm_lin = 1.0;
    if (L.diffusion) {                                                 // :505-512, d enters below
        fail |= (on && m.m_lin > 0.0 && d < md.d_min) ? FAIL_GRAIN_SIZE : 0;
        L.B_lin = m.F_lin * ph.A_lin * exp((m.Q_lin + P * m.V_lin) / md.R / m.n_lin / T) * ph.f_lin *
                  exp_or_1(-m.a_lin * phi / m.n_lin);
        L.C_lin = L.k_lin ? 1.0 / pow_k(2.0 * L.B_lin, m.n_lin, L.k_lin) : pow_call(2.0 * L.B_lin, -m.n_lin);
        L.dm_lin = pow_or_1(d, -m.m_lin);
    }
    if (L.gbs)                                                         // :513-515
        L.B_gbs = m.F_gbs * ph.A_gbs * exp((m.Q_gbs + P * m.V_gbs) / md.R / m.n_gbs / T) *
                  pow_or_1(d, m.m_gbs / m.n_gbs) * ph.f_gbs * exp_or_1(-m.a_gbs * phi / m.n_gbs);
    L.nST = m.n_exp;
    if (__any(L.peierls)) {                                            // :516-523
        const double g = m.G_exp;
        const double ST = m.Q_exp / md.R / T * 2.0 * g * (1 - g);
        const double Arr = exp(-m.Q_exp / md.R / T * ((1.0 - g) * (1.0 - g)));
        L.nST = ST + m.n_exp;
        const double F_exp = pow_call(pow_call(2.0, 1.0 - ST - m.n_exp) / pow_call(sqrt(3.0), ST + m.n_exp + 1.0), 1.0 / L.nST);
        L.B_exp = F_exp * (pow_call(g * m.S_exp, ST / L.nST) / pow_call(m.E_exp * Arr, 1.0 / L.nST));
        L.C_exp = pow_call(2.0 * L.B_exp, -L.nST);
    }
    return L;
}

// ViscosityConcise (RheologyDensity.c:385-1080) for one (node, phase) with
// the laws of laws_at: returns the dissipative viscosity; etaVE, Pcorr and
// Eii_pl by reference.  fr holds sin and cos of the friction angle and sin of
// the dilation angle.
struct friction {
    double sin_fric, cos_fric, sin_dil;
};
template <bool EXT>
__device__ __forceinline__ double viscosity_concise(const rheo_phase &ph, const creep_laws &L, const rheo_ctl &md, bool on,
                                                    double P, double d, double Exx, double Ezz, double Exz, const friction &fr,
                                                    double C, double &etaVE, double &Pcorr, double &Eii_pl,
                                                    int &fail) {
    const mdg_phase_prop &m = ph.m;
    const double dt = (md.step == 0) ? 1e100 : md.dt;
    const bool plastic = m.plast == 1 && md.step != 0;                // :483
    const double K = L.elastic ? 1.0 / m.beta : 1e10;                  // :493
    const double sin_fric = fr.sin_fric, sin_dil = L.elastic ? fr.sin_dil : 0.0;
    const double Eyy = -(Exx + Ezz);
    double Eii = sqrt(0.5 * (Exx * Exx + Ezz * Ezz + Eyy * Eyy) + Exz * Exz);   // :457-459
    Eii = Eii * md.scale_E < 1e-30 ? 1e-30 / md.scale_E : Eii;
    Pcorr = P;
    double Tyield = 0.0;
    if (plastic) {                                                     // :530-539
        Tyield = C * fr.cos_fric + P * sin_fric;
        Tyield = m.Slim < Tyield ? m.Slim : Tyield;
    }
    double eta_up = 1.0e100 / md.scale_eta;                        // :585-592
    if (L.constant) eta_up = fmin(eta_up, L.eta_cst);
    if (L.dislocation) eta_up = fmin(eta_up, L.B_pwl * pow_call(Eii, 1.0 / m.n_pwl - 1.0));
    if (L.elastic) eta_up = fmin(eta_up, L.eta_el);
    if (__any(L.peierls)) {
        const double up = fmin(eta_up, L.B_exp * pow_call(Eii, 1.0 / L.nST - 1.0));
        eta_up = L.peierls ? up : eta_up;
    }
    if (L.diffusion)
        eta_up = fmin(eta_up, L.B_lin * pow_or_1(Eii, 1.0 / m.n_lin - 1.0) * pow_or_1(d, m.m_lin / m.n_lin));
    if (L.gbs) eta_up = fmin(eta_up, L.B_gbs * pow_call(Eii, 1.0 / m.n_gbs - 1.0));
    double eta_ve = eta_up;
    double Eii_pwl = 0.0, Eii_exp = 0.0, Eii_lin = 0.0;
    fail |= local_ve(L, on, Eii, eta_ve, Eii_pwl, Eii_exp, Eii_lin) ? 0 : FAIL_LOCAL_ITER;
    double Tii = 2.0 * eta_ve * Eii;
    bool is_pl = false;
    double eta_vep = eta_ve, gdot = 0.0;
    if (plastic) {                                                     // :655-707
        const double F0 = Tii - Tyield, tol = md.eta_tol;
        is_pl = on && F0 > 1e-17;
        if (__any(is_pl)) {
            const double Kdt_ss = K * dt * sin_fric * sin_dil;
            double g = F0 / (eta_ve + m.eta_vp * pow_or_1(Eii, 1.0 / m.n_vp - 1) + Kdt_ss);
            double Pc = P, Tiic = Tii;
            bool run = is_pl;
            for (int it = 0; it < 20; it++) {
                const double eta_vp = m.eta_vp * pow_or_1(fabs(g), 1.0 / m.n_vp - 1.0);
                Pc = run ? P + K * dt * (g * sin_dil) : Pc;
                Tyield = run ? Tyield + g * eta_vp : Tyield;    // accumulates, as in the reference
                Tiic = run ? Tii - eta_ve * g : Tiic;
                const double F_trial = Tiic - Tyield, res = fabs(F_trial);
                run = run && !(res < tol || res / F0 < tol);
                if (!__any(run)) break;
                const double next = g - F_trial / (-eta_ve - eta_vp / m.n_vp - Kdt_ss);
                g = run ? next : g;
            }
            const bool neg = Tiic < 0.0;                               // :694-701
            g = neg ? (Tii - md.Tiimin) / eta_ve : g;
            Tiic = neg ? md.Tiimin : Tiic;
            Pc = neg ? P : Pc;
            gdot = is_pl ? g : 0.0;
            Pcorr = is_pl ? Pc : P;
            eta_vep = Tiic / (2.0 * Eii);
            Tii = is_pl ? Tiic : Tii;
        }
    }
    etaVE = is_pl ? eta_vep : eta_ve;                                  // :962-970
    Eii_pl = is_pl ? gdot / 2.0 : 0.0;
    // dissipative viscosity (:987-1032): each law's viscosity at its own
    // strain-rate share; diffusion creep at the phase's reference grain size
    double inv = 0.0;
    if (__any(L.peierls)) {
        const double i_exp = 1.0 / (L.B_exp * pow_call(Eii_exp, 1.0 / L.nST - 1.0));
        inv = L.peierls ? i_exp : inv;
    }
    if (L.dislocation) inv += 1.0 / (L.B_pwl * pow_call(Eii_pwl, 1.0 / m.n_pwl - 1.0));
    if (L.diffusion)
        inv += 1.0 / (L.B_lin * pow_or_1(Eii_lin, 1.0 / m.n_lin - 1.0) * pow_or_1(m.gs_ref, m.m_lin / m.n_lin));
    if (L.constant) inv += 1.0 / L.eta_cst;
    if (__any(is_pl)) {
        const double i_pl = inv + 1.0 / (Tii / gdot);
        inv = is_pl ? i_pl : inv;
    }
    double eta = 1.0 / inv;
    etaVE = fmax(fmin(etaVE, md.max_eta), md.min_eta);                 // :1058-1073
    eta = eta > md.max_eta ? md.max_eta : eta;
    eta = eta < md.min_eta ? md.min_eta : eta;
    return eta;
}

// Friction terms of a node: the phase's own, or those of the node's angles.
__device__ __forceinline__ friction friction_at(const rheo_phase &ph, const mdg_rheo_nodes &f, int i) {
    friction r{ph.sin_fric, ph.cos_fric, ph.sin_dil};
    if (f.fric) {
        r.sin_fric = sin(f.fric[i]);
        r.cos_fric = cos(f.fric[i]);
    }
    if (f.dil) r.sin_dil = sin(f.dil[i]);
    return r;
}

// The phase table of a call on the device (a buffer kept with the context).
struct phase_buf : dbuf<rheo_phase> {
    std::vector<rheo_phase> h;    // lives until the copy has run
};
inline int upload_phases(mdg_ctx *c, const mdg_phase_prop *phases, int nph, phase_buf &buf) {
    buf.h.resize(nph);
    for (int p = 0; p < nph; p++) buf.h[p] = make_phase(phases[p]);
    HIPCHK(c, buf.reserve(nph));
    HIPCHK(c, hipMemcpyAsync(buf.p, buf.h.data(), nph * sizeof(rheo_phase), hipMemcpyHostToDevice, c->stream));
    return MDG_OK;
}

// Whether any phase needs the EXT instantiation of viscosity_concise.
inline bool needs_ext(const mdg_phase_prop *ph, int nph) {
    for (int p = 0; p < nph; p++)
        if (ph[p].linv || ph[p].gbsv || ph[p].expv || ph[p].m_pwl != 0.0 || ph[p].r_pwl != 0.0 ||
            ph[p].a_pwl != 0.0)
            return true;
    return false;
}

// The kernel-side constants of one call.
inline rheo_ctl make_ctl(const mdg_rheo_params *prm, int nph) {
    return {prm->step,     prm->elastic, prm->average, nph,           prm->dt,
            prm->R,        prm->zeroC,   prm->min_eta, prm->max_eta,  prm->eta_tol,
            prm->Tiimin,   prm->scale_E, prm->scale_eta, prm->T_peierls, prm->d_min};
}

// Status of a call from the or-ed failure codes of its nodes.
inline int fail_status(mdg_ctx *c, int fail) {
    if (fail & FAIL_GRAIN_SIZE)
        return mdg_fail(c, MDG_ERR_ARG, "grain size below d_min with grain-size dependent diffusion creep");
    if (fail & FAIL_LOCAL_ITER)
        return mdg_fail(c, MDG_ERR_DIVERGED, "visco-elastic local iterations failed to converge");
    return MDG_OK;
}

}  // namespace rheo
