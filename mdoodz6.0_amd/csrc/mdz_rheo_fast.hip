/*
 * mdz_rheo_fast.hip -- gfx950 grid rheology for the common case: arithmetic
 * phase averaging (eta_average = 0), isotropic, no grain-size evolution, no
 * phase mixing, no reaction softening.  Same local constitutive update as
 * RheologyDensity.c:44-707 (Viscosity) and the same phase accumulation as
 * RheologyDensity.c:961-1415 (NonNewtonianViscosityGrid), organised for the
 * GPU:
 *
 *  - Creep laws in log space.  The node-independent part of each prefactor
 *    is folded once per phase into log B0 (k_phase_constants).  Per node and
 *    phase: one log(Eii); per local iteration one log(Tii) shared by all
 *    mechanisms and one exp per active mechanism.  Viscosity evaluates each
 *    prefactor with pow/exp per factor and each mechanism with its own pow
 *    per iteration; both forms agree to rounding (~1e-15 relative).
 *  - The phase-averaged outputs are streamed to HBM as each phase finishes
 *    (stored for the first active phase, added for the later ones in phase
 *    order: the reference's summation order), so no accumulators stay live
 *    across the local solve.
 *  - Phase constants are read with wave-uniform indices (scalar loads).
 *  - Mixed precision (MDZ_RHEO_MIXED / LEARNED): the visco-elastic Newton
 *    iteration first runs in FP32 (Newton in log eta, hardware log/exp) from
 *    the reference guess (or the network's guess) to |r/Eii| < 1e-5; FP64
 *    Newton steps then finish to the reference tolerance |r/Eii| < 1e-13.  The
 *    tangent, the plastic return and every output stay FP64.
 */
#include "mdz_kernels.h"
#include "mdz_mlp_dev.h"

#define ZEROC 273.15
#define LN2 0.69314718055994530942
#define LN3 1.09861228866810969140

/* -(r / n) ln f, with pow(f, -0) = 1 for every f */
__device__ __forceinline__ double lnpow_neg(double r_over_n, double f) {
    return r_over_n == 0.0 ? 0.0 : -r_over_n * log(f);
}

__global__ void k_phase_constants(const mat_prop *__restrict__ mt, int nph, PhaseK *pk) {
    int p = threadIdx.x;
    if (p >= nph) return;
    PhaseK k;
    k.cst = mt->cstv[p] != 0;
    k.pwl = mt->pwlv[p] != 0;
    k.expv = mt->expv[p] != 0;
    k.lin = mt->linv[p] != 0;
    k.gbs = mt->gbsv[p] != 0;
    k.tensile = mt->is_tensile[p] == 1;
    k.eta_cst = mt->eta0[p];
    double n = mt->npwl[p];
    k.n_pwl = n; k.Ea_pwl = mt->Qpwl[p]; k.Va_pwl = mt->Vpwl[p];
    k.lnB0_pwl = k.pwl ? log(mt->pref_pwl[p] * mt->Fpwl[p] * pow(mt->Apwl[p], -1.0 / n)) : 0.0;
    k.mn_pwl = mt->mpwl[p] / n;
    k.lnfr_pwl = k.pwl ? lnpow_neg(mt->rpwl[p] / n, mt->fpwl[p]) : 0.0;
    k.an_pwl = mt->apwl[p] / n;
    n = mt->nlin[p];
    k.n_lin = n; k.Ea_lin = mt->Qlin[p]; k.Va_lin = mt->Vlin[p]; k.m_lin = mt->mlin[p];
    k.lnB0_lin = k.lin ? log(mt->Flin[p] * pow(mt->Alin[p], -1.0 / n)) : 0.0;
    k.lnfr_lin = k.lin ? lnpow_neg(mt->rlin[p] / n, mt->flin[p]) : 0.0;
    k.an_lin = mt->alin[p] / n;
    n = mt->ngbs[p];
    k.n_gbs = n; k.Ea_gbs = mt->Qgbs[p]; k.Va_gbs = mt->Vgbs[p];
    k.lnB0_gbs = k.gbs ? log(mt->Fgbs[p] * pow(mt->Agbs[p], -1.0 / n)) : 0.0;
    k.mn_gbs = mt->mgbs[p] / n;
    k.lnfr_gbs = k.gbs ? lnpow_neg(mt->rgbs[p] / n, mt->fgbs[p]) : 0.0;
    k.an_gbs = mt->agbs[p] / n;
    k.Ea_exp = mt->Qexp[p]; k.gamma = mt->Gexp[p]; k.n_exp = mt->nexp[p];
    k.ln_gS = k.expv ? log(mt->Gexp[p] * mt->Sexp[p]) : 0.0;
    k.ln_E = k.expv ? log(mt->Eexp[p]) : 0.0;
    k.Slim = mt->Slim[p]; k.eta_vp0 = mt->eta_vp[p]; k.n_vp = mt->n_vp[p];
    k.gs_ref = mt->gs_ref[p];
    k.ln_gs_ref = log(mt->gs_ref[p]);
    k.inv_n_pwl = 1.0 / k.n_pwl;
    k.inv_n_lin = 1.0 / k.n_lin;
    k.inv_n_gbs = 1.0 / k.n_gbs;
    k.inv_eta_cst = 1.0 / k.eta_cst;
    k.inv_n_vp = 1.0 / k.n_vp;
    k.vp_exp = 1.0 / k.n_vp - 1.0;
    /* the diffusion creep's d1^-m / n term of its inverse viscosity */
    k.ginv_lin = k.m_lin != 0.0 ? k.m_lin / k.n_lin * k.ln_gs_ref : 0.0;
    pk[p] = k;
}

/* The rheology outputs are two runs of consecutive fields in the slab
 * (eta_n .. drhodp_n on centroids, VE_s .. OverS_s on vertices), so each
 * output is addressed as run base + position * stride + node. */
template <int FIRST, int LAST, int FAM>
struct FieldRun {
    static constexpr bool same_family() {
        constexpr int fam[] = {
#define MDZ_FFAM(name, fam, role) MDZ_FAM_##fam,
            MDZ_ALL_DOUBLE_FIELDS(MDZ_FFAM)
#undef MDZ_FFAM
        };
        for (int i = FIRST; i <= LAST; i++)
            if (fam[i] != FAM) return false;
        return true;
    }
};
static_assert(FieldRun<FI_eta_n, FI_drhodp_n, MDZ_FAM_C>::same_family(), "centroid rheology outputs must be one run");
static_assert(FieldRun<FI_VE_s, FI_OverS_s, MDZ_FAM_V>::same_family(), "vertex rheology outputs must be one run");

/* Output stream of one node: fr * v stored (first active phase) or added. */
struct Out {
    double *base; /* first field of the run */
    long long stride;
    int c, first_fi;
    double fr;
    bool first;
    __device__ __forceinline__ double *at(int fi) const { return base + (long long)(fi - first_fi) * stride + c; }
    __device__ __forceinline__ void put(int fi, double v) const {
        double x = fr * v;
        double *f = at(fi);
        if (first) *f = x;
        else *f += x;
    }
};

/* Node inputs; the friction and dilatancy angles enter as sines/cosines,
 * evaluated once per node.  (Txx0, Tzz0, Txz0 feed only the visco-elastic
 * rates; the diagnostic outputs read the old stresses again, see DiagSrc.) */
struct NodeIn {
    double G, T, P, d, phi, Exx, Ezz, Exz, Gxx, Gzz, Gxz, Txx0, Tzz0, Txz0, sin_dil, sin_fric, cos_fric, C, beta;
};

/* Effective visco-elastic strain rates for an isotropic node: the inverse
 * anisotropy tensor of RheologyDensity.c:1061-1094 is diag(1/2, 1/2, 1). */
__device__ __forceinline__ void ve_rates_iso(double exx, double ezz, double exz, double sxx0, double szz0, double sxz0,
                                             double etae, NodeIn &in) {
    in.Exx = exx + (0.5 * sxx0) / etae;
    in.Ezz = ezz + (0.5 * szz0) / etae;
    in.Exz = exz + sxz0 / 2.0 / etae;
    double gxz = 2.0 * exz + sxz0 / etae;
    in.Gxx = in.Exx;
    in.Gzz = in.Ezz;
    in.Gxz = gxz * 0.5;
}

/* Local update of one node and one phase (RheologyDensity.c:44-707 with
 * gs = 0, constant_mix = 0); outputs go through o.  CELL selects the
 * centroid output set, otherwise the vertex set.  DIAG: all outputs;
 * otherwise only those the rest of a Newton-iteration unit reads (eta, the
 * tangent, the plastic divergence derivatives, p_corr). */
/* Node-independent constants of the local update, from the scales of the
 * model (computed on the host, read as kernel arguments). */
struct FastConst {
    double T_peierls; /* (1200 + 273.15) K, scaled */
    double T_min;     /* 273.15 K, scaled */
    double eta_start; /* 1e100 Pa s, scaled */
    double P_tens;    /* -25 MPa, scaled */
    double E_floor;   /* 1e-30 s^-1, scaled */
};

/* Local update of one node and one phase (RheologyDensity.c:44-707 with
 * gs = 0, constant_mix = 0); outputs go through o.  CELL selects the
 * centroid output set, otherwise the vertex set.  DIAG: all outputs;
 * otherwise only those the rest of a Newton-iteration unit reads (eta, the
 * tangent, the plastic divergence derivatives, p_corr).  Divisions by
 * quantities used more than once are products with one reciprocal (a
 * rounding-level difference from the reference's expressions). */
/* Inputs that only the diagnostic outputs read (old stresses, P0, X0, the
 * deviatoric strain rates).  They sit in the block's LDS stash from the
 * node's load batch on and are read where those outputs are computed,
 * behind a compiler barrier, instead of staying in registers through the
 * local solve (that is what keeps the all-outputs centroid kernel within
 * its register budget).  Slot k of the lane at s[k * stride]. */
enum { DS_SXX0 = 0, DS_SZZ0, DS_SXZ0, DS_P0, DS_X0, DS_EXX, DS_EZZ, DS_EXZ };
struct DiagSrc {
    const double *s;
    int stride;
    __device__ __forceinline__ double get(int k) const { return s[k * stride]; }
};

/* Outputs accumulated over the phases in registers and stored once: the
 * grain-size sum (the reference's d = 1 / sum fr / d_ref) and X. */
struct NodeAcc {
    double d, x;
};

template <bool CELL, bool DIAG>
__device__ __forceinline__ void local_update(const PhaseK &k, double R, const DevParams &prm, const FastConst &fc,
                                             const NodeIn &in, bool Xout, const Out &o, const DiagSrc &ds,
                                             double guess, double gdot_guess, const BlockHist &hist, NodeAcc &acc) {
    const double dt = prm.dt;
    int elastic = prm.iselastic;
    double G = in.G, T = in.T, P = in.P, C = in.C, K = 1.0 / in.beta;
    const double Exx = in.Exx, Ezz = in.Ezz, Exz = in.Exz;
    double Eyy = -(Exx + Ezz), Gyy = -(in.Gxx + in.Gzz);
    double Eii = sqrt(1.0 / 2.0 * (Exx * Exx + Ezz * Ezz + Eyy * Eyy) + Exz * Exz);
    double Gii = sqrt(1.0 / 2.0 * (in.Gxx * in.Gxx + in.Gzz * in.Gzz + Gyy * Gyy) + in.Gxz * in.Gxz);
    if (Eii * prm.sE < 1e-30) Eii = fc.E_floor;
    if (Gii * prm.sE < 1e-30) Gii = fc.E_floor;
    const double inv_Eii = 1.0 / Eii;
    const double f_ani = Gii * inv_Eii;
    const int peierls = k.expv && T < fc.T_peierls;
    if (prm.step == 0) elastic = 0;
    if (elastic == 0) { G = 1e1; K = 1e1; } /* and dil = 0 (sin_dil set by the caller) */
    if (T < fc.T_min) T = fc.T_min;
    const double inv_RT = 1.0 / (R * T);
    const double lnEii = log(Eii), lnf2 = log(2.0 * f_ani), lnd = log(in.d);

    /* prefactors B and compliances C = (2 f B)^-n, in logs */
    double lnB_pwl = 0, lnC_pwl = 0, lnB_lin = 0, lnC_lin = 0, lnB_gbs = 0, lnC_gbs = 0, lnB_exp = 0, lnC_exp = 0;
    double nST = 0, inv_nST = 0;
    if (k.pwl) {
        lnB_pwl = k.lnB0_pwl + (k.Ea_pwl + P * k.Va_pwl) * inv_RT * k.inv_n_pwl
                + (k.mn_pwl != 0.0 ? k.mn_pwl * lnd : 0.0) + k.lnfr_pwl - k.an_pwl * in.phi;
        lnC_pwl = -k.n_pwl * (lnf2 + lnB_pwl);
    }
    if (k.lin) {
        lnB_lin = k.lnB0_lin + (k.Ea_lin + P * k.Va_lin) * inv_RT * k.inv_n_lin + k.lnfr_lin - k.an_lin * in.phi;
        /* the diffusion rate carries d1^-m with d1 the reference grain size */
        lnC_lin = -k.n_lin * (lnf2 + lnB_lin) - (k.m_lin != 0.0 ? k.m_lin * k.ln_gs_ref : 0.0);
    }
    if (k.gbs) {
        lnB_gbs = k.lnB0_gbs + (k.Ea_gbs + P * k.Va_gbs) * inv_RT * k.inv_n_gbs
                + (k.mn_gbs != 0.0 ? k.mn_gbs * lnd : 0.0) + k.lnfr_gbs - k.an_gbs * in.phi;
        lnC_gbs = -k.n_gbs * (lnf2 + lnB_gbs);
    }
    if (peierls) {
        const double EaRT = k.Ea_exp * inv_RT;
        double ST = EaRT * 2.0 * k.gamma * (1 - k.gamma);
        nST = ST + k.n_exp;
        inv_nST = 1.0 / nST;
        double lnArr = -EaRT * (1.0 - k.gamma) * (1.0 - k.gamma);
        double lnF = ((1.0 - nST) * LN2 - 0.5 * (nST + 1.0) * LN3) * inv_nST;
        lnB_exp = lnF + (ST * inv_nST) * k.ln_gS - (k.ln_E + lnArr) * inv_nST;
        lnC_exp = -nST * (lnf2 + lnB_exp);
    }

    /* Drucker-Prager yield with the von Mises and tension cut-offs */
    double cos_fric = in.cos_fric, sin_fric = in.sin_fric, sin_dil = in.sin_dil;
    double Tyield = C * cos_fric + P * sin_fric;
    if (k.Slim < Tyield) { sin_fric = 0.0; cos_fric = 1.0; sin_dil = 0.0; C = k.Slim; Tyield = k.Slim; }
    int tens = 0;
    {
        double sft = -C * cos_fric / fc.P_tens;
        if (C * cos_fric + P * sft < Tyield && k.tensile) { sin_fric = sft; Tyield = C * cos_fric + P * sft; tens = 1; }
    }

    /* initial guess: the smallest isolated viscosity */
    const double eta_el = G * dt, inv_eel = 1.0 / eta_el;
    double eta_ve = fc.eta_start;
    if (k.cst) eta_ve = fmin(eta_ve, k.eta_cst);
    if (k.pwl) eta_ve = fmin(eta_ve, exp(lnB_pwl + (k.inv_n_pwl - 1.0) * lnEii));
    if (elastic) eta_ve = fmin(eta_ve, eta_el);
    if (peierls) eta_ve = fmin(eta_ve, exp(lnB_exp + (inv_nST - 1.0) * lnEii));
    if (k.lin)
        eta_ve = fmin(eta_ve, exp(lnB_lin + (k.inv_n_lin - 1.0) * lnEii + (k.m_lin != 0.0 ? k.m_lin * k.inv_n_lin * lnd : 0.0)));
    if (k.gbs) eta_ve = fmin(eta_ve, exp(lnB_gbs + (k.inv_n_gbs - 1.0) * lnEii));

    /* FP32 pre-iterations */
    int it32 = 0;
    if (prm.rheo_mode != MDZ_RHEO_FP64) {
        float e = guess > 0.0 ? (float)(guess * eta_ve) : (float)eta_ve;
        const float Ef = (float)Eii, ff = (float)f_ani, ecst = (float)k.eta_cst;
        const float iEf = 1.0f / Ef, heel = (float)(0.5 * inv_eel), iecst = (float)k.inv_eta_cst;
        const float lcp = (float)lnC_pwl, lce = (float)lnC_exp, lcl = (float)lnC_lin, lcg = (float)lnC_gbs;
        const float np_ = (float)k.n_pwl, ne = (float)nST, nl = (float)k.n_lin, ng = (float)k.n_gbs;
        #pragma unroll 1
        for (it32 = 0; it32 < 20; it32++) {
            float Tf = 2.0f * ff * e * Ef;
            float lt = __logf(Tf);
            float Ep = k.pwl ? __expf(lcp + np_ * lt) : 0.0f;
            float Ee = peierls ? __expf(lce + ne * lt) : 0.0f;
            float El = k.lin ? __expf(lcl + nl * lt) : 0.0f;
            float Eg = k.gbs ? __expf(lcg + ng * lt) : 0.0f;
            float Ec = k.cst ? e * Ef * iecst : 0.0f;
            float r = Ef - (elastic ? Tf * heel : 0.0f) - (Ep + Ee + El + Eg + Ec);
            if (fabsf(r * iEf) < MDZ_F32_TOL) break;
            /* e * d r / d e and its derivative in log(eta): each term of
             * the strain-rate sum is proportional to eta^n */
            float dfe = 0.0f, d2 = 0.0f;
            if (elastic) { const float t = Ef * 2.0f * heel * e; dfe -= t; d2 -= t; }
            if (peierls) { dfe -= Ee * ne; d2 -= Ee * ne * ne; }
            if (k.lin) { dfe -= El * nl; d2 -= El * nl * nl; }
            if (k.pwl) { dfe -= Ep * np_; d2 -= Ep * np_ * np_; }
            if (k.gbs) { dfe -= Eg * ng; d2 -= Eg * ng * ng; }
            if (k.cst) { const float t = Ef * iecst * e; dfe -= t; d2 -= t; }
            (void)ecst;
            /* step in log(eta): the strain-rate sum is convex and increasing
             * in log(eta), so the iteration converges from either side
             * without leaving eta > 0; Halley's step (cubic) near the root,
             * Newton's further away */
            const float st = fabsf(r * iEf) < 0.5f ? -2.0f * r * dfe / (2.0f * dfe * dfe - r * d2) : -r / dfe;
            const float ds = fminf(fmaxf(st, -10.0f), 10.0f);
            e *= __expf(ds);
        }
        if (e > 0.0f && e < 3.0e38f) eta_ve = (double)e;
    } else if (guess > 0.0) {
        eta_ve *= guess;
    }

    /* FP64 visco-elastic Newton iteration (RheologyDensity.c:330-370) */
    const double half_inv_eel = 0.5 * inv_eel;
    double Ep = 0, Ee = 0, El = 0, Eg = 0, Ec = 0, lT = 0;
    int it;
    #pragma unroll 1
    for (it = 0; it < 20; it++) {
        double Ti = 2.0 * f_ani * eta_ve * Eii;
        lT = log(Ti);
        if (k.cst) Ec = Ti / f_ani * 0.5 * k.inv_eta_cst;
        if (k.pwl) Ep = exp(lnC_pwl + k.n_pwl * lT);
        if (k.gbs) Eg = exp(lnC_gbs + k.n_gbs * lT);
        if (peierls) Ee = exp(lnC_exp + nST * lT);
        if (k.lin) El = exp(lnC_lin + k.n_lin * lT);
        double r = Eii - elastic * Ti * half_inv_eel - (Ep + Ee + El + Eg + Ec);
        if (fabs(r * inv_Eii) < 1.0e-13) break;
        /* eta_ve * d r / d eta_ve */
        double dfe = 0.0;
        if (elastic) dfe += -Eii * inv_eel * eta_ve;
        if (peierls) dfe += -Ee * nST;
        if (k.lin) dfe += -El * k.n_lin;
        if (k.pwl) dfe += -Ep * k.n_pwl;
        if (k.cst) dfe += -Eii * k.inv_eta_cst * eta_ve;
        if (prm.rheo_mode != MDZ_RHEO_FP64 && fabs(r * inv_Eii) < 1.0e-3) {
            /* polish of an FP32 root: Halley's step (cubic convergence), so
             * that one step from |r/Eii| ~ 1e-5 meets the 1e-13 stop; with
             * eta^2 d2r/deta2 = -sum n (n - 1) E of the power-law terms */
            double d2 = 0.0;
            if (peierls) d2 -= Ee * nST * (nST - 1.0);
            if (k.lin) d2 -= El * k.n_lin * (k.n_lin - 1.0);
            if (k.pwl) d2 -= Ep * k.n_pwl * (k.n_pwl - 1.0);
            eta_ve -= 2.0 * r * dfe * eta_ve / (2.0 * dfe * dfe - r * d2);
        } else {
            eta_ve -= r * eta_ve / dfe;
        }
    }
    hist.add(0, it);
    hist.add(2, it32);
    /* stresses at the converged eta_ve */
    double Tii = 2.0 * eta_ve * f_ani * Eii;
    const double sfac = Tii / f_ani * inv_Eii;
    double Txx = in.Gxx * sfac, Tzz = in.Gzz * sfac, Txz = in.Gxz * sfac;
    /* creep rates at this Tii: the loop's values unless it ran out of
     * iterations (then eta_ve moved after the last evaluation) */
    double lTp = lT, Epp = Ep, Eep = Ee, Elp = El;
    if (it == 20) {
        lTp = log(Tii);
        if (k.pwl) Epp = exp(lnC_pwl + k.n_pwl * lTp);
        if (peierls) Eep = exp(lnC_exp + nST * lTp);
        if (k.lin) Elp = exp(lnC_lin + k.n_lin * lTp);
    }
    /* inverse viscosities of the creep mechanisms */
    const double inv_lin = k.lin ? exp(-(lnB_lin + (k.inv_n_lin - 1.0) * (lnC_lin + k.n_lin * lT) + k.ginv_lin)) : 0.0;
    const double inv_exp = peierls ? exp(-(lnB_exp + (inv_nST - 1.0) * (lnC_exp + nST * lT))) : 0.0;
    double inv_pwl = k.pwl ? exp(LN2 + lnC_pwl - (1.0 - k.n_pwl) * lTp) : 0.0;

    /* tangent of the visco-elastic update (RheologyDensity.c:425-447) */
    const double inv_Tii = 1.0 / Tii;
    const double inv_Ti3 = inv_Tii * inv_Tii * inv_Tii;
    double deta = 0.0;
    if (k.pwl) deta -= Epp * inv_Ti3 * (k.n_pwl - 1.0);
    if (peierls) deta -= Eep * inv_Ti3 * (nST - 1.0);
    if (k.lin) deta -= Elp * inv_Ti3 * (k.n_lin - 1.0);
    const double e2 = eta_ve * eta_ve;
    double dTxx = deta * (2.0 * Txx + Tzz) * e2, dTzz = deta * (2.0 * Tzz + Txx) * e2, dTxz = 2.0 * deta * Txz * e2;
    double den = 1.0 - 2.0 * (dTxx * Exx + dTzz * Ezz + dTxz * Exz);
    const double tden = 2.0 * eta_ve / den;
    const double de_xx = dTxx * tden, de_zz = dTzz * tden, de_xz = dTxz * tden;
    double dummy = 0.0;
    if (k.pwl) dummy += 2.0 * Epp * inv_Tii * k.Va_pwl * inv_RT;
    if (k.lin) dummy += 2.0 * Elp * inv_Tii * (k.m_lin != 0.0 ? exp(k.m_lin * (k.ln_gs_ref - lnd)) : 1.0) * k.Va_lin * inv_RT;
    const double de_p = e2 * dummy;

    /* plastic return map (RheologyDensity.c:468-531) */
    const double vp_exp = k.vp_exp;
    double F_trial = Tii - Tyield, gdot = 0.0, eta_vp = 0.0, Pc = P, divp = 0.0;
    double dQdtxx = 0, dQdtzz = 0, dQdtxz = 0;
    const double Kdt = K * dt;
    if (tens == 1) {
        eta_vp = k.eta_vp0 * (vp_exp == 0.0 ? 1.0 : pow(Eii, vp_exp));
        double Pc_chk = -(C * cos_fric) / (-Tii / P + sin_fric);
        sin_dil = (P * eta_ve + P * eta_vp - Pc_chk * eta_ve - Pc_chk * eta_vp)
                / (Kdt * (C * cos_fric + Pc_chk * sin_fric - Tii));
    }
    /* the diffusion, Peierls and constant-viscosity parts of the strain-rate
     * partition use the visco-elastic stresses (before the return map) */
    /* (the visco-elastic stresses are in.Gxx * sfac, ... : recomputed below) */
    const bool is_pl = F_trial > 1e-17;
    if (is_pl) {
        eta_vp = k.eta_vp0 * (vp_exp == 0.0 ? 1.0 : pow(Eii, vp_exp));
        const double Kds_dil = Kdt * sin_fric * sin_dil;
        gdot = F_trial / (eta_ve + eta_vp + Kds_dil);
        /* the network's correction of this start begins a nonlinear return
         * map (n_vp != 1); a linear one (n_vp = 1, with or without
         * dilation) is solved exactly by the start itself */
        if (gdot_guess > 0.0 && vp_exp != 0.0) gdot *= gdot_guess;
        const double hinv_Tii = 0.5 * inv_Tii;
        dQdtxx = Txx * hinv_Tii; dQdtzz = Tzz * hinv_Tii; dQdtxz = Txz * inv_Tii;
        const double F0 = F_trial;
        int itp;
        #pragma unroll 1
        for (itp = 0; itp < 20; itp++) {
            divp = gdot * sin_dil;
            Pc = P + Kdt * divp;
            eta_vp = k.eta_vp0 * (vp_exp == 0.0 ? 1.0 : pow(fabs(gdot), vp_exp));
            Tyield = C * cos_fric + Pc * sin_fric + gdot * eta_vp;
            double F = Tii - eta_ve * gdot - Tyield;
            double res = fabs(F);
            if (res < 1.0e-11 || res < 1.0e-11 * F0) break;
            gdot -= F / (-eta_ve - eta_vp * k.inv_n_vp - Kds_dil);
        }
        hist.add(1, itp + 1);
        Txx = 2.0 * eta_ve * (Exx - gdot * dQdtxx);
        Tzz = 2.0 * eta_ve * (Ezz - gdot * dQdtzz);
        double Tyy = -(Txx + Tzz);
        Txz = 2.0 * eta_ve * (Exz - gdot * dQdtxz * 0.5);
        Tii = sqrt(0.5 * (Txx * Txx + Tzz * Tzz + Tyy * Tyy) + Txz * Txz);
    } else {
        hist.add(1, 0);
    }
    const double hinv_Eii = 0.5 * inv_Eii;
    const double eta_vep = Tii * hinv_Eii;
    if (is_pl) Tii = 2.0 * eta_vep * Eii;

    /* dissipative viscosity: Peierls, dislocation, diffusion, constant,
     * visco-plastic, in this order */
    double inv_diss = 0.0;
    if (peierls) inv_diss += inv_exp;
    if (k.pwl) inv_diss += inv_pwl;
    if (k.lin) inv_diss += inv_lin;
    if (k.cst) inv_diss += k.inv_eta_cst;

    /* consistent tangent and plastic divergence derivatives */
    double etaVE = eta_ve, dexx = de_xx, dezz = de_zz, dexz = de_xz, dp = de_p;
    double ddxx = 0, ddzz = 0, ddxz = 0, ddp = 0;
    if (is_pl) {
        double dsx = 0, dsz = 0, dsxz = 0, dsp = 0;
        if (tens == 1) {
            const double dE[3] = {(2.0 * Exx + Ezz) * hinv_Eii, (2.0 * Ezz + Exx) * hinv_Eii, Exz * inv_Eii};
            const double dev[3] = {de_xx, de_zz, de_xz};
            double a2 = 2 * Eii * eta_ve - P * sin_fric;
            double bden = Kdt * a2 * (C * P * cos_fric * sin_fric + (C * cos_fric - 2 * Eii * eta_ve) * a2);
            const double inv_bden = 1.0 / bden;
            double q1 = C * P * cos_fric * sin_fric + a2 * a2;
            double od[3];
#pragma unroll
            for (int i = 0; i < 3; i++) {
                double dT = Eii * dev[i] + dE[i] * eta_ve;
                od[i] = (2 * Kdt * sin_dil * dT * q1
                         + P * (-C * cos_fric * dev[i] * a2 + 2 * C * cos_fric * (eta_ve + eta_vp) * dT + dev[i] * a2 * a2)) * inv_bden;
            }
            dsx = od[0]; dsz = od[1]; dsxz = od[2];
            dsp = (2 * C * Eii * cos_fric * (eta_ve + eta_vp) * (P * de_p - eta_ve) - C * P * cos_fric * de_p * a2
                   + 2 * Eii * Kdt * sin_dil * (C * cos_fric * sin_fric * (P * de_p - eta_ve) + de_p * a2 * a2)
                   + a2 * a2 * (P * de_p + eta_ve + eta_vp)) * inv_bden;
        }
        const double gg = 1.0 / (eta_ve + eta_vp * k.inv_n_vp + Kdt * sin_fric * sin_dil);
        const double Kds = Kdt * sin_fric;
        const double eE = eta_ve * inv_Eii;
        double lx = gg * (((2.0 * Exx + Ezz) * eE + 2.0 * Eii * de_xx) - gdot * (de_xx + Kds * dsx));
        double lz = gg * (((2.0 * Ezz + Exx) * eE + 2.0 * Eii * de_zz) - gdot * (de_zz + Kds * dsz));
        double lxz = gg * ((2.0 * Exz * eE + 2.0 * Eii * de_xz) - gdot * (de_xz + Kds * dsxz));
        double lp = gg * ((-sin_fric + 2.0 * Eii * de_p) - gdot * (de_p + Kds * dsp));
        const double evg = vp_exp == 0.0 ? 0.0 : eta_vp / gdot * vp_exp;
        double vx = evg * lx, vz = evg * lz, vxz = evg * lxz, vpp = evg * lp;
        double a = eta_vp + Kdt * sin_fric * sin_dil;
        const double tyE3 = Tyield * (hinv_Eii * inv_Eii * inv_Eii);
        dexx = -0.5 * (2.0 * Exx + Ezz) * tyE3 + (a * lx + gdot * vx + gdot * Kds * dsx) * hinv_Eii;
        dezz = -0.5 * (2.0 * Ezz + Exx) * tyE3 + (a * lz + gdot * vz + gdot * Kds * dsz) * hinv_Eii;
        dexz = -Exz * tyE3 + (a * lxz + gdot * vxz + gdot * Kds * dsxz) * hinv_Eii;
        dp = (sin_fric + a * lp + gdot * vpp + gdot * Kds * dsp) * hinv_Eii;
        etaVE = eta_vep;
        ddxx = sin_dil * lx + gdot * dsx;
        ddzz = sin_dil * lz + gdot * dsz;
        ddxz = sin_dil * lxz + gdot * dsxz;
        ddp = sin_dil * lp + gdot * dsp + 0.0;
        inv_diss += 1.0 / eta_vep;
        /* the dislocation viscosity of the strain-rate partition is
         * evaluated at the post-return stress */
        if (k.pwl) inv_pwl = exp(LN2 + lnC_pwl - (1.0 - k.n_pwl) * log(Tii));
    }
    double eta = 1.0 / inv_diss;
    const double VE = elastic ? eta_ve * inv_eel : 0.0;
    if (prm.step == 0) etaVE = eta;
    eta = fmin(fmax(eta, prm.mineta), prm.maxeta);
    etaVE = fmin(fmax(etaVE, prm.mineta), prm.maxeta);

    /* The output addresses depend on the node index; making it opaque here
     * keeps the compiler from computing the ~40 64-bit addresses before the
     * phase loop and holding them in registers through the local solve. */
    Out w = o;
    __asm__ volatile("" : "+v"(w.c));
    if (DIAG) __asm__ volatile("" ::: "memory");
    double Txx0 = 0, Tzz0 = 0, Txz0 = 0, P0 = 0, X0 = 0, exxd = 0, ezzd = 0, exzc = 0;
    if (DIAG) {
        Txx0 = ds.get(DS_SXX0); Tzz0 = ds.get(DS_SZZ0); Txz0 = ds.get(DS_SXZ0);
        P0 = ds.get(DS_P0); X0 = ds.get(DS_X0);
        if (CELL) { exxd = ds.get(DS_EXX); ezzd = ds.get(DS_EZZ); exzc = ds.get(DS_EXZ); }
    }
    const double Txx_ve = in.Gxx * sfac, Tzz_ve = in.Gzz * sfac, Txz_ve = in.Gxz * sfac;
    /* strain-rate partition (RheologyDensity.c:640-690) */
    const double ex_el = (double)elastic * (Txx - Txx0) * half_inv_eel;
    const double ez_el = (double)elastic * (Tzz - Tzz0) * half_inv_eel;
    const double exz_el = (double)elastic * (Txz - Txz0) * half_inv_eel;
    const double h_lin = 0.5 * inv_lin, h_pwl = 0.5 * inv_pwl, h_exp = 0.5 * inv_exp;
    const double h_cst = k.cst ? 0.5 * k.inv_eta_cst : 0.0;
    const double ex_d = gdot * dQdtxx + Txx_ve * h_lin + Txx * h_pwl + Txx_ve * h_exp + 0.0 + Txx_ve * h_cst;
    const double ez_d = gdot * dQdtzz + Tzz_ve * h_lin + Tzz * h_pwl + Tzz_ve * h_exp + 0.0 + Tzz_ve * h_cst;
    const double exz_d = gdot * dQdtxz / 2.0 + Txz_ve * h_lin + Txz * h_pwl + Txz_ve * h_exp + 0.0 + Txz_ve * h_cst;

    if (CELL) {
        w.put(FI_eta_n, etaVE);
        if (DIAG) w.put(FI_eta_phys_n, eta);
        w.put(FI_detadexx_n, dexx);
        w.put(FI_detadezz_n, dezz);
        w.put(FI_detadgxz_n, dexz / 2.0);
        w.put(FI_detadp_n, dp);
        if (DIAG) {
            w.put(FI_sxxd, Txx);
            w.put(FI_szzd, Tzz);
            w.put(FI_sxz_n, Txz);
            w.put(FI_VE_n, VE);
            w.put(FI_eII_el, (double)elastic * fabs(Tii - sqrt(Txx0 * Txx0 + Txz0 * Txz0)) * half_inv_eel);
            w.put(FI_eII_pl, gdot / 2.0);
            w.put(FI_eII_pwl, Tii * h_pwl);
            w.put(FI_eII_exp, Ee);
            w.put(FI_eII_lin, El);
            w.put(FI_eII_gbs, Eg);
            w.put(FI_eII_cst, Ec);
            acc.d = w.first ? w.fr * 1.0 / k.gs_ref : acc.d + w.fr * 1.0 / k.gs_ref;
            w.put(FI_exx_el, ex_el);
            w.put(FI_exx_diss, ex_d);
            w.put(FI_ezz_el, ez_el);
            w.put(FI_ezz_diss, ez_d);
            w.put(FI_Wtot, Txx * exxd + Tzz * ezzd + (Txx + Tzz) * (exxd + ezzd) + 2.0 * Txz * exzc);
            w.put(FI_Wdiss, Txx * ex_d + Tzz * ez_d + (Txx + Tzz) * (ex_d + ez_d) + 2.0 * Txz * exz_d);
            w.put(FI_Wel, Txx * ex_el + Tzz * ez_el + (Txx + Tzz) * (ex_el + ez_el) + 2.0 * Txz * exz_el);
        }
        w.put(FI_ddivpdexx_n, ddxx);
        w.put(FI_ddivpdezz_n, ddzz);
        w.put(FI_ddivpdgxz_n, ddxz / 2.0);
        w.put(FI_ddivpdp_n, ddp);
        w.put(FI_p_corr, Pc);
        if (DIAG) {
            w.put(FI_div_u_el, -(Pc - P0) / Kdt);
            w.put(FI_div_u_pl, divp);
            w.put(FI_div_u_r, 0.0);
            if (Xout) acc.x = w.first ? w.fr * X0 : acc.x + w.fr * X0;
            w.put(FI_OverS_n, is_pl ? eta_vp * gdot : 0.0);
        }
    } else {
        w.put(FI_eta_s, etaVE);
        if (DIAG) w.put(FI_eta_phys_s, eta);
        w.put(FI_detadexx_s, dexx);
        w.put(FI_detadezz_s, dezz);
        w.put(FI_detadgxz_s, dexz / 2.0);
        w.put(FI_detadp_s, dp);
        if (DIAG) {
            w.put(FI_sxz, Txz);
            w.put(FI_VE_s, VE);
            w.put(FI_exz_el, exz_el);
            w.put(FI_exz_diss, exz_d);
            w.put(FI_OverS_s, is_pl ? eta_vp * gdot : 0.0);
            if (Xout) acc.x = w.first ? w.fr * X0 : acc.x + w.fr * X0;
        }
    }
}

/* sines and cosines of the node's friction and dilatancy angles; dil = 0
 * when elasticity is off (RheologyDensity.c:160) */
__device__ __forceinline__ void node_angles(const DevParams &prm, double fric, double dil, NodeIn &in) {
    const int elastic = prm.step == 0 ? 0 : prm.iselastic;
    in.sin_fric = sin(fric);
    in.cos_fric = cos(fric);
    in.sin_dil = elastic == 0 ? 0.0 : sin(dil);
}

/* Initial-guess source of the local iterations: per-phase arrays written by
 * k_mlp_guess (factor on the reference's eta_ve guess, then the factor on
 * the return map's closed-form start at offset nph * n), or the network
 * evaluated in the kernel's own prologue (ph = the node's dominant phase,
 * fac and gd its factors), or none. */
struct GuessIn {
    const float *arr;
    int ph;
    float fac, gd;
    __device__ __forceinline__ double at(int p, int n, int node) const {
        return arr ? (double)arr[(size_t)p * n + node] : (p == ph ? (double)fac : 0.0);
    }
    __device__ __forceinline__ double gdot_at(int p, int nph, int n, int node) const {
        return arr ? (double)arr[(size_t)(nph + p) * n + node] : (p == ph ? (double)gd : 0.0);
    }
};

/* wave-wide minimum / maximum of an int */
__device__ __forceinline__ int wave_min_i(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ int wave_max_i(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    return v;
}

/* LDS ordering between the lanes of one wave: the wave's LDS writes are
 * complete (and the compiler keeps its LDS accesses on their side) before
 * any lane reads what another lane wrote. */
__device__ __forceinline__ void wave_lds_sync() {
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}

/* The phase fractions of one node (1 <= nph phases, checked at context
 * creation) into its LDS stash slots nd, nd + 1, ... (slot k of the lane at
 * sl[k * NT]; the stash holds at least nd + 4 slots): the first four in the
 * node's load batch, with no branch (phase index clamped, so every load is
 * in bounds; slots past nph receive copies nobody reads), the others after
 * it. */
template <int NT>
__device__ __forceinline__ void stash_fractions(const double *__restrict__ frac, int n, int node, int nph, int nd,
                                                double *sl) {
    double f[4];
#pragma unroll
    for (int q = 0; q < 4; q++) f[q] = frac[(size_t)min(q, nph - 1) * n + node];
#pragma unroll
    for (int q = 0; q < 4; q++) sl[(nd + q) * NT] = f[q];
    for (int p = 4; p < nph; p++) sl[(nd + p) * NT] = frac[(size_t)p * n + node];
}

/* Inputs of one node, loaded in one batch (index clamped into the grid, so
 * that every load is in bounds) before any branch or store: a wave waits
 * for memory once per node, not once per dependent branch and phase. */
struct NodeLoad {
    int tag;
    double mu, exx, ezz, exz, sxx0, szz0, sxz0, T, P, d, phi, C, bet, fric, dil;
};

/* The network's guess for the wave's centroids, one node per lane (all
 * lanes take part in the matrix instructions, those without a guess with
 * their features or zeros), from the node's loaded inputs; the outputs are
 * kept in w.cn for the vertices.  Weights and biases are read from global
 * memory (they stay in the caches).  The features and the choice of the
 * nodes (spread_wants_net, then features_from inside the sampled domain)
 * are those of k_mlp_guess, so both routes give the same guess bit for
 * bit.  A wave none of whose nodes takes the guess skips the features and
 * the network. */
template <int NT>
__device__ __forceinline__ GuessIn net_prologue(const DevGrid &g, const DevParams &prm, const DevMLPI &w,
                                                const PhaseK *__restrict__ pk, const SpreadConst &sc, bool act,
                                                int node, int n, const NodeLoad &v, const double *frac_sl) {
    __shared__ __attribute__((aligned(16))) unsigned short sX[NT / 64][64 * GS];
    __shared__ float sY0[NT / 64][64], sY1[NT / 64][64];
    const int wv = threadIdx.x >> 6, l = threadIdx.x & 63;
    int ph = act ? dominant_of(frac_sl, NT, min(prm.Nb_phases, g.nph)) : -1;
    /* the spread first (with the phase constants read by scalar loads when
     * the wave's nodes share one phase), the features only in a wave where
     * some node takes the network's guess */
    const VeEii e = ve_eii(prm, v.mu, v.exx, v.ezz, v.exz, v.sxx0, v.szz0, v.sxz0);
    const int phmin = wave_min_i(ph >= 0 ? ph : MDZ_MAX_PHASES), phmax = wave_max_i(ph);
    bool want;
    if (phmin == phmax) {
        const int phu = __builtin_amdgcn_readfirstlane(phmin);
        want = ph >= 0 && spread_wants_net(pk[phu], sc, e.lnEii, v.T, v.P, v.mu, v.d, v.phi);
    } else {
        want = ph >= 0 && spread_wants_net(pk[ph >= 0 ? ph : 0], sc, e.lnEii, v.T, v.P, v.mu, v.d, v.phi);
    }
    if (!want) ph = -1;
    float f[MLP_IN];
#pragma unroll
    for (int k = 0; k < MLP_IN; k++) f[k] = 0.0f;
    float y0 = 0.0f, y1 = 0.0f;
    if (__any(ph >= 0)) {
        if (ph >= 0 && !features_from(prm, ph, e, v.T, v.P, v.C, v.fric, f)) ph = -1;
        stage_features(sX[wv], f);
        wave_lds_sync();
        net_infer64(w.w + MLI_W1, 16, w.w + MLI_W2, w.w + MLI_W3, w.w + MLI_W4, 64, w.b, sX[wv], sY0[wv], sY1[wv]);
        wave_lds_sync();
        if (ph >= 0) {
            y0 = sY0[wv][l];
            y1 = sY1[wv][l];
        }
    }
    if (node < n) w.cn[node] = CellNet{y0, y1, ph, 0};
    return GuessIn{nullptr, ph, guess_factor(ph, y0), guess_gdot(ph, y1)};
}

/* The centroid output fields the rest of a unit reads (all of them are
 * written when DIAG). */
__device__ __constant__ const int k_unit_fields_n[10] = {FI_eta_n, FI_detadexx_n, FI_detadezz_n, FI_detadgxz_n,
                                                         FI_detadp_n, FI_ddivpdexx_n, FI_ddivpdezz_n,
                                                         FI_ddivpdgxz_n, FI_ddivpdp_n, FI_p_corr};
__device__ __constant__ const int k_unit_fields_s[5] = {FI_eta_s, FI_detadexx_s, FI_detadezz_s, FI_detadgxz_s,
                                                        FI_detadp_s};

/* LDS stash slots of a node: the diagnostic-only inputs (DIAG), then the
 * phase fractions. */
template <bool CELL, bool DIAG>
struct StashSlots {
    static constexpr int nd = DIAG ? (CELL ? 8 : 5) : 0;
};

/* The local update of one node over its phases, from the loaded inputs v
 * and the stash sl (the reference's accumulation over the phases, outputs
 * stored for the first active phase and added for the later ones). */
template <int NT, bool CELL, bool DIAG>
__device__ __forceinline__ void rheo_node(const DevGrid &g, const DevParams &prm, const PhaseK *__restrict__ pk,
                                          const FastConst &fc, double R, const GuessIn &gi, const BlockHist &hist,
                                          int node, int n, const NodeLoad &v, const double *sl) {
    constexpr int ND = StashSlots<CELL, DIAG>::nd;
    const bool active = CELL ? (v.tag != 30 && v.tag != 31) : v.tag != 30;
    const bool Xout = DIAG && prm.UnsplitDiffReac == 0;
    double *base = CELL ? g.eta_n : g.VE_s;
    const long long stride = CELL ? g.cstride : g.vstride;
    const int first_fi = CELL ? FI_eta_n : FI_VE_s;
    bool any = false;
    NodeAcc acc{0.0, 0.0};
    if (active) {
        const double etae = prm.iselastic == 1 ? prm.dt * v.mu : 1.0;
        NodeIn in;
        in.Txx0 = v.sxx0; in.Tzz0 = v.szz0; in.Txz0 = v.sxz0;
        ve_rates_iso(v.exx, v.ezz, v.exz, v.sxx0, v.szz0, v.sxz0, etae, in);
        in.G = v.mu; in.T = v.T; in.P = v.P; in.d = v.d; in.phi = v.phi; in.C = v.C; in.beta = v.bet;
        node_angles(prm, v.fric, v.dil, in);
        const DiagSrc ds{sl, NT};
        for (int p = 0; p < prm.Nb_phases; p++) {
            const double fr = sl[(ND + p) * NT];
            if (!(fabs(fr) > 1.0e-13)) continue;
            const Out o{base, stride, node, first_fi, fr, !any};
            const double gs = gi.at(p, n, node), gd = gi.gdot_at(p, g.nph, n, node);
            local_update<CELL, DIAG>(pk[p], R, prm, fc, in, Xout, o, ds, gs, gd, hist, acc);
            any = true;
        }
    }
    double *X = CELL ? g.X_n : g.X_s;
    if (!any) {
        /* air node, or no phase above the fraction threshold */
        if (DIAG) {
            const int last = CELL ? FI_OverS_n - FI_eta_n : FI_OverS_s - FI_VE_s;
            for (int i = 0; i <= last; i++) base[(long long)i * stride + node] = 0.0;
        } else if (CELL) {
            for (int i = 0; i < 10; i++) base[(long long)(k_unit_fields_n[i] - FI_eta_n) * stride + node] = 0.0;
        } else {
            for (int i = 0; i < 5; i++) base[(long long)(k_unit_fields_s[i] - FI_VE_s) * stride + node] = 0.0;
        }
        if (Xout) X[node] = 0.0;
        /* 1 / (empty sum) */
        if (CELL && DIAG && active) base[(long long)(FI_d_n - FI_eta_n) * stride + node] = 1.0 / 0.0;
    } else {
        if (Xout) X[node] = acc.x;
        if (CELL && DIAG) base[(long long)(FI_d_n - FI_eta_n) * stride + node] = 1.0 / acc.d;
    }
}

/* centroid `c0` of the lane (c0 >= nc: no node) */
template <int NT, bool DIAG, bool NET>
__device__ __forceinline__ void rheo_cell_fast(const DevGrid &g, const DevParams &prm, const FastConst &fc,
                                               const PhaseK *__restrict__ pk, double R,
                                               const float *__restrict__ guess, const DevMLPI &w,
                                               const SpreadConst &sc, const BlockHist &bh, double *stash, int c0) {
    constexpr int ND = StashSlots<true, DIAG>::nd;
    const int nc = g.ncx * g.ncz;
    const int c = c0 < nc ? c0 : nc - 1;
    double *sl = stash + threadIdx.x;
    NodeLoad v;
    v.tag = g.BCp[c];
    v.mu = g.mu_n[c]; v.exx = g.exxd[c]; v.ezz = g.ezzd[c]; v.exz = g.exz_n[c];
    v.sxx0 = g.sxxd0[c]; v.szz0 = g.szzd0[c]; v.sxz0 = g.sxz0_n[c];
    v.T = g.T[c]; v.P = g.p_in[c]; v.d = g.d0_n[c]; v.phi = g.phi0_n[c]; v.C = g.C_n[c]; v.bet = g.bet_n[c];
    v.fric = g.fric_n[c]; v.dil = g.dil_n[c];
    if (DIAG) {
        const double P0 = g.p0_n[c], X0 = g.X0_n[c];
        sl[DS_SXX0 * NT] = v.sxx0; sl[DS_SZZ0 * NT] = v.szz0; sl[DS_SXZ0 * NT] = v.sxz0;
        sl[DS_P0 * NT] = P0; sl[DS_X0 * NT] = X0;
        sl[DS_EXX * NT] = v.exx; sl[DS_EZZ * NT] = v.ezz; sl[DS_EXZ * NT] = v.exz;
    }
    stash_fractions<NT>(g.phase_n, nc, c, prm.Nb_phases, ND, sl);
    GuessIn gi{guess, -1, 0.0f, 0.0f};
    if constexpr (NET)
        gi = net_prologue<NT>(g, prm, w, pk, sc, c0 < nc && v.tag != 30 && v.tag != 31, c0, nc, v, sl + ND * NT);
    if (c0 < nc) rheo_node<NT, true, DIAG>(g, prm, pk, fc, R, gi, bh, c0, nc, v, sl);
}

/* vertex `c1` of the lane (c1 >= nv: no node) */
template <int NT, bool DIAG, bool NET>
__device__ __forceinline__ void rheo_vertex_fast(const DevGrid &g, const DevParams &prm, const FastConst &fc,
                                                 const PhaseK *__restrict__ pk, double R,
                                                 const float *__restrict__ guess, const DevMLPI &w,
                                                 const BlockHist &bh, double *stash, int c1) {
    constexpr int ND = StashSlots<false, DIAG>::nd;
    const int nv = g.Nx * g.Nz;
    const int c = c1 < nv ? c1 : nv - 1;
    double *sl = stash + threadIdx.x;
    NodeLoad v;
    v.tag = g.BCg[c];
    v.mu = g.mu_s[c]; v.exx = g.exxd_s[c]; v.ezz = g.ezzd_s[c]; v.exz = g.exz[c];
    v.sxx0 = g.sxxd0_s[c]; v.szz0 = g.szzd0_s[c]; v.sxz0 = g.sxz0[c];
    v.T = g.T_s[c]; v.P = g.P_s[c]; v.d = g.d0_s[c]; v.phi = g.phi0_s[c]; v.C = g.C_s[c]; v.bet = g.bet_s[c];
    v.fric = g.fric_s[c]; v.dil = g.dil_s[c];
    /* the network outputs of the four centroids around the vertex */
    CellNet cnb[4];
    bool inb[4];
    if constexpr (NET) {
        const int i = c % g.Nx, j = c / g.Nx;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int ic = i - 1 + (k & 1), jc = j - 1 + (k >> 1);
            inb[k] = ic >= 0 && ic < g.ncx && jc >= 0 && jc < g.ncz;
            cnb[k] = w.cn[inb[k] ? jc * g.ncx + ic : 0];
        }
    }
    if (DIAG) {
        const double P0 = g.p0_s[c], X0 = g.X0_s[c];
        sl[DS_SXX0 * NT] = v.sxx0; sl[DS_SZZ0 * NT] = v.szz0; sl[DS_SXZ0 * NT] = v.sxz0;
        sl[DS_P0 * NT] = P0; sl[DS_X0 * NT] = X0;
    }
    stash_fractions<NT>(g.phase_s, nv, c, prm.Nb_phases, ND, sl);
    GuessIn gi{guess, -1, 0.0f, 0.0f};
    if constexpr (NET) {
        /* vertex_net on the loaded values */
        int ph = c1 < nv && v.tag != 30 ? dominant_of(sl + ND * NT, NT, min(prm.Nb_phases, g.nph)) : -1;
        float y0 = 0.0f, y1 = 0.0f;
        if (ph >= 0) ph = vertex_mean(cnb, inb, ph, y0, y1);
        gi = GuessIn{nullptr, ph, guess_factor(ph, y0), guess_gdot(ph, y1)};
    }
    if (c1 < nv) rheo_node<NT, false, DIAG>(g, prm, pk, fc, R, gi, bh, c1, nv, v, sl);
}

enum { RHEO_BOTH, RHEO_CELLS, RHEO_VERTICES };

/* The local iterations at the centroids, then at the vertices, as block
 * ranges of one launch: the two are independent, so the last centroid waves
 * and the first vertex waves share the chip (41 x 41 nodes: 13 us against
 * 13 + 10, 1001 x 501: 119 against 79 + 62).  With the network's guess in the
 * pass (NET) a vertex reads the network outputs of its centroids, which the
 * centroid blocks write: then each has its own launch.  Two waves per SIMD:
 * every variant fits 256 registers (with both ranges and every output, 36
 * bytes of scratch); one wave per SIMD left the FP64 latency exposed.
 * Dynamic LDS: the stash, (StashSlots::nd + max(Nb_phases, 4)) * NT doubles. */
template <int NT, bool DIAG, bool NET, int PART>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2)))
k_rheo_fast(DevGrid g, DevParams prm, FastConst fc, const PhaseK *__restrict__ pk, double R,
            const float *__restrict__ guess_n, const float *__restrict__ guess_s, DevMLPI w, SpreadConst sc,
            unsigned long long *hist) {
    __shared__ unsigned int lh[3 * MDZ_HIST_BINS];
    extern __shared__ double stash[];
    const BlockHist bh = hist_begin(lh, hist);
    const int b = blockIdx.x, nbc = PART == RHEO_VERTICES ? 0 : mdz_div_up(g.ncx * g.ncz, NT);
    if (PART != RHEO_VERTICES && b < nbc)
        rheo_cell_fast<NT, DIAG, NET>(g, prm, fc, pk, R, guess_n, w, sc, bh, stash, b * NT + (int)threadIdx.x);
    if (PART != RHEO_CELLS && b >= nbc)
        rheo_vertex_fast<NT, DIAG, NET>(g, prm, fc, pk, R, guess_s, w, bh, stash, (b - nbc) * NT + (int)threadIdx.x);
    hist_flush(bh, hist);
}

int mdz_rheo_fast_eligible(const DevParams &prm, const mat_prop *host_mt) {
    if (prm.eta_avg != 0 || prm.aniso != 0 || prm.Nb_phases > MDZ_MAX_PHASES || prm.VolChangeReac != 0) return 0;
    for (int p = 0; p < prm.Nb_phases; p++) {
        if (host_mt->gs[p] != 0 || host_mt->reac_soft[p] == 1) return 0;
        if (prm.diffuse_X != 0 && host_mt->phase_mix[p] != 0) return 0;
    }
    return 1;
}

size_t mdz_phasek_bytes(void) { return MDZ_MAX_PHASES * sizeof(PhaseK); }

void mdz_launch_phase_constants(const mat_prop *d_mt, int nph, void *d_pk, hipStream_t s) {
    hipLaunchKernelGGL(k_phase_constants, dim3(1), dim3(64), 0, s, d_mt, nph < MDZ_MAX_PHASES ? nph : MDZ_MAX_PHASES,
                       (PhaseK *)d_pk);
}

template <int NT, bool DIAG, bool NET>
static void launch_fast(const DevGrid &g, const DevParams &prm, const PhaseK *pk, double R, const float *guess_n,
                        const float *guess_s, const DevMLPI &w, unsigned long long *hist, hipStream_t s) {
    int nc = g.ncx * g.ncz, nv = g.Nx * g.Nz;
    FastConst fc;
    fc.T_peierls = (1200.0 + ZEROC) / prm.sT;
    fc.T_min = ZEROC / prm.sT;
    fc.eta_start = 1.0e100 / prm.seta;
    fc.P_tens = -25e6 / prm.sS;
    fc.E_floor = 1e-30 / prm.sE;
    const SpreadConst sc = spread_const(R, prm.sT, prm.dt, prm.iselastic != 0 && prm.step != 0);
    const int nph = prm.Nb_phases > 4 ? prm.Nb_phases : 4; /* stash_fractions writes at least four slots */
    const size_t lds_c = (size_t)(StashSlots<true, DIAG>::nd + nph) * NT * sizeof(double);
    const size_t lds_v = (size_t)(StashSlots<false, DIAG>::nd + nph) * NT * sizeof(double);
    const int nbc = mdz_div_up(nc, NT), nbv = mdz_div_up(nv, NT);
    if constexpr (NET) {
        hipLaunchKernelGGL((k_rheo_fast<NT, DIAG, NET, RHEO_CELLS>), dim3(nbc), dim3(NT), lds_c, s, g, prm, fc, pk, R,
                           guess_n, guess_s, w, sc, hist);
        hipLaunchKernelGGL((k_rheo_fast<NT, DIAG, NET, RHEO_VERTICES>), dim3(nbv), dim3(NT), lds_v, s, g, prm, fc, pk,
                           R, guess_n, guess_s, w, sc, hist);
    } else {
        hipLaunchKernelGGL((k_rheo_fast<NT, DIAG, NET, RHEO_BOTH>), dim3(nbc + nbv), dim3(NT),
                           lds_c > lds_v ? lds_c : lds_v, s, g, prm, fc, pk, R, guess_n, guess_s, w, sc, hist);
    }
}

template <int NT, bool DIAG>
static void launch_fast(const DevGrid &g, const DevParams &prm, const PhaseK *pk, double R, const float *guess_n,
                        const float *guess_s, const DevMLPI *net, unsigned long long *hist, hipStream_t s) {
    if (net) launch_fast<NT, DIAG, true>(g, prm, pk, R, nullptr, nullptr, *net, hist, s);
    else
        launch_fast<NT, DIAG, false>(g, prm, pk, R, guess_n, guess_s, DevMLPI{nullptr, nullptr, nullptr}, hist, s);
}

int mdz_launch_rheology_fast(const DevGrid &g, const DevParams &prm, const void *d_pk, double R, const float *guess_n,
                             const float *guess_s, unsigned long long *hist, int nt, int diag, hipStream_t s,
                             const DevMLPI *net) {
    const PhaseK *pk = (const PhaseK *)d_pk;
    if (net && (!net->w || !net->b || !net->cn)) return mdz_error(MDZ_EINVAL, "rheology: network without weights");
    switch (nt * 2 + (diag ? 1 : 0)) {
    case 129: launch_fast<64, true>(g, prm, pk, R, guess_n, guess_s, net, hist, s); return MDZ_OK;
    case 128: launch_fast<64, false>(g, prm, pk, R, guess_n, guess_s, net, hist, s); return MDZ_OK;
    case 257: launch_fast<128, true>(g, prm, pk, R, guess_n, guess_s, net, hist, s); return MDZ_OK;
    case 256: launch_fast<128, false>(g, prm, pk, R, guess_n, guess_s, net, hist, s); return MDZ_OK;
    case 513: launch_fast<256, true>(g, prm, pk, R, guess_n, guess_s, net, hist, s); return MDZ_OK;
    case 512: launch_fast<256, false>(g, prm, pk, R, guess_n, guess_s, net, hist, s); return MDZ_OK;
    default: return mdz_error(MDZ_EINVAL, "rheology block size: 64, 128 or 256 threads");
    }
}
