/*
 * mdz_assembly.hip -- gfx950 kernels of the decoupled Stokes assembly and
 * residual of the Newton-iteration path.
 *
 * One lane per CSR row (equation).  Every row is emitted by one templated
 * device function through a sink: SINK_COUNT counts the appended entries,
 * SINK_PATTERN writes the column indices, SINK_VALUES writes the values and
 * folds Dirichlet neighbours into bbc.  Which neighbours are appended, and
 * in which order, depends only on the boundary tags, so the pattern built
 * once per boundary-condition set stays valid for every Newton iteration
 * and the value pass writes in place into it.
 *
 *   equation numbering              StokesRoutines.c:1134-1187
 *   AddCoeff2 folding               StokesAssemblyCoupled.c:47-57
 *   continuity rows                 StokesAssemblyDecoupled.c:62-103
 *   Picard X rows, W/E Neumann      StokesAssemblyDecoupled.c:109-234, 476-790
 *   Picard Z rows, S/N Neumann      StokesAssemblyDecoupled.c:796-972, 1168-1428
 *   Jacobian X / Z rows             StokesAssemblyDecoupled.c:3034-3421, 3427-3825
 *   row order / append order        StokesAssemblyCoupled.c:1446-1492
 *   residual norms                  StokesRoutines.c:839-916
 *
 * The Jacobian rows are the composition of the linear operators they
 * linearise (staggered strain rates, masked centroid<->vertex means with
 * the weights wE/wW/wS/wN, the tangent blocks, the stress divergence);
 * each neighbour's coefficient accumulates its contributions through it.
 */
#include "mdz_kernels.h"

#define BLK 256
#define OUTSIDE 99

/* Emission of one row: COUNT counts the entries, PATTERN writes the column
 * indices, VALUES the coefficients.  A neighbour of Dirichlet type (0, 31,
 * 11, 13) is folded into the row's bbc instead of appended.  In VALUES mode
 * the choice is made without a branch: a folded coefficient is stored to
 * the lane's own dump slot, so every append is one store and one select. */
template <int MODE>
struct Sink {
    int n;
    int *J;
    double *A;
    double bbc;
    double *dump; /* VALUES: per-lane slot for folded coefficients */
    /* val(): the neighbour's boundary value, read only when it is folded */
    template <class V>
    __device__ __forceinline__ void add(int jeq, double coeff, int type, V val) {
        const bool fold = type == 0 || type == 31 || type == 11 || type == 13;
        if (MODE == SINK_VALUES) {
            if (fold) bbc -= coeff * val();
            *(fold ? dump : A + n) = coeff;
            n += fold ? 0 : 1;
        } else if (!fold) {
            if (MODE == SINK_PATTERN) J[n] = jeq;
            n++;
        }
    }
};

/* Tag reads with the reference's out-of-array reads mapped to OUTSIDE; the
 * index is clamped instead of branched around, so the load is always in
 * bounds and the lanes stay converged. */
struct Tags {
    const int8_t *u, *v, *p, *gv;
    int nu, nw, nc, nv;
    __device__ __forceinline__ static int rd(const int8_t *t, int i, int n) {
        const bool in = (unsigned)i < (unsigned)n;
        const int x = t[in ? i : 0];
        return in ? x : OUTSIDE;
    }
    __device__ __forceinline__ int U(int i) const { return rd(u, i, nu); }
    __device__ __forceinline__ int V(int i) const { return rd(v, i, nw); }
    __device__ __forceinline__ int P(int i) const { return rd(p, i, nc); }
    __device__ __forceinline__ int G(int i) const { return rd(gv, i, nv); }
};

/* Tag source of a row whose every tag read is a free degree of freedom
 * (-1): no loads, and the row code specialises to the interior stencil. */
struct FreeTags {
    __device__ __forceinline__ int U(int) const { return -1; }
    __device__ __forceinline__ int V(int) const { return -1; }
    __device__ __forceinline__ int P(int) const { return -1; }
    __device__ __forceinline__ int G(int) const { return -1; }
};

/* Real tag reads that also record whether every one of them was -1. */
struct CheckTags : Tags {
    mutable bool all_free;
    __device__ __forceinline__ int note(int t) const { all_free = all_free && t == -1; return t; }
    __device__ __forceinline__ int U(int i) const { return note(Tags::U(i)); }
    __device__ __forceinline__ int V(int i) const { return note(Tags::V(i)); }
    __device__ __forceinline__ int P(int i) const { return note(Tags::P(i)); }
    __device__ __forceinline__ int G(int i) const { return note(Tags::G(i)); }
};

__device__ __forceinline__ Tags make_tags(const DevGrid &g) {
    Tags t;
    t.u = g.BCu; t.v = g.BCv; t.p = g.BCp; t.gv = g.BCg;
    t.nu = g.Nx * g.nzvx; t.nw = g.nxvz * g.Nz; t.nc = g.ncx * g.ncz; t.nv = g.Nx * g.Nz;
    return t;
}

/* ------------------------------------------------------------------ */
/* continuity                                                           */
/* ------------------------------------------------------------------ */
template <bool ASM, int MODE>
__device__ void continuity_row(const DevAsm &a, int comp, int c1, int c2, int c3, Sink<MODE> &rc, double &b, double &F) {
    const DevGrid &g = a.g;
    int nxvz = g.nxvz;
    int tW = g.BCu[c1], tE = g.BCu[c1 + 1], tS = g.BCv[c3], tN = g.BCv[c3 + nxvz];
    double uW = tW != 13 ? -a.one_dx * 1e0 : 0.0, uE = tE != 13 ? a.one_dx * 1e0 : 0.0;
    double vS = tS != 13 ? -a.one_dz * 1e0 : 0.0, vN = tN != 13 ? a.one_dz * 1e0 : 0.0;
    if (ASM) {
        b *= a.celvol;
        if (tW != 13) rc.add(a.e.eqn_u[c1], uW * a.celvol, tW, [&] { return g.BCu_val[c1]; });
        if (tE != 13) rc.add(a.e.eqn_u[c1 + 1], uE * a.celvol, tE, [&] { return g.BCu_val[c1 + 1]; });
        if (tS != 13) rc.add(a.e.eqn_v[c3], vS * a.celvol, tS, [&] { return g.BCv_val[c3]; });
        if (tN != 13) rc.add(a.e.eqn_v[c3 + nxvz], vN * a.celvol, tN, [&] { return g.BCv_val[c3 + nxvz]; });
    } else {
        double pc = comp == 0 ? 0.0 : g.bet_n[c2] / a.dt;
        double f = pc * a.p_cont[c2] + uW * a.u[c1] + uE * a.u[c1 + 1] + vS * a.v[c3] + vN * a.v[c3 + nxvz];
        f -= b;
        F = f * a.celvol;
    }
}

/* Coefficients of a Picard momentum row in the residual pass (Assemble =
 * 0), with the reference's divisions by dx, dz: F is a small difference
 * of large terms, so its parity needs the same roundings.  X rows
 * (StokesAssemblyDecoupled.c:210-233): D11 of the west and east centroids,
 * D33 of the north and south vertices and their in-domain flags. */
struct XRes {
    double uW, uC, uE, uS, uN, vSW, vSE, vNW, vNE;
};
__device__ __forceinline__ XRes xres_coeffs(double D11W, double D11E, double D33N, double D33S, double inW,
                                            double inE, double inS, double inN, double dx, double dz) {
    const double comp = 1.0;
    XRes r;
    r.uW = D11W * inW * ((1.0 / 3.0) * comp / dx - 1.0 / dx) / dx;
    r.uC = -(-D33N * inN / dz - D33S * inS / dz) / dz
         - (D11E * inE * ((1.0 / 3.0) * comp / dx - 1 / dx) - D11W * inW * (-1.0 / 3.0 * comp / dx + 1.0 / dx)) / dx;
    r.uE = -D11E * inE * (-1.0 / 3.0 * comp / dx + 1.0 / dx) / dx;
    r.uS = -D33S * inS / (dz * dz);
    r.uN = -D33N * inN / (dz * dz);
    r.vSW = (1.0 / 3.0) * D11W * comp * inW / (dx * dz) - D33S * inS / (dx * dz);
    r.vSE = -1.0 / 3.0 * D11E * comp * inE / (dx * dz) + D33S * inS / (dx * dz);
    r.vNW = -1.0 / 3.0 * D11W * comp * inW / (dx * dz) + D33N * inN / (dx * dz);
    r.vNE = (1.0 / 3.0) * D11E * comp * inE / (dx * dz) - D33N * inN / (dx * dz);
    return r;
}
/* Z rows (StokesAssemblyDecoupled.c:939-971): D22 of the south and north
 * centroids, D33 of the west and east vertices. */
struct ZRes {
    double vW, vC, vE, vS, vN, uSW, uSE, uNW, uNE;
};
__device__ __forceinline__ ZRes zres_coeffs(double D22S, double D22N, double D33W, double D33E, double inS,
                                            double inN, double inW, double inE, double dx, double dz) {
    const double comp = 1.0;
    ZRes r;
    r.vW = -D33W * inW / (dx * dx);
    r.vC = -(D22N * inN * ((1.0 / 3.0) * comp / dz - 1 / dz) - D22S * inS * (-1.0 / 3.0 * comp / dz + 1.0 / dz)) / dz
         - (-D33E * inE / dx - D33W * inW / dx) / dx;
    r.vE = -D33E * inE / (dx * dx);
    r.vS = D22S * inS * ((1.0 / 3.0) * comp / dz - 1 / dz) / dz;
    r.vN = -D22N * inN * (-1.0 / 3.0 * comp / dz + 1.0 / dz) / dz;
    r.uSW = (1.0 / 3.0) * D22S * comp * inS / (dx * dz) - D33W * inW / (dx * dz);
    r.uSE = -1.0 / 3.0 * D22S * comp * inS / (dx * dz) + D33E * inE / (dx * dz);
    r.uNW = -1.0 / 3.0 * D22N * comp * inN / (dx * dz) + D33W * inW / (dx * dz);
    r.uNE = (1.0 / 3.0) * D22N * comp * inN / (dx * dz) - D33E * inE / (dx * dz);
    return r;
}

/* ------------------------------------------------------------------ */
/* Picard X rows                                                        */
/* ------------------------------------------------------------------ */
template <bool ASM, int MODE, class TG>
__device__ void xmom_inner(const DevAsm &a, const TG &T, int c1, int c2, int c3, int eqn, Sink<MODE> &ra, Sink<MODE> &rb,
                           double &b, double &F) {
    const DevGrid &g = a.g;
    int nx = g.Nx, ncx = g.ncx, nxvz = g.nxvz;
    int iVxC = c1, iVxW = iVxC - 1, iVxE = iVxC + 1, iVxS = iVxC - nx, iVxN = iVxC + nx;
    int iVzSW = c3 - nxvz, iVzSE = c3 - nxvz + 1, iVzNW = c3, iVzNE = c3 + 1;
    int iPrW = c2, iPrE = c2 + 1, ixyN = c1, ixyS = c1 - nx;
    if (T.U(iVxC) == -2) { iVxW = c1 + nx - 2; iPrW = c2 + ncx; iVzSW = c3 - 2; iVzNW = c3 + nxvz - 2; }
    double D11E = a.d11p[iPrE], D11W = a.d11p[iPrW], D33N = a.d33p[ixyN], D33S = a.d33p[ixyS];
    double inW = T.P(iPrW) == -1 ? 1.0 : 0.0, inE = T.P(iPrE) == -1 ? 1.0 : 0.0;
    double inS = (T.G(ixyS) != 30 && T.U(ixyS) != 13) ? 1.0 : 0.0;
    double inN = (T.G(c1) != 30 && T.U(c1 + nx) != 13) ? 1.0 : 0.0;
    const double comp = 1.0;
    double uW, uC, uE, uS, uN, vSW, vSE, vNW, vNE;
    if (ASM) {
        /* matrix values: the reference's divisions by dx, dz, dx dz and dz^2
         * as products with the per-grid reciprocals (one rounding apart) */
        const double idx = a.one_dx, idz = a.one_dz, idxz = a.one_dx_dz, idzz = a.one_dz_dz;
        uW = D11W * inW * ((1.0 / 3.0) * comp * idx - idx) * idx;
        uC = -(-D33N * inN * idz - D33S * inS * idz) * idz
           - (D11E * inE * ((1.0 / 3.0) * comp * idx - idx) - D11W * inW * (-1.0 / 3.0 * comp * idx + idx)) * idx;
        uE = -D11E * inE * (-1.0 / 3.0 * comp * idx + idx) * idx;
        uS = -D33S * inS * idzz;
        uN = -D33N * inN * idzz;
        vSW = (1.0 / 3.0) * D11W * comp * inW * idxz - D33S * inS * idxz;
        vSE = -1.0 / 3.0 * D11E * comp * inE * idxz + D33S * inS * idxz;
        vNW = -1.0 / 3.0 * D11W * comp * inW * idxz + D33N * inN * idxz;
        vNE = (1.0 / 3.0) * D11E * comp * inE * idxz - D33N * inN * idxz;
    } else {
        const XRes r = xres_coeffs(D11W, D11E, D33N, D33S, inW, inE, inS, inN, g.dx, g.dz);
        uW = r.uW; uC = r.uC; uE = r.uE; uS = r.uS; uN = r.uN;
        vSW = r.vSW; vSE = r.vSE; vNW = r.vNW; vNE = r.vNE;
    }
    double pW = 0, pE = 0;
    if (a.stab == 1) {
        double drhodx = (g.rho_n[c2 + 1] - g.rho_n[c2]) * a.one_dx;
        double uC_corr = 1.00 * a.om * a.dt * g.gx[c1] * drhodx;
        if (uC + uC_corr > 0.0) uC += uC_corr;
    }
    int tS = T.U(iVxS), tN = T.U(iVxN);
    if (tS == 11) uC -= uS;
    if (tN == 11) uC -= uN;
    bool pgrad = T.P(iPrE) != 30 && T.P(iPrW) != 30;
    if (pgrad) { pW = -a.one_dx * 1e0; pE = a.one_dx * 1e0; }
    double cv = a.celvol;
    if (ASM) {
        b *= cv;
        if (tS != 30) ra.add(a.e.eqn_u[iVxS], uS * cv, tS, [&] { return (tS != 11 ? 1.0 : 2.0) * g.BCu_val[iVxS]; });
        if (T.U(iVxW) != 30) ra.add(a.e.eqn_u[iVxW], uW * cv, T.U(iVxW), [&] { return g.BCu_val[iVxW]; });
        ra.add(eqn, uC * cv, T.U(iVxC), [&] { return g.BCu_val[iVxC]; });
        if (T.U(iVxE) != 30) ra.add(a.e.eqn_u[iVxE], uE * cv, T.U(iVxE), [&] { return g.BCu_val[iVxE]; });
        if (T.U(c1 + nx) != 30) ra.add(a.e.eqn_u[iVxN], uN * cv, tN, [&] { return (tN != 11 ? 1.0 : 2.0) * g.BCu_val[iVxN]; });
        if (T.V(iVzSW) != 30) ra.add(a.e.eqn_v[iVzSW], vSW * cv, T.V(iVzSW), [&] { return g.BCv_val[iVzSW]; });
        if (T.V(iVzSE) != 30) ra.add(a.e.eqn_v[iVzSE], vSE * cv, T.V(iVzSE), [&] { return g.BCv_val[iVzSE]; });
        if (T.V(iVzNW) != 30) ra.add(a.e.eqn_v[iVzNW], vNW * cv, T.V(iVzNW), [&] { return g.BCv_val[iVzNW]; });
        if (T.V(iVzNE) != 30) ra.add(a.e.eqn_v[iVzNE], vNE * cv, T.V(iVzNE), [&] { return g.BCv_val[iVzNE]; });
        if (pgrad) {
            rb.add(a.e.eqn_p[iPrW] - a.e.neq_mom, pW * cv, T.P(iPrW), [&] { return g.BCp_val[iPrW]; });
            rb.add(a.e.eqn_p[iPrE] - a.e.neq_mom, pE * cv, T.P(iPrE), [&] { return g.BCp_val[iPrE]; });
        }
    } else {
        const double *u = a.u, *v = a.v, *p = a.p_mom;
        double f = uC * u[iVxC];
        if (pgrad) f += pW * p[iPrW] + pE * p[iPrE];
        if (T.V(iVzSE) != 30) f += vSE * v[iVzSE];
        if (T.V(iVzSW) != 30) f += vSW * v[iVzSW];
        if (T.V(iVzNE) != 30) f += vNE * v[iVzNE];
        if (T.V(iVzNW) != 30) f += vNW * v[iVzNW];
        if (tS != 30 && tS != 11) f += uS * u[iVxS];
        if (tS == 11) f += 2.0 * uS * g.BCu_val[iVxS];
        if (tN != 30 && tN != 11) f += uN * u[iVxN];
        if (tN == 11) f += 2.0 * uN * g.BCu_val[iVxN];
        if (T.U(iVxW) != 30) f += uW * u[iVxW];
        if (T.U(iVxE) != 30) f += uE * u[iVxE];
        f -= b;
        F = f * cv;
    }
}

template <bool ASM, int MODE, class TG>
__device__ void xmom_neumann(const DevAsm &a, const TG &T, int c1, int c2, int c3, int eqn, int east, int comp, Sink<MODE> &ra,
                             Sink<MODE> &rb, double &b, double bbc_in, double &F) {
    const DevGrid &g = a.g;
    int nx = g.Nx, nxvz = g.nxvz;
    double etaE, etaW, etaN = g.eta_s[c1], etaS = g.eta_s[c1 - nx];
    if (!east) { etaE = g.eta_n[c2 + 1]; etaW = etaE; }
    else { etaW = g.eta_n[c2]; etaE = etaW; }
    double uS = 0, uN = 0, uW = 0, uE = 0, uC = 0, vSW = 0, vSE = 0, vNW = 0, vNE = 0, pE = 0, pW = 0;
    double dxx = a.one_dx_dx, dzz = a.one_dz_dz, dxz = a.one_dx_dz;
    if (!east) {
        b -= g.BCu_val[c1] * a.one_dx;
        if (T.U(c1 + 1) != 30) {
            uC = -2.0 * dxx * (etaE) + comp * 2.0 / 3.0 * dxx * etaE;
            uE = 2.0 * dxx * etaE - comp * 2.0 / 3.0 * dxx * etaE;
        }
    } else {
        b += g.BCu_val[c1] * a.one_dx;
        if (T.U(c1 - 1) != 30) {
            uW = 2.0 * dxx * etaW - comp * 2.0 / 3.0 * dxx * etaW;
            uC = -2.0 * dxx * (etaW) + comp * 2.0 / 3.0 * dxx * etaW;
        }
    }
    int tS = T.U(c1 - nx), tN = T.U(c1 + nx);
    if (tS != 30 && tN != 30) {
        if (tS != 13) { uS = dzz * etaS; uC += -dzz * etaS; }
        if (tN != 13) { uN = dzz * etaN; uC += -dzz * etaN; }
    }
    if (tS == 30 && tN != 30) {
        if (tN != 13) uC += -dzz * etaN;
        if (tN != 13) uN = dzz * etaN;
    }
    if (tS != 30 && tN == 30) {
        if (tS != 13) uC += -dzz * etaS;
        if (tS != 13) uS = dzz * etaS;
    }
    if (tS == 11) uC += -dzz * etaS;
    if (tN == 11) uC += -dzz * etaN;
    bool vs = T.V(c3 - nxvz) != 30 && T.V(c3 - nxvz + 1) != 30;
    bool vn = T.V(c3 + 1) != 30 && T.V(c3) != 30;
    if (vs) {
        vSE = -dxz * etaS + comp * 2.0 / 3.0 * dxz * etaE;
        vSW = dxz * etaS - comp * 2.0 / 3.0 * dxz * etaW;
    }
    if (vn) {
        vNE = dxz * etaN - comp * 2.0 / 3.0 * dxz * etaE;
        vNW = -dxz * etaN + comp * 2.0 / 3.0 * dxz * etaW;
    }
    int ip = east ? c2 : c2 + 1;
    if (!east) { if (T.P(c2 + 1) != 30) { pW = a.one_dx; pE = -pW; } }
    else { if (T.P(c2) != 30) pW = a.one_dx; }
    uS = -uS; uN = -uN; uW = -uW; uE = -uE; uC = -uC; vSW = -vSW; vSE = -vSE; vNW = -vNW; vNE = -vNE; pE = -pE; pW = -pW;
    double pcoef = east ? pW : pE;
    double cv = a.celvol;
    if (ASM) {
        b *= cv;
        if (tS != 30) ra.add(a.e.eqn_u[c1 - nx], uS * cv, tS, [&] { return (tS != 11 ? 1.0 : 2.0) * g.BCu_val[c1 - nx]; });
        if (east && T.U(c1 - 1) != 30) ra.add(a.e.eqn_u[c1 - 1], uW * cv, T.U(c1 - 1), [&] { return g.BCu_val[c1 - 1]; });
        ra.add(eqn, uC * cv, T.U(c1), [&] { return g.BCu_val[c1]; });
        if (!east && T.U(c1 + 1) != 30) ra.add(a.e.eqn_u[c1 + 1], uE * cv, T.U(c1 + 1), [&] { return g.BCu_val[c1 + 1]; });
        if (tN != 30) ra.add(a.e.eqn_u[c1 + nx], uN * cv, tN, [&] { return (tN != 11 ? 1.0 : 2.0) * g.BCu_val[c1 + nx]; });
        if (vs) {
            ra.add(a.e.eqn_v[c3 - nxvz], vSW * cv, T.V(c3 - nxvz), [&] { return g.BCv_val[c3 - nxvz]; });
            ra.add(a.e.eqn_v[c3 - nxvz + 1], vSE * cv, T.V(c3 - nxvz + 1), [&] { return g.BCv_val[c3 - nxvz + 1]; });
        }
        if (vn) {
            ra.add(a.e.eqn_v[c3], vNW * cv, T.V(c3), [&] { return g.BCv_val[c3]; });
            ra.add(a.e.eqn_v[c3 + 1], vNE * cv, T.V(c3 + 1), [&] { return g.BCv_val[c3 + 1]; });
        }
        if (T.P(ip) != 30) rb.add(a.e.eqn_p[ip] - a.e.neq_mom, pcoef * cv, T.P(ip), [&] { return g.BCp_val[ip]; });
    } else {
        const double *u = a.u, *v = a.v, *p = a.p_mom;
        double f = -(b + bbc_in / cv);
        f += uC * u[c1];
        if (tS != 30 && tS != 11) f += uS * u[c1 - nx];
        if (east && T.U(c1 - 1) != 30) f += uW * u[c1 - 1];
        if (!east && T.U(c1 + 1) != 30) f += uE * u[c1 + 1];
        if (tN != 30 && tN != 11) f += uN * u[c1 + nx];
        if (vs) {
            int t1 = T.V(c3 - nxvz + 1), t0 = T.V(c3 - nxvz);
            if (t1 != 11 && t1 != 0) f += vSE * v[c3 - nxvz + 1];
            if (t0 != 11 && t0 != 0) f += vSW * v[c3 - nxvz];
        }
        if (vn) {
            int t1 = T.V(c3 + 1), t0 = T.V(c3);
            if (t1 != 11 && t1 != 0) f += vNE * v[c3 + 1];
            if (t0 != 11 && t0 != 0) f += vNW * v[c3];
        }
        if (T.P(ip) != 30) f += pcoef * p[ip];
        F = f * cv;
    }
}

/* ------------------------------------------------------------------ */
/* Picard Z rows                                                        */
/* ------------------------------------------------------------------ */
template <bool ASM, int MODE, class TG>
__device__ void zmom_inner(const DevAsm &a, const TG &T, int c1, int c2, int c3, int eqn, Sink<MODE> &ra, Sink<MODE> &rb,
                           double &b, double &F) {
    const DevGrid &g = a.g;
    int nx = g.Nx, ncx = g.ncx, nxvz = g.nxvz;
    double D22S = a.d22p[c2], D22N = a.d22p[c2 + ncx], D33E = a.d33p[c1], D33W = a.d33p[c1 - 1];
    if (T.P(c2 + ncx) == 31) b += g.BCv_val[c3] * a.one_dz;
    int tVS = T.V(c3 - nxvz), tVN = T.V(c3 + nxvz);
    double inS = 0, inN = 0;
    if (tVS != 30 && tVN != 30) { inS = 1.0; inN = 1.0; }
    if (tVS == 30 && tVN != 30) inN = 1.0;
    if (tVS != 30 && tVN == 30) inS = 1.0;
    if (T.P(c2) == -1) inS = 1.0;
    if (T.P(c2 + ncx) == -1) inN = 1.0;
    double inW = (T.G(c1 - 1) != 30 && T.V(c3 - 1) != 13) ? 1.0 : 0.0;
    double inE = (T.G(c1) != 30 && T.V(c3 + 1) != 13) ? 1.0 : 0.0;
    const double comp = 1.0;
    double vW, vC, vE, vS, vN, uSW, uSE, uNW, uNE;
    if (ASM) {
        /* matrix values with the per-grid reciprocals, as in the X rows */
        const double idx = a.one_dx, idz = a.one_dz, idxz = a.one_dx_dz, idxx = a.one_dx_dx;
        vW = -D33W * inW * idxx;
        vC = -(D22N * inN * ((1.0 / 3.0) * comp * idz - idz) - D22S * inS * (-1.0 / 3.0 * comp * idz + idz)) * idz
           - (-D33E * inE * idx - D33W * inW * idx) * idx;
        vE = -D33E * inE * idxx;
        vS = D22S * inS * ((1.0 / 3.0) * comp * idz - idz) * idz;
        vN = -D22N * inN * (-1.0 / 3.0 * comp * idz + idz) * idz;
        uSW = (1.0 / 3.0) * D22S * comp * inS * idxz - D33W * inW * idxz;
        uSE = -1.0 / 3.0 * D22S * comp * inS * idxz + D33E * inE * idxz;
        uNW = -1.0 / 3.0 * D22N * comp * inN * idxz + D33W * inW * idxz;
        uNE = (1.0 / 3.0) * D22N * comp * inN * idxz - D33E * inE * idxz;
    } else {
        const ZRes r = zres_coeffs(D22S, D22N, D33W, D33E, inS, inN, inW, inE, g.dx, g.dz);
        vW = r.vW; vC = r.vC; vE = r.vE; vS = r.vS; vN = r.vN;
        uSW = r.uSW; uSE = r.uSE; uNW = r.uNW; uNE = r.uNE;
    }
    int tW = T.V(c3 - 1), tE = T.V(c3 + 1);
    if (tW == 11) vC -= vW;
    if (tE == 11) vC -= vE;
    if (a.stab == 1) {
        double drhodz = (g.rho_n[c2 + ncx] - g.rho_n[c2]) * a.one_dz;
        double vC_corr = 1.00 * a.om * a.dt * g.gz[c3] * drhodz;
        if (vC + vC_corr > 0.0) vC += vC_corr;
    }
    double pS = 0, pN = 0;
    bool pgrad = T.P(c2) != 30 && T.P(c2 + ncx) != 30;
    if (pgrad) { pS = -a.one_dz * 1e0; pN = a.one_dz * 1e0; }
    double cv = a.celvol;
    if (ASM) {
        b *= cv;
        if (T.U(c1 + nx) != 30) ra.add(a.e.eqn_u[c1 + nx], uNE * cv, T.U(c1 + nx), [&] { return g.BCu_val[c1 + nx]; });
        if (T.U(c1) != 30) ra.add(a.e.eqn_u[c1], uSE * cv, T.U(c1), [&] { return g.BCu_val[c1]; });
        if (T.U(c1 + nx - 1) != 30) ra.add(a.e.eqn_u[c1 + nx - 1], uNW * cv, T.U(c1 + nx - 1), [&] { return g.BCu_val[c1 + nx - 1]; });
        if (T.U(c1 - 1) != 30) ra.add(a.e.eqn_u[c1 - 1], uSW * cv, T.U(c1 - 1), [&] { return g.BCu_val[c1 - 1]; });
        if (tVS != 30) ra.add(a.e.eqn_v[c3 - nxvz], vS * cv, tVS, [&] { return g.BCv_val[c3 - nxvz]; });
        if (tW != 30 && tW != -12) ra.add(a.e.eqn_v[c3 - 1], vW * cv, tW, [&] { return (tW != 11 ? 1.0 : 2.0) * g.BCv_val[c3 - 1]; });
        if (tW == -12) ra.add(a.e.eqn_v[c3 + nxvz - 3], vW * cv, T.V(c3 + nxvz - 3), [&] { return g.BCv_val[c3 + nxvz - 3]; });
        ra.add(eqn, vC * cv, T.V(c3), [&] { return g.BCv_val[c3]; });
        if (tE != 30 && tE != -12) ra.add(a.e.eqn_v[c3 + 1], vE * cv, tE, [&] { return (tE != 11 ? 1.0 : 2.0) * g.BCv_val[c3 + 1]; });
        if (tE == -12) ra.add(a.e.eqn_v[c3 - nxvz + 3], vE * cv, T.V(c3 - nxvz + 3), [&] { return g.BCv_val[c3 - nxvz + 3]; });
        if (tVN != 30) ra.add(a.e.eqn_v[c3 + nxvz], vN * cv, tVN, [&] { return g.BCv_val[c3 + nxvz]; });
        if (pgrad) {
            rb.add(a.e.eqn_p[c2] - a.e.neq_mom, pS * cv, T.P(c2), [&] { return g.BCp_val[c2]; });
            rb.add(a.e.eqn_p[c2 + ncx] - a.e.neq_mom, pN * cv, T.P(c2 + ncx), [&] { return g.BCp_val[c2 + ncx]; });
        }
    } else {
        const double *u = a.u, *v = a.v, *p = a.p_mom;
        double f = vC * v[c3];
        if (pgrad) f += pS * p[c2] + pN * p[c2 + ncx];
        if (tVS != 30) f += vS * v[c3 - nxvz];
        if (tW != 30 && tW != 11 && tW != -12) f += vW * v[c3 - 1];
        if (tE != 30 && tE != 11 && tE != -12) f += vE * v[c3 + 1];
        if (tVN != 30) f += vN * v[c3 + nxvz];
        if (T.U(c1 - 1) != 30) f += uSW * u[c1 - 1];
        if (T.U(c1) != 30) f += uSE * u[c1];
        if (T.U(c1 + nx - 1) != 30) f += uNW * u[c1 + nx - 1];
        if (T.U(c1 + nx) != 30) f += uNE * u[c1 + nx];
        if (tW == 11) f += -2 * D33W * a.one_dx_dx * g.BCv_val[c3 - 1];
        if (tE == 11) f += -2 * D33E * a.one_dx_dx * g.BCv_val[c3 + 1];
        if (tW == -12) f += vW * v[c3 + nxvz - 3];
        if (tE == -12) f += vE * v[c3 - nxvz + 3];
        f -= b;
        F = f * cv;
    }
}

template <bool ASM, int MODE, class TG>
__device__ void zmom_neumann(const DevAsm &a, const TG &T, int c1, int c2, int c3, int eqn, int north, int comp, Sink<MODE> &ra,
                             Sink<MODE> &rb, double &b, double bbc_in, double &F) {
    const DevGrid &g = a.g;
    int nx = g.Nx, ncx = g.ncx, nxvz = g.nxvz;
    double etaS, etaN, etaE = g.eta_s[c1], etaW = g.eta_s[c1 - 1];
    if (!north) { etaN = g.eta_n[c2 + ncx]; etaS = etaN; }
    else { etaS = g.eta_n[c2]; etaN = etaS; }
    double uSW = 0, uSE = 0, uNW = 0, uNE = 0, vS = 0, vW = 0, vC = 0, vE = 0, vN = 0, pN = 0, pS = 0;
    double dxx = a.one_dx_dx, dzz = a.one_dz_dz, dxz = a.one_dx_dz;
    if (!north) b -= g.BCv_val[c3] * a.one_dz;
    else b += g.BCv_val[c3] * a.one_dz;
    bool us = T.U(c1 - 1) != 30 && T.U(c1) != 30;
    bool un = T.U(c1 + nx - 1) != 30 && T.U(c1 + nx) != 30;
    if (us) {
        uSW = dxz * etaW - comp * 2.0 / 3.0 * etaS * dxz;
        uSE = -dxz * etaE + comp * 2.0 / 3.0 * etaS * dxz;
    }
    if (un) {
        uNW = -dxz * etaW + comp * 2.0 / 3.0 * etaN * dxz;
        uNE = dxz * etaE - comp * 2.0 / 3.0 * etaN * dxz;
    }
    if (!north) {
        if (T.V(c3 + nxvz) != 30) {
            vC = -2.0 * dzz * (etaN) + comp * 2.0 / 3.0 * etaS * dzz;
            vN = 2.0 * dzz * etaN - comp * 2.0 / 3.0 * etaN * dzz;
        }
    } else {
        if (T.V(c3 - nxvz) != 30) {
            vS = 2.0 * dzz * etaS - comp * 2.0 / 3.0 * etaS * dzz;
            vC = -2.0 * dzz * (etaS) + comp * 2.0 / 3.0 * etaS * dzz;
        }
    }
    int tW = T.V(c3 - 1), tE = T.V(c3 + 1);
    if (tW != 30 && tE != 30) {
        if (tW != 13) { vW = dxx * etaW; vC += -dxx * etaW; }
        if (tE != 13) { vE = dxx * etaE; vC += -dxx * etaE; }
    }
    if (tW == 30 && tE != 30) {
        if (tE != 13) vE = dxx * etaE;
        if (tE != 13) vC += -dxx * etaE;
    }
    if (tW != 30 && tE == 30) {
        if (tW != 13) vW = dxx * etaW;
        if (tW != 13) vC += -dxx * etaW;
    }
    if (tW == 11) vC += -dxx * etaW;
    if (tE == 11) vC += -dxx * etaE;
    if (a.stab == 1) {
        /* density-gradient stabilisation with the model's scalar gz */
        double drhodz = (g.rho_n[c2 + ncx] - g.rho_n[c2]) * a.one_dz;
        if (!north) vC += 1.00 * a.om * a.dt * a.gz_model * drhodz;
        else vC += -1.00 * a.om * a.dt * a.gz_model * drhodz;
    }
    if (!north) { if (T.P(c2 + ncx) != 30) pN = -a.one_dz; }
    else { if (T.P(c2) != 30) pS = a.one_dz; }
    uSW = -uSW; uSE = -uSE; uNW = -uNW; uNE = -uNE; vS = -vS; vW = -vW; vC = -vC; vE = -vE; vN = -vN; pN = -pN; pS = -pS;
    double cv = a.celvol;
    if (ASM) {
        b *= cv;
        if (us) {
            ra.add(a.e.eqn_u[c1 - 1], uSW * cv, T.U(c1 - 1), [&] { return g.BCu_val[c1 - 1]; });
            ra.add(a.e.eqn_u[c1], uSE * cv, T.U(c1), [&] { return g.BCu_val[c1]; });
        }
        if (un) {
            ra.add(a.e.eqn_u[c1 + nx - 1], uNW * cv, T.U(c1 + nx - 1), [&] { return g.BCu_val[c1 + nx - 1]; });
            ra.add(a.e.eqn_u[c1 + nx], uNE * cv, T.U(c1 + nx), [&] { return g.BCu_val[c1 + nx]; });
        }
        if (north && T.V(c3 - nxvz) != 30) ra.add(a.e.eqn_v[c3 - nxvz], vS * cv, T.V(c3 - nxvz), [&] { return g.BCv_val[c3 - nxvz]; });
        if (tW != 30) ra.add(a.e.eqn_v[c3 - 1], vW * cv, tW, [&] { return (tW != 11 ? 1.0 : 2.0) * g.BCv_val[c3 - 1]; });
        ra.add(eqn, vC * cv, T.V(c3), [&] { return g.BCv_val[c3]; });
        if (tE != 30) ra.add(a.e.eqn_v[c3 + 1], vE * cv, tE, [&] { return (tE != 11 ? 1.0 : 2.0) * g.BCv_val[c3 + 1]; });
        if (!north && T.V(c3 + nxvz) != 30) ra.add(a.e.eqn_v[c3 + nxvz], vN * cv, T.V(c3 + nxvz), [&] { return g.BCv_val[c3 + nxvz]; });
        if (!north) {
            if (T.P(c2 + ncx) != 30) rb.add(a.e.eqn_p[c2 + ncx] - a.e.neq_mom, pN * cv, T.P(c2 + ncx), [&] { return g.BCp_val[c2 + ncx]; });
        } else {
            if (T.P(c2) != 30) rb.add(a.e.eqn_p[c2] - a.e.neq_mom, pS * cv, T.P(c2), [&] { return g.BCp_val[c2]; });
        }
    } else {
        const double *u = a.u, *v = a.v, *p = a.p_mom;
        double f = -(b + bbc_in / cv);
        f += vC * v[c3];
        if (tW != 30 && tW != 11) f += vW * v[c3 - 1];
        if (!north && T.V(c3 + nxvz) != 30) f += vN * v[c3 + nxvz];
        if (north && T.V(c3 - nxvz) != 30) f += vS * v[c3 - nxvz];
        if (tE != 30 && tE != 11) f += vE * v[c3 + 1];
        if (us) {
            int t0 = T.U(c1 - 1), t1 = T.U(c1);
            if (t0 != 11 && t0 != 0) f += uSW * u[c1 - 1];
            if (t1 != 11 && t1 != 0) f += uSE * u[c1];
        }
        if (un) {
            int t0 = T.U(c1 + nx - 1), t1 = T.U(c1 + nx);
            if (t0 != 11 && t0 != 0) f += uNW * u[c1 + nx - 1];
            if (t1 != 11 && t1 != 0) f += uNE * u[c1 + nx];
        }
        if (!north) { if (T.P(c2 + ncx) != 30) f += pN * p[c2 + ncx]; }
        else {
            /* the reference reads the pressure one row below (c2 - ncx) here */
            if (T.P(c2 - ncx) != 30) f += pS * p[c2 - ncx];
        }
        F = f * cv;
    }
}

/* ------------------------------------------------------------------ */
/* Jacobian X rows                                                      */
/* ------------------------------------------------------------------ */
/* u slots [dj+1][di+1] around the row's Vx node; v slots [b+2][a+1]
 * around vz(k, l); p slots [b+1][a] for centroid (k-1+a, l-1+b). */
struct XAcc { double u[3][3]; double v[4][4]; double p[3][2]; };

/* stencil factors of the Jacobian rows, one division each per row:
 * (1 - cmp/3)/dx, (1 - cmp/3)/dz, (cmp/3)/dx, (cmp/3)/dz, 1/dx, 1/dz */
/* Averaging weight of the Jacobian rows: the count w of in-domain
 * neighbours (a sum of four 0/1 flags) becomes 1/w when w > 1
 * (StokesAssemblyDecoupled.c:3157-3160); the quotients are the constants
 * 1/2, 1/3, 1/4, so no division is needed. */
__device__ __forceinline__ double inv_weight(double w) {
    return w > 3.5 ? 0.25 : (w > 2.5 ? 1.0 / 3.0 : (w > 1.5 ? 0.5 : w));
}

struct JK { double e1x, e1z, e3x, e3z, idx, idz; };
/* the per-grid factors (1 - cmp/3)/dx, (1 - cmp/3)/dz, (cmp/3)/dx, (cmp/3)/dz,
 * 1/dx, 1/dz with cmp = 1, computed on the host */
__device__ __forceinline__ JK make_jk(const DevAsm &a) {
    return JK{a.jk_e1x, a.jk_e1z, a.jk_e3x, a.jk_e3z, a.one_dx, a.one_dz};
}

__device__ __forceinline__ void xa_exx(XAcc &c, int a, int b, double w, const JK &K) {
    double f = w * K.e1x, h = w * K.e3z;
    c.u[b + 1][a + 1] += f; c.u[b + 1][a] -= f;
    c.v[b + 2][a + 1] -= h; c.v[b + 1][a + 1] += h;
}
__device__ __forceinline__ void xa_ezz(XAcc &c, int a, int b, double w, const JK &K) {
    double f = w * K.e1z, h = w * K.e3x;
    c.v[b + 2][a + 1] += f; c.v[b + 1][a + 1] -= f;
    c.u[b + 1][a + 1] -= h; c.u[b + 1][a] += h;
}
__device__ __forceinline__ void xa_gxz(XAcc &c, int a, int b, double w, const JK &K) {
    const double wz = w * K.idz, wx = w * K.idx;
    c.u[b + 2][a + 1] += wz; c.u[b + 1][a + 1] -= wz;
    c.v[b + 2][a + 2] += wx; c.v[b + 2][a + 1] -= wx;
}

template <bool ASM, int MODE, class TG>
__device__ void xjac_row(const DevAsm &a, const TG &T, int c1, int c2, int c3, int eqn, int k, int l,
                         Sink<MODE> &ra, Sink<MODE> &rb, double &b, double &F) {
    const DevGrid &g = a.g;
    int nx = g.Nx, ncx = g.ncx, nxvz = g.nxvz;
    int iVxC = c1, iVxW = iVxC - 1, iVxE = iVxC + 1, iVxS = iVxC - nx, iVxN = iVxC + nx;
    int iVxSW = iVxS - 1, iVxSE = iVxS + 1, iVxNW = iVxN - 1, iVxNE = iVxN + 1;
    int iVzSW = c3 - nxvz, iVzSE = c3 - nxvz + 1, iVzNW = c3, iVzNE = c3 + 1;
    int iVzSWW = iVzSW - 1, iVzSEE = iVzSE + 1, iVzNWW = iVzNW - 1, iVzNEE = iVzNE + 1;
    int iVzNNW = iVzNW + nxvz, iVzSSW = iVzSW - nxvz, iVzNNE = iVzNE + nxvz, iVzSSE = iVzSE - nxvz;
    int iPrW = c2, iPrE = c2 + 1, ixyN = c1, ixyS = c1 - nx;
    int ixySW = ixyS - 1, ixySE = ixyS + 1, ixyNW = ixyN - 1, ixyNE = ixyN + 1;
    int iPrSW = iPrW - ncx, iPrSE = iPrE - ncx, iPrNW = iPrW + ncx, iPrNE = iPrE + ncx;
    if (T.V(iVzSWW) == -12) iVzSWW = iVzSW + (nx - 2);
    if (T.V(iVzNWW) == -12) iVzNWW = iVzNW + (nx - 2);
    if (T.V(iVzSEE) == -12) iVzSEE = iVzSE - (nx - 2);
    if (T.V(iVzNEE) == -12) iVzNEE = iVzNE - (nx - 2);
    if (T.U(iVxC) == -2) {
        iVxW = c1 + nx - 2; iPrW = c2 + ncx; iVzSW = c3 - 2; iVzNW = c3 + nxvz - 2;
        iPrNW = iPrW + ncx; iPrSW = iPrW - ncx;
        iVxSW = iVxW - nx; iVxNW = iVxW + nx;
        iVzNNW = iVzNW + nxvz; iVzSSW = iVzSW - nxvz;
        iVzSWW = iVzSW - 1; iVzNWW = iVzNW - 1;
    }
    double inW = T.P(iPrW) == -1 ? 1.0 : 0.0, inE = T.P(iPrE) == -1 ? 1.0 : 0.0;
    double inS = (T.G(ixyS) != 30 && T.U(iVxS) != 13) ? 1.0 : 0.0;
    double inN = (T.G(ixyN) != 30 && T.U(iVxN) != 13) ? 1.0 : 0.0;
    double inSWc = 0, inSEc = 0, inNWc = 0, inNEc = 0, inSWv = 0, inSEv = 0, inNWv = 0, inNEv = 0;
    int nzvx = a.Nz_model + 1, nz = a.Nz_model;
    if (l > 1 || (l == 1 && T.U(iVxS) == 11)) {
        if (T.P(iPrSW) == -1) inSWc = 1.0;
        if (T.P(iPrSE) == -1) inSEc = 1.0;
    }
    if (l < nzvx - 2 || (l == nzvx - 2 && T.U(iVxN) == 11)) {
        if (T.P(iPrNW) == -1) inNWc = 1.0;
        if (T.P(iPrNE) == -1) inNEc = 1.0;
    }
    if ((k > 0) || (k == 0 && (T.V(iVzSW) == -1 || T.V(iVzSW) == 0))) {
        if (T.G(ixySW) != 30) inSWv = 1.0;
        if (T.G(ixyNW) != 30) inNWv = 1.0;
    }
    if ((k < nx - 1) || (k == nx - 1 && (T.V(iVzSE) == -1 || T.V(iVzSE) == 0))) {
        if (T.G(ixySE) != 30) inSEv = 1.0;
        if (T.G(ixyNE) != 30) inNEv = 1.0;
    }
    double wE = inN + inS + inNEv + inSEv, wW = inN + inS + inNWv + inSWv;
    double wS = inW + inE + inSWc + inSEc, wN = inW + inE + inNWc + inNEc;
    wW = inv_weight(wW); wE = inv_weight(wE); wS = inv_weight(wS); wN = inv_weight(wN);

    double uSW = 0, uS = 0, uSE = 0, uW = 0, uC = 0, uE = 0, uNW = 0, uN = 0, uNE = 0;
    double vSSW = 0, vSSE = 0, vSWW = 0, vSW = 0, vSE = 0, vSEE = 0, vNWW = 0, vNW = 0, vNE = 0, vNEE = 0, vNNW = 0, vNNE = 0;
    double pSW = 0, pSE = 0, pW = 0, pE = 0, pNW = 0, pNE = 0;
    if (MODE == SINK_VALUES) {
        const JK K = make_jk(a);
        double D11E = g.D11_n[iPrE], D12E = g.D12_n[iPrE], D13E = g.D13_n[iPrE], D14E = g.D14_n[iPrE];
        double D11W = g.D11_n[iPrW], D12W = g.D12_n[iPrW], D13W = g.D13_n[iPrW], D14W = g.D14_n[iPrW];
        double D31N = g.D31_s[ixyN], D32N = g.D32_s[ixyN], D33N = g.D33_s[ixyN], D34N = g.D34_s[ixyN];
        double D31S = g.D31_s[ixyS], D32S = g.D32_s[ixyS], D33S = g.D33_s[ixyS], D34S = g.D34_s[ixyS];
        XAcc c;
#pragma unroll
        for (int i = 0; i < 3; i++) {
#pragma unroll
            for (int j = 0; j < 3; j++) c.u[i][j] = 0.0;
#pragma unroll
            for (int j = 0; j < 2; j++) c.p[i][j] = 0.0;
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) c.v[i][j] = 0.0;
        /* normal stress at centroids W (aa=0) and E (aa=1) */
#pragma unroll
        for (int aa = 0; aa < 2; aa++) {
            double f = aa == 0 ? inW * K.idx : -inE * K.idx;
            double D1 = aa == 0 ? D11W : D11E, D2 = aa == 0 ? D12W : D12E, D3 = aa == 0 ? D13W : D13E, D4 = aa == 0 ? D14W : D14E;
            double w = aa == 0 ? wW : wE;
            xa_exx(c, aa, 0, f * D1, K);
            xa_ezz(c, aa, 0, f * D2, K);
            double fSo = aa == 0 ? inSWv : inSEv, fNo = aa == 0 ? inNWv : inNEv;
            xa_gxz(c, 0, -1, f * D3 * w * inS, K);
            xa_gxz(c, 0, 0, f * D3 * w * inN, K);
            xa_gxz(c, aa == 0 ? -1 : 1, -1, f * D3 * w * fSo, K);
            xa_gxz(c, aa == 0 ? -1 : 1, 0, f * D3 * w * fNo, K);
            c.p[1][aa] += f * D4;
        }
        /* shear stress at vertices S (bb=0) and N (bb=1) */
#pragma unroll
        for (int bb = 0; bb < 2; bb++) {
            int bv = bb == 0 ? -1 : 0;
            double f = bb == 0 ? inS * K.idz : -inN * K.idz;
            double D1 = bb == 0 ? D31S : D31N, D2 = bb == 0 ? D32S : D32N, D3 = bb == 0 ? D33S : D33N, D4 = bb == 0 ? D34S : D34N;
            double w = bb == 0 ? wS : wN;
            int cb = bb == 0 ? -1 : 1;
            double fl[4] = {inW, inE, bb == 0 ? inSWc : inNWc, bb == 0 ? inSEc : inNEc};
            const int ca[4] = {0, 1, 0, 1};
            int cr[4] = {0, 0, cb, cb};
#pragma unroll
            for (int q = 0; q < 4; q++) {
                double wq = w * fl[q];
                xa_exx(c, ca[q], cr[q], f * D1 * wq, K);
                xa_ezz(c, ca[q], cr[q], f * D2 * wq, K);
                c.p[cr[q] + 1][ca[q]] += f * D4 * wq;
            }
            xa_gxz(c, 0, bv, f * D3, K);
        }
        c.p[1][0] += -inW * K.idx;
        c.p[1][1] += inE * K.idx;
        uSW = c.u[0][0]; uS = c.u[0][1]; uSE = c.u[0][2]; uW = c.u[1][0]; uC = c.u[1][1]; uE = c.u[1][2];
        uNW = c.u[2][0]; uN = c.u[2][1]; uNE = c.u[2][2];
        vSSW = c.v[0][1]; vSSE = c.v[0][2]; vSWW = c.v[1][0]; vSW = c.v[1][1]; vSE = c.v[1][2]; vSEE = c.v[1][3];
        vNWW = c.v[2][0]; vNW = c.v[2][1]; vNE = c.v[2][2]; vNEE = c.v[2][3]; vNNW = c.v[3][1]; vNNE = c.v[3][2];
        pSW = c.p[0][0]; pSE = c.p[0][1]; pW = c.p[1][0]; pE = c.p[1][1]; pNW = c.p[2][0]; pNE = c.p[2][1];
        if (a.stab == 1) {
            double drhodx = (g.rho_n[c2 + 1] - g.rho_n[c2]) * a.one_dx;
            double uC_corr = 1.00 * a.om * a.dt * g.gx[c1] * drhodx;
            if (uC + uC_corr > 0.0) uC += uC_corr;
        }
        if (T.U(iVxS) == 11) uC -= uS;
        if (T.U(iVxN) == 11) uC -= uN;
        if (T.U(iVxSW) == 11) uW -= uSW;
        if (T.U(iVxSE) == 11) uE -= uSE;
        if (T.U(iVxNW) == 11) uW -= uNW;
        if (T.U(iVxNE) == 11) uE -= uNE;
        if (T.V(iVzNWW) == 11) vNW -= vNWW;
        if (T.V(iVzNEE) == 11) vNE -= vNEE;
        if (T.V(iVzSWW) == 11) vSW -= vSWW;
        if (T.V(iVzSEE) == 11) vSE -= vSEE;
    }
    double cv = a.celvol;
    if (ASM) {
        b *= cv;
        const int *eu = a.e.eqn_u, *ev = a.e.eqn_v, *ep = a.e.eqn_p;
        const double *uv = g.BCu_val, *vv = g.BCv_val, *pv = g.BCp_val;
#define UADD11(idx, coef) \
    if (T.U(idx) != 30) ra.add(eu[idx], (coef)*cv, T.U(idx), [&] { return (T.U(idx) != 11 ? 1.0 : 2.0) * uv[idx]; });
        UADD11(iVxSW, uSW)
        UADD11(iVxS, uS)
        UADD11(iVxSE, uSE)
        if (T.U(iVxW) != 30) ra.add(eu[iVxW], uW * cv, T.U(iVxW), [&] { return uv[iVxW]; });
        ra.add(eqn, uC * cv, T.U(iVxC), [&] { return uv[iVxC]; });
        if (T.U(iVxE) != 30) ra.add(eu[iVxE], uE * cv, T.U(iVxE), [&] { return uv[iVxE]; });
        UADD11(iVxNW, uNW)
        UADD11(iVxN, uN)
        UADD11(iVxNE, uNE)
#undef UADD11
#define VADD(idx, coef) ra.add(ev[idx], (coef)*cv, T.V(idx), [&] { return vv[idx]; })
        if (l > 1 && T.V(iVzSSW) != 30) VADD(iVzSSW, vSSW);
        if (l > 1 && T.V(iVzSSE) != 30) VADD(iVzSSE, vSSE);
        if ((k > 1) || ((k == 0 || k == 1) && T.V(iVzSWW) == -1))
            if (T.V(iVzSWW) != 30) VADD(iVzSWW, vSWW);
        if (T.V(iVzSW) != 30) VADD(iVzSW, vSW);
        if (T.V(iVzSE) != 30) VADD(iVzSE, vSE);
        if ((k < nx - 2) || ((k == nx - 2 || k == nx - 1) && T.V(iVzSEE) == -1))
            if (T.V(iVzSEE) != 30) VADD(iVzSEE, vSEE);
        if ((k > 1) || ((k == 0 || k == 1) && T.V(iVzNWW) == -1))
            if (T.V(iVzNWW) != 30) VADD(iVzNWW, vNWW);
        if (T.V(iVzNW) != 30) VADD(iVzNW, vNW);
        if (T.V(iVzNE) != 30) VADD(iVzNE, vNE);
        if ((k < nx - 2) || ((k == nx - 2 || k == nx - 1) && T.V(iVzNEE) == -1))
            if (T.V(iVzNEE) != 30) VADD(iVzNEE, vNEE);
        if (l < nz - 1 && T.V(iVzNNW) != 30) VADD(iVzNNW, vNNW);
        if (l < nz - 1 && T.V(iVzNNE) != 30) VADD(iVzNNE, vNNE);
#undef VADD
#define PADD(idx, coef) rb.add(ep[idx] - a.e.neq_mom, (coef)*cv, T.P(idx), [&] { return pv[idx]; })
        if (l > 1) {
            if (T.P(iPrSW) != 30) PADD(iPrSW, pSW);
            if (T.P(iPrSE) != 30) PADD(iPrSE, pSE);
        }
        if (T.P(iPrE) != 30 && T.P(c2) != 30) { PADD(iPrW, pW); PADD(iPrE, pE); }
        if (l < nz - 1) {
            if (T.P(iPrNW) != 30) PADD(iPrNW, pNW);
            if (T.P(iPrNE) != 30) PADD(iPrNE, pNE);
        }
#undef PADD
    } else {
        double f = 0.0;
        f += (g.sxxd[iPrE] - g.sxxd[iPrW]) / g.dx;
        f -= (g.p_in[iPrE] - g.p_in[iPrW]) / g.dx;
        f += (g.sxz[ixyN] - g.sxz[ixyS]) / g.dz;
        f *= -1.0;
        f -= b;
        F = f * cv;
    }
}

/* ------------------------------------------------------------------ */
/* Jacobian Z rows                                                      */
/* ------------------------------------------------------------------ */
/* v slots [dj+1][di+1] around the row's Vz node; u slots [b+1][a+2]
 * around u(k, l); p slots [b][a+1] for centroid (k-1+a, l-1+b). */
struct ZAcc { double v[3][3]; double u[4][4]; double p[2][3]; };

__device__ __forceinline__ void za_exx(ZAcc &c, int a, int b, double w, const JK &K) {
    double f = w * K.e1x, h = w * K.e3z;
    c.u[b + 1][a + 2] += f; c.u[b + 1][a + 1] -= f;
    c.v[b + 1][a + 1] -= h; c.v[b][a + 1] += h;
}
__device__ __forceinline__ void za_ezz(ZAcc &c, int a, int b, double w, const JK &K) {
    double f = w * K.e1z, h = w * K.e3x;
    c.v[b + 1][a + 1] += f; c.v[b][a + 1] -= f;
    c.u[b + 1][a + 2] -= h; c.u[b + 1][a + 1] += h;
}
__device__ __forceinline__ void za_gxz(ZAcc &c, int a, int b, double w, const JK &K) {
    const double wz = w * K.idz, wx = w * K.idx;
    c.u[b + 2][a + 1] += wz; c.u[b + 1][a + 1] -= wz;
    c.v[b + 1][a + 1] += wx; c.v[b + 1][a] -= wx;
}

template <bool ASM, int MODE, class TG>
__device__ void zjac_row(const DevAsm &a, const TG &T, int c1, int c2, int c3, int eqn, int k, int l,
                         Sink<MODE> &ra, Sink<MODE> &rb, double &b, double &F) {
    const DevGrid &g = a.g;
    int nx = g.Nx, ncx = g.ncx, nxvz = g.nxvz;
    int periodix = a.periodic;
    int iVzC = c3, iVzW = iVzC - 1, iVzE = iVzC + 1, iVzS = c3 - nxvz, iVzN = c3 + nxvz;
    int iVzSW = iVzS - 1, iVzSE = iVzS + 1, iVzNW = iVzN - 1, iVzNE = iVzN + 1;
    int iVxNW = c1 + nx - 1, iVxNE = c1 + nx, iVxSW = c1 - 1, iVxSE = c1;
    int iVxNWW = iVxNW - 1, iVxNEE = iVxNE + 1, iVxSWW = iVxSW - 1, iVxSEE = iVxSE + 1;
    int iVxNNW = iVxNW + nx, iVxNNE = iVxNE + nx, iVxSSW = iVxSW - nx, iVxSSE = iVxSE - nx;
    int iPrS = c2, iPrSW = iPrS - 1, iPrSE = iPrS + 1, iPrN = c2 + ncx, iPrNW = iPrN - 1, iPrNE = iPrN + 1;
    int ixyW = c1 - 1, ixySW = ixyW - nx, ixyNW = ixyW + nx, ixyE = c1, ixySE = ixyE - nx, ixyNE = ixyE + nx;
    if (k == 1 && T.V(iVzW) == -12) {
        iVxNWW = iVxNW + (nx - 2); iVxSWW = iVxSW + (nx - 2);
        iPrNW = iPrN + (ncx - 1); iPrSW = iPrS + (ncx - 1);
        iVzW = iVzC + (nx - 2); iVzSW = iVzW - nxvz; iVzNW = iVzW + nxvz;
    }
    if (k == nx - 1 && T.V(iVzE) == -12) {
        iVxNEE = iVxNE - (nx - 2); iVxSEE = iVxSE - (nx - 2);
        iPrNE = iPrN - (ncx - 1); iPrSE = iPrS - (ncx - 1);
        iVzE = iVzC - (nx - 2); iVzNE = iVzE + nxvz; iVzSE = iVzE - nxvz;
    }
    double inS = T.P(iPrS) == -1 ? 1.0 : 0.0, inN = T.P(iPrN) == -1 ? 1.0 : 0.0;
    double inW = (T.G(ixyW) != 30 && T.V(iVzW) != 13) ? 1.0 : 0.0;
    double inE = (T.G(ixyE) != 30 && T.V(iVzE) != 13) ? 1.0 : 0.0;
    double inSWc = 0, inSEc = 0, inNWc = 0, inNEc = 0, inSWv = 0, inSEv = 0, inNWv = 0, inNEv = 0;
    int nz = a.Nz_model;
    if ((k > 1) || (k == 1 && T.V(iVzW) == -1)) {
        if (T.P(iPrSW) == -1) inSWc = 1.0;
        if (T.P(iPrNW) == -1) inNWc = 1.0;
    }
    if ((k < nxvz - 2) || (k == nxvz - 2 && T.V(iVzE) == -1)) {
        if (T.P(iPrSE) == -1) inSEc = 1.0;
        if (T.P(iPrNE) == -1) inNEc = 1.0;
    }
    if (l > 0) {
        if (T.G(ixySW) != 30) inSWv = 1.0;
        if (T.G(ixySE) != 30) inSEv = 1.0;
    }
    if (l < nz - 1) {
        if (T.G(ixyNW) != 30) inNWv = 1.0;
        if (T.G(ixyNE) != 30) inNEv = 1.0;
    }
    double wE = inN + inS + inNEc + inSEc, wW = inN + inS + inNWc + inSWc;
    double wS = inW + inE + inSWv + inSEv, wN = inW + inE + inNWv + inNEv;
    wW = inv_weight(wW); wE = inv_weight(wE); wS = inv_weight(wS); wN = inv_weight(wN);

    double vSW = 0, vS = 0, vSE = 0, vW = 0, vC = 0, vE = 0, vNW = 0, vN = 0, vNE = 0;
    double uSSW = 0, uSSE = 0, uSWW = 0, uSW = 0, uSE = 0, uSEE = 0, uNWW = 0, uNW = 0, uNE = 0, uNEE = 0, uNNW = 0, uNNE = 0;
    double pSW = 0, pS = 0, pSE = 0, pNW = 0, pN = 0, pNE = 0;
    if (MODE == SINK_VALUES) {
        const JK K = make_jk(a);
        double D31W = g.D31_s[ixyW], D32W = g.D32_s[ixyW], D33W = g.D33_s[ixyW], D34W = g.D34_s[ixyW];
        double D31E = g.D31_s[ixyE], D32E = g.D32_s[ixyE], D33E = g.D33_s[ixyE], D34E = g.D34_s[ixyE];
        double D21S = g.D21_n[iPrS], D22S = g.D22_n[iPrS], D23S = g.D23_n[iPrS], D24S = g.D24_n[iPrS];
        double D21N = g.D21_n[iPrN], D22N = g.D22_n[iPrN], D23N = g.D23_n[iPrN], D24N = g.D24_n[iPrN];
        ZAcc c;
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) c.v[i][j] = 0.0;
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) c.u[i][j] = 0.0;
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 3; j++) c.p[i][j] = 0.0;
        /* normal stress at centroids S (bb=0) and N (bb=1) */
#pragma unroll
        for (int bb = 0; bb < 2; bb++) {
            double f = bb == 0 ? inS * K.idz : -inN * K.idz;
            double D1 = bb == 0 ? D21S : D21N, D2 = bb == 0 ? D22S : D22N, D3 = bb == 0 ? D23S : D23N, D4 = bb == 0 ? D24S : D24N;
            double w = bb == 0 ? wS : wN;
            za_exx(c, 0, bb, f * D1, K);
            za_ezz(c, 0, bb, f * D2, K);
            int vb = bb == 0 ? -1 : 1;
            double fo_w = bb == 0 ? inSWv : inNWv, fo_e = bb == 0 ? inSEv : inNEv;
            za_gxz(c, 0, 0, f * D3 * w * inW, K);
            za_gxz(c, 1, 0, f * D3 * w * inE, K);
            za_gxz(c, 0, vb, f * D3 * w * fo_w, K);
            za_gxz(c, 1, vb, f * D3 * w * fo_e, K);
            c.p[bb][1] += f * D4;
        }
        /* shear stress at vertices W (aa=0) and E (aa=1) */
#pragma unroll
        for (int aa = 0; aa < 2; aa++) {
            double f = aa == 0 ? inW * K.idx : -inE * K.idx;
            double D1 = aa == 0 ? D31W : D31E, D2 = aa == 0 ? D32W : D32E, D3 = aa == 0 ? D33W : D33E, D4 = aa == 0 ? D34W : D34E;
            double w = aa == 0 ? wW : wE;
            int co = aa == 0 ? -1 : 1;
            double fl[4] = {inS, inN, aa == 0 ? inSWc : inSEc, aa == 0 ? inNWc : inNEc};
            int ca[4] = {0, 0, co, co};
            const int cb[4] = {0, 1, 0, 1};
#pragma unroll
            for (int q = 0; q < 4; q++) {
                double wq = w * fl[q];
                za_exx(c, ca[q], cb[q], f * D1 * wq, K);
                za_ezz(c, ca[q], cb[q], f * D2 * wq, K);
                c.p[cb[q]][ca[q] + 1] += f * D4 * wq;
            }
            za_gxz(c, aa, 0, f * D3, K);
        }
        c.p[0][1] += -inS * K.idz;
        c.p[1][1] += inN * K.idz;
        vSW = c.v[0][0]; vS = c.v[0][1]; vSE = c.v[0][2]; vW = c.v[1][0]; vC = c.v[1][1]; vE = c.v[1][2];
        vNW = c.v[2][0]; vN = c.v[2][1]; vNE = c.v[2][2];
        uSSW = c.u[0][1]; uSSE = c.u[0][2]; uSWW = c.u[1][0]; uSW = c.u[1][1]; uSE = c.u[1][2]; uSEE = c.u[1][3];
        uNWW = c.u[2][0]; uNW = c.u[2][1]; uNE = c.u[2][2]; uNEE = c.u[2][3]; uNNW = c.u[3][1]; uNNE = c.u[3][2];
        pSW = c.p[0][0]; pS = c.p[0][1]; pSE = c.p[0][2]; pNW = c.p[1][0]; pN = c.p[1][1]; pNE = c.p[1][2];
        if (a.stab == 1) {
            double drhodz = (g.rho_n[c2 + ncx] - g.rho_n[c2]) * a.one_dz;
            double vC_corr = 1.00 * a.om * a.dt * g.gz[c3] * drhodz;
            if (vC + vC_corr > 0.0) vC += vC_corr;
        }
        if (T.V(iVzW) == 11) vC -= vW;
        if (T.V(iVzE) == 11) vC -= vE;
        if (T.V(iVzSW) == 11) vW -= vSW;
        if (T.V(iVzSE) == 11) vE -= vSE;
        if (T.V(iVzNW) == 11) vW -= vNW;
        if (T.V(iVzNE) == 11) vE -= vNE;
        if (T.U(iVxNNW) == 11) uNW -= uNNW;
        if (T.U(iVxNNE) == 11) uNE -= uNNE;
        if (T.U(iVxSSW) == 11) uSW -= uSSW;
        if (T.U(iVxSSE) == 11) uSE -= uSSE;
    }
    double cv = a.celvol;
    if (ASM) {
        b *= cv;
        const int *eu = a.e.eqn_u, *ev = a.e.eqn_v, *ep = a.e.eqn_p;
        const double *uv = g.BCu_val, *vv = g.BCv_val, *pv = g.BCp_val;
#define UADD(idx, coef) ra.add(eu[idx], (coef)*cv, T.U(idx), [&] { return uv[idx]; })
#define VADD(idx, coef) ra.add(ev[idx], (coef)*cv, T.V(idx), [&] { return vv[idx]; })
        if (T.U(iVxSSW) != 30) UADD(iVxSSW, uSSW);
        if (T.U(iVxSSE) != 30) UADD(iVxSSE, uSSE);
        if ((k > 1) || (k == 1 && T.U(iVxSWW) == -1))
            if (T.U(iVxSWW) != 30) UADD(iVxSWW, uSWW);
        if (T.U(iVxSW) != 30) UADD(iVxSW, uSW);
        if (T.U(iVxSE) != 30) UADD(iVxSE, uSE);
        if ((k < nx - 1) || (k == nx - 1 && T.U(iVxSEE) == -1))
            if (T.U(c1 + 1) != 30) UADD(iVxSEE, uSEE);
        if ((k > 1) || (k == 1 && T.U(iVxNWW) == -1))
            if (T.U(c1 + nx - 2) != 30) UADD(iVxNWW, uNWW);
        if (T.U(iVxNW) != 30) UADD(iVxNW, uNW);
        if (T.U(iVxNE) != 30) UADD(iVxNE, uNE);
        if ((k < nx - 1) || (k == nx - 1 && T.U(iVxNEE) == -1))
            if (T.U(iVxNEE) != 30) UADD(iVxNEE, uNEE);
        if (T.U(iVxNNW) != 30) UADD(iVxNNW, uNNW);
        if (T.U(iVxNNE) != 30) UADD(iVxNNE, uNNE);
        if (T.V(iVzSW) == -1) VADD(iVzSW, vSW);
        if (T.V(iVzS) != 30) VADD(iVzS, vS);
        if (T.V(iVzSE) == -1) VADD(iVzSE, vSE);
        if (T.V(iVzW) == -1) VADD(iVzW, vW);
        ra.add(eqn, vC * cv, T.V(iVzC), [&] { return vv[iVzC]; });
        if (T.V(iVzE) == -1) VADD(iVzE, vE);
        if (T.V(iVzNW) == -1) VADD(iVzNW, vNW);
        if (T.V(iVzN) != 30) VADD(iVzN, vN);
        if (T.V(iVzNE) == -1) VADD(iVzNE, vNE);
#undef UADD
#undef VADD
#define PADD(idx, coef, vidx) rb.add(ep[idx] - a.e.neq_mom, (coef)*cv, T.P(idx), [&] { return pv[vidx]; })
        if (k > 1 || (k == 1 && periodix == 1))
            if (T.P(iPrSW) != 30) PADD(iPrSW, pSW, iPrSW);
        if (T.P(iPrS) != 30 && T.P(iPrN) != 30) PADD(iPrS, pS, iPrS);
        if (k < nx - 1 || (k == nx - 1 && periodix == 1))
            if (T.P(iPrSE) != 30) PADD(iPrSE, pSE, iPrSE);
        if (k > 1 || (k == 1 && periodix == 1))
            if (T.P(iPrNW) != 30) PADD(iPrNW, pNW, iPrNW);
        if (T.P(iPrS) != 30 && T.P(iPrN) != 30) PADD(iPrN, pN, c2 + ncx);
        if (k < nx - 1 || (k == nx - 1 && periodix == 1))
            if (T.P(iPrNE) != 30) PADD(iPrNE, pNE, iPrNE);
#undef PADD
    } else {
        double f = 0.0;
        f += (g.szzd[iPrN] - g.szzd[iPrS]) / g.dz;
        f -= (g.p_in[iPrN] - g.p_in[iPrS]) / g.dz;
        f += (g.sxz[ixyE] - g.sxz[ixyW]) / g.dx;
        f *= -1.0;
        f -= b;
        F = f * cv;
    }
}

/* ------------------------------------------------------------------ */
/* row dispatch                                                         */
/* ------------------------------------------------------------------ */

/* One momentum row: which stencil applies (StokesAssemblyDecoupled.c:1691-1729,
 * 1763-1800, 3952-4060). */
template <bool ASM, int MODE, class TG>
__device__ void momentum_row(int kind, const DevAsm &a, const TG &T, int eqn, int node, Sink<MODE> &ra, Sink<MODE> &rb,
                             double &b, double bbc_in, double &F) {
    const DevGrid &g = a.g;
    int nx = g.Nx, ncx = g.ncx, nxvz = g.nxvz, nz = g.Nz, nzvx = g.nzvx;
    int nu = nx * nzvx;
    int comp_builder = kind == 1 ? 1 : a.comp_model;
    if (node < nu) {
        int c1 = node, k = c1 % nx, l = c1 / nx;
        int c2 = k - 1 + (l - 1) * ncx, c3 = k + l * nxvz;
        int t = T.U(c1);
        bool inner = l > 0 && l < nzvx - 1 && k > 0 && k < nx - 1;
        if (inner || (k == 0 && t == -2)) {
            if (kind == 0) xmom_inner<ASM, MODE>(a, T, c1, c2, c3, eqn, ra, rb, b, F);
            else xjac_row<ASM, MODE>(a, T, c1, c2, c3, eqn, k, l, ra, rb, b, F);
        }
        if (k == 0 && t == 2) xmom_neumann<ASM, MODE>(a, T, c1, c2, c3, eqn, 0, comp_builder, ra, rb, b, bbc_in, F);
        if (k == nx - 1 && t == 2) xmom_neumann<ASM, MODE>(a, T, c1, c2, c3, eqn, 1, comp_builder, ra, rb, b, bbc_in, F);
    } else {
        int c3 = node - nu, k = c3 % nxvz, l = c3 / nxvz;
        int c1 = k + l * nx, c2 = k - 1 + (l - 1) * ncx;
        int t = T.V(c3);
        bool inner = k > 0 && k < nxvz - 1 && l > 0 && l < nz - 1;
        if (inner) {
            if (kind == 0) zmom_inner<ASM, MODE>(a, T, c1, c2, c3, eqn, ra, rb, b, F);
            else zjac_row<ASM, MODE>(a, T, c1, c2, c3, eqn, k, l, ra, rb, b, F);
        }
        if (l == 0 && t == 2) zmom_neumann<ASM, MODE>(a, T, c1, c2, c3, eqn, 0, comp_builder, ra, rb, b, bbc_in, F);
        if (l == nz - 1 && t == 2) zmom_neumann<ASM, MODE>(a, T, c1, c2, c3, eqn, 1, comp_builder, ra, rb, b, bbc_in, F);
    }
}

/* right-hand side of the momentum row of node (mom_node of its equation) */
__device__ __forceinline__ double mom_rhs(const DevAsm &a, int node) {
    const int nu = a.g.Nx * a.g.nzvx;
    return node < nu ? a.g.roger_x[node] : a.g.roger_z[node - nu];
}

__device__ __forceinline__ int wave_max(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    return v;
}

/* pattern: per-row counts; the largest row length of each block goes to
 * cnt[neq] (one atomic per wave) */
__global__ void __launch_bounds__(BLK) k_count_mom(int kind, DevAsm a, int *cntA, int *cntB) {
    const int eqn = blockIdx.x * BLK + threadIdx.x;
    const int neq = a.e.neq_mom;
    int na = 0, nb = 0;
    if (eqn < neq) {
        Tags T = make_tags(a.g);
        Sink<SINK_COUNT> ra{0, nullptr, nullptr, 0.0}, rb{0, nullptr, nullptr, 0.0};
        double b = 0.0, F = 0.0;
        momentum_row<true, SINK_COUNT>(kind, a, T, eqn, a.e.mom_node[eqn], ra, rb, b, 0.0, F);
        na = ra.n;
        nb = rb.n;
        cntA[eqn] = na;
        cntB[eqn] = nb;
    }
    na = wave_max(na);
    nb = wave_max(nb);
    if ((threadIdx.x & 63) == 0) {
        atomicMax(&cntA[neq], na);
        atomicMax(&cntB[neq], nb);
    }
}

__device__ __forceinline__ void cont_geom(const DevAsm &a, int eqn, int &c1, int &c2, int &c3) {
    c2 = a.e.cont_node[eqn];
    int k = c2 % a.g.ncx, l = c2 / a.g.ncx;
    c1 = k + (l + 1) * a.g.Nx;
    c3 = k + l * a.g.nxvz + 1;
}

__global__ void __launch_bounds__(BLK) k_count_cont(DevAsm a, int *cntC) {
    const int eqn = blockIdx.x * BLK + threadIdx.x;
    const int neq = a.e.neq_cont;
    int nc = 0;
    if (eqn < neq) {
        int c1, c2, c3;
        cont_geom(a, eqn, c1, c2, c3);
        Sink<SINK_COUNT> rc{0, nullptr, nullptr, 0.0};
        double b = 0.0, F = 0.0;
        continuity_row<true, SINK_COUNT>(a, 0, c1, c2, c3, rc, b, F);
        nc = rc.n;
        cntC[eqn] = nc;
    }
    nc = wave_max(nc);
    if ((threadIdx.x & 63) == 0) atomicMax(&cntC[neq], nc);
}

__global__ void __launch_bounds__(BLK) k_pattern_mom(int kind, DevAsm a, DevBlock A, DevBlock B) {
    int eqn = blockIdx.x * BLK + threadIdx.x;
    if (eqn >= a.e.neq_mom) return;
    Tags T = make_tags(a.g);
    Sink<SINK_PATTERN> ra{0, A.J + A.Ic[eqn], nullptr, 0.0}, rb{0, B.J + B.Ic[eqn], nullptr, 0.0};
    double b = 0.0, F = 0.0;
    momentum_row<true, SINK_PATTERN>(kind, a, T, eqn, a.e.mom_node[eqn], ra, rb, b, 0.0, F);
}

__global__ void __launch_bounds__(BLK) k_pattern_cont(DevAsm a, DevBlock C) {
    int eqn = blockIdx.x * BLK + threadIdx.x;
    if (eqn >= a.e.neq_cont) return;
    int c1, c2, c3;
    cont_geom(a, eqn, c1, c2, c3);
    Sink<SINK_PATTERN> rc{0, C.J + C.Ic[eqn], nullptr, 0.0};
    double b = 0.0, F = 0.0;
    continuity_row<true, SINK_PATTERN>(a, 0, c1, c2, c3, rc, b, F);
}

/* values (Assemble = 1): A/B values, bbc, final b = rhs*celvol (+/- Neumann) + bbc.
 * Rows of one block are consecutive, so their values are one contiguous
 * range of A (and of B): each thread writes its row into LDS and the block
 * copies the range out with coalesced stores.  Needs every row length
 * within the LDS slot (CAPA, CAPB); KIND 0 = Picard, 1 = Jacobian. */
/* the continuity rows of a value pass (C and D blocks), one lane per row */
__device__ __forceinline__ void values_cont_row(const DevAsm &a, DevBlock &C, DevBlock &D, int eqn, double *dump) {
    int c1, c2, c3;
    cont_geom(a, eqn, c1, c2, c3);
    Sink<SINK_VALUES> rc{0, nullptr, C.A + C.Ic[eqn], 0.0, dump};
    double b = a.g.rhs_p[c2], F = 0.0;
    continuity_row<true, SINK_VALUES>(a, 0, c1, c2, c3, rc, b, F);
    C.bbc[eqn] = rc.bbc;
    D.bbc[eqn] = 0.0;
    double bf = b + rc.bbc;
    C.b[eqn] = bf;
    D.b[eqn] = bf;
}

/* Blocks [0, nbm) take VBLK momentum rows each; the blocks after them take
 * VBLK continuity rows each, so that the continuity pass runs in the tail of
 * the momentum pass instead of after it. */
template <int KIND, int VBLK, int CAPA, int CAPB>
__global__ void __launch_bounds__(VBLK) k_values_mom(DevAsm a, DevBlock A, DevBlock B, DevBlock C, DevBlock D,
                                                     int nbm) {
    __shared__ double sA[VBLK * CAPA];
    __shared__ double sB[VBLK * CAPB];
    __shared__ double sDump[VBLK];
    if ((int)blockIdx.x >= nbm) {
        const int eqn = ((int)blockIdx.x - nbm) * VBLK + threadIdx.x;
        if (eqn < a.e.neq_cont) values_cont_row(a, C, D, eqn, sDump + threadIdx.x);
        return;
    }
    const int r0 = xcd_tile_of(blockIdx.x, nbm) * VBLK;
    const int r1 = min(r0 + VBLK, a.e.neq_mom);
    const int eqn = r0 + threadIdx.x;
    /* the row's own indices in one batch of loads (row index clamped into
     * the block), before the wave's vote and the row code: its field loads
     * then wait on one round trip (the node), not on the vote as well */
    const int er = eqn < r1 ? eqn : r1 - 1;
    const int node = a.e.mom_node[er];
    const int ia = A.Ic[er], ib = B.Ic[er];
    const int a0 = A.Ic[r0], b0 = B.Ic[r0], a1 = A.Ic[r1], b1 = B.Ic[r1];
    const int frow = A.free_row ? A.free_row[er] : 0;
    /* A wave whose rows read only free degrees of freedom (every tag -1, as
     * recorded with the pattern) takes the tag-free instance of the row
     * code: no tag loads, whose branch-dependent chain is otherwise the
     * row's latency.  Same values bit for bit. */
    const bool free_wave = A.free_row && __all(frow);
    if (eqn < r1) {
        Sink<SINK_VALUES> ra{0, nullptr, sA + (ia - a0), 0.0, sDump + threadIdx.x},
            rb{0, nullptr, sB + (ib - b0), 0.0, sDump + threadIdx.x};
        double b = mom_rhs(a, node), F = 0.0;
        if (free_wave) momentum_row<true, SINK_VALUES>(KIND, a, FreeTags{}, eqn, node, ra, rb, b, 0.0, F);
        else momentum_row<true, SINK_VALUES>(KIND, a, make_tags(a.g), eqn, node, ra, rb, b, 0.0, F);
        A.bbc[eqn] = ra.bbc;
        B.bbc[eqn] = rb.bbc;
        double bf = b + ra.bbc;
        A.b[eqn] = bf;
        B.b[eqn] = bf;
    }
    __syncthreads();
    /* coalesced copy-out; streaming (non-temporal) stores, as nothing in the
     * unit reads the values again and the stencil inputs keep the L2 */
    const int na = a1 - a0, nb = b1 - b0;
    for (int i = threadIdx.x; i < na; i += VBLK) __builtin_nontemporal_store(sA[i], A.A + a0 + i);
    for (int i = threadIdx.x; i < nb; i += VBLK) __builtin_nontemporal_store(sB[i], B.A + b0 + i);
}

/* The staged value pass over 64-row blocks (one wave each), for patterns
 * whose free-row flags and list of general waves are built: blocks [0, ngen)
 * take the listed general waves (A.gen_waves) with the general row code, the
 * next nbm blocks every wave whose rows are all free with the tag-free row
 * code (a general wave returns at once there), the blocks after them the
 * continuity rows.  A general wave is one long chain of dependent tag and
 * field loads: first in the grid, it runs beside the tag-free waves
 * instead of in a launch of its own after them (Jacobian, 1001 x 501 nodes:
 * 92 us against 77 + 24; 2049 x 1025: 389 either way, the stores bound it).
 * Same row code and staging as k_values_mom, so the same values bit for bit. */
template <bool GEN, int KIND, int CAPA, int CAPB>
__device__ __forceinline__ void values_wave(const DevAsm &a, DevBlock &A, DevBlock &B, int wv, double *sA, double *sB,
                                            double *sDump) {
    const int r0 = wv * 64;
    const int r1 = min(r0 + 64, a.e.neq_mom);
    const int eqn = r0 + threadIdx.x;
    const int er = eqn < r1 ? eqn : r1 - 1;
    /* wave-uniform (scalar) loads: the wave's kind, its first and last
     * rows' nodes and its row ranges */
    if (!GEN) {
        const int *pos = A.gen_waves + mdz_div_up(a.e.neq_mom, 64) + 1; /* scanned general-wave flags */
        if (pos[wv + 1] != pos[wv]) return; /* a general wave: listed, taken above */
    }
    const int a0 = A.Ic[r0], b0 = B.Ic[r0], a1 = A.Ic[r1], b1 = B.Ic[r1];
    const int n0 = a.e.mom_node[r0], nl = a.e.mom_node[r1 - 1];
    /* a regular wave -- 64 rows of consecutive nodes, each of full length --
     * needs no per-row index loads: its rows' nodes and offsets follow from
     * the first row's (mom_node increases with the row) */
    const bool regular = r1 - r0 == 64 && nl - n0 == 63 && a1 - a0 == 64 * CAPA && b1 - b0 == 64 * CAPB;
    int node, ia, ib;
    if (regular) {
        node = n0 + (int)threadIdx.x;
        ia = a0 + (int)threadIdx.x * CAPA;
        ib = b0 + (int)threadIdx.x * CAPB;
    } else {
        node = a.e.mom_node[er];
        ia = A.Ic[er];
        ib = B.Ic[er];
    }
    if (eqn < r1) {
        Sink<SINK_VALUES> ra{0, nullptr, sA + (ia - a0), 0.0, sDump + threadIdx.x},
            rb{0, nullptr, sB + (ib - b0), 0.0, sDump + threadIdx.x};
        double b = mom_rhs(a, node), F = 0.0;
        if (GEN) momentum_row<true, SINK_VALUES>(KIND, a, make_tags(a.g), eqn, node, ra, rb, b, 0.0, F);
        else momentum_row<true, SINK_VALUES>(KIND, a, FreeTags{}, eqn, node, ra, rb, b, 0.0, F);
        A.bbc[eqn] = ra.bbc;
        B.bbc[eqn] = rb.bbc;
        double bf = b + ra.bbc;
        A.b[eqn] = bf;
        B.b[eqn] = bf;
    }
    __syncthreads();
    const int na = a1 - a0, nb = b1 - b0;
    for (int i = threadIdx.x; i < na; i += 64) __builtin_nontemporal_store(sA[i], A.A + a0 + i);
    for (int i = threadIdx.x; i < nb; i += 64) __builtin_nontemporal_store(sB[i], B.A + b0 + i);
}

template <int KIND, int CAPA, int CAPB, int WAVES>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WAVES)))
k_values_split(DevAsm a, DevBlock A, DevBlock B, DevBlock C, DevBlock D, int ngen, int nbm) {
    __shared__ double sA[64 * CAPA];
    __shared__ double sB[64 * CAPB];
    __shared__ double sDump[64];
    int b = blockIdx.x;
    if (b < ngen) { values_wave<true, KIND, CAPA, CAPB>(a, A, B, A.gen_waves[b], sA, sB, sDump); return; }
    b -= ngen;
    if (b < nbm) { values_wave<false, KIND, CAPA, CAPB>(a, A, B, xcd_tile_of(b, nbm), sA, sB, sDump); return; }
    const int eqn = (b - nbm) * 64 + threadIdx.x;
    if (eqn < a.e.neq_cont) values_cont_row(a, C, D, eqn, sDump + threadIdx.x);
}

/* The value passes of the Picard (P) and Jacobian (J) families in one launch
 * of 64-row blocks: their general waves, tag-free waves and continuity rows
 * in turn.  Picard rows read the J = 0 components of `a`, Jacobian rows the
 * tensor of the grid, so the two need no order. */
struct ValuesPair {
    DevBlock A[2], B[2], C[2], D[2]; /* 0 Picard, 1 Jacobian */
};

template <int CAPA0, int CAPB0, int CAPA1, int CAPB1>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
k_values_pair(DevAsm a, ValuesPair p, int nbm, int nbc) {
    __shared__ double sA[64 * CAPA1];
    __shared__ double sB[64 * CAPB1];
    __shared__ double sDump[64];
    int b = blockIdx.x;
    if (b < p.A[1].n_gen) {
        values_wave<true, 1, CAPA1, CAPB1>(a, p.A[1], p.B[1], p.A[1].gen_waves[b], sA, sB, sDump);
        return;
    }
    b -= p.A[1].n_gen;
    if (b < p.A[0].n_gen) {
        values_wave<true, 0, CAPA0, CAPB0>(a, p.A[0], p.B[0], p.A[0].gen_waves[b], sA, sB, sDump);
        return;
    }
    b -= p.A[0].n_gen;
    if (b < nbm) { values_wave<false, 1, CAPA1, CAPB1>(a, p.A[1], p.B[1], xcd_tile_of(b, nbm), sA, sB, sDump); return; }
    b -= nbm;
    if (b < nbm) { values_wave<false, 0, CAPA0, CAPB0>(a, p.A[0], p.B[0], xcd_tile_of(b, nbm), sA, sB, sDump); return; }
    b -= nbm;
    const int k = b < nbc ? 0 : 1;
    const int eqn = (b - k * nbc) * 64 + threadIdx.x;
    if (eqn < a.e.neq_cont) values_cont_row(a, p.C[k], p.D[k], eqn, sDump + threadIdx.x);
}

/* the same without staging, for patterns with longer rows */
template <int KIND>
__global__ void __launch_bounds__(BLK) k_values_mom_direct(DevAsm a, DevBlock A, DevBlock B) {
    __shared__ double sDump[BLK];
    int eqn = xcd_tile() * BLK + threadIdx.x;
    const int neq = a.e.neq_mom;
    const bool in = eqn < neq;
    /* indices in one batch (row clamped), then the tag-free instance for
     * waves of free rows, as in k_values_mom */
    const int er = in ? eqn : neq - 1;
    const int node = a.e.mom_node[er], ia = A.Ic[er], ib = B.Ic[er];
    const int frow = A.free_row ? A.free_row[er] : 0;
    const bool free_wave = A.free_row && __all(in ? frow : 1);
    if (!in) return;
    Sink<SINK_VALUES> ra{0, nullptr, A.A + ia, 0.0, sDump + threadIdx.x},
        rb{0, nullptr, B.A + ib, 0.0, sDump + threadIdx.x};
    double b = mom_rhs(a, node), F = 0.0;
    if (free_wave) momentum_row<true, SINK_VALUES>(KIND, a, FreeTags{}, eqn, node, ra, rb, b, 0.0, F);
    else momentum_row<true, SINK_VALUES>(KIND, a, make_tags(a.g), eqn, node, ra, rb, b, 0.0, F);
    A.bbc[eqn] = ra.bbc;
    B.bbc[eqn] = rb.bbc;
    double bf = b + ra.bbc;
    A.b[eqn] = bf;
    B.b[eqn] = bf;
}

__global__ void __launch_bounds__(BLK) k_values_cont(DevAsm a, DevBlock C, DevBlock D) {
    __shared__ double sDump[BLK];
    int eqn = xcd_tile() * BLK + threadIdx.x;
    if (eqn >= a.e.neq_cont) return;
    values_cont_row(a, C, D, eqn, sDump + threadIdx.x);
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

/* Slots of the per-block sums of a fused residual + norm pass:
 * partial[q * nsm + slot], q = 0..3 (u F^2, u count, v F^2, v count), for
 * the momentum launches, then partial[4 * nsm + q * nsc + slot], q = 0..1
 * (p F^2, p count), for the continuity launch. */
struct NormSlots {
    double *partial;
    int nsm, nsc;
    int slot0;        /* first momentum slot of this launch */
    const int *waves; /* general momentum launch: its waves, one per block */
};

/* NQ per-thread values summed over the block in a fixed order (waves by
 * shuffles, then the waves in order); thread 0 gets the sums */
template <int NQ>
__device__ __forceinline__ void block_sums(double (&v)[NQ]) {
    __shared__ double ws[BLK / 64][NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) v[q] = wave_sum(v[q]);
    const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int q = 0; q < NQ; q++) ws[w][q] = v[q];
    __syncthreads();
    if (threadIdx.x == 0)
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            double t = 0.0;
            for (int k = 0; k < nw; k++) t += ws[k][q];
            v[q] = t;
        }
}

/* residual (Assemble = 0): b = rhs (Neumann rows adjusted), F.  Waves
 * whose rows are all free take the tag-free instance (FREE), the others the
 * general one.  NORM: the norm pass of EvaluateStokesResidualDecoupled
 * (StokesRoutines.c:1390-1452) on the row as well: ru / rv of its node = F,
 * F *= d, and per-block sums of F^2 and of the rows per family.  The
 * general NORM instance runs one 64-row wave per block, the waves listed in
 * ns.waves; the others run 256-row tiles. */
template <int KIND, bool FREE, bool NORM>
__global__ void __launch_bounds__(BLK) k_residual_mom(DevAsm a, DevBlock A, NormSlots ns) {
    const int eqn = (NORM && !FREE) ? ns.waves[blockIdx.x] * 64 + (int)threadIdx.x : xcd_tile() * BLK + (int)threadIdx.x;
    const int neq = a.e.neq_mom;
    bool run = eqn < neq;
    /* the row's inputs that do not depend on its node, in one batch with
     * the node (row clamped), before the wave's vote */
    const int er = run ? eqn : neq - 1;
    const int node = a.e.mom_node[er];
    const double bbc_in = A.bbc[er], F0 = A.F[er], dr = NORM ? A.d[er] : 1.0;
    const int frow = A.free_row ? A.free_row[er] : 1;
    if (A.free_row) {
        if ((__all(run ? frow : 1) != 0) != FREE) run = false;
    } else if (FREE) {
        run = false;
    }
    if (!NORM && !run) return;
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    if (run) {
        Sink<SINK_COUNT> ra{0, nullptr, nullptr, 0.0}, rb{0, nullptr, nullptr, 0.0};
        double b = mom_rhs(a, node), F = F0;
        if (FREE) momentum_row<false, SINK_COUNT>(KIND, a, FreeTags{}, eqn, node, ra, rb, b, bbc_in, F);
        else momentum_row<false, SINK_COUNT>(KIND, a, make_tags(a.g), eqn, node, ra, rb, b, bbc_in, F);
        A.b[eqn] = b;
        if (NORM) {
            const int nu = a.g.Nx * a.g.nzvx;
            if (node < nu) { a.g.ru[node] = F; v[0] = F * F; v[1] = 1.0; }
            else { a.g.rv[node - nu] = F; v[2] = F * F; v[3] = 1.0; }
            A.F[eqn] = F * dr;
        } else {
            A.F[eqn] = F;
        }
    }
    if (NORM) {
        block_sums<4>(v);
        if (threadIdx.x == 0) {
            const int slot = ns.slot0 + (FREE ? xcd_tile() : (int)blockIdx.x);
#pragma unroll
            for (int q = 0; q < 4; q++) ns.partial[q * ns.nsm + slot] = v[q];
        }
    }
}

/* The general Picard rows (kind 0, Assemble = 0, with the norm work) of
 * listed wave `slot`, in one wave; its sums go to slot ns.slot0 + slot. */
__device__ __forceinline__ void residual_general_wave(const DevAsm &a, const DevBlock &A, const NormSlots &ns, int slot) {
    const int lane = threadIdx.x & 63;
    const int eqn = ns.waves[slot] * 64 + lane;
    const bool in = eqn < a.e.neq_mom;
    const int er = in ? eqn : a.e.neq_mom - 1;
    const int node = a.e.mom_node[er];
    const double bbc_in = A.bbc[er], F0 = A.F[er], dr = A.d[er];
    const bool run = in && !A.free_row[er];
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    if (run) {
        Sink<SINK_COUNT> ra{0, nullptr, nullptr, 0.0}, rb{0, nullptr, nullptr, 0.0};
        double b = mom_rhs(a, node), F = F0;
        momentum_row<false, SINK_COUNT>(0, a, make_tags(a.g), eqn, node, ra, rb, b, bbc_in, F);
        A.b[eqn] = b;
        const int nu = a.g.Nx * a.g.nzvx;
        if (node < nu) { a.g.ru[node] = F; v[0] = F * F; v[1] = 1.0; }
        else { a.g.rv[node - nu] = F; v[2] = F * F; v[3] = 1.0; }
        A.F[eqn] = F * dr;
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const double t = wave_sum(v[q]);
        if (lane == 0) ns.partial[q * ns.nsm + ns.slot0 + slot] = t;
    }
}

/* The residual pass (Picard, kind 0) with its norm work over tiles of
 * RT_TX x RT_TZ grid positions: lane (i, j) takes the x-momentum row of
 * u-node (i, j) and the z-momentum row of v-node (i, j) when their rows
 * are free (every tag they read is -1: free_node, from the pattern build;
 * the other momentum rows are left to the blocks of the listed
 * waves), and the continuity row of centroid (i, j).  The block stages
 * u, v, p_corr, the J = 0 D11 (= D22) at the centroids and D33 at the
 * vertices, and the u, v tags, of its tile with a one-node halo in LDS
 * (coalesced row loads, one batch), so a row's stencil is read from LDS
 * and the row -> node map is not on the load path.  The row arithmetic is
 * that of the tag-free instance of xmom_inner / zmom_inner / continuity_row
 * (same expressions and summation order), so the values are bit for bit
 * those of k_residual_mom<0, true, .> and k_residual_cont.  Per-block sums
 * of F^2 and of the rows go to slot `tile` of each family.  The first ngb
 * blocks take the listed general waves, one per wave.  The tiles stream from
 * HBM and want eight waves per SIMD; the general rows then spill, which their
 * few waves hide behind the tiles (2049 x 1025 nodes: 111 us, 129 without the
 * bound, 110 + 15 in two launches; 1001 x 501: 37 against 33 + 12). */
#define RT_TX 64
#define RT_TZ 4
struct ResTile {
    double u[RT_TZ + 2][RT_TX + 2];  /* u(i0 - 1 + a, j0 - 1 + b) */
    double v[RT_TZ + 2][RT_TX + 3];  /* v(i0 - 1 + a, j0 - 1 + b) */
    double p[RT_TZ + 1][RT_TX + 1];  /* p_corr at centroid (i0 - 1 + a, j0 - 1 + b) */
    double d11[RT_TZ + 1][RT_TX + 1]; /* D11 = D22 (J = 0) at centroid (i0 - 1 + a, j0 - 1 + b) */
    double d33[RT_TZ + 1][RT_TX + 1]; /* D33 (J = 0) at vertex (i0 - 1 + a, j0 - 1 + b) */
    signed char tu[RT_TZ + 2][RT_TX + 2], tv[RT_TZ + 2][RT_TX + 3];
};

template <int N, int W, int H>
__device__ __forceinline__ void tile_load(double (&dst)[H][W], signed char (*tdst)[W], const double *__restrict__ src,
                                          const int8_t *__restrict__ tsrc, int x0, int z0, int nx, int nz) {
    constexpr int R = (W * H + N - 1) / N;
    double v[R];
    int8_t t[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int q = threadIdx.x + N * r, a = q % W, b = q / W, x = x0 + a, z = z0 + b;
        const bool in = q < W * H && x >= 0 && x < nx && z >= 0 && z < nz;
        const int idx = in ? x + z * nx : 0;
        v[r] = src[idx];
        if (tdst) t[r] = in ? tsrc[idx] : (int8_t)OUTSIDE;
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int q = threadIdx.x + N * r;
        if (q < W * H) {
            dst[q / W][q % W] = v[r];
            if (tdst) tdst[q / W][q % W] = (signed char)t[r];
        }
    }
}

__global__ void __launch_bounds__(RT_TX * RT_TZ) __attribute__((amdgpu_waves_per_eu(8)))
k_residual_tile(DevAsm a, DevBlock A, DevBlock C, DevBlock D, const unsigned char *__restrict__ free_node, int scaled,
                int ntx, int ngb, NormSlots ns) {
    __shared__ ResTile T;
    const DevGrid &g = a.g;
    const int Nx = g.Nx, Nz = g.Nz, ncx = g.ncx, ncz = g.ncz, nxvz = g.nxvz, nzvx = g.nzvx;
    const int nu = Nx * nzvx;
    /* the listed general waves first, one per wave of the block: their long
     * load chains run beside the tiles */
    if ((int)blockIdx.x < ngb) {
        const int slot = blockIdx.x * (RT_TX * RT_TZ / 64) + ((int)threadIdx.x >> 6);
        if (slot < A.n_gen) residual_general_wave(a, A, ns, slot);
        return;
    }
    const int tile = blockIdx.x - ngb;
    const int i0 = (tile % ntx) * RT_TX, j0 = (tile / ntx) * RT_TZ;
    const int tx = threadIdx.x % RT_TX, ty = threadIdx.x / RT_TX;
    const int i = i0 + tx, j = j0 + ty;
    /* the lane's own rows: node indices, flags, equation numbers, rhs */
    const bool hu = i < Nx && j < nzvx, hv = i < nxvz && j < Nz, hc = i < ncx && j < ncz;
    const int un = hu ? i + j * Nx : 0, vn = hv ? i + j * nxvz : 0, cn = hc ? i + j * ncx : 0;
    const bool fu = hu && free_node[un], fv = hv && free_node[nu + vn];
    const int equ = a.e.eqn_u[un], eqv = a.e.eqn_v[vn], eqp = a.e.eqn_p[cn];
    const double bu = g.roger_x[un], bv = g.roger_z[vn];
    const double pc = a.p_cont[cn], bet = g.bet_n[cn], rp = g.rhs_p[cn];
    const int comp = g.comp_cells[cn];
    /* the tile and its halo */
    constexpr int N = RT_TX * RT_TZ;
    tile_load<N>(T.u, T.tu, a.u, g.BCu, i0 - 1, j0 - 1, Nx, nzvx);
    tile_load<N>(T.v, T.tv, a.v, g.BCv, i0 - 1, j0 - 1, nxvz, Nz);
    tile_load<N>(T.p, (signed char (*)[RT_TX + 1]) nullptr, a.p_mom, nullptr, i0 - 1, j0 - 1, ncx, ncz);
    tile_load<N>(T.d11, (signed char (*)[RT_TX + 1]) nullptr, a.d11p, nullptr, i0 - 1, j0 - 1, ncx, ncz);
    tile_load<N>(T.d33, (signed char (*)[RT_TX + 1]) nullptr, a.d33p, nullptr, i0 - 1, j0 - 1, Nx, Nz);
    __syncthreads();
    const int X = tx + 1, Z = ty + 1;
    const double cv = a.celvol;
    double vsum[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (fu) {
        /* x-momentum row of u(i, j) (xmom_inner, tag-free) */
        const double D11W = T.d11[Z - 1][X - 1], D11E = T.d11[Z - 1][X], D33N = T.d33[Z][X], D33S = T.d33[Z - 1][X];
        const XRes r = xres_coeffs(D11W, D11E, D33N, D33S, 1.0, 1.0, 1.0, 1.0, g.dx, g.dz);
        double uC = r.uC;
        if (a.stab == 1) {
            const int c2 = i - 1 + (j - 1) * ncx;
            double drhodx = (g.rho_n[c2 + 1] - g.rho_n[c2]) * a.one_dx;
            double uC_corr = 1.00 * a.om * a.dt * g.gx[un] * drhodx;
            if (uC + uC_corr > 0.0) uC += uC_corr;
        }
        const double pW = -a.one_dx * 1e0, pE = a.one_dx * 1e0;
        double f = uC * T.u[Z][X];
        f += pW * T.p[Z - 1][X - 1] + pE * T.p[Z - 1][X];
        f += r.vSE * T.v[Z - 1][X + 1];
        f += r.vSW * T.v[Z - 1][X];
        f += r.vNE * T.v[Z][X + 1];
        f += r.vNW * T.v[Z][X];
        f += r.uS * T.u[Z - 1][X];
        f += r.uN * T.u[Z + 1][X];
        f += r.uW * T.u[Z][X - 1];
        f += r.uE * T.u[Z][X + 1];
        f -= bu;
        const double F = f * cv;
        A.b[equ] = bu;
        g.ru[un] = F;
        vsum[0] = F * F; vsum[1] = 1.0;
        A.F[equ] = scaled ? F * A.d[equ] : F;
    }
    if (fv) {
        /* z-momentum row of v(i, j) (zmom_inner, tag-free) */
        const double D22S = T.d11[Z - 1][X - 1], D22N = T.d11[Z][X - 1], D33W = T.d33[Z][X - 1], D33E = T.d33[Z][X];
        const ZRes r = zres_coeffs(D22S, D22N, D33W, D33E, 1.0, 1.0, 1.0, 1.0, g.dx, g.dz);
        double vC = r.vC;
        if (a.stab == 1) {
            const int c2 = i - 1 + (j - 1) * ncx;
            double drhodz = (g.rho_n[c2 + ncx] - g.rho_n[c2]) * a.one_dz;
            double vC_corr = 1.00 * a.om * a.dt * g.gz[vn] * drhodz;
            if (vC + vC_corr > 0.0) vC += vC_corr;
        }
        const double pS = -a.one_dz * 1e0, pN = a.one_dz * 1e0;
        double f = vC * T.v[Z][X];
        f += pS * T.p[Z - 1][X - 1] + pN * T.p[Z][X - 1];
        f += r.vS * T.v[Z - 1][X];
        f += r.vW * T.v[Z][X - 1];
        f += r.vE * T.v[Z][X + 1];
        f += r.vN * T.v[Z + 1][X];
        f += r.uSW * T.u[Z][X - 1];
        f += r.uSE * T.u[Z][X];
        f += r.uNW * T.u[Z + 1][X - 1];
        f += r.uNE * T.u[Z + 1][X];
        f -= bv;
        const double F = f * cv;
        A.b[eqv] = bv;
        g.rv[vn] = F;
        vsum[2] = F * F; vsum[3] = 1.0;
        A.F[eqv] = scaled ? F * A.d[eqv] : F;
    }
    if (hc && eqp >= 0) {
        /* continuity row of centroid (i, j) (continuity_row, Assemble = 0) */
        const int row = eqp - a.e.neq_mom;
        const int tW = T.tu[Z + 1][X], tE = T.tu[Z + 1][X + 1], tS = T.tv[Z][X + 1], tN = T.tv[Z + 1][X + 1];
        double uW = tW != 13 ? -a.one_dx * 1e0 : 0.0, uE = tE != 13 ? a.one_dx * 1e0 : 0.0;
        double vS = tS != 13 ? -a.one_dz * 1e0 : 0.0, vN = tN != 13 ? a.one_dz * 1e0 : 0.0;
        double pcoef = comp == 0 ? 0.0 : bet / a.dt;
        double f = pcoef * pc + uW * T.u[Z + 1][X] + uE * T.u[Z + 1][X + 1] + vS * T.v[Z][X + 1] + vN * T.v[Z + 1][X + 1];
        f -= rp;
        const double F = f * cv;
        C.b[row] = rp;
        C.F[row] = F;
        g.rp[cn] = F;
        vsum[4] = F * F; vsum[5] = 1.0;
        D.F[row] = scaled ? F * D.d[row] : F;
    }
    block_sums<6>(vsum);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int q = 0; q < 4; q++) ns.partial[q * ns.nsm + tile] = vsum[q];
        ns.partial[4 * ns.nsm + tile] = vsum[4];
        ns.partial[4 * ns.nsm + ns.nsc + tile] = vsum[5];
    }
}

/* free_row[eqn] = 1 when every tag the row reads, in the value and in the
 * residual pass, is a free degree of freedom (-1) (the residual kernels
 * use it; the value pass is checked too so that the flag describes the
 * whole row).  Rows longer than the
 * 32-entry scratch slot are never free (the host checks the pattern's
 * longest row before the launch). */
#define FREE_SLOT 33
__global__ void __launch_bounds__(64) k_free_rows(int kind, DevAsm a, unsigned char *free_row) {
    __shared__ double scr[64 * FREE_SLOT];
    const int eqn = blockIdx.x * 64 + threadIdx.x;
    if (eqn >= a.e.neq_mom) return;
    CheckTags T;
    static_cast<Tags &>(T) = make_tags(a.g);
    T.all_free = true;
    double *mine = scr + threadIdx.x * FREE_SLOT;
    Sink<SINK_VALUES> ra{0, nullptr, mine, 0.0, mine + FREE_SLOT - 1}, rb{0, nullptr, mine, 0.0, mine + FREE_SLOT - 1};
    const int node = a.e.mom_node[eqn];
    double b = mom_rhs(a, node), F = 0.0;
    momentum_row<true, SINK_VALUES>(kind, a, T, eqn, node, ra, rb, b, 0.0, F);
    Sink<SINK_COUNT> rc{0, nullptr, nullptr, 0.0}, rd{0, nullptr, nullptr, 0.0};
    double b2 = mom_rhs(a, node), F2 = 0.0;
    momentum_row<false, SINK_COUNT>(kind, a, T, eqn, node, rc, rd, b2, 0.0, F2);
    free_row[eqn] = T.all_free ? 1 : 0;
}

template <bool NORM>
__global__ void __launch_bounds__(BLK) k_residual_cont(int kind, DevAsm a, DevBlock C, DevBlock D, NormSlots ns) {
    int eqn = xcd_tile() * BLK + threadIdx.x;
    if (!NORM && eqn >= a.e.neq_cont) return;
    double v[2] = {0.0, 0.0};
    if (eqn < a.e.neq_cont) {
        int c1, c2, c3;
        cont_geom(a, eqn, c1, c2, c3);
        /* the Jacobian builder reads comp_cells at the vertex-family index c1 */
        int comp = kind == 1 ? a.g.comp_cells[c1] : a.g.comp_cells[c2];
        Sink<SINK_COUNT> rc{0, nullptr, nullptr, 0.0};
        double b = a.g.rhs_p[c2], F = 0.0;
        continuity_row<false, SINK_COUNT>(a, comp, c1, c2, c3, rc, b, F);
        C.b[eqn] = b;
        C.F[eqn] = F;
        if (NORM) {
            a.g.rp[c2] = F;
            v[0] = F * F; v[1] = 1.0;
            D.F[eqn] = F * D.d[eqn];
        } else {
            D.F[eqn] = F;
        }
    }
    if (NORM) {
        block_sums<2>(v);
        if (threadIdx.x == 0) {
            const int slot = xcd_tile();
            ns.partial[4 * ns.nsm + slot] = v[0];
            ns.partial[4 * ns.nsm + ns.nsc + slot] = v[1];
        }
    }
}

/* ------------------------------------------------------------------ */
/* scan, numbering                                                      */
/* ------------------------------------------------------------------ */
#define SCAN_BLK 1024

__device__ __forceinline__ int wave_incl_scan(int v) {
    int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        int t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    return v;
}

/* block-local exclusive scan; writes the block total */
__global__ void __launch_bounds__(SCAN_BLK) k_scan_local(int *data, int n, int *block_sums) {
    __shared__ int wsum[SCAN_BLK / 64];
    int i = blockIdx.x * SCAN_BLK + threadIdx.x;
    int v = i < n ? data[i] : 0;
    int inc = wave_incl_scan(v);
    int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    if (w == 0) {
        int s = lane < SCAN_BLK / 64 ? wsum[lane] : 0;
        int si = wave_incl_scan(s);
        if (lane < SCAN_BLK / 64) wsum[lane] = si - s;
    }
    __syncthreads();
    int excl = inc - v + wsum[w];
    if (i < n) data[i] = excl;
    if (threadIdx.x == SCAN_BLK - 1) block_sums[blockIdx.x] = excl + v;
}

/* single-block exclusive scan of the block sums (any count) */
__global__ void __launch_bounds__(SCAN_BLK) k_scan_sums(int *sums, int nb, int *total) {
    __shared__ int carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (int base = 0; base < nb; base += SCAN_BLK) {
        __shared__ int wsum[SCAN_BLK / 64];
        int i = base + threadIdx.x;
        int v = i < nb ? sums[i] : 0;
        int inc = wave_incl_scan(v);
        int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
        if (lane == 63) wsum[w] = inc;
        __syncthreads();
        if (w == 0) {
            int s = lane < SCAN_BLK / 64 ? wsum[lane] : 0;
            int si = wave_incl_scan(s);
            if (lane < SCAN_BLK / 64) wsum[lane] = si - s;
        }
        __syncthreads();
        int excl = inc - v + wsum[w] + carry;
        if (i < nb) sums[i] = excl;
        __syncthreads();
        if (threadIdx.x == SCAN_BLK - 1) carry = excl + v;
        __syncthreads();
    }
    if (threadIdx.x == 0) *total = carry;
}

__global__ void __launch_bounds__(SCAN_BLK) k_scan_add(int *data, int n, const int *block_sums) {
    int i = blockIdx.x * SCAN_BLK + threadIdx.x;
    if (i < n) data[i] += block_sums[blockIdx.x];
}

int mdz_scan_exclusive(int *data, int n, int *scratch, size_t scratch_len, hipStream_t s, int *total) {
    int nb = mdz_div_up(n > 0 ? n : 1, SCAN_BLK);
    if ((size_t)nb + 1 > scratch_len) return MDZ_ENOMEM;
    int *sums = scratch, *dtot = scratch + nb;
    hipLaunchKernelGGL(k_scan_local, dim3(nb), dim3(SCAN_BLK), 0, s, data, n, sums);
    hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(SCAN_BLK), 0, s, sums, nb, dtot);
    hipLaunchKernelGGL(k_scan_add, dim3(nb), dim3(SCAN_BLK), 0, s, data, n, (const int *)sums);
    if (total) {
        if (hipMemcpyAsync(total, dtot, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess) return MDZ_EHIP;
        if (hipStreamSynchronize(s) != hipSuccess) return MDZ_EHIP;
    }
    return MDZ_OK;
}

/* flags of u, v (momentum) and p (continuity) DOFs, concatenated */
__global__ void __launch_bounds__(BLK) k_eqn_flags(DevGrid g, int *flags) {
    int i = blockIdx.x * BLK + threadIdx.x;
    int nu = g.Nx * g.nzvx, nw = g.nxvz * g.Nz, nc = g.ncx * g.ncz;
    if (i >= nu + nw + nc) return;
    int f = 0;
    if (i < nu) { int t = g.BCu[i]; f = (t == -1 || t == 2 || t == -2); }
    else if (i < nu + nw) { int t = g.BCv[i - nu]; f = (t == -1 || t == 2); }
    else { f = g.BCp[i - nu - nw] == -1; }
    flags[i] = f;
}

/* eqn from the scanned flags; row->node maps */
__global__ void __launch_bounds__(BLK) k_eqn_assign(DevGrid g, const int *scan, DevEqn e) {
    int i = blockIdx.x * BLK + threadIdx.x;
    int nu = g.Nx * g.nzvx, nw = g.nxvz * g.Nz, nc = g.ncx * g.ncz;
    if (i >= nu + nw + nc) return;
    if (i < nu) {
        int t = g.BCu[i];
        int eq = (t == -1 || t == 2 || t == -2) ? scan[i] : -1;
        e.eqn_u[i] = eq;
        if (eq >= 0) e.mom_node[eq] = i;
    } else if (i < nu + nw) {
        int c = i - nu, t = g.BCv[c];
        int eq = (t == -1 || t == 2) ? scan[i] : -1;
        e.eqn_v[c] = eq;
        if (eq >= 0) e.mom_node[eq] = i;
    } else {
        int c = i - nu - nw;
        int eq = g.BCp[c] == -1 ? scan[i] : -1;
        e.eqn_p[c] = eq;
        if (eq >= 0) e.cont_node[eq - e.neq_mom] = c;
    }
}

/* -12 nodes copy the equation number of the node Nx-1 to their left
 * (StokesRoutines.c:1156); sequential dependence along a row resolved by
 * walking left until a non-copy node */
__global__ void __launch_bounds__(BLK) k_eqn_periodic(DevGrid g, DevEqn e) {
    int i = blockIdx.x * BLK + threadIdx.x;
    int nu = g.Nx * g.nzvx;
    if (i >= nu) return;
    if (g.BCu[i] != -12) return;
    int j = i - g.Nx + 1;
    e.eqn_u[i] = j >= 0 ? (g.BCu[j] == -12 ? -1 : e.eqn_u[j]) : -1;
}

int mdz_number_equations(const DevGrid &g, DevEqn &e, int *scratch, size_t scratch_len, hipStream_t s) {
    int nu = g.Nx * g.nzvx, nw = g.nxvz * g.Nz, nc = g.ncx * g.ncz, n = nu + nw + nc;
    if ((size_t)n + (size_t)mdz_div_up(n, SCAN_BLK) + 2 > scratch_len) return MDZ_ENOMEM;
    int *flags = scratch, *rest = scratch + n;
    hipLaunchKernelGGL(k_eqn_flags, dim3(mdz_div_up(n, BLK)), dim3(BLK), 0, s, g, flags);
    /* counts of momentum DOFs: scan of the u+v part gives neq_mom */
    int total = 0;
    int rc = mdz_scan_exclusive(flags, n, rest, scratch_len - n, s, &total);
    if (rc) return rc;
    /* neq_mom = scanned value at the first p flag */
    int neq_mom = 0;
    if (hipMemcpyAsync(&neq_mom, flags + nu + nw, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess) return MDZ_EHIP;
    if (hipStreamSynchronize(s) != hipSuccess) return MDZ_EHIP;
    e.neq_mom = neq_mom;
    e.neq_cont = total - neq_mom;
    hipLaunchKernelGGL(k_eqn_assign, dim3(mdz_div_up(n, BLK)), dim3(BLK), 0, s, g, (const int *)flags, e);
    hipLaunchKernelGGL(k_eqn_periodic, dim3(mdz_div_up(nu, BLK)), dim3(BLK), 0, s, g, e);
    return MDZ_OK;
}

/* ------------------------------------------------------------------ */
/* pattern, values, residual launchers                                  */
/* ------------------------------------------------------------------ */
int mdz_build_pattern(int kind, const DevAsm &a, DevBlock *A, DevBlock *B, DevBlock *C, int *scratch,
                      size_t scratch_len, hipStream_t s) {
    int nm = a.e.neq_mom, ncnt = a.e.neq_cont;
    int gm = mdz_div_up(nm > 0 ? nm : 1, BLK), gc = mdz_div_up(ncnt > 0 ? ncnt : 1, BLK);
    /* counts go into Ic[0..neq-1], scanned in place; the largest row length
     * is collected in Ic[neq] (later overwritten with nnz) */
    if (hipMemsetAsync(A->Ic + nm, 0, sizeof(int), s) != hipSuccess) return MDZ_EHIP;
    if (hipMemsetAsync(B->Ic + nm, 0, sizeof(int), s) != hipSuccess) return MDZ_EHIP;
    if (C && hipMemsetAsync(C->Ic + ncnt, 0, sizeof(int), s) != hipSuccess) return MDZ_EHIP;
    hipLaunchKernelGGL(k_count_mom, dim3(gm), dim3(BLK), 0, s, kind, a, A->Ic, B->Ic);
    if (C) hipLaunchKernelGGL(k_count_cont, dim3(gc), dim3(BLK), 0, s, a, C->Ic);
    int mx[3] = {0, 0, 0};
    if (hipMemcpyAsync(&mx[0], A->Ic + nm, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess) return MDZ_EHIP;
    if (hipMemcpyAsync(&mx[1], B->Ic + nm, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess) return MDZ_EHIP;
    if (C && hipMemcpyAsync(&mx[2], C->Ic + ncnt, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess) return MDZ_EHIP;
    if (hipStreamSynchronize(s) != hipSuccess) return MDZ_EHIP;
    A->maxrow = mx[0];
    B->maxrow = mx[1];
    if (C) C->maxrow = mx[2];
    int tot = 0, rc;
    if ((rc = mdz_scan_exclusive(A->Ic, nm, scratch, scratch_len, s, &tot))) return rc;
    A->nnz = tot;
    if ((rc = mdz_scan_exclusive(B->Ic, nm, scratch, scratch_len, s, &tot))) return rc;
    B->nnz = tot;
    if (C) {
        if ((rc = mdz_scan_exclusive(C->Ic, ncnt, scratch, scratch_len, s, &tot))) return rc;
        C->nnz = tot;
    }
    return MDZ_OK;
}

/* second half of the pattern build, once J has been allocated for the nnz */
void mdz_fill_pattern(int kind, const DevAsm &a, DevBlock *A, DevBlock *B, DevBlock *C, hipStream_t s) {
    int nm = a.e.neq_mom, ncnt = a.e.neq_cont;
    if (nm > 0) hipLaunchKernelGGL(k_pattern_mom, dim3(mdz_div_up(nm, BLK)), dim3(BLK), 0, s, kind, a, *A, *B);
    if (C && ncnt > 0) hipLaunchKernelGGL(k_pattern_cont, dim3(mdz_div_up(ncnt, BLK)), dim3(BLK), 0, s, a, *C);
}

/* LDS slots of the staged value kernels: the reference's row budgets
 * (StokesAssemblyDecoupled.c:1632-1635, :3887-3890) */
#define PIC_CAPA 9
#define PIC_CAPB 2
#define JAC_CAPA 21
#define JAC_CAPB 6

template <int KIND, int VBLK, int CAPA, int CAPB>
static void launch_staged(const DevAsm &a, DevBlock *A, DevBlock *B, DevBlock *C, DevBlock *D, hipStream_t s) {
    /* one launch: each wave picks the tag-free or the general row code (a
     * separate launch for the blocks of free rows, with only the tag-free
     * code and fewer registers, was measured slower) */
    const int nbm = mdz_div_up(a.e.neq_mom, VBLK), nbc = mdz_div_up(a.e.neq_cont, VBLK);
    hipLaunchKernelGGL((k_values_mom<KIND, VBLK, CAPA, CAPB>), dim3(nbm + nbc), dim3(VBLK), 0, s, a, *A, *B, *C, *D,
                       nbm);
}

/* WAVES per SIMD of the launch: the Jacobian's general row code takes 207
 * registers and spills at three waves per SIMD, where the tag-free code runs
 * best; a grid that two waves per SIMD hold at once (1024 SIMDs) has nothing
 * to gain from a third (41 x 41 nodes: 17.4 us against 23.0) */
#define SPLIT_ROUND2 2048

template <int KIND, int CAPA, int CAPB>
static void launch_split(const DevAsm &a, DevBlock *A, DevBlock *B, DevBlock *C, DevBlock *D, hipStream_t s) {
    const int nbm = mdz_div_up(a.e.neq_mom, 64), nbc = mdz_div_up(a.e.neq_cont, 64);
    const int grid = A->n_gen + nbm + nbc;
    if constexpr (KIND == 1)
        if (grid <= SPLIT_ROUND2) {
            hipLaunchKernelGGL((k_values_split<KIND, CAPA, CAPB, 2>), dim3(grid), dim3(64), 0, s, a, *A, *B, *C, *D,
                               A->n_gen, nbm);
            return;
        }
    hipLaunchKernelGGL((k_values_split<KIND, CAPA, CAPB, KIND == 1 ? 3 : 6>), dim3(grid), dim3(64), 0, s, a, *A, *B,
                       *C, *D, A->n_gen, nbm);
}

/* One launch up to the size where two waves per SIMD hold both passes at
 * once: there each pass is the latency of its general waves (18 and 9 us at
 * 41 x 41 nodes), which overlap.  Beyond it the Picard pass would lose the six
 * waves per SIMD that it has on its own. */
bool mdz_launch_values_pair(const DevAsm &a, DevBlock *P, DevBlock *J, const LaunchShape &shape, hipStream_t s) {
    const bool split = P->free_row && P->gen_waves && J->free_row && J->gen_waves;
    const bool fits = P[0].maxrow <= PIC_CAPA && P[1].maxrow <= PIC_CAPB && J[0].maxrow <= JAC_CAPA &&
                      J[1].maxrow <= JAC_CAPB;
    const bool rows64 = shape.jac == 64 && (shape.asked ? shape.pic == 64 : shape.pic != 0);
    if (a.e.neq_mom <= 0 || !rows64 || !split || !fits) return false;
    const int nbm = mdz_div_up(a.e.neq_mom, 64), nbc = mdz_div_up(a.e.neq_cont, 64);
    const int grid = P->n_gen + J->n_gen + 2 * (nbm + nbc);
    if (grid > SPLIT_ROUND2) return false;
    const ValuesPair p{{P[0], J[0]}, {P[1], J[1]}, {P[2], J[2]}, {P[3], J[3]}};
    hipLaunchKernelGGL((k_values_pair<PIC_CAPA, PIC_CAPB, JAC_CAPA, JAC_CAPB>), dim3(grid), dim3(64), 0, s, a, p, nbm,
                       nbc);
    return true;
}

__global__ void __launch_bounds__(BLK) k_fill_bytes(unsigned char *p, int n) {
    const int i = blockIdx.x * BLK + threadIdx.x;
    if (i < n) p[i] = 0;
}
/* free_node[node] = free_row of the momentum row the node owns (u nodes,
 * then v nodes; 0 for nodes without a row of their own) */
__global__ void __launch_bounds__(BLK) k_free_nodes(DevAsm a, const unsigned char *free_row, unsigned char *free_node) {
    const int eq = blockIdx.x * BLK + threadIdx.x;
    if (eq < a.e.neq_mom) free_node[a.e.mom_node[eq]] = free_row[eq];
}

int mdz_launch_free_rows(int kind, const DevAsm &a, DevBlock *A, DevBlock *B, hipStream_t s) {
    if (!A->free_row) return MDZ_OK;
    const int nm = a.e.neq_mom;
    if (nm <= 0) return MDZ_OK;
    if (A->maxrow > FREE_SLOT - 1 || B->maxrow > FREE_SLOT - 1) {
        /* rows beyond the scratch slot: every row takes the general kernels */
        if (hipMemsetAsync(A->free_row, 0, nm, s) != hipSuccess) return MDZ_EHIP;
        return MDZ_OK;
    }
    hipLaunchKernelGGL(k_free_rows, dim3(mdz_div_up(nm, 64)), dim3(64), 0, s, kind, a, A->free_row);
    if (A->free_node) {
        const int nn = a.g.Nx * a.g.nzvx + a.g.nxvz * a.g.Nz;
        hipLaunchKernelGGL(k_fill_bytes, dim3(mdz_div_up(nn, BLK)), dim3(BLK), 0, s, A->free_node, nn);
        hipLaunchKernelGGL(k_free_nodes, dim3(mdz_div_up(nm, BLK)), dim3(BLK), 0, s, a, (const unsigned char *)A->free_row,
                           A->free_node);
    }
    return MDZ_OK;
}

int mdz_shape_valid(const LaunchShape &sh) {
    return (sh.rheo == 64 || sh.rheo == 128 || sh.rheo == 256) &&
           (sh.pic == 0 || sh.pic == 64 || sh.pic == 128 || sh.pic == 256) &&
           (sh.jac == 0 || sh.jac == 64 || sh.jac == 128);
}

void mdz_launch_values(int kind, const DevAsm &a, DevBlock *A, DevBlock *B, DevBlock *C, DevBlock *D, int vblk,
                       hipStream_t s) {
    int nm = a.e.neq_mom, ncnt = a.e.neq_cont;
    if (nm > 0) {
        const bool fits = kind == 0 ? A->maxrow <= PIC_CAPA && B->maxrow <= PIC_CAPB
                                    : A->maxrow <= JAC_CAPA && B->maxrow <= JAC_CAPB;
        const int v = fits ? vblk : 0;
        /* the staged kernels also take the continuity rows; 64-row blocks
         * take the split pass where the free-row flags and the list of
         * general waves are built */
        const bool split = A->free_row && A->gen_waves;
        if (kind == 0 && v == 64 && split) { launch_split<0, PIC_CAPA, PIC_CAPB>(a, A, B, C, D, s); return; }
        if (kind == 1 && v == 64 && split) { launch_split<1, JAC_CAPA, JAC_CAPB>(a, A, B, C, D, s); return; }
        if (kind == 0 && v == 64) { launch_staged<0, 64, PIC_CAPA, PIC_CAPB>(a, A, B, C, D, s); return; }
        if (kind == 0 && v == 128) { launch_staged<0, 128, PIC_CAPA, PIC_CAPB>(a, A, B, C, D, s); return; }
        if (kind == 0 && v == 256) { launch_staged<0, 256, PIC_CAPA, PIC_CAPB>(a, A, B, C, D, s); return; }
        if (kind == 1 && v == 64) { launch_staged<1, 64, JAC_CAPA, JAC_CAPB>(a, A, B, C, D, s); return; }
        if (kind == 1 && v == 128) { launch_staged<1, 128, JAC_CAPA, JAC_CAPB>(a, A, B, C, D, s); return; }
        if (kind == 0)
            hipLaunchKernelGGL(k_values_mom_direct<0>, dim3(mdz_div_up(nm, BLK)), dim3(BLK), 0, s, a, *A, *B);
        else
            hipLaunchKernelGGL(k_values_mom_direct<1>, dim3(mdz_div_up(nm, BLK)), dim3(BLK), 0, s, a, *A, *B);
    }
    if (ncnt > 0) hipLaunchKernelGGL(k_values_cont, dim3(mdz_div_up(ncnt, BLK)), dim3(BLK), 0, s, a, *C, *D);
}

void mdz_launch_residual(int kind, const DevAsm &a, DevBlock *A, DevBlock *C, DevBlock *D, hipStream_t s) {
    int nm = a.e.neq_mom, ncnt = a.e.neq_cont;
    if (nm > 0) {
        const dim3 grid(mdz_div_up(nm, BLK));
        const NormSlots ns{};
        if (kind == 0) {
            if (A->free_row) hipLaunchKernelGGL((k_residual_mom<0, true, false>), grid, dim3(BLK), 0, s, a, *A, ns);
            hipLaunchKernelGGL((k_residual_mom<0, false, false>), grid, dim3(BLK), 0, s, a, *A, ns);
        } else {
            if (A->free_row) hipLaunchKernelGGL((k_residual_mom<1, true, false>), grid, dim3(BLK), 0, s, a, *A, ns);
            hipLaunchKernelGGL((k_residual_mom<1, false, false>), grid, dim3(BLK), 0, s, a, *A, ns);
        }
    }
    if (ncnt > 0)
        hipLaunchKernelGGL(k_residual_cont<false>, dim3(mdz_div_up(ncnt, BLK)), dim3(BLK), 0, s, kind, a, *C, *D,
                           NormSlots{});
}

/* flag[w] = 1 when wave w (rows 64 w .. 64 w + 63) holds a row that is not free */
__global__ void __launch_bounds__(BLK) k_general_wave_flags(const unsigned char *free_row, int nm, int *flag) {
    const int w = blockIdx.x * BLK + threadIdx.x;
    if (w >= mdz_div_up(nm, 64)) return;
    int f = 0;
    for (int r = w * 64; r < min(nm, w * 64 + 64); r++) f |= free_row[r] == 0;
    flag[w] = f;
}

/* list[pos[w]] = w for the flagged waves (pos: exclusive scan of the flags, pos[nw] = total) */
__global__ void __launch_bounds__(BLK) k_general_wave_list(const int *pos, int nwv, int *list) {
    const int w = blockIdx.x * BLK + threadIdx.x;
    if (w < nwv && pos[w + 1] != pos[w]) list[pos[w]] = w;
}

int mdz_build_general_waves(DevBlock *A, int nm, int *scratch, size_t scratch_len, hipStream_t s) {
    A->n_gen = 0;
    if (nm <= 0) return MDZ_OK;
    if (!A->free_row || !A->gen_waves) return MDZ_EINVAL;
    const int nwv = mdz_div_up(nm, 64);
    int *list = A->gen_waves, *pos = A->gen_waves + nwv + 1;
    hipLaunchKernelGGL(k_general_wave_flags, dim3(mdz_div_up(nwv, BLK)), dim3(BLK), 0, s,
                       (const unsigned char *)A->free_row, nm, pos);
    int total = 0;
    int rc = mdz_scan_exclusive(pos, nwv, scratch, scratch_len, s, &total);
    if (rc) return rc;
    if (hipMemcpyAsync(pos + nwv, &total, sizeof(int), hipMemcpyHostToDevice, s) != hipSuccess) return MDZ_EHIP;
    hipLaunchKernelGGL(k_general_wave_list, dim3(mdz_div_up(nwv, BLK)), dim3(BLK), 0, s, (const int *)pos, nwv, list);
    if (hipStreamSynchronize(s) != hipSuccess) return MDZ_EHIP;
    A->n_gen = total;
    return MDZ_OK;
}

size_t mdz_residual_norm_partials(int nm, int n_gen, int ncnt) {
    return 4 * ((size_t)mdz_div_up(nm, BLK) + (size_t)n_gen) + 2 * (size_t)mdz_div_up(ncnt, BLK);
}

/* one block per family: the slots of its sums and counts, in slot order;
 * copy6 (optional): a second place for them, in device or pinned host
 * memory, so that a caller needs no copy after the launch (5 us) */
__global__ void __launch_bounds__(1024) k_norms_final_slots(const double *partial, int nsm, int nsc, double *out6,
                                                            double *copy6) {
    const int f = blockIdx.x;
    const double *ps = f == 2 ? partial + 4 * (size_t)nsm : partial + 2 * f * (size_t)nsm;
    const int n = f == 2 ? nsc : nsm;
    const double *pc = ps + n;
    double s = 0, c = 0;
    /* unrolled so that the loads of several iterations are in flight; the
     * additions keep their order */
#pragma unroll 8
    for (int i = threadIdx.x; i < n; i += 1024) { s += ps[i]; c += pc[i]; }
    __shared__ double ws[1024 / 64][2];
    s = wave_sum(s);
    c = wave_sum(c);
    if ((threadIdx.x & 63) == 0) { ws[threadIdx.x >> 6][0] = s; ws[threadIdx.x >> 6][1] = c; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double ts = 0, tc = 0;
        for (int q = 0; q < 1024 / 64; q++) { ts += ws[q][0]; tc += ws[q][1]; }
        out6[f] = ts;
        out6[3 + f] = tc;
        if (copy6) {
            copy6[f] = ts;
            copy6[3 + f] = tc;
        }
    }
}

int mdz_launch_residual_norms(int kind, const DevAsm &a, DevBlock *A, DevBlock *C, DevBlock *D, double *partial,
                              size_t partial_len, double *out6, hipStream_t s, int d_scaled, double *copy6) {
    const int nm = a.e.neq_mom, ncnt = a.e.neq_cont;
    if (nm > 0 && (!A->free_row || !A->gen_waves)) return MDZ_EINVAL;
    if (kind == 0 && nm > 0 && A->free_node && a.d11p == a.d22p) {
        /* tiles for the free momentum rows and every continuity row, then
         * the general rows of the listed waves */
        const int ntx = mdz_div_up(a.g.Nx + 1, RT_TX), ntz = mdz_div_up(a.g.Nz + 1, RT_TZ), nt = ntx * ntz;
        const int ngen = A->n_gen;
        if ((size_t)(4 * (nt + ngen) + 2 * nt) <= partial_len) {
            NormSlots ns{partial, nt + ngen, nt, nt, A->gen_waves};
            const int ngb = mdz_div_up(ngen, RT_TX * RT_TZ / 64);
            hipLaunchKernelGGL(k_residual_tile, dim3(ngb + nt), dim3(RT_TX * RT_TZ), 0, s, a, *A, *C, *D,
                               (const unsigned char *)A->free_node, d_scaled, ntx, ngb, ns);
            hipLaunchKernelGGL(k_norms_final_slots, dim3(3), dim3(1024), 0, s, (const double *)partial, nt + ngen, nt,
                               out6, copy6);
            return MDZ_OK;
        }
    }
    const int nbf = mdz_div_up(nm, BLK), ngen = nm > 0 ? A->n_gen : 0, nbc = mdz_div_up(ncnt, BLK);
    if (mdz_residual_norm_partials(nm, ngen, ncnt) > partial_len) return MDZ_ENOMEM;
    NormSlots ns{partial, nbf + ngen, nbc, 0, A->gen_waves};
    if (nm > 0) {
        if (kind == 0) hipLaunchKernelGGL((k_residual_mom<0, true, true>), dim3(nbf), dim3(BLK), 0, s, a, *A, ns);
        else hipLaunchKernelGGL((k_residual_mom<1, true, true>), dim3(nbf), dim3(BLK), 0, s, a, *A, ns);
        if (ngen > 0) {
            ns.slot0 = nbf;
            if (kind == 0) hipLaunchKernelGGL((k_residual_mom<0, false, true>), dim3(ngen), dim3(64), 0, s, a, *A, ns);
            else hipLaunchKernelGGL((k_residual_mom<1, false, true>), dim3(ngen), dim3(64), 0, s, a, *A, ns);
        }
    }
    if (ncnt > 0) hipLaunchKernelGGL(k_residual_cont<true>, dim3(nbc), dim3(BLK), 0, s, kind, a, *C, *D, ns);
    hipLaunchKernelGGL(k_norms_final_slots, dim3(3), dim3(1024), 0, s, (const double *)partial, nbf + ngen, nbc, out6,
                       copy6);
    return MDZ_OK;
}

/* ------------------------------------------------------------------ */
/* diagonal scaling (StokesRoutines.c:1232-1342)                        */
/* ------------------------------------------------------------------ */
/* X.d[i] = last diagonal entry of row i of X (kept when there is none);
 * Y.d[i] = X.d[i] */
__global__ void __launch_bounds__(BLK) k_extract_diag(DevBlock X, DevBlock Y, int nrows) {
    const int i = blockIdx.x * BLK + threadIdx.x;
    if (i >= nrows) return;
    double d = X.d[i];
    for (int k = X.Ic[i]; k < X.Ic[i + 1]; k++)
        if (X.J[k] == i) d = X.A[k];
    X.d[i] = d;
    Y.d[i] = d;
}

/* row i: b, F scaled by M.d[i]; values by dr[i] * dc[j] */
__global__ void __launch_bounds__(BLK) k_scale_rows(DevBlock M, int nrows, const double *__restrict__ dr,
                                                    const double *__restrict__ dc) {
    const int i = blockIdx.x * BLK + threadIdx.x;
    if (i >= nrows) return;
    const double di = M.d[i];
    M.b[i] *= di;
    M.F[i] *= di;
    const double ri = dr[i];
    for (int k = M.Ic[i]; k < M.Ic[i + 1]; k++) M.A[k] *= ri * dc[M.J[k]];
}

void mdz_launch_extract_diagonal(DevBlock *A, DevBlock *B, DevBlock *C, DevBlock *D, hipStream_t s) {
    int nm = A->neq, nc = C->neq;
    if (nm > 0) hipLaunchKernelGGL(k_extract_diag, dim3(mdz_div_up(nm, BLK)), dim3(BLK), 0, s, *A, *B, nm);
    if (nc > 0) hipLaunchKernelGGL(k_extract_diag, dim3(mdz_div_up(nc, BLK)), dim3(BLK), 0, s, *D, *C, nc);
}

void mdz_launch_scale_matrix(DevBlock *A, DevBlock *B, DevBlock *C, DevBlock *D, hipStream_t s) {
    int nm = A->neq, nc = C->neq;
    if (nm > 0) {
        hipLaunchKernelGGL(k_scale_rows, dim3(mdz_div_up(nm, BLK)), dim3(BLK), 0, s, *A, nm, (const double *)A->d,
                           (const double *)A->d);
        hipLaunchKernelGGL(k_scale_rows, dim3(mdz_div_up(nm, BLK)), dim3(BLK), 0, s, *B, nm, (const double *)A->d,
                           (const double *)D->d);
    }
    if (nc > 0) {
        hipLaunchKernelGGL(k_scale_rows, dim3(mdz_div_up(nc, BLK)), dim3(BLK), 0, s, *C, nc, (const double *)D->d,
                           (const double *)A->d);
        hipLaunchKernelGGL(k_scale_rows, dim3(mdz_div_up(nc, BLK)), dim3(BLK), 0, s, *D, nc, (const double *)D->d,
                           (const double *)D->d);
    }
}

/* ------------------------------------------------------------------ */
/* norms                                                                */
/* ------------------------------------------------------------------ */
#define NRM_BLK 256

/* per node family: F^2 sums and DOF counts, residual fields, F *= d.
 * block partials: [3 families][2 quantities][nblocks] */
__global__ void __launch_bounds__(NRM_BLK) k_norms(DevAsm a, DevBlock A, DevBlock D, double *partial, int nbu,
                                                   int nbv, int nbp) {
    const DevGrid &g = a.g;
    int nu = g.Nx * g.nzvx, nw = g.nxvz * g.Nz, nc = g.ncx * g.ncz;
    int bid = blockIdx.x, fam, base;
    if (bid < nbu) { fam = 0; base = bid; }
    else if (bid < nbu + nbv) { fam = 1; base = bid - nbu; }
    else { fam = 2; base = bid - nbu - nbv; }
    int i = base * NRM_BLK + threadIdx.x;
    double s = 0.0, cnt = 0.0;
    if (fam == 0 && i < nu) {
        int t = g.BCu[i];
        if (t != 0 && t != 30 && t != 11 && t != 13 && t != -12) {
            int e = a.e.eqn_u[i];
            double f = A.F[e];
            s = f * f; cnt = 1.0;
            g.ru[i] = f;
            A.F[e] = f * A.d[e];
        }
    } else if (fam == 1 && i < nw) {
        int t = g.BCv[i];
        if (t != 0 && t != 30 && t != 11 && t != 13 && t != -12) {
            int e = a.e.eqn_v[i];
            double f = A.F[e];
            s = f * f; cnt = 1.0;
            g.rv[i] = f;
            A.F[e] = f * A.d[e];
        }
    } else if (fam == 2 && i < nc) {
        int t = g.BCp[i];
        if (t != 0 && t != 30 && t != 31) {
            int e = a.e.eqn_p[i] - a.e.neq_mom;
            double f = D.F[e];
            s = f * f; cnt = 1.0;
            g.rp[i] = f;
            D.F[e] = f * D.d[e];
        }
    }
    __shared__ double ws[NRM_BLK / 64][2];
    s = wave_sum(s);
    cnt = wave_sum(cnt);
    int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { ws[w][0] = s; ws[w][1] = cnt; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double ts = 0, tc = 0;
        for (int q = 0; q < NRM_BLK / 64; q++) { ts += ws[q][0]; tc += ws[q][1]; }
        int nbf = fam == 0 ? nbu : (fam == 1 ? nbv : nbp);
        int off = fam == 0 ? 0 : (fam == 1 ? 2 * nbu : 2 * (nbu + nbv));
        partial[off + base] = ts;
        partial[off + nbf + base] = tc;
    }
}

/* one block per family (u, v, p): fixed summation order, so the norms are
 * deterministic */
#define NRM_FIN 1024
__global__ void __launch_bounds__(NRM_FIN) k_norms_final(const double *partial, int nbu, int nbv, int nbp, double *out6) {
    const int f = blockIdx.x;
    const int nbf = f == 0 ? nbu : (f == 1 ? nbv : nbp);
    const int off = f == 0 ? 0 : (f == 1 ? 2 * nbu : 2 * (nbu + nbv));
    double s = 0, c = 0;
    for (int i = threadIdx.x; i < nbf; i += NRM_FIN) { s += partial[off + i]; c += partial[off + nbf + i]; }
    __shared__ double ws[NRM_FIN / 64][2];
    s = wave_sum(s);
    c = wave_sum(c);
    if ((threadIdx.x & 63) == 0) { ws[threadIdx.x >> 6][0] = s; ws[threadIdx.x >> 6][1] = c; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double ts = 0, tc = 0;
        for (int q = 0; q < NRM_FIN / 64; q++) { ts += ws[q][0]; tc += ws[q][1]; }
        out6[f] = ts;
        out6[3 + f] = tc;
    }
}

size_t mdz_norm_partials(const DevGrid &g) {
    int nbu = mdz_div_up(g.Nx * g.nzvx, NRM_BLK), nbv = mdz_div_up(g.nxvz * g.Nz, NRM_BLK), nbp = mdz_div_up(g.ncx * g.ncz, NRM_BLK);
    return 2 * (size_t)(nbu + nbv + nbp);
}

void mdz_launch_norms(const DevAsm &a, DevBlock *A, DevBlock *D, double *partial, double *out6, hipStream_t s) {
    const DevGrid &g = a.g;
    int nbu = mdz_div_up(g.Nx * g.nzvx, NRM_BLK), nbv = mdz_div_up(g.nxvz * g.Nz, NRM_BLK), nbp = mdz_div_up(g.ncx * g.ncz, NRM_BLK);
    hipLaunchKernelGGL(k_norms, dim3(nbu + nbv + nbp), dim3(NRM_BLK), 0, s, a, *A, *D, partial, nbu, nbv, nbp);
    hipLaunchKernelGGL(k_norms_final, dim3(3), dim3(NRM_FIN), 0, s, (const double *)partial, nbu, nbv, nbp, out6);
}
