/*
 * mdz_rheology.hip -- gfx950 kernels of the rheology half of the
 * Newton-iteration path: strain rates, centroid->vertex interpolation,
 * grid rheology (one lane per centroid / vertex, phase loop, averaging),
 * D-tensor assembly (Picard and consistent tangent) and the momentum /
 * continuity right-hand sides.
 *
 *   k_strain_tile                                   RheologyDensity.c:1902-1982 (+ GridRoutines.c:106)
 *   k_interp_c2v                                    GridRoutines.c:106-196
 *   k_rheo_cells / k_rheo_vertices                  RheologyDensity.c:961-1415
 *   dtensor_cell / dtensor_vertex (k_rhs_dtensor)   RheologyDensity.c:713-954
 *   rhs_u / rhs_v / rhs_p (k_rhs_dtensor)           StokesRoutines.c:922-1128
 *
 * All HBM-bound except the rheology, which is FP64-VALU bound
 * (transcendentals of the local iterations).
 */
#include "mdz_kernels.h"
#include "mdz_viscosity.h"

#define BLK 256

/* ---------------------------------------------------------------- */
/* strain rates                                                      */
/* ---------------------------------------------------------------- */
/* padded-centroid value at padded coordinates (i, j), i in [0, ncx+1],
 * j in [0, ncz+1]: zero-flux (or periodic in x) ghost ring */
__device__ __forceinline__ double padded(const double *__restrict__ c, int i, int j, int ncx, int ncz, int per) {
    int ci, cj = j - 1;
    if (i == 0) ci = per ? ncx - 1 : 0;
    else if (i == ncx + 1) ci = per ? 0 : ncx - 1;
    else ci = i - 1;
    cj = cj < 0 ? 0 : (cj > ncz - 1 ? ncz - 1 : cj);
    return c[ci + cj * ncx];
}

/* Up to four centroid fields interpolated to vertices in one pass. */
__global__ void __launch_bounds__(BLK) k_interp_c2v(DevGrid g, int per, int nf, const double *__restrict__ s0,
                                                    double *__restrict__ d0, const double *__restrict__ s1,
                                                    double *__restrict__ d1, const double *__restrict__ s2,
                                                    double *__restrict__ d2, const double *__restrict__ s3,
                                                    double *__restrict__ d3, const double *__restrict__ s4,
                                                    double *__restrict__ d4) {
    int c1 = xcd_tile() * BLK + threadIdx.x;
    int Nx = g.Nx;
    if (c1 >= Nx * g.Nz) return;
    int k = c1 % Nx, l = c1 / Nx;
    bool air = g.BCg[c1] == 30;
    const double *src[5] = {s0, s1, s2, s3, s4};
    double *dst[5] = {d0, d1, d2, d3, d4};
#pragma unroll
    for (int f = 0; f < 5; f++) {
        if (f >= nf) break;
        double v = 0.0;
        if (!air) {
            const double *c = src[f];
            /* same summation order as the padded-array formulation */
            v = 0.25 * (padded(c, k, l, g.ncx, g.ncz, per) + padded(c, k + 1, l, g.ncx, g.ncz, per)
                        + padded(c, k, l + 1, g.ncx, g.ncz, per) + padded(c, k + 1, l + 1, g.ncx, g.ncz, per));
        }
        dst[f][c1] = v;
    }
}

/* ---------------------------------------------------------------- */
/* strain rates and vertex interpolation in one pass                 */
/* ---------------------------------------------------------------- */
/* Strain rates of centroid c0 (RheologyDensity.c:1914-1936), 0 for air and
 * surface-pressure cells; the velocity loads do not wait for the tag load. */
struct CellStrain {
    double div, exx, ezz;
};
__device__ __forceinline__ CellStrain cell_strain(const DevGrid &g, int c0) {
    const int Ncx = g.ncx, Nx = g.Nx;
    const int k = c0 % Ncx, l = c0 / Ncx;
    const int c1 = k + l * Nx, c2 = k + l * (Nx + 1);
    const double dudx = (g.u_in[c1 + 1 + Nx] - g.u_in[c1 + Nx]) / g.dx;
    const double dvdz = (g.v_in[c2 + Nx + 1 + 1] - g.v_in[c2 + 1]) / g.dz;
    const double div = dudx + dvdz;
    const double exx = dudx - 1.0 / 3.0 * div;
    const double ezz = (g.v_in[c2 + 1 + (Nx + 1)] - g.v_in[c2 + 1]) / g.dz - 1.0 / 3.0 * div;
    const int t = g.BCp[c0];
    const bool in = t != 30 && t != 31;
    return CellStrain{in ? div : 0.0, in ? exx : 0.0, in ? ezz : 0.0};
}

/* index of the centroid behind padded coordinates (i, j) (padded()) */
__device__ __forceinline__ int padded_index(int i, int j, int ncx, int ncz, int per) {
    int ci, cj = j - 1;
    if (i == 0) ci = per ? ncx - 1 : 0;
    else if (i == ncx + 1) ci = per ? 0 : ncx - 1;
    else ci = i - 1;
    cj = cj < 0 ? 0 : (cj > ncz - 1 ? ncz - 1 : cj);
    return ci + cj * ncx;
}

/* StrainRateComponents (RheologyDensity.c:1902-1982) and, with INTERP5,
 * the vertex values of div_u, T, P, d and phi that NonNewtonianViscosity-
 * Grid interpolates first (RheologyDensity.c:979-983, GridRoutines.c:106),
 * in one launch over tiles of ST_TX x ST_TZ vertices (and the centroids of
 * the same indices), one of each per thread.  A block stages the
 * velocities, the tags and (with INTERP5) T, P, d, phi of its tile with a
 * one-node halo in LDS (coalesced row loads), computes the strain rates of
 * the tile's centroids and of the ring below and to the left of it and the
 * shear rates of the tile's vertices and of the ring above and to the
 * right, once each, in LDS; a vertex then averages the strain rates of its
 * four padded centroids, a centroid the shear rates of its four vertices.
 * Nothing is written and read back between kernels, and each output takes
 * the expressions and summation order of the reference's sequence (strain
 * rates, then padded 4-point averages).  Periodic-x vertices on the left
 * and right edges average centroids of the far edge, outside the tile:
 * those are read from global memory. */
#define ST_TX 64
#define ST_TZ 4
#define ST_HX (ST_TX + 2) /* u and v tile widths */
#define ST_HZ (ST_TZ + 2) /* u and v tile heights */
#define ST_CX (ST_TX + 1) /* centroid ring [i0 - 1, i0 + TX) and vertex ring [i0, i0 + TX] widths */
#define ST_CZ (ST_TZ + 1)

/* the tile of one block in LDS */
struct StrainTile {
    double u[ST_HZ][ST_HX];                      /* u(x = i0 - 1 + a, z = j0 + b) */
    double v[ST_HZ][ST_HX];                      /* v(x = i0 + a, z = j0 - 1 + b) */
    double div[ST_CZ][ST_CX], exx[ST_CZ][ST_CX], ezz[ST_CZ][ST_CX]; /* centroid (i0 - 1 + a, j0 - 1 + b) */
    double exz[ST_CZ][ST_CX];                    /* vertex (i0 + a, j0 + b) */
    double f[4][ST_CZ][ST_CX];                   /* T, P, d, phi at centroid (i0 - 1 + a, j0 - 1 + b) */
    signed char tu[ST_HZ][ST_HX], tv[ST_HZ][ST_HX]; /* BCu, BCv at the u, v nodes */
    signed char tg[ST_CZ][ST_CX];                /* BCg at vertex (i0 + a, j0 + b) */
    signed char tp[ST_CZ][ST_CX];                /* BCp at centroid (i0 - 1 + a, j0 - 1 + b) */
};

template <bool INTERP5>
__global__ void __launch_bounds__(256) k_strain_tile(DevGrid g, int per, int ntx) {
    __shared__ StrainTile T;
    const int Nx = g.Nx, Nz = g.Nz, ncx = g.ncx, ncz = g.ncz, nxv = Nx + 1;
    const int t = xcd_tile();
    const int i0 = (t % ntx) * ST_TX, j0 = (t / ntx) * ST_TZ;
    const int tid = threadIdx.x;
    /* 1. velocities, tags and centroid fields of the tile and its halo: all
     * loads of the thread into registers first (one round trip), then the
     * LDS stores */
    constexpr int NUV = (ST_HZ * ST_HX + 255) / 256, NR = (ST_CZ * ST_CX + 255) / 256;
    double ul[NUV], vl[NUV], fl[NR][4];
    signed char tul[NUV], tvl[NUV], tgl[NR], tpl[NR];
#pragma unroll
    for (int r = 0; r < NUV; r++) {
        const int q = tid + 256 * r, a = q % ST_HX, b = q / ST_HX;
        const int xu = i0 - 1 + a, zu = j0 + b;
        const bool inu = q < ST_HZ * ST_HX && xu >= 0 && xu < Nx && zu <= Nz;
        const int iu = inu ? xu + zu * Nx : 0;
        ul[r] = g.u_in[iu];
        tul[r] = inu ? g.BCu[iu] : (signed char)30;
        const int xv = i0 + a, zv = j0 - 1 + b;
        const bool inv = q < ST_HZ * ST_HX && xv < nxv && zv >= 0 && zv < Nz;
        const int iv = inv ? xv + zv * nxv : 0;
        vl[r] = g.v_in[iv];
        tvl[r] = inv ? g.BCv[iv] : (signed char)30;
    }
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const int q = tid + 256 * r, a = q % ST_CX, b = q / ST_CX;
        const int xg = i0 + a, zg = j0 + b;
        const bool ing = q < ST_CZ * ST_CX && xg < Nx && zg < Nz;
        tgl[r] = ing ? g.BCg[xg + zg * Nx] : (signed char)30;
        const int xc = i0 - 1 + a, zc = j0 - 1 + b;
        const bool inc = q < ST_CZ * ST_CX && xc >= 0 && xc < ncx && zc >= 0 && zc < ncz;
        const int c = inc ? xc + zc * ncx : 0;
        tpl[r] = inc ? g.BCp[c] : (signed char)30;
        if (INTERP5) {
            fl[r][0] = g.T[c];
            fl[r][1] = g.p_in[c];
            fl[r][2] = g.d0_n[c];
            fl[r][3] = g.phi0_n[c];
        }
    }
#pragma unroll
    for (int r = 0; r < NUV; r++) {
        const int q = tid + 256 * r;
        if (q < ST_HZ * ST_HX) {
            const int a = q % ST_HX, b = q / ST_HX;
            T.u[b][a] = ul[r];
            T.tu[b][a] = tul[r];
            T.v[b][a] = vl[r];
            T.tv[b][a] = tvl[r];
        }
    }
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const int q = tid + 256 * r;
        if (q < ST_CZ * ST_CX) {
            const int a = q % ST_CX, b = q / ST_CX;
            T.tg[b][a] = tgl[r];
            T.tp[b][a] = tpl[r];
            if (INTERP5)
#pragma unroll
                for (int f = 0; f < 4; f++) T.f[f][b][a] = fl[r][f];
        }
    }
    __syncthreads();
    /* 2. strain rates of the centroid ring (the expressions of cell_strain)
     * and shear rates of the vertex ring (RheologyDensity.c:1939-1954: both
     * terms formed for every vertex and applied by their tags; e never
     * holds -0, so e + 0 leaves it unchanged) */
    for (int q = tid; q < ST_CZ * ST_CX; q += 256) {
        const int a = q % ST_CX, b = q / ST_CX;
        const double dudx = (T.u[b][a + 1] - T.u[b][a]) / g.dx;
        const double dvdz = (T.v[b + 1][a] - T.v[b][a]) / g.dz;
        const double div = dudx + dvdz;
        const double exx = dudx - 1.0 / 3.0 * div;
        const double ezz = (T.v[b + 1][a] - T.v[b][a]) / g.dz - 1.0 / 3.0 * div;
        const bool in = T.tp[b][a] != 30 && T.tp[b][a] != 31;
        T.div[b][a] = in ? div : 0.0;
        T.exx[b][a] = in ? exx : 0.0;
        T.ezz[b][a] = in ? ezz : 0.0;
        const double du = 0.5 * (T.u[b + 1][a + 1] - T.u[b][a + 1]) / g.dz;
        const double dv = 0.5 * (T.v[b + 1][a + 1] - T.v[b + 1][a]) / g.dx;
        double e = 0.0;
        if (T.tg[b][a] != 30) {
            e += (T.tu[b][a + 1] != 30 && T.tu[b + 1][a + 1] != 30) ? du : 0.0;
            e += (T.tv[b + 1][a] != 30 && T.tv[b + 1][a + 1] != 30) ? dv : 0.0;
        }
        T.exz[b][a] = e;
    }
    __syncthreads();
    /* 3. one vertex and one centroid per thread */
    const int tx = tid % ST_TX, ty = tid / ST_TX;
    const int i = i0 + tx, j = j0 + ty;
    if (i < Nx && j < Nz) {
        const int c1 = i + j * Nx;
        const bool air = T.tg[ty][tx] == 30;
        const int pc[4] = {padded_index(i, j, ncx, ncz, per), padded_index(i + 1, j, ncx, ncz, per),
                           padded_index(i, j + 1, ncx, ncz, per), padded_index(i + 1, j + 1, ncx, ncz, per)};
        CellStrain cs[4];
        double fv[4][4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int a = pc[k] % ncx - (i0 - 1), b = pc[k] / ncx - (j0 - 1);
            if (a >= 0 && a < ST_CX && b >= 0 && b < ST_CZ) {
                cs[k] = CellStrain{T.div[b][a], T.exx[b][a], T.ezz[b][a]};
                if (INTERP5)
#pragma unroll
                    for (int f = 0; f < 4; f++) fv[f][k] = T.f[f][b][a];
            } else {
                /* periodic wrap: a centroid of the far edge, from global memory */
                cs[k] = cell_strain(g, pc[k]);
                if (INTERP5) {
                    fv[0][k] = g.T[pc[k]];
                    fv[1][k] = g.p_in[pc[k]];
                    fv[2][k] = g.d0_n[pc[k]];
                    fv[3][k] = g.phi0_n[pc[k]];
                }
            }
        }
        g.exz[c1] = T.exz[ty][tx];
        g.exxd_s[c1] = air ? 0.0 : 0.25 * (cs[0].exx + cs[1].exx + cs[2].exx + cs[3].exx);
        g.ezzd_s[c1] = air ? 0.0 : 0.25 * (cs[0].ezz + cs[1].ezz + cs[2].ezz + cs[3].ezz);
        if (INTERP5) {
            g.div_u_s[c1] = air ? 0.0 : 0.25 * (cs[0].div + cs[1].div + cs[2].div + cs[3].div);
            double *dst[4] = {g.T_s, g.P_s, g.d0_s, g.phi0_s};
#pragma unroll
            for (int f = 0; f < 4; f++) dst[f][c1] = air ? 0.0 : 0.25 * (fv[f][0] + fv[f][1] + fv[f][2] + fv[f][3]);
        }
    }
    if (i < ncx && j < ncz) {
        const int c0 = i + j * ncx;
        /* exz_n: the mean of the shear rates of the cell's non-air vertices */
        double sm = 0.0, n = 0.0;
        const int tc = T.tp[ty + 1][tx + 1];
        if (tc != 30 && tc != 31) {
            const bool a0 = T.tg[ty][tx] != 30, a1 = T.tg[ty][tx + 1] != 30, a2 = T.tg[ty + 1][tx] != 30,
                       a3 = T.tg[ty + 1][tx + 1] != 30;
            sm += a0 ? T.exz[ty][tx] : 0.0; n += a0 ? 1 : 0;
            sm += a1 ? T.exz[ty][tx + 1] : 0.0; n += a1 ? 1 : 0;
            sm += a2 ? T.exz[ty + 1][tx] : 0.0; n += a2 ? 1 : 0;
            sm += a3 ? T.exz[ty + 1][tx + 1] : 0.0; n += a3 ? 1 : 0;
            if (n > 0) sm /= n;
        }
        g.div_u[c0] = T.div[ty + 1][tx + 1];
        g.exxd[c0] = T.exx[ty + 1][tx + 1];
        g.ezzd[c0] = T.ezz[ty + 1][tx + 1];
        g.exz_n[c0] = sm;
    }
}

/* ---------------------------------------------------------------- */
/* grid rheology                                                     */
/* ---------------------------------------------------------------- */

/* Effective visco-elastic strain rates through the inverse anisotropy
 * tensor (RheologyDensity.c:1061-1094). */
__device__ __forceinline__ void ve_rates(const DevParams &prm, double nx, double nz, double af, double fs,
                                         double exx, double ezz, double exz, double sxx0, double szz0,
                                         double sxz0, double etae, double &Exx, double &Ezz, double &Exz,
                                         double &Gxx, double &Gzz, double &Gxz) {
    double ani = 0.0, d0 = 0.0, d1 = 0.0;
    if (prm.aniso != 0) {
        if (prm.aniso_fstrain == 0) ani = 1.0 - 1.0 / af;
        if (prm.aniso_fstrain == 1) ani = 1.0 - 1.0 / fs;
        d0 = 2.0 * pow(nx, 2.0) * pow(nz, 2.0);
        d1 = nx * nz * (-pow(nx, 2.0) + pow(nz, 2.0));
    }
    double Da11 = 2.0 - 2.0 * ani * d0, Da12 = 2.0 * ani * d0, Da13 = 2.0 * ani * d1;
    double Da22 = 2.0 - 2.0 * ani * d0, Da23 = -2.0 * ani * d1, Da33 = 1.0 + 2.0 * ani * (d0 - 0.5);
    double a11 = Da33 * Da22 - Da23 * Da23, a12 = Da13 * Da23 - Da33 * Da12, a13 = Da12 * Da23 - Da13 * Da22;
    double a22 = Da33 * Da11 - Da13 * Da13, a23 = Da12 * Da13 - Da11 * Da23, a33 = Da11 * Da22 - Da12 * Da12;
    double det = (Da11 * a11) + (Da12 * a12) + (Da13 * a13);
    double i11 = a11 / det, i12 = a12 / det, i13 = a13 / det, i22 = a22 / det, i23 = a23 / det, i33 = a33 / det;
    Exx = exx + (i11 * sxx0 + i12 * szz0 + i13 * sxz0) / etae;
    Ezz = ezz + (i12 * sxx0 + i22 * szz0 + i23 * sxz0) / etae;
    Exz = exz + (i13 * sxx0 + i23 * szz0 + i33 * sxz0) / 2.0 / etae;
    double gxz = 2.0 * exz + (i13 * sxx0 + i23 * szz0 + i33 * sxz0) / etae;
    Gxx = Exx * (1.0 - ani * d0) + Ezz * ani * d0 + gxz * ani * d1;
    Gzz = Ezz * (1.0 - ani * d0) + Exx * ani * d0 - gxz * ani * d1;
    Gxz = Exx * ani * d1 - Exx * ani * d1 + gxz * (ani * (d0 - 0.5) + 0.5);
}


__device__ __forceinline__ void rheo_cell_generic(const DevGrid &g, const DevParams &prm,
                                                  const mat_prop *__restrict__ mt, const float *__restrict__ guess_n,
                                                  const BlockHist &hist, int c0, int nc) {
    const int average = prm.eta_avg;
    double eta_n = 0, eta_phys_n = 0, VE_n = 0, sxxd = 0, szzd = 0, sxz_n = 0;
    double eII_el = 0, eII_pl = 0, eII_pwl = 0, eII_exp = 0, eII_lin = 0, eII_gbs = 0, eII_cst = 0, d_n = 0;
    double exx_el = 0, ezz_el = 0, exx_diss = 0, ezz_diss = 0;
    double dexx = 0, dezz = 0, dgxz = 0, dp = 0, ddxx = 0, ddzz = 0, ddgxz = 0, ddp = 0;
    double p_corr = 0, div_el = 0, div_pl = 0, div_r = 0, Wtot = 0, Wel = 0, Wdiss = 0, X_n = 0, OverS = 0;
    int t = g.BCp[c0];
    bool active = t != 30 && t != 31;
    if (active) {
        double etae = prm.iselastic == 1 ? prm.dt * g.mu_n[c0] : 1.0;
        double Exx, Ezz, Exz, Gxx, Gzz, Gxz;
        double exxd = g.exxd[c0], ezzd = g.ezzd[c0], exz_c = g.exz_n[c0];
        ve_rates(prm, g.nx0_n[c0], g.nz0_n[c0], g.aniso_factor_n[c0], g.FS_AR_n[c0], exxd, ezzd, exz_c,
                 g.sxxd0[c0], g.szzd0[c0], g.sxz0_n[c0], etae, Exx, Ezz, Exz, Gxx, Gzz, Gxz);
        const double mu = g.mu_n[c0], T = g.T[c0], P = g.p_in[c0], d0 = g.d0_n[c0], phi0 = g.phi0_n[c0];
        const double X0 = g.X0_n[c0], s0xx = g.sxxd0[c0], s0zz = g.szzd0[c0], s0xz = g.sxz0_n[c0];
        const double dil = g.dil_n[c0], fric = g.fric_n[c0], C = g.C_n[c0], P0 = g.p0_n[c0], bet = g.bet_n[c0];
        for (int p = 0; p < prm.Nb_phases; p++) {
            double fr = g.phase_n[(size_t)p * nc + c0];
            if (!(fabs(fr) > 1.0e-13)) continue;
            VGuess gs;
            gs.mode = prm.rheo_mode;
            gs.factor = guess_n ? (double)guess_n[(size_t)p * nc + c0] : 0.0;
            gs.gdot = guess_n ? (double)guess_n[(size_t)(g.nph + p) * nc + c0] : 0.0;
            VOut o;
            mdz_viscosity(p, mu, T, P, d0, phi0, X0, Exx, Ezz, Exz, Gxx, Gzz, Gxz, s0xx, s0zz, s0xz, mt, prm, dil,
                          fric, C, P0, bet, gs, o);
            hist.add(0, o.it_ve & 0xff);
            hist.add(1, o.it_pl);
            hist.add(2, o.it_ve >> 8);
            if (average == 0) {
                eta_n += fr * o.etaVE;
                eta_phys_n += fr * o.eta;
                dexx += fr * o.detadexx;
                dezz += fr * o.detadezz;
                dgxz += fr * o.detadexz / 2.0;
                dp += fr * o.detadp;
            }
            if (average == 0 || average == 2) {
                sxxd += fr * o.txx;
                szzd += fr * o.tzz;
                sxz_n += fr * o.txz;
            }
            VE_n += fr * o.VEcoeff;
            eII_el += fr * o.Eii_el;
            eII_pl += fr * o.Eii_pl;
            eII_pwl += fr * o.Eii_pwl;
            eII_exp += fr * o.Eii_exp;
            eII_lin += fr * o.Eii_lin;
            eII_gbs += fr * o.Eii_gbs;
            eII_cst += fr * o.Eii_cst;
            d_n += fr * 1.0 / o.d1;
            exx_el += fr * o.Exx_el;
            exx_diss += fr * o.Exx_diss;
            ezz_el += fr * o.Ezz_el;
            ezz_diss += fr * o.Ezz_diss;
            double txx1 = o.txx, tzz1 = o.tzz, txz1 = o.txz;
            Wtot += fr * (txx1 * exxd + tzz1 * ezzd + (txx1 + tzz1) * (exxd + ezzd) + 2.0 * txz1 * exz_c);
            Wdiss += fr * (txx1 * o.Exx_diss + tzz1 * o.Ezz_diss + (txx1 + tzz1) * (o.Exx_diss + o.Ezz_diss) + 2.0 * txz1 * o.Exz_diss);
            Wel += fr * (txx1 * o.Exx_el + tzz1 * o.Ezz_el + (txx1 + tzz1) * (o.Exx_el + o.Ezz_el) + 2.0 * txz1 * o.Exz_el);
            ddxx += fr * o.ddivpdexx;
            ddzz += fr * o.ddivpdezz;
            ddgxz += fr * o.ddivpdexz / 2.0;
            ddp += fr * o.ddivpdp;
            p_corr += fr * o.Pcorr;
            div_el += fr * o.div_el;
            div_pl += fr * o.div_pl;
            div_r += fr * o.div_r;
            X_n += fr * o.X1;
            OverS += fr * o.OverS;
            if (average == 1) {
                sxxd += fr * 1.0 / txx1;
                szzd += fr * 1.0 / tzz1;
                sxz_n += fr * 1.0 / txz1;
                eta_n += fr * 1.0 / o.etaVE;
                eta_phys_n += fr * 1.0 / o.eta;
                double e2 = pow(o.etaVE, 2.0);
                dexx += fr * o.detadexx / e2;
                dezz += fr * o.detadezz / e2;
                dgxz += fr * o.detadexz / 2.0 / e2;
                dp += fr * o.detadp / e2;
            }
            if (average == 2) {
                eta_n += fr * log(o.etaVE);
                eta_phys_n += fr * log(o.eta);
                dexx += fr * o.detadexx / o.etaVE;
                dezz += fr * o.detadezz / o.etaVE;
                dgxz += fr * o.detadexz / 2.0 / o.etaVE;
                dp += fr * o.detadp / o.etaVE;
            }
        }
        d_n = 1.0 / d_n;
        if (average == 1) {
            sxxd = 1.0 / sxxd; szzd = 1.0 / szzd; sxz_n = 1.0 / sxz_n;
            eta_n = 1.0 / eta_n; eta_phys_n = 1.0 / eta_phys_n;
            double e2 = pow(eta_n, 2.0);
            dexx *= e2; dezz *= e2; dgxz *= e2; dp *= e2;
        }
        if (average == 2) {
            eta_n = exp(eta_n); eta_phys_n = exp(eta_phys_n);
            dexx *= eta_n; dezz *= eta_n; dgxz *= eta_n; dp *= eta_n;
        }
    }
    g.eta_n[c0] = eta_n; g.eta_phys_n[c0] = eta_phys_n; g.VE_n[c0] = VE_n;
    g.sxxd[c0] = sxxd; g.szzd[c0] = szzd; g.sxz_n[c0] = sxz_n;
    g.eII_el[c0] = eII_el; g.eII_pl[c0] = eII_pl; g.eII_pwl[c0] = eII_pwl; g.eII_exp[c0] = eII_exp;
    g.eII_lin[c0] = eII_lin; g.eII_gbs[c0] = eII_gbs; g.eII_cst[c0] = eII_cst; g.d_n[c0] = d_n;
    g.exx_el[c0] = exx_el; g.exx_diss[c0] = exx_diss; g.ezz_el[c0] = ezz_el; g.ezz_diss[c0] = ezz_diss;
    g.detadexx_n[c0] = dexx; g.detadezz_n[c0] = dezz; g.detadgxz_n[c0] = dgxz; g.detadp_n[c0] = dp;
    g.ddivpdexx_n[c0] = ddxx; g.ddivpdezz_n[c0] = ddzz; g.ddivpdgxz_n[c0] = ddgxz; g.ddivpdp_n[c0] = ddp;
    g.p_corr[c0] = p_corr; g.div_u_el[c0] = div_el; g.div_u_pl[c0] = div_pl; g.div_u_r[c0] = div_r;
    g.Wtot[c0] = Wtot; g.Wel[c0] = Wel; g.Wdiss[c0] = Wdiss;
    if (prm.UnsplitDiffReac == 0) g.X_n[c0] = X_n;
    g.OverS_n[c0] = OverS;
}

__device__ __forceinline__ void rheo_vertex_generic(const DevGrid &g, const DevParams &prm,
                                                    const mat_prop *__restrict__ mt, const float *__restrict__ guess_s,
                                                    const BlockHist &hist, int c1, int nv) {
    const int average = prm.eta_avg;
    double VE_s = 0, sxz = 0, eta_phys_s = 0, eta_s = 0, exz_el = 0, exz_diss = 0;
    double dexx = 0, dezz = 0, dgxz = 0, dp = 0, X_s = 0, OverS = 0;
    if (g.BCg[c1] != 30) {
        double etae = prm.iselastic == 1 ? prm.dt * g.mu_s[c1] : 1.0;
        double Exx, Ezz, Exz, Gxx, Gzz, Gxz;
        ve_rates(prm, g.nx0_s[c1], g.nz0_s[c1], g.aniso_factor_s[c1], g.FS_AR_s[c1], g.exxd_s[c1], g.ezzd_s[c1],
                 g.exz[c1], g.sxxd0_s[c1], g.szzd0_s[c1], g.sxz0[c1], etae, Exx, Ezz, Exz, Gxx, Gzz, Gxz);
        const double mu = g.mu_s[c1], T = g.T_s[c1], P = g.P_s[c1], d0 = g.d0_s[c1], phi0 = g.phi0_s[c1];
        const double X0 = g.X0_s[c1], s0xx = g.sxxd0_s[c1], s0zz = g.szzd0_s[c1], s0xz = g.sxz0[c1];
        const double dil = g.dil_s[c1], fric = g.fric_s[c1], C = g.C_s[c1], P0 = g.p0_s[c1], bet = g.bet_s[c1];
        for (int p = 0; p < prm.Nb_phases; p++) {
            double fr = g.phase_s[(size_t)p * nv + c1];
            if (!(fabs(fr) > 1.0e-13)) continue;
            VGuess gs;
            gs.mode = prm.rheo_mode;
            gs.factor = guess_s ? (double)guess_s[(size_t)p * nv + c1] : 0.0;
            gs.gdot = guess_s ? (double)guess_s[(size_t)(g.nph + p) * nv + c1] : 0.0;
            VOut o;
            mdz_viscosity(p, mu, T, P, d0, phi0, X0, Exx, Ezz, Exz, Gxx, Gzz, Gxz, s0xx, s0zz, s0xz, mt, prm, dil,
                          fric, C, P0, bet, gs, o);
            hist.add(0, o.it_ve & 0xff);
            hist.add(1, o.it_pl);
            hist.add(2, o.it_ve >> 8);
            if (average == 0) {
                eta_s += fr * o.etaVE;
                eta_phys_s += fr * o.eta;
                dexx += fr * o.detadexx;
                dezz += fr * o.detadezz;
                dgxz += fr * o.detadexz / 2.0;
                dp += fr * o.detadp;
            }
            if (average == 0 || average == 2) sxz += fr * o.txz;
            VE_s += fr * o.VEcoeff;
            exz_el += fr * o.Exz_el;
            exz_diss += fr * o.Exz_diss;
            OverS += fr * o.OverS;
            X_s += fr * o.X1;
            if (average == 1) {
                sxz += fr * 1.0 / o.txz;
                eta_s += fr * 1.0 / o.etaVE;
                eta_phys_s += fr * 1.0 / o.eta;
                double e2 = pow(o.etaVE, 2.0);
                dexx += fr * o.detadexx / e2;
                dezz += fr * o.detadezz / e2;
                dgxz += fr * o.detadexz / 2.0 / e2;
                dp += fr * o.detadp / e2;
            }
            if (average == 2) {
                eta_s += fr * log(o.etaVE);
                eta_phys_s += fr * log(o.eta);
                dexx += fr * o.detadexx / o.etaVE;
                dezz += fr * o.detadezz / o.etaVE;
                dgxz += fr * o.detadexz / 2.0 / o.etaVE;
                dp += fr * o.detadp / o.etaVE;
            }
        }
        if (average == 1) {
            sxz = 1.0 / sxz; eta_s = 1.0 / eta_s; eta_phys_s = 1.0 / eta_phys_s;
            double e2 = pow(eta_s, 2.0);
            dexx *= e2; dezz *= e2; dgxz *= e2; dp *= e2;
        }
        if (average == 2) {
            eta_s = exp(eta_s); eta_phys_s = exp(eta_phys_s);
            dexx *= eta_s; dezz *= eta_s; dgxz *= eta_s; dp *= eta_s;
        }
    }
    g.VE_s[c1] = VE_s; g.sxz[c1] = sxz; g.eta_phys_s[c1] = eta_phys_s; g.eta_s[c1] = eta_s;
    g.exz_el[c1] = exz_el; g.exz_diss[c1] = exz_diss;
    g.detadexx_s[c1] = dexx; g.detadezz_s[c1] = dezz; g.detadgxz_s[c1] = dgxz; g.detadp_s[c1] = dp;
    if (prm.UnsplitDiffReac == 0) g.X_s[c1] = X_s;
    g.OverS_s[c1] = OverS;
}

__global__ void __launch_bounds__(BLK) k_rheo_cells(DevGrid g, DevParams prm, const mat_prop *__restrict__ mt,
                                                    const float *__restrict__ guess_n, unsigned long long *hist) {
    __shared__ unsigned int lh[3 * MDZ_HIST_BINS];
    const BlockHist bh = hist_begin(lh, hist);
    const int c0 = blockIdx.x * BLK + threadIdx.x;
    const int nc = g.ncx * g.ncz;
    if (c0 < nc) rheo_cell_generic(g, prm, mt, guess_n, bh, c0, nc);
    hist_flush(bh, hist);
}

__global__ void __launch_bounds__(BLK) k_rheo_vertices(DevGrid g, DevParams prm, const mat_prop *__restrict__ mt,
                                                       const float *__restrict__ guess_s, unsigned long long *hist) {
    __shared__ unsigned int lh[3 * MDZ_HIST_BINS];
    const BlockHist bh = hist_begin(lh, hist);
    const int c1 = blockIdx.x * BLK + threadIdx.x;
    const int nv = g.Nx * g.Nz;
    if (c1 < nv) rheo_vertex_generic(g, prm, mt, guess_s, bh, c1, nv);
    hist_flush(bh, hist);
}

/* ---------------------------------------------------------------- */
/* D tensor                                                          */
/* ---------------------------------------------------------------- */
__device__ __forceinline__ void aniso_factors(const DevParams &prm, double nx, double nz, double af, double fs,
                                              double &ani, double &d0, double &d1) {
    ani = 0.0; d0 = 0.0; d1 = 0.0;
    if (prm.aniso != 0) {
        if (prm.aniso_fstrain == 0) ani = 1.0 - 1.0 / af;
        if (prm.aniso_fstrain == 1) ani = 1.0 - 1.0 / fs;
        d0 = 2.0 * pow(nx, 2.0) * pow(nz, 2.0);
        d1 = nx * nz * (-pow(nx, 2.0) + pow(nz, 2.0));
    }
}

/* MODE as for mdz_launch_dtensor: 0 J = 0, 1 J = 1, 2 J = 1 plus the J = 0
 * Picard components into dp, 3 only those.  The node's inputs are loaded
 * in one batch before its tag test (the anisotropy fields and the
 * compressibility only where the model uses them, after that batch). */
template <int MODE>
__device__ __forceinline__ void dtensor_cell(const DevGrid &g, const DevParams &prm, double *__restrict__ dp, int k) {
    constexpr bool JAC = MODE == 1 || MODE == 2, PIC = MODE >= 2;
    if (k >= g.ncx * g.ncz) return;
    const int t = g.BCp[k];
    const double eta = g.eta_n[k];
    double mu = 0, exx = 0, ezz = 0, exz = 0, sxx0 = 0, szz0 = 0, sxz0 = 0;
    double a = 0, b = 0, c = 0, dpp = 0, q1 = 0, q2 = 0, q3 = 0, q4 = 0;
    if (JAC) {
        mu = g.mu_n[k]; exx = g.exxd[k]; ezz = g.ezzd[k]; exz = g.exz_n[k];
        sxx0 = g.sxxd0[k]; szz0 = g.szzd0[k]; sxz0 = g.sxz0_n[k];
        a = g.detadexx_n[k]; b = g.detadezz_n[k]; c = g.detadgxz_n[k]; dpp = g.detadp_n[k];
        q1 = g.ddivpdexx_n[k]; q2 = g.ddivpdezz_n[k]; q3 = g.ddivpdgxz_n[k]; q4 = g.ddivpdp_n[k];
    }
    double nx0 = 0, nz0 = 0, af = 0, fs = 0, bet = 0;
    if (prm.aniso != 0) { nx0 = g.nx0_n[k]; nz0 = g.nz0_n[k]; af = g.aniso_factor_n[k]; fs = g.FS_AR_n[k]; }
    if (JAC && prm.compressible == 1) bet = g.bet_n[k];
    double D11 = 0, D12 = 0, D13 = 0, D14 = 0, D21 = 0, D22 = 0, D23 = 0, D24 = 0;
    if (t != 30 && t != 31) {
        double ani, d0, d1;
        aniso_factors(prm, nx0, nz0, af, fs, ani, d0, d1);
        D11 = 2.0 * eta - 2.0 * ani * d0 * eta;
        D12 = 2.0 * ani * d0 * eta;
        D13 = 2.0 * ani * d1 * eta;
        D21 = 2.0 * ani * d0 * eta;
        D22 = 2.0 * eta - 2.0 * ani * d0 * eta;
        D23 = -2.0 * ani * d1 * eta;
        if (JAC) {
            if (PIC) dp[k] = D11;  /* J = 0: D22 has the same expression */
            double etae = prm.iselastic == 1 ? prm.dt * mu : 1.0;
            double K = prm.compressible == 1 ? 1.0 / bet : 0.0;
            double Exx, Ezz, Exz, Gxx, Gzz, Gxz;
            ve_rates(prm, nx0, nz0, af, fs, exx, ezz, exz, sxx0, szz0, sxz0, etae, Exx, Ezz, Exz, Gxx, Gzz, Gxz);
            double Kdt = K * prm.dt;
            D11 = D11 + 2.0 * a * Gxx - Kdt * q1;
            D12 = D12 + 2.0 * b * Gxx - Kdt * q2;
            D13 = D13 + 2.0 * c * Gxx - Kdt * q3;
            D14 = 2.0 * dpp * Exx - Kdt * q4;
            D21 = D21 + 2.0 * a * Gzz - Kdt * q1;
            D22 = D22 + 2.0 * b * Gzz - Kdt * q2;
            D23 = D23 + 2.0 * c * Gzz - Kdt * q3;
            D24 = 2.0 * dpp * Ezz - Kdt * q4;
        }
    } else if (PIC) {
        dp[k] = 0.0;
    }
    if (MODE == 3) {
        if (t != 30 && t != 31) dp[k] = D11;
        return;
    }
    g.D11_n[k] = D11; g.D12_n[k] = D12; g.D13_n[k] = D13; g.D14_n[k] = D14;
    g.D21_n[k] = D21; g.D22_n[k] = D22; g.D23_n[k] = D23; g.D24_n[k] = D24;
}

template <int MODE>
__device__ __forceinline__ void dtensor_vertex(const DevGrid &g, const DevParams &prm, int *status,
                                               double *__restrict__ dp, int k) {
    constexpr bool JAC = MODE == 1 || MODE == 2, PIC = MODE >= 2;
    if (k >= g.Nx * g.Nz) return;
    const int t = g.BCg[k];
    const double eta = g.eta_s[k];
    double mu = 0, exx = 0, ezz = 0, exz = 0, sxx0 = 0, szz0 = 0, sxz0 = 0, a = 0, b = 0, c = 0, dpp = 0;
    if (JAC) {
        mu = g.mu_s[k]; exx = g.exxd_s[k]; ezz = g.ezzd_s[k]; exz = g.exz[k];
        sxx0 = g.sxxd0_s[k]; szz0 = g.szzd0_s[k]; sxz0 = g.sxz0[k];
        a = g.detadexx_s[k]; b = g.detadezz_s[k]; c = g.detadgxz_s[k]; dpp = g.detadp_s[k];
    }
    double nx0 = 0, nz0 = 0, af = 0, fs = 0;
    if (prm.aniso != 0) { nx0 = g.nx0_s[k]; nz0 = g.nz0_s[k]; af = g.aniso_factor_s[k]; fs = g.FS_AR_s[k]; }
    double D31 = 0, D32 = 0, D33 = 0, D34 = 0;
    if (t != 30) {
        double ani, d0, d1;
        aniso_factors(prm, nx0, nz0, af, fs, ani, d0, d1);
        D31 = 2.0 * ani * d1 * eta;
        D32 = -2.0 * ani * d1 * eta;
        D33 = eta + 2.0 * ani * (d0 - 0.5) * eta;
        if (JAC) {
            if (PIC) dp[k] = D33;
            double etae = prm.iselastic == 1 ? prm.dt * mu : 1.0;
            double Exx, Ezz, Exz, Gxx, Gzz, Gxz;
            ve_rates(prm, nx0, nz0, af, fs, exx, ezz, exz, sxx0, szz0, sxz0, etae, Exx, Ezz, Exz, Gxx, Gzz, Gxz);
            D31 = D31 + 2.0 * a * Gxz;
            D32 = D32 + 2.0 * b * Gxz;
            D33 = D33 + 2.0 * c * Gxz;
            D34 = 2.0 * dpp * Exz;
        }
    } else if (PIC) {
        dp[k] = 0.0;
    }
    if (MODE == 3) {
        if (t != 30) dp[k] = D33;
        return;
    }
    g.D31_s[k] = D31; g.D32_s[k] = D32; g.D33_s[k] = D33; g.D34_s[k] = D34;
    if (JAC && status) {
        if (isnan(D34)) atomicOr(status, 1);
        if (isinf(D34)) atomicOr(status, 2);
    }
}

/* ---------------------------------------------------------------- */
/* right-hand sides                                                  */
/* ---------------------------------------------------------------- */
/* Index i clamped into [0, n): the loads of the right-hand-side kernels are
 * issued for every row with in-range indices, before the tag tests that
 * decide which of them are used, so that a wave waits for memory once. */
__device__ __forceinline__ int clampi(int i, int n) { return i < 0 ? 0 : (i >= n ? n - 1 : i); }

__device__ __forceinline__ void rhs_u(const DevGrid &g, const DevParams &prm, const double *__restrict__ xg,
                                      const double *__restrict__ zvx, int c) {
    int Nx = g.Nx, NzVx = g.nzvx, Ncx = g.ncx;
    if (c >= Nx * NzVx) return;
    int k = c % Nx, l = c / Nx;
    int c2 = k + (l - 1) * Ncx;
    const int nc = Ncx * g.ncz, nv = Nx * g.Nz, nu = Nx * NzVx;
    const int t = g.BCu[c];
    int iPrW = c2 - 1, iPrE = c2, ixyN = c, ixyS = c - Nx, iVxS = c - Nx, iVxN = c + Nx;
    if (t == -2) iPrW = c2 + Ncx - 1;
    /* every input in one batch (clamped indices); on wall nodes the
     * reference reads one cell outside the centroid array (unused there:
     * the elastic terms skip k = 0, Nx-1) */
    const int jW = clampi(iPrW, nc), jE = clampi(iPrE, nc), vS = clampi(ixyS, nv), vN = clampi(ixyN, nv);
    const int uS = clampi(iVxS, nu), uN = clampi(iVxN, nu);
    const int pW = g.BCp[jW], pE = g.BCp[jE], gS = g.BCg[vS], gN = g.BCg[vN], tuS = g.BCu[uS], tuN = g.BCu[uN];
    const double rsS = g.rho_s[vS], rsN = g.rho_s[vN], rnW = g.rho_n[jW], rnE = g.rho_n[jE];
    const double eE = g.eta_n[jE], mE = g.mu_n[jE], sE = g.sxxd0[jE];
    const double eW = g.eta_n[jW], mW = g.mu_n[jW], sW = g.sxxd0[jW];
    const double eN = g.eta_s[vN], mN = g.mu_s[vN], sN = g.sxz0[vN];
    const double eS = g.eta_s[vS], mS = g.mu_s[vS], sS = g.sxz0[vS];
    double gx = prm.gx, r = 0.0;
    if (prm.polar == 1) {
        double x = xg[k], z = zvx[l], tet = atan(z / x);
        if (tet > 0.0) gx = prm.gz * cos(tet);
        if (tet < 0.0) gx = -prm.gz * cos(tet);
    }
    g.gx[c] = gx;
    if (l > 0 && l < NzVx - 1 && (t == -1 || t == 2 || t == -2)) {
        bool inW = iPrW >= 0 && iPrW < nc && pW == -1;
        bool inE = iPrE >= 0 && iPrE < nc && pE == -1;
        bool inS = gS != 30 && tuS != 13;
        bool inN = gN != 30 && tuN != 13;
        double rhoVx = prm.polar == 0 ? 0.5 * (rsS + rsN) : 0.5 * (rnW + rnE);
        r = -gx * rhoVx;
        if (prm.iselastic == 1 && k > 0 && k < Nx - 1) {
            double dx = g.dx, dz = g.dz, dt = prm.dt;
            /* the four terms are formed for every row and applied by their
             * flags; r - 0 leaves r unchanged */
            const double tE = 1.0 / dx * (eE / (mE * dt) * sE);
            const double tW = 1.0 / dx * (-eW / (mW * dt) * sW);
            const double tN = 1.0 / dz * (eN / (mN * dt) * sN);
            const double tS = 1.0 / dz * (-eS / (mS * dt) * sS);
            r -= inE ? tE : 0.0;
            r -= inW ? tW : 0.0;
            r -= inN ? tN : 0.0;
            r -= inS ? tS : 0.0;
        }
    }
    g.roger_x[c] = -r;
}

__device__ __forceinline__ void rhs_v(const DevGrid &g, const DevParams &prm, const double *__restrict__ xvz,
                                      const double *__restrict__ zg, int c) {
    int Nx = g.Nx, NxVz = g.nxvz, Nz = g.Nz, Ncx = g.ncx;
    if (c >= NxVz * Nz) return;
    int k = c % NxVz, l = c / NxVz;
    int c1 = k + l * Nx - 1, c2 = k - 1 + (l - 1) * Ncx;
    const int nc = Ncx * g.ncz, nv = Nx * Nz, nw = NxVz * Nz;
    int iPrS = c2, iPrN = c2 + Ncx, ixyE = c1 + 1, ixyW = c1, iVyW = c - 1, iVyE = c + 1;
    /* every input in one batch (clamped indices), as in rhs_u */
    const int tv = g.BCv[c];
    const int jS = clampi(iPrS, nc), jN = clampi(iPrN, nc), vW = clampi(ixyW, nv), vE = clampi(ixyE, nv);
    const int wW = clampi(iVyW, nw), wE = clampi(iVyE, nw);
    const int pS = g.BCp[jS], pN = g.BCp[jN], gW = g.BCg[vW], gE = g.BCg[vE], tvW = g.BCv[wW], tvE = g.BCv[wE];
    const double rS = g.rho_n[jS], rN = g.rho_n[jN];
    const double eN = g.eta_n[jN], mN = g.mu_n[jN], sN = g.szzd0[jN];
    const double eS = g.eta_n[jS], mS = g.mu_n[jS], sS = g.szzd0[jS];
    const double eE = g.eta_s[vE], mE = g.mu_s[vE], sE = g.sxz0[vE];
    const double eW = g.eta_s[vW], mW = g.mu_s[vW], sW = g.sxz0[vW];
    double gz = prm.gz, r = 0.0;
    if (prm.polar == 1) {
        double x = xvz[k], z = zg[l], tet = atan(z / x);
        if (tet > 0.0) gz = prm.gz * sin(tet);
        if (tet < 0.0) gz = -prm.gz * sin(tet);
    }
    g.gz[c] = gz;
    if (k > 0 && k < NxVz - 1 && tv == -1) {
        if (iPrS < 0 || iPrN >= nc) { g.roger_z[c] = 0.0; return; } /* no interior Vz row outside the cells */
        bool inS = pS == -1, inN = pN == -1;
        bool inW = gW != 30 && tvW != 13;
        bool inE = gE != 30 && tvE != 13;
        double rhoVz = 0.5 * (rS + rN);
        r = -gz * rhoVz;
        if (prm.iselastic == 1 && l > 0 && l < Nz - 1) {
            double dx = g.dx, dz = g.dz, dt = prm.dt;
            /* every term formed, applied by its flag (as in rhs_u) */
            const double tN = 1.0 / dz * (eN / (mN * dt) * (sN));
            const double tS = 1.0 / dz * (-eS / (mS * dt) * (sS));
            const double tE = 1.0 / dx * (eE / (mE * dt) * sE);
            const double tW = 1.0 / dx * (-eW / (mW * dt) * sW);
            r -= inN ? tN : 0.0;
            r -= inS ? tS : 0.0;
            r -= inE ? tE : 0.0;
            r -= inW ? tW : 0.0;
        }
    }
    g.roger_z[c] = -r;
}

__device__ __forceinline__ void rhs_p(const DevGrid &g, const DevParams &prm, int c) {
    if (c >= g.ncx * g.ncz) return;
    int t = g.BCp[c];
    if (t != 30 && t != 31) {
        g.rhs_t[c] = g.T[c];
        g.Qrho[c] = 0.0;
        double r = 0.0;
        if (prm.compressible == 1 && g.comp_cells[c] == 1) {
            if (prm.VolChangeReac == 0) r += g.p0_n[c] * g.bet_n[c] / prm.dt;
            if (prm.VolChangeReac == 1) r += log(g.rho0_n[c]) / prm.dt;
            if (prm.adiab_heat > 0) r += g.divth0_n[c];
        }
        g.rhs_p[c] = r;
    }
}

/* The right-hand sides (RHS) and the D tensor (MODE 0..3 as above, -1 none)
 * in one launch: both read only what the rheology wrote, so that their five
 * passes -- u rows, v rows, cells, vertices, p rows -- are block ranges of
 * one grid and run side by side: 4 us against 17 in five launches at 41 x 41
 * nodes, 50 against 64 at 1001 x 501, 198 against 213 at 2049 x 1025 (HBM).
 * Five waves per SIMD hold the u rows' 96 registers; four or six, with spills,
 * are slower (50.1, 53.2 us). */
template <int MODE, bool RHS>
__global__ void __launch_bounds__(BLK) __attribute__((amdgpu_waves_per_eu(5)))
k_rhs_dtensor(DevGrid g, DevParams prm, const double *__restrict__ xg, const double *__restrict__ zvx,
              const double *__restrict__ xvz, const double *__restrict__ zg, int *status, double *__restrict__ dp_n,
              double *__restrict__ dp_s) {
    int b = blockIdx.x;
    const int nbc = mdz_div_up(g.ncx * g.ncz, BLK), nbs = mdz_div_up(g.Nx * g.Nz, BLK);
    if (RHS) {
        const int nbu = mdz_div_up(g.Nx * g.nzvx, BLK), nbv = mdz_div_up(g.nxvz * g.Nz, BLK);
        if (b < nbu) { rhs_u(g, prm, xg, zvx, xcd_tile_of(b, nbu) * BLK + threadIdx.x); return; }
        b -= nbu;
        if (b < nbv) { rhs_v(g, prm, xvz, zg, xcd_tile_of(b, nbv) * BLK + threadIdx.x); return; }
        b -= nbv;
    }
    if constexpr (MODE >= 0) {
        if (b < nbc) { dtensor_cell<MODE>(g, prm, dp_n, xcd_tile_of(b, nbc) * BLK + threadIdx.x); return; }
        b -= nbc;
        if (b < nbs) { dtensor_vertex<MODE>(g, prm, status, dp_s, xcd_tile_of(b, nbs) * BLK + threadIdx.x); return; }
        b -= nbs;
    }
    if (RHS) rhs_p(g, prm, xcd_tile_of(b, nbc) * BLK + threadIdx.x);
}

/* ---------------------------------------------------------------- */
/* launchers                                                         */
/* ---------------------------------------------------------------- */
void mdz_launch_strain_rates(const DevGrid &g, const DevParams &prm, hipStream_t s) {
    const int ntx = mdz_div_up(g.Nx, ST_TX), ntz = mdz_div_up(g.Nz, ST_TZ);
    hipLaunchKernelGGL(k_strain_tile<false>, dim3(ntx * ntz), dim3(256), 0, s, g, prm.isperiodic_x, ntx);
}

void mdz_launch_strain_interp5(const DevGrid &g, const DevParams &prm, hipStream_t s) {
    const int ntx = mdz_div_up(g.Nx, ST_TX), ntz = mdz_div_up(g.Nz, ST_TZ);
    hipLaunchKernelGGL(k_strain_tile<true>, dim3(ntx * ntz), dim3(256), 0, s, g, prm.isperiodic_x, ntx);
}

void mdz_launch_interp(const DevGrid &g, const DevParams &prm, const double *src, double *dst, hipStream_t s) {
    int nv = g.Nx * g.Nz;
    hipLaunchKernelGGL(k_interp_c2v, dim3(mdz_div_up(nv, BLK)), dim3(BLK), 0, s, g, prm.isperiodic_x, 1, src, dst,
                       (const double *)nullptr, (double *)nullptr, (const double *)nullptr, (double *)nullptr,
                       (const double *)nullptr, (double *)nullptr, (const double *)nullptr, (double *)nullptr);
}

void mdz_launch_interp5(const DevGrid &g, const DevParams &prm, hipStream_t s) {
    int nv = g.Nx * g.Nz;
    hipLaunchKernelGGL(k_interp_c2v, dim3(mdz_div_up(nv, BLK)), dim3(BLK), 0, s, g, prm.isperiodic_x, 5,
                       (const double *)g.div_u, g.div_u_s, (const double *)g.T, g.T_s, (const double *)g.p_in, g.P_s,
                       (const double *)g.d0_n, g.d0_s, (const double *)g.phi0_n, g.phi0_s);
}

void mdz_launch_rheology(const DevGrid &g, const DevParams &prm, const mat_prop *mt, const float *guess_n,
                         const float *guess_s, unsigned long long *hist, hipStream_t s) {
    int nc = g.ncx * g.ncz, nv = g.Nx * g.Nz;
    hipLaunchKernelGGL(k_rheo_cells, dim3(mdz_div_up(nc, BLK)), dim3(BLK), 0, s, g, prm, mt, guess_n, hist);
    hipLaunchKernelGGL(k_rheo_vertices, dim3(mdz_div_up(nv, BLK)), dim3(BLK), 0, s, g, prm, mt, guess_s, hist);
}

/* mode: 0..3 (mdz_launch_dtensor) or -1; rhs: with the right-hand sides */
static void launch_rhs_dtensor(const DevGrid &g, const DevParams &prm, int mode, bool rhs, const double *xg,
                               const double *zvx, const double *xvz, const double *zg, int *status, double *dp_n,
                               double *dp_s, hipStream_t s) {
    const int nc = mdz_div_up(g.ncx * g.ncz, BLK);
    int nb = 0;
    if (rhs) nb += mdz_div_up(g.Nx * g.nzvx, BLK) + mdz_div_up(g.nxvz * g.Nz, BLK) + nc;
    if (mode >= 0) nb += nc + mdz_div_up(g.Nx * g.Nz, BLK);
#define MDZ_RD(M, R)                                                                                               \
    hipLaunchKernelGGL((k_rhs_dtensor<M, R>), dim3(nb), dim3(BLK), 0, s, g, prm, xg, zvx, xvz, zg, status, dp_n, dp_s)
    switch (mode * 2 + (rhs ? 1 : 0)) {
    case -1: MDZ_RD(-1, true); break;
    case 0: MDZ_RD(0, false); break;
    case 1: MDZ_RD(0, true); break;
    case 2: MDZ_RD(1, false); break;
    case 4: MDZ_RD(2, false); break;
    case 5: MDZ_RD(2, true); break;
    case 6: MDZ_RD(3, false); break;
    default: MDZ_RD(3, true); break;
    }
#undef MDZ_RD
}

void mdz_launch_dtensor(const DevGrid &g, const DevParams &prm, int mode, int *status, hipStream_t s, double *dp_n,
                        double *dp_s) {
    launch_rhs_dtensor(g, prm, mode, false, nullptr, nullptr, nullptr, nullptr, status, dp_n, dp_s, s);
}

void mdz_launch_rhs(const DevGrid &g, const DevParams &prm, const double *xg, const double *zvx,
                    const double *xvz, const double *zg, hipStream_t s) {
    launch_rhs_dtensor(g, prm, -1, true, xg, zvx, xvz, zg, nullptr, nullptr, nullptr, s);
}

void mdz_launch_rhs_dtensor(const DevGrid &g, const DevParams &prm, int mode, const double *xg, const double *zvx,
                            const double *xvz, const double *zg, int *status, hipStream_t s, double *dp_n,
                            double *dp_s) {
    launch_rhs_dtensor(g, prm, mode, true, xg, zvx, xvz, zg, status, dp_n, dp_s, s);
}
