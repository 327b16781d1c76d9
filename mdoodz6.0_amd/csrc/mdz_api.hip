/*
 * mdz_api.hip -- C ABI of libmdz_hot.so: the reference-named drop-in entry
 * points and the device-resident interface (include/mdoodz_hot.h).
 *
 * Drop-in entry points keep the reference's contract: host structs in,
 * host structs out, CSR arrays returned in malloc() buffers the caller
 * frees, errors reported by printing the reference's message and calling
 * exit() with the reference's code (switchable with mdz_set_exit_on_error).
 * Each call uploads the fields it reads and downloads the fields it writes;
 * the device mirror of a host grid is kept between calls (keyed by the grid
 * pointer and its dimensions) so that allocations are not repeated.
 */
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "mdz_kernels.h"
#include "mdz_mlp.h"
#include "mdz_viscosity.h"
#include "mdz_h5.h"
#include "mdz_solver.h"

/* ------------------------------------------------------------------ */
/* errors                                                               */
/* ------------------------------------------------------------------ */
static char g_err[512];
static int g_status = 0;
static int g_exit_on_error = 1;

extern "C" const char *mdz_last_error(void) { return g_err; }
extern "C" void mdz_set_exit_on_error(int on) { g_exit_on_error = on; }
extern "C" int mdz_last_status(void) { return g_status; }

static int set_err(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    g_status = code;
    return code;
}

/* error reporting for the other translation units of the library */
int mdz_error(int code, const char *msg) { return set_err(code, "%s", msg); }

#define HIPCHK(x)                                                                                  \
    do {                                                                                           \
        hipError_t _e = (x);                                                                       \
        if (_e != hipSuccess) return set_err(MDZ_EHIP, "%s: %s", #x, hipGetErrorString(_e));      \
    } while (0)

/* Drop-in failure: the reference prints and exits; kernels cannot, so the
 * host wrapper reproduces its message and exit code. */
static void dropin_fail(int code, int exit_code, const char *msg) {
    if (msg) printf("%s", msg);
    if (g_exit_on_error) {
        fflush(stdout);
        exit(exit_code);
    }
    if (!g_status) set_err(code, "%s", msg ? msg : "error");
}

static void dropin_check(int rc) {
    if (rc != MDZ_OK) {
        fprintf(stderr, "mdz: %s\n", g_err);
        if (g_exit_on_error) exit(1);
    }
}

/* ------------------------------------------------------------------ */
/* field table                                                          */
/* ------------------------------------------------------------------ */
struct FieldRef {
    size_t host_off, dev_off;
    int fam, role;
};
static const FieldRef FREF[] = {
#define MDZ_FREF(name, fam, role) {offsetof(grid, name), offsetof(DevGrid, name), MDZ_FAM_##fam, MDZ_ROLE_##role},
    MDZ_ALL_DOUBLE_FIELDS(MDZ_FREF)
#undef MDZ_FREF
};

static size_t fam_len(int fam, int Nx, int Nz) {
    switch (fam) {
    case MDZ_FAM_C: return (size_t)(Nx - 1) * (Nz - 1);
    case MDZ_FAM_V: return (size_t)Nx * Nz;
    case MDZ_FAM_U: return (size_t)Nx * (Nz + 1);
    default: return (size_t)(Nx + 1) * Nz;
    }
}

static size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

/* ------------------------------------------------------------------ */
/* context                                                              */
/* ------------------------------------------------------------------ */
struct mdz_ctx {
    int Nx, Nz, nph;
    hipStream_t stream;
    char *slab;          /* field arrays, tags, phases, coords, numbering */
    size_t slab_bytes;
    DevGrid g;
    DevParams prm;
    mat_prop *d_mat;
    void *d_pk;          /* per-phase constants of the log-space rheology */
    double *xg, *zg, *xvz, *zvx;
    DevEqn e;
    DevBlock blk[8];     /* 0..3 Picard A, B, C, D; 4..7 Jacobian A, B, C, D */
    size_t blk_cap[8];   /* allocated nnz capacity */
    int pattern_ready[2];
    int d_scaled[2];     /* the scaling vectors d of a block family may differ from 1 */
    int *scratch;
    size_t scratch_len;
    double *norm_partial, *norm_out;
    double *norm_host; /* pinned: the six sums of the last eager unit */
    size_t norm_partial_len;
    int *status;
    unsigned long long *hist;
    int hist_on;         /* collect local-iteration histograms (off by default) */
    float *guess_n, *guess_s;
    CellNet *cellnet;        /* the network's outputs at the centroids, read by the vertices */
    double *tmp_c, *tmp_v;  /* staging for InterpCentroidsToVerticesDouble */
    double *dpic_n, *dpic_s; /* J = 0 D11 (= D22) at the centroids and D33 at the vertices (fused D passes) */
    int d_jac;               /* D11_n..D34_s hold the J = 1 tensor (left by a fused unit) */
    int defer_diag;          /* units write only the rheology outputs the unit itself reads */
    int guess_fused;         /* learned guess evaluated in the log-space rheology kernels' prologue */
    int diag_stale;          /* the other rheology outputs are not those of the last rheology pass */
    double *p_snap;          /* p_in as the last rheology pass read it, once p_in has changed since */
    int p_snapped;
    params model;
    mat_prop materials;
    scale scaling;
    /* surrogate network (set by mdz_ctx_set_network): blob and inference form */
    float *d_net;
    size_t net_floats;
    unsigned short *net_wp;
    float *net_bp;
    LaunchShape shape;   /* block shapes of the tunable kernels (set by the ensemble autotuner) */
    unsigned version;    /* bumped by every setter that changes what a unit launches */
    /* line-search batch: saved iterate, correction, step lengths, norms per
     * trial, and the captured graph of the trials */
    double *ls_base, *ls_dx, *ls_alpha, *ls_res;
    hipGraph_t ls_graph;
    hipGraphExec_t ls_exec;
    int ls_ntry, ls_kernel, ls_stale, ls_snapped;
    unsigned ls_version;
    MarkerStore *ms;     /* markers and their bins (marker-to-grid), allocated at first use */
    /* device solve (mdz_ctx_solve): solver state, the Picard pattern it was
     * ordered for, per continuity row diagonals, and the last correction */
    MdzSolver *sv;
    unsigned pattern_gen, sv_gen;
    int sv_nb;
    double *sv_pd, *sol;
    int sol_ready;
};

static void fill_params(mdz_ctx *c, const params *m, const scale *s) {
    DevParams &p = c->prm;
    p.dt = m->dt; p.mineta = m->mineta; p.maxeta = m->maxeta; p.gx = m->gx; p.gz = m->gz;
    p.free_surf_stab = m->free_surf_stab; p.compressible = m->compressible;
    p.sT = s->T; p.sE = s->E; p.seta = s->eta; p.sS = s->S; p.sL = s->L; p.st = s->t;
    p.step = m->step; p.iselastic = m->iselastic; p.eta_avg = m->eta_avg; p.aniso = m->aniso;
    p.aniso_fstrain = m->aniso_fstrain; p.isperiodic_x = m->isperiodic_x; p.UnsplitDiffReac = m->UnsplitDiffReac;
    p.diffuse_X = m->diffuse_X; p.diffuse_avg = m->diffuse_avg; p.polar = m->polar;
    p.VolChangeReac = m->VolChangeReac; p.adiab_heat = m->adiab_heat; p.Nb_phases = m->Nb_phases;
    p.Nx = m->Nx; p.Nz = m->Nz;
    c->model = *m;
    c->scaling = *s;
}

static int check_supported(const params *m, const mat_prop *mt) {
    if (m->VolChangeReac == 1)
        return set_err(MDZ_EUNSUPPORTED, "VolChangeReac = 1 (reaction volume changes) is not supported");
    if (m->aniso == 1)
        return set_err(MDZ_EUNSUPPORTED, "aniso = 1 (anisotropic viscosity and the stress-divergence residual) is not "
                                         "supported");
    if (mt) {
        for (int p = 0; p < m->Nb_phases; p++)
            if (mt->reac_soft[p] == 1)
                return set_err(MDZ_EUNSUPPORTED, "reac_soft = 1 (progressive reactions) is not supported (phase %d)", p);
    }
    if (m->Nb_phases < 1 || m->Nb_phases > 20) return set_err(MDZ_EINVAL, "Nb_phases = %d", m->Nb_phases);
    return MDZ_OK;
}

static DevAsm make_asm(const mdz_ctx *c) {
    DevAsm a;
    memset(&a, 0, sizeof(a));
    a.g = c->g;
    a.e = c->e;
    double dx = c->g.dx, dz = c->g.dz;
    a.celvol = dx * dz;
    a.one_dx = 1.0 / dx; a.one_dz = 1.0 / dz;
    a.one_dx_dx = 1.0 / dx / dx; a.one_dz_dz = 1.0 / dz / dz; a.one_dx_dz = 1.0 / dx / dz;
    const double cmp = 1.0; /* the Jacobian rows' compressibility switch (StokesAssemblyDecoupled.c:3165) */
    a.jk_e1x = (1.0 - cmp / 3.0) / dx; a.jk_e1z = (1.0 - cmp / 3.0) / dz;
    a.jk_e3x = cmp / 3.0 / dx; a.jk_e3z = cmp / 3.0 / dz;
    a.om = c->model.free_surf_stab; a.dt = c->model.dt; a.gz_model = c->model.gz;
    a.stab = c->model.free_surf_stab > 0 ? 1 : 0;
    a.comp_model = c->model.compressible == 1 ? 1 : 0;
    a.periodic = c->model.isperiodic_x;
    a.Nz_model = c->model.Nz;
    a.u = c->g.u_in; a.v = c->g.v_in; a.p_mom = c->g.p_corr; a.p_cont = c->g.p_in;
    a.d11p = c->g.D11_n; a.d22p = c->g.D22_n; a.d33p = c->g.D33_s;
    return a;
}

/* Isotropic models (aniso = 0) take fused D passes in a Newton unit: one
 * pass writes the J = 1 tensor and keeps the J = 0 components that the
 * Picard rows and the residual read (D11 = D22 = 2 eta, D33 = eta) in
 * dpic_n / dpic_s, so the J = 0 tensor is not computed twice.  Models with
 * aniso = 1 compute the J = 0 tensor again after the Jacobian values, for
 * the residual, which reads every component. */
static bool fused_dtensor(const mdz_ctx *c) { return c->model.aniso == 0; }

/* assembly arguments of the Picard values and the residual of a unit */
static DevAsm picard_asm(const mdz_ctx *c) {
    DevAsm a = make_asm(c);
    if (fused_dtensor(c)) { a.d11p = c->dpic_n; a.d22p = c->dpic_n; a.d33p = c->dpic_s; }
    return a;
}

static void ctx_free_blocks(mdz_ctx *c) {
    for (int i = 0; i < 8; i++) {
        hipFree(c->blk[i].Ic); hipFree(c->blk[i].J); hipFree(c->blk[i].A);
        hipFree(c->blk[i].b); hipFree(c->blk[i].bbc); hipFree(c->blk[i].F); hipFree(c->blk[i].d);
        hipFree(c->blk[i].free_row); hipFree(c->blk[i].gen_waves); hipFree(c->blk[i].free_node);
        memset(&c->blk[i], 0, sizeof(DevBlock));
        c->blk_cap[i] = 0;
    }
    c->pattern_ready[0] = c->pattern_ready[1] = 0;
}

/* Allocates the device mirror for an Nx x Nz grid with nph phases. */
static int ctx_alloc(mdz_ctx **out, int Nx, int Nz, int nph) {
    if (Nx < 4 || Nz < 4) return set_err(MDZ_EINVAL, "grid too small: %d x %d", Nx, Nz);
    mdz_ctx *c = (mdz_ctx *)calloc(1, sizeof(mdz_ctx));
    if (!c) return set_err(MDZ_ENOMEM, "host allocation");
    c->shape = MDZ_SHAPE_DEFAULT;
    c->guess_fused = 1; /* learned mode: the network in the rheology kernels' prologue (measured faster) */
    c->Nx = Nx; c->Nz = Nz; c->nph = nph;
    size_t nc = fam_len(MDZ_FAM_C, Nx, Nz), nv = fam_len(MDZ_FAM_V, Nx, Nz);
    size_t nu = fam_len(MDZ_FAM_U, Nx, Nz), nw = fam_len(MDZ_FAM_W, Nx, Nz);
    /* slab layout */
    size_t off = 0;
    std::vector<size_t> foff(FI_COUNT);
    for (int i = 0; i < FI_COUNT; i++) { foff[i] = off; off += align256(fam_len(FREF[i].fam, Nx, Nz) * sizeof(double)); }
    size_t o_uval = off; off += align256(nu * 8);
    size_t o_vval = off; off += align256(nw * 8);
    size_t o_pval = off; off += align256(nc * 8);
    size_t o_tu = off; off += align256(nu);
    size_t o_tv = off; off += align256(nw);
    size_t o_tp = off; off += align256(nc);
    size_t o_tg = off; off += align256(nv);
    size_t o_comp = off; off += align256(nc * 4);
    size_t o_phn = off; off += align256(nc * nph * 8);
    size_t o_phs = off; off += align256(nv * nph * 8);
    size_t o_xg = off; off += align256((size_t)Nx * 8);
    size_t o_zg = off; off += align256((size_t)Nz * 8);
    size_t o_xvz = off; off += align256((size_t)(Nx + 1) * 8);
    size_t o_zvx = off; off += align256((size_t)(Nz + 1) * 8);
    size_t o_eu = off; off += align256(nu * 4);
    size_t o_ev = off; off += align256(nw * 4);
    size_t o_ep = off; off += align256(nc * 4);
    size_t o_mn = off; off += align256((nu + nw) * 4);
    size_t o_cn = off; off += align256(nc * 4);
    size_t o_tc = off; off += align256(nc * 8);
    size_t o_tvv = off; off += align256(nv * 8);
    size_t o_dpn = off; off += align256(nc * 8);
    size_t o_psn = off; off += align256(nc * 8);
    size_t o_dps = off; off += align256(nv * 8);
    c->slab_bytes = off;
    if (hipMalloc((void **)&c->slab, off) != hipSuccess) { free(c); return set_err(MDZ_ENOMEM, "device slab of %zu bytes", off); }
    hipMemset(c->slab, 0, off);
    DevGrid &g = c->g;
    g.Nx = Nx; g.Nz = Nz; g.ncx = Nx - 1; g.ncz = Nz - 1; g.nxvz = Nx + 1; g.nzvx = Nz + 1; g.nph = nph;
    for (int i = 0; i < FI_COUNT; i++) *(double **)((char *)&g + FREF[i].dev_off) = (double *)(c->slab + foff[i]);
    g.BCu_val = (double *)(c->slab + o_uval); g.BCv_val = (double *)(c->slab + o_vval); g.BCp_val = (double *)(c->slab + o_pval);
    g.BCu = (int8_t *)(c->slab + o_tu); g.BCv = (int8_t *)(c->slab + o_tv); g.BCp = (int8_t *)(c->slab + o_tp);
    g.BCg = (int8_t *)(c->slab + o_tg);
    g.comp_cells = (int *)(c->slab + o_comp);
    g.phase_n = (double *)(c->slab + o_phn); g.phase_s = (double *)(c->slab + o_phs);
    g.cstride = (long long)(align256(nc * sizeof(double)) / sizeof(double));
    g.vstride = (long long)(align256(nv * sizeof(double)) / sizeof(double));
    c->xg = (double *)(c->slab + o_xg); c->zg = (double *)(c->slab + o_zg);
    c->xvz = (double *)(c->slab + o_xvz); c->zvx = (double *)(c->slab + o_zvx);
    c->e.eqn_u = (int *)(c->slab + o_eu); c->e.eqn_v = (int *)(c->slab + o_ev); c->e.eqn_p = (int *)(c->slab + o_ep);
    c->e.mom_node = (int *)(c->slab + o_mn); c->e.cont_node = (int *)(c->slab + o_cn);
    c->tmp_c = (double *)(c->slab + o_tc); c->tmp_v = (double *)(c->slab + o_tvv);
    c->dpic_n = (double *)(c->slab + o_dpn); c->dpic_s = (double *)(c->slab + o_dps);
    c->p_snap = (double *)(c->slab + o_psn);
    c->scratch_len = (nu + nw + nc) + 4096 + (nu + nw + nc) / 512;
    if (hipMalloc((void **)&c->scratch, c->scratch_len * sizeof(int)) != hipSuccess) return set_err(MDZ_ENOMEM, "scratch");
    size_t np = 0;
    {
        int nbu = mdz_div_up((int)nu, 256), nbv = mdz_div_up((int)nw, 256), nbp = mdz_div_up((int)nc, 256);
        np = 2 * (size_t)(nbu + nbv + nbp);
        /* fused residual norms: 256-row tiles and at most one 64-row wave
         * per 64 momentum rows, then the continuity tiles */
        np = std::max(np, mdz_residual_norm_partials((int)(nu + nw), mdz_div_up((int)(nu + nw), 64), (int)nc));
    }
    c->norm_partial_len = np;
    if (hipMalloc((void **)&c->norm_partial, np * sizeof(double) + 256) != hipSuccess) return set_err(MDZ_ENOMEM, "norms");
    if (hipMalloc((void **)&c->norm_out, 8 * sizeof(double)) != hipSuccess) return set_err(MDZ_ENOMEM, "norms");
    if (hipHostMalloc((void **)&c->norm_host, 8 * sizeof(double), hipHostMallocDefault) != hipSuccess)
        return set_err(MDZ_ENOMEM, "norms");
    if (hipMalloc((void **)&c->status, 4 * sizeof(int)) != hipSuccess) return set_err(MDZ_ENOMEM, "status");
    if (hipMalloc((void **)&c->hist, 3 * MDZ_HIST_BINS * sizeof(unsigned long long)) != hipSuccess) return set_err(MDZ_ENOMEM, "hist");
    if (hipMalloc((void **)&c->d_mat, sizeof(mat_prop)) != hipSuccess) return set_err(MDZ_ENOMEM, "materials");
    if (hipMalloc(&c->d_pk, mdz_phasek_bytes()) != hipSuccess) return set_err(MDZ_ENOMEM, "phase constants");
    hipMemset(c->status, 0, 4 * sizeof(int));
    hipMemset(c->hist, 0, 3 * MDZ_HIST_BINS * sizeof(unsigned long long));
    if (hipStreamCreate(&c->stream) != hipSuccess) return set_err(MDZ_EHIP, "stream");
    *out = c;
    return MDZ_OK;
}

static void ctx_release(mdz_ctx *c) {
    if (!c) return;
    hipStreamSynchronize(c->stream);
    ctx_free_blocks(c);
    hipFree(c->slab); hipFree(c->scratch); hipFree(c->norm_partial); hipFree(c->norm_out);
    if (c->norm_host) hipHostFree(c->norm_host);
    hipFree(c->status); hipFree(c->hist); hipFree(c->d_mat); hipFree(c->d_pk); hipFree(c->guess_n); hipFree(c->guess_s);
    hipFree(c->cellnet);
    hipFree(c->d_net); hipFree(c->net_wp); hipFree(c->net_bp);
    hipFree(c->ls_base); hipFree(c->ls_dx); hipFree(c->ls_alpha); hipFree(c->ls_res);
    if (c->ls_exec) hipGraphExecDestroy(c->ls_exec);
    if (c->ls_graph) hipGraphDestroy(c->ls_graph);
    mdz_mstore_destroy(c->ms);
    mdz_solver_destroy(c->sv);
    hipFree(c->sv_pd); hipFree(c->sol);
    hipStreamDestroy(c->stream);
    free(c);
}

/* ---- transfers ---- */
static int up(mdz_ctx *c, const grid *m, int fi) {
    const double *h = *(double *const *)((const char *)m + FREF[fi].host_off);
    double *d = *(double **)((char *)&c->g + FREF[fi].dev_off);
    if (!h) return set_err(MDZ_EINVAL, "host field %d is NULL", fi);
    HIPCHK(hipMemcpyAsync(d, h, fam_len(FREF[fi].fam, c->Nx, c->Nz) * sizeof(double), hipMemcpyHostToDevice, c->stream));
    return MDZ_OK;
}
static int down(mdz_ctx *c, grid *m, int fi) {
    double *h = *(double **)((char *)m + FREF[fi].host_off);
    const double *d = *(double *const *)((const char *)&c->g + FREF[fi].dev_off);
    if (!h) return set_err(MDZ_EINVAL, "host field %d is NULL", fi);
    HIPCHK(hipMemcpyAsync(h, d, fam_len(FREF[fi].fam, c->Nx, c->Nz) * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    return MDZ_OK;
}
static int up_list(mdz_ctx *c, const grid *m, std::initializer_list<int> l) {
    for (int fi : l) { int rc = up(c, m, fi); if (rc) return rc; }
    return MDZ_OK;
}
static int down_list(mdz_ctx *c, grid *m, std::initializer_list<int> l) {
    for (int fi : l) { int rc = down(c, m, fi); if (rc) return rc; }
    return MDZ_OK;
}

static int up_tags(mdz_ctx *c, const grid *m) {
    size_t nc = fam_len(MDZ_FAM_C, c->Nx, c->Nz), nv = fam_len(MDZ_FAM_V, c->Nx, c->Nz);
    size_t nu = fam_len(MDZ_FAM_U, c->Nx, c->Nz), nw = fam_len(MDZ_FAM_W, c->Nx, c->Nz);
    HIPCHK(hipMemcpyAsync(c->g.BCu, m->BCu.type, nu, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->g.BCv, m->BCv.type, nw, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->g.BCp, m->BCp.type, nc, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->g.BCg, m->BCg.type, nv, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->g.BCu_val, m->BCu.val, nu * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->g.BCv_val, m->BCv.val, nw * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->g.BCp_val, m->BCp.val, nc * 8, hipMemcpyHostToDevice, c->stream));
    if (m->comp_cells) HIPCHK(hipMemcpyAsync(c->g.comp_cells, m->comp_cells, nc * 4, hipMemcpyHostToDevice, c->stream));
    return MDZ_OK;
}

static int up_phases(mdz_ctx *c, const grid *m, int nph) {
    size_t nc = fam_len(MDZ_FAM_C, c->Nx, c->Nz), nv = fam_len(MDZ_FAM_V, c->Nx, c->Nz);
    for (int p = 0; p < nph; p++) {
        HIPCHK(hipMemcpyAsync(c->g.phase_n + p * nc, m->phase_perc_n[p], nc * 8, hipMemcpyHostToDevice, c->stream));
        HIPCHK(hipMemcpyAsync(c->g.phase_s + p * nv, m->phase_perc_s[p], nv * 8, hipMemcpyHostToDevice, c->stream));
    }
    return MDZ_OK;
}

static int up_coords(mdz_ctx *c, const grid *m) {
    if (m->xg_coord) HIPCHK(hipMemcpyAsync(c->xg, m->xg_coord, c->Nx * 8, hipMemcpyHostToDevice, c->stream));
    if (m->zg_coord) HIPCHK(hipMemcpyAsync(c->zg, m->zg_coord, c->Nz * 8, hipMemcpyHostToDevice, c->stream));
    if (m->xvz_coord) HIPCHK(hipMemcpyAsync(c->xvz, m->xvz_coord, (c->Nx + 1) * 8, hipMemcpyHostToDevice, c->stream));
    if (m->zvx_coord) HIPCHK(hipMemcpyAsync(c->zvx, m->zvx_coord, (c->Nz + 1) * 8, hipMemcpyHostToDevice, c->stream));
    return MDZ_OK;
}

static int up_materials(mdz_ctx *c, const mat_prop *mt) {
    c->materials = *mt;
    HIPCHK(hipMemcpyAsync(c->d_mat, &c->materials, sizeof(mat_prop), hipMemcpyHostToDevice, c->stream));
    mdz_launch_phase_constants(c->d_mat, MDZ_MAX_PHASES, c->d_pk, c->stream);
    HIPCHK(hipGetLastError());
    return MDZ_OK;
}

static int sync(mdz_ctx *c) {
    HIPCHK(hipStreamSynchronize(c->stream));
    HIPCHK(hipGetLastError());
    return MDZ_OK;
}

/* ---- blocks ---- */
static int block_alloc_rows(DevBlock *b, int neq) {
    b->neq = neq;
    size_t n = (size_t)neq + 1;
    HIPCHK(hipMalloc((void **)&b->Ic, n * sizeof(int)));
    HIPCHK(hipMalloc((void **)&b->b, n * sizeof(double)));
    HIPCHK(hipMalloc((void **)&b->bbc, n * sizeof(double)));
    HIPCHK(hipMalloc((void **)&b->F, n * sizeof(double)));
    HIPCHK(hipMalloc((void **)&b->d, n * sizeof(double)));
    HIPCHK(hipMemset(b->Ic, 0, n * sizeof(int)));
    HIPCHK(hipMemset(b->bbc, 0, n * sizeof(double)));
    HIPCHK(hipMemset(b->F, 0, n * sizeof(double)));
    return MDZ_OK;
}

__global__ void k_fill(double *p, double v, int n) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = v;
}

static int ensure_rows(mdz_ctx *c) {
    int nm = c->e.neq_mom, ncn = c->e.neq_cont;
    for (int i = 0; i < 8; i++) {
        int neq = (i % 4) < 2 ? nm : ncn;
        if (c->blk[i].Ic && c->blk[i].neq == neq) continue;
        hipFree(c->blk[i].Ic); hipFree(c->blk[i].J); hipFree(c->blk[i].A);
        hipFree(c->blk[i].b); hipFree(c->blk[i].bbc); hipFree(c->blk[i].F); hipFree(c->blk[i].d);
        hipFree(c->blk[i].free_row); hipFree(c->blk[i].gen_waves); hipFree(c->blk[i].free_node);
        memset(&c->blk[i], 0, sizeof(DevBlock));
        c->blk_cap[i] = 0;
        int rc = block_alloc_rows(&c->blk[i], neq);
        if (rc) return rc;
        hipLaunchKernelGGL(k_fill, dim3(mdz_div_up(neq + 1, 256)), dim3(256), 0, c->stream, c->blk[i].d, 1.0, neq + 1);
        c->pattern_ready[0] = c->pattern_ready[1] = 0;
    }
    return MDZ_OK;
}

/* builds the Picard (kind 0) or Jacobian (kind 1) pattern into blocks
 * 4*kind + {0,1,2}; block 4*kind+3 (D) stays empty */
static int build_pattern(mdz_ctx *c, int kind) {
    int rc = ensure_rows(c);
    if (rc) return rc;
    DevAsm a = make_asm(c);
    DevBlock *A = &c->blk[4 * kind], *B = &c->blk[4 * kind + 1], *C = &c->blk[4 * kind + 2], *D = &c->blk[4 * kind + 3];
    HIPCHK(hipMemsetAsync(A->Ic, 0, ((size_t)A->neq + 1) * 4, c->stream));
    HIPCHK(hipMemsetAsync(B->Ic, 0, ((size_t)B->neq + 1) * 4, c->stream));
    HIPCHK(hipMemsetAsync(C->Ic, 0, ((size_t)C->neq + 1) * 4, c->stream));
    HIPCHK(hipMemsetAsync(D->Ic, 0, ((size_t)D->neq + 1) * 4, c->stream));
    rc = mdz_build_pattern(kind, a, A, B, C, c->scratch, c->scratch_len, c->stream);
    if (rc) return rc;
    DevBlock *blks[3] = {A, B, C};
    for (int q = 0; q < 3; q++) {
        DevBlock *b = blks[q];
        int idx = 4 * kind + q;
        HIPCHK(hipMemcpyAsync(b->Ic + b->neq, &b->nnz, sizeof(int), hipMemcpyHostToDevice, c->stream));
        if ((size_t)b->nnz > c->blk_cap[idx] || !b->J) {
            hipFree(b->J); hipFree(b->A);
            size_t cap = (size_t)b->nnz + 64;
            HIPCHK(hipMalloc((void **)&b->J, cap * sizeof(int)));
            HIPCHK(hipMalloc((void **)&b->A, cap * sizeof(double)));
            c->blk_cap[idx] = cap;
        }
    }
    D->nnz = 0;
    HIPCHK(hipStreamSynchronize(c->stream));
    mdz_fill_pattern(kind, a, A, B, C, c->stream);
    /* rows whose stencil touches only free degrees of freedom take the
     * tag-free value and residual kernels */
    if (!A->free_row && A->neq > 0) HIPCHK(hipMalloc((void **)&A->free_row, (size_t)A->neq));
    if (kind == 0 && !A->free_node && A->neq > 0)
        HIPCHK(hipMalloc((void **)&A->free_node, (size_t)c->g.Nx * c->g.nzvx + (size_t)c->g.nxvz * c->g.Nz));
    if (!A->gen_waves && A->neq > 0)
        HIPCHK(hipMalloc((void **)&A->gen_waves, 2 * ((size_t)A->neq / 64 + 2) * sizeof(int)));
    if ((rc = mdz_launch_free_rows(kind, a, A, B, c->stream))) return set_err(rc, "free-row flags");
    if ((rc = mdz_build_general_waves(A, A->neq, c->scratch, c->scratch_len, c->stream)))
        return set_err(rc, "general-wave list");
    c->pattern_ready[kind] = 1;
    c->pattern_gen++;
    c->sol_ready = 0;
    c->version++; /* captured graphs hold the block pointers */
    return sync(c);
}

/* ------------------------------------------------------------------ */
/* drop-in registry                                                     */
/* ------------------------------------------------------------------ */
struct RegEntry { const grid *key; mdz_ctx *ctx; };
static std::vector<RegEntry> g_reg;
static std::mutex g_reg_mu;

static mdz_ctx *dropin_ctx(const grid *mesh, int nph) {
    std::lock_guard<std::mutex> lk(g_reg_mu);
    for (auto &r : g_reg)
        if (r.key == mesh) {
            if (r.ctx->Nx == mesh->Nx && r.ctx->Nz == mesh->Nz && r.ctx->nph >= nph) return r.ctx;
            ctx_release(r.ctx);
            r.ctx = nullptr;
            int rc = ctx_alloc(&r.ctx, mesh->Nx, mesh->Nz, nph);
            if (rc) { dropin_check(rc); return nullptr; }
            return r.ctx;
        }
    mdz_ctx *c = nullptr;
    int rc = ctx_alloc(&c, mesh->Nx, mesh->Nz, nph);
    if (rc) { dropin_check(rc); return nullptr; }
    g_reg.push_back({mesh, c});
    return c;
}

static void dropin_geometry(mdz_ctx *c, const grid *mesh) {
    c->g.dx = mesh->dx;
    c->g.dz = mesh->dz;
}

/* ------------------------------------------------------------------ */
/* drop-in entry points                                                 */
/* ------------------------------------------------------------------ */
#define STRAIN_IN FI_u_in, FI_v_in
#define STRAIN_OUT FI_div_u, FI_exxd, FI_ezzd, FI_exz, FI_exz_n, FI_exxd_s, FI_ezzd_s

extern "C" void StrainRateComponents(grid *mesh, scale scaling, params *model) {
    g_status = 0;
    mdz_ctx *c = dropin_ctx(mesh, model->Nb_phases > 0 ? model->Nb_phases : 1);
    if (!c) return;
    dropin_geometry(c, mesh);
    fill_params(c, model, &scaling);
    dropin_check(up_tags(c, mesh));
    dropin_check(up_list(c, mesh, {STRAIN_IN}));
    mdz_launch_strain_rates(c->g, c->prm, c->stream);
    dropin_check(down_list(c, mesh, {STRAIN_OUT}));
    dropin_check(sync(c));
}

extern "C" void InterpCentroidsToVerticesDouble(double *CentroidArray, double *VertexArray, grid *mesh, params *model) {
    g_status = 0;
    mdz_ctx *c = dropin_ctx(mesh, model->Nb_phases > 0 ? model->Nb_phases : 1);
    if (!c) return;
    dropin_geometry(c, mesh);
    size_t nc = fam_len(MDZ_FAM_C, c->Nx, c->Nz), nv = fam_len(MDZ_FAM_V, c->Nx, c->Nz);
    if (hipMemcpyAsync(c->g.BCg, mesh->BCg.type, nv, hipMemcpyHostToDevice, c->stream) != hipSuccess ||
        hipMemcpyAsync(c->tmp_c, CentroidArray, nc * 8, hipMemcpyHostToDevice, c->stream) != hipSuccess) {
        dropin_check(set_err(MDZ_EHIP, "upload"));
        return;
    }
    DevParams prm = c->prm;
    prm.isperiodic_x = model->isperiodic_x;
    mdz_launch_interp(c->g, prm, c->tmp_c, c->tmp_v, c->stream);
    if (hipMemcpyAsync(VertexArray, c->tmp_v, nv * 8, hipMemcpyDeviceToHost, c->stream) != hipSuccess) {
        dropin_check(set_err(MDZ_EHIP, "download"));
        return;
    }
    dropin_check(sync(c));
}

#define RHEO_IN                                                                                                \
    FI_p_in, FI_T, FI_mu_n, FI_mu_s, FI_sxxd0, FI_szzd0, FI_sxz0, FI_sxz0_n, FI_sxxd0_s, FI_szzd0_s, FI_d0_n,  \
        FI_phi0_n, FI_X0_n, FI_X0_s, FI_strain_n, FI_strain_s, FI_dil_n, FI_dil_s, FI_fric_n, FI_fric_s, FI_C_n, \
        FI_C_s, FI_p0_n, FI_p0_s, FI_bet_n, FI_bet_s, FI_nx0_n, FI_nz0_n, FI_nx0_s, FI_nz0_s, FI_aniso_factor_n,  \
        FI_aniso_factor_s, FI_FS_AR_n, FI_FS_AR_s, FI_X_n, FI_X_s, FI_div_u, FI_exxd, FI_ezzd, FI_exz, FI_exz_n, \
        FI_exxd_s, FI_ezzd_s
#define RHEO_OUT                                                                                                   \
    FI_div_u_s, FI_T_s, FI_P_s, FI_d0_s, FI_phi0_s, FI_eta_n, FI_eta_phys_n, FI_VE_n, FI_sxxd, FI_szzd, FI_sxz_n,    \
        FI_eII_el, FI_eII_pl, FI_eII_pwl, FI_eII_exp, FI_eII_lin, FI_eII_gbs, FI_eII_cst, FI_d_n, FI_exx_el,          \
        FI_ezz_el, FI_exx_diss, FI_ezz_diss, FI_detadexx_n, FI_detadezz_n, FI_detadgxz_n, FI_detadp_n,              \
        FI_ddivpdexx_n, FI_ddivpdezz_n, FI_ddivpdgxz_n, FI_ddivpdp_n, FI_p_corr, FI_div_u_el, FI_div_u_pl,           \
        FI_div_u_r, FI_Wtot, FI_Wel, FI_Wdiss, FI_X_n, FI_OverS_n, FI_VE_s, FI_sxz, FI_eta_phys_s, FI_eta_s,         \
        FI_exz_el, FI_exz_diss, FI_detadexx_s, FI_detadezz_s, FI_detadgxz_s, FI_detadp_s, FI_X_s, FI_OverS_s

/* kernel selection: 0 = log-space kernel where eligible, 1 = generic kernel */
static int g_rheo_kernel = 0;
extern "C" int mdz_set_rheology_kernel(int which) {
    if (which < 0 || which > 1) return set_err(MDZ_EINVAL, "rheology kernel %d", which);
    g_rheo_kernel = which;
    return MDZ_OK;
}

/* With mdz_ctx_fuse_guess the log-space kernels evaluate the network in
 * their own prologue; otherwise (and always for the generic kernel)
 * k_mlp_guess writes the guess arrays first. */
static bool fused_guess(const mdz_ctx *c, int use_guess) {
    return use_guess && c->guess_fused && g_rheo_kernel == 0 && mdz_rheo_fast_eligible(c->prm, &c->materials);
}

/* first part of the rheology: vertex values of div_u, T, P, d and phi
 * (NonNewtonianViscosityGrid :979-983; interp_done: already written by
 * mdz_launch_strain_interp5), then the network's guess when it is not
 * evaluated inside the rheology kernels */
static int rheology_prep(mdz_ctx *c, int use_guess, hipStream_t s, bool interp_done = false) {
    if (!interp_done) mdz_launch_interp5(c->g, c->prm, s);
    if (use_guess && !c->net_wp) return set_err(MDZ_EINVAL, "learned guess without a network");
    if (use_guess && !fused_guess(c, use_guess)) {
        if (!c->net_wp || !c->guess_n || !c->guess_s || !c->cellnet)
            return set_err(MDZ_EINVAL, "learned guess without a network");
        mdz_launch_mlp_guess(c->g, c->prm, DevMLPI{c->net_wp, c->net_bp, c->cellnet}, c->d_pk, c->materials.R,
                             c->guess_n, c->guess_s, s);
    }
    return MDZ_OK;
}

/* second part: the local iterations at centroids and vertices, with every
 * output field, or with deferred diagnostics only the unit's own */
static int rheology_kernels(mdz_ctx *c, int use_guess, hipStream_t s) {
    const float *gn = use_guess ? c->guess_n : nullptr, *gs = use_guess ? c->guess_s : nullptr;
    unsigned long long *hist = c->hist_on ? c->hist : nullptr;
    c->p_snapped = 0;
    if (g_rheo_kernel == 0 && mdz_rheo_fast_eligible(c->prm, &c->materials)) {
        const int diag = !c->defer_diag;
        const DevMLPI net{c->net_wp, c->net_bp, c->cellnet};
        const bool fused = fused_guess(c, use_guess);
        int rc = mdz_launch_rheology_fast(c->g, c->prm, c->d_pk, c->materials.R, fused ? nullptr : gn,
                                          fused ? nullptr : gs, hist, c->shape.rheo, diag, s,
                                          fused ? &net : nullptr);
        if (rc) return rc;
        c->diag_stale = !diag;
        return MDZ_OK;
    }
    mdz_launch_rheology(c->g, c->prm, c->d_mat, gn, gs, hist, s);
    c->diag_stale = 0;
    return MDZ_OK;
}

/* Deferred diagnostics: the last rheology pass again with every output, on
 * the inputs it read (strain rates, interpolated fields and the guess are
 * still in place; p_in from its snapshot when it has changed since), so
 * that the fields the unit used come out unchanged. */
static int flush_diagnostics(mdz_ctx *c) {
    if (!c->diag_stale) return MDZ_OK;
    DevGrid g = c->g;
    if (c->p_snapped) g.p_in = c->p_snap;
    const int guess = c->prm.rheo_mode == MDZ_RHEO_LEARNED;
    const DevMLPI net{c->net_wp, c->net_bp, c->cellnet};
    const bool fused = fused_guess(c, guess);
    int rc = mdz_launch_rheology_fast(g, c->prm, c->d_pk, c->materials.R, guess && !fused ? c->guess_n : nullptr,
                                      guess && !fused ? c->guess_s : nullptr, nullptr, c->shape.rheo, 1, c->stream,
                                      fused ? &net : nullptr);
    if (rc) return rc;
    c->diag_stale = 0;
    c->p_snapped = 0;
    return MDZ_OK;
}

__global__ void __launch_bounds__(256) k_copy_doubles(const double *__restrict__ src, double *__restrict__ dst, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

/* p_in is about to change while the diagnostics are deferred: keep the
 * values the last rheology pass read (a kernel, so that it can be captured) */
static int snapshot_p(mdz_ctx *c, hipStream_t s) {
    if (!c->diag_stale || c->p_snapped) return MDZ_OK;
    const int n = (int)fam_len(MDZ_FAM_C, c->Nx, c->Nz);
    hipLaunchKernelGGL(k_copy_doubles, dim3(mdz_div_up(n, 256)), dim3(256), 0, s, (const double *)c->g.p_in,
                       c->p_snap, n);
    c->p_snapped = 1;
    return MDZ_OK;
}

static int rheology_pass(mdz_ctx *c, int use_guess, hipStream_t s, bool interp_done = false) {
    int rc = rheology_prep(c, use_guess, s, interp_done);
    return rc ? rc : rheology_kernels(c, use_guess, s);
}

extern "C" void NonNewtonianViscosityGrid(grid *mesh, mat_prop *materials, params *model, Nparams Nmodel, scale *scaling) {
    g_status = 0;
    (void)Nmodel;
    int rc = check_supported(model, materials);
    if (rc) { dropin_check(rc); return; }
    mdz_ctx *c = dropin_ctx(mesh, model->Nb_phases);
    if (!c) return;
    dropin_geometry(c, mesh);
    fill_params(c, model, scaling);
    c->prm.rheo_mode = MDZ_RHEO_FP64;
    dropin_check(up_tags(c, mesh));
    dropin_check(up_phases(c, mesh, model->Nb_phases));
    dropin_check(up_materials(c, materials));
    dropin_check(up_list(c, mesh, {RHEO_IN}));
    dropin_check(rheology_pass(c, 0, c->stream));
    dropin_check(down_list(c, mesh, {RHEO_OUT}));
    dropin_check(sync(c));
}

#define DT_IN                                                                                                   \
    FI_eta_n, FI_eta_s, FI_detadexx_n, FI_detadezz_n, FI_detadgxz_n, FI_detadp_n, FI_ddivpdexx_n, FI_ddivpdezz_n, \
        FI_ddivpdgxz_n, FI_ddivpdp_n, FI_detadexx_s, FI_detadezz_s, FI_detadgxz_s, FI_detadp_s, FI_exxd, FI_ezzd,  \
        FI_exz_n, FI_exz, FI_exxd_s, FI_ezzd_s, FI_sxxd0, FI_szzd0, FI_sxz0_n, FI_sxz0, FI_sxxd0_s, FI_szzd0_s,    \
        FI_mu_n, FI_mu_s, FI_bet_n, FI_nx0_n, FI_nz0_n, FI_nx0_s, FI_nz0_s, FI_aniso_factor_n, FI_aniso_factor_s,  \
        FI_FS_AR_n, FI_FS_AR_s
#define DT_OUT FI_D11_n, FI_D12_n, FI_D13_n, FI_D14_n, FI_D21_n, FI_D22_n, FI_D23_n, FI_D24_n, FI_D31_s, FI_D32_s, FI_D33_s, FI_D34_s

static int dtensor_status(mdz_ctx *c) {
    int st = 0;
    HIPCHK(hipMemcpyAsync(&st, c->status, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipMemsetAsync(c->status, 0, sizeof(int), c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return st;
}

extern "C" void RheologicalOperators(grid *mesh, params *model, scale *scaling, int Jacobian) {
    g_status = 0;
    mdz_ctx *c = dropin_ctx(mesh, model->Nb_phases > 0 ? model->Nb_phases : 1);
    if (!c) return;
    dropin_geometry(c, mesh);
    fill_params(c, model, scaling);
    dropin_check(up_tags(c, mesh));
    dropin_check(up_list(c, mesh, {DT_IN}));
    mdz_launch_dtensor(c->g, c->prm, Jacobian ? 1 : 0, c->status, c->stream);
    dropin_check(down_list(c, mesh, {DT_OUT}));
    int st = dtensor_status(c);
    if (Jacobian && st < 0) { dropin_check(st); return; }
    if (Jacobian && (st & 1)) { dropin_fail(MDZ_ED34, 1, "EXIT: D34 is NAN!\n"); return; }
    if (Jacobian && (st & 2)) { dropin_fail(MDZ_ED34, 1, "EXIT: D34 is INF!\n"); return; }
}

#define RHS_IN                                                                                                 \
    FI_rho_n, FI_rho_s, FI_eta_n, FI_eta_s, FI_mu_n, FI_mu_s, FI_sxxd0, FI_szzd0, FI_sxz0, FI_T, FI_p0_n,       \
        FI_bet_n, FI_rho0_n, FI_divth0_n, FI_rhs_t, FI_rhs_p, FI_Qrho
#define RHS_OUT FI_roger_x, FI_roger_z, FI_gx, FI_gz, FI_rhs_p, FI_rhs_t, FI_Qrho

extern "C" void EvaluateRHS(grid *mesh, params model, scale scaling, double RHO_REF) {
    g_status = 0;
    (void)RHO_REF;
    mdz_ctx *c = dropin_ctx(mesh, model.Nb_phases > 0 ? model.Nb_phases : 1);
    if (!c) return;
    dropin_geometry(c, mesh);
    fill_params(c, &model, &scaling);
    dropin_check(up_tags(c, mesh));
    dropin_check(up_coords(c, mesh));
    dropin_check(up_list(c, mesh, {RHS_IN}));
    mdz_launch_rhs(c->g, c->prm, c->xg, c->zvx, c->xvz, c->zg, c->stream);
    dropin_check(down_list(c, mesh, {RHS_OUT}));
    dropin_check(sync(c));
}

extern "C" void UpdateNonLinearity(grid *mesh, markers *particles, markers *topo_chain, surface *topo,
                                   mat_prop materials, params *model, Nparams *Nmodel, scale scaling, int mode,
                                   double h_contin) {
    g_status = 0;
    (void)particles; (void)topo_chain; (void)topo; (void)Nmodel; (void)mode; (void)h_contin;
    int rc = check_supported(model, &materials);
    if (rc) { dropin_check(rc); return; }
    mdz_ctx *c = dropin_ctx(mesh, model->Nb_phases);
    if (!c) return;
    dropin_geometry(c, mesh);
    fill_params(c, model, &scaling);
    c->prm.rheo_mode = MDZ_RHEO_FP64;
    dropin_check(up_tags(c, mesh));
    dropin_check(up_coords(c, mesh));
    dropin_check(up_phases(c, mesh, model->Nb_phases));
    dropin_check(up_materials(c, &materials));
    dropin_check(up_list(c, mesh, {STRAIN_IN}));
    dropin_check(up_list(c, mesh, {RHEO_IN}));
    dropin_check(up_list(c, mesh, {RHS_IN}));
    dropin_check(up_list(c, mesh, {DT_IN}));
    mdz_launch_strain_interp5(c->g, c->prm, c->stream);
    dropin_check(rheology_pass(c, 0, c->stream, true));
    mdz_launch_rhs_dtensor(c->g, c->prm, 0, c->xg, c->zvx, c->xvz, c->zg, c->status, c->stream);
    dropin_check(down_list(c, mesh, {STRAIN_OUT}));
    dropin_check(down_list(c, mesh, {RHEO_OUT}));
    dropin_check(down_list(c, mesh, {RHS_OUT}));
    dropin_check(down_list(c, mesh, {DT_OUT}));
    dropin_check(sync(c));
}

/* numbering on the device; host arrays malloc()ed as in the reference */
__global__ void k_nodes_from_eqn(DevGrid g, DevEqn e) {
    int i = blockIdx.x * 256 + threadIdx.x;
    int nu = g.Nx * g.nzvx, nw = g.nxvz * g.Nz, nc = g.ncx * g.ncz;
    if (i >= nu + nw + nc) return;
    if (i < nu) {
        int t = g.BCu[i], eq = e.eqn_u[i];
        if ((t == -1 || t == 2 || t == -2) && eq >= 0 && eq < e.neq_mom) e.mom_node[eq] = i;
    } else if (i < nu + nw) {
        int c = i - nu, t = g.BCv[c], eq = e.eqn_v[c];
        if ((t == -1 || t == 2) && eq >= 0 && eq < e.neq_mom) e.mom_node[eq] = i;
    } else {
        int c = i - nu - nw, eq = e.eqn_p[c];
        if (g.BCp[c] == -1 && eq >= e.neq_mom && eq < e.neq_mom + e.neq_cont) e.cont_node[eq - e.neq_mom] = c;
    }
}

/* tags the numbering and the stencils accept; anything else would make the
 * right-hand-side order of the reference differ from the equation order */
static int validate_tags(const grid *m) {
    int Nx = m->Nx, Nz = m->Nz;
    for (int i = 0; i < Nx * (Nz + 1); i++) {
        int t = m->BCu.type[i];
        if (!(t == -1 || t == 0 || t == 2 || t == -2 || t == -12 || t == 11 || t == 13 || t == 30))
            return set_err(MDZ_EUNSUPPORTED, "Vx tag %d at node %d", t, i);
    }
    for (int i = 0; i < (Nx + 1) * Nz; i++) {
        int t = m->BCv.type[i];
        if (!(t == -1 || t == 0 || t == 2 || t == -12 || t == 11 || t == 13 || t == 30))
            return set_err(MDZ_EUNSUPPORTED, "Vz tag %d at node %d", t, i);
    }
    for (int i = 0; i < (Nx - 1) * (Nz - 1); i++) {
        int t = m->BCp.type[i];
        if (!(t == -1 || t == 0 || t == 30 || t == 31)) return set_err(MDZ_EUNSUPPORTED, "P tag %d at cell %d", t, i);
    }
    return MDZ_OK;
}

extern "C" void EvalNumberOfEquations(grid *mesh, SparseMat *Stokes) {
    g_status = 0;
    mdz_ctx *c = dropin_ctx(mesh, 1);
    if (!c) return;
    dropin_geometry(c, mesh);
    dropin_check(validate_tags(mesh));
    dropin_check(up_tags(c, mesh));
    dropin_check(mdz_number_equations(c->g, c->e, c->scratch, c->scratch_len, c->stream));
    size_t nc = fam_len(MDZ_FAM_C, c->Nx, c->Nz), nu = fam_len(MDZ_FAM_U, c->Nx, c->Nz), nw = fam_len(MDZ_FAM_W, c->Nx, c->Nz);
    Stokes->eqn_u = (int *)malloc(nu * sizeof(int));
    Stokes->eqn_v = (int *)malloc(nw * sizeof(int));
    Stokes->eqn_p = (int *)malloc(nc * sizeof(int));
    hipMemcpyAsync(Stokes->eqn_u, c->e.eqn_u, nu * 4, hipMemcpyDeviceToHost, c->stream);
    hipMemcpyAsync(Stokes->eqn_v, c->e.eqn_v, nw * 4, hipMemcpyDeviceToHost, c->stream);
    hipMemcpyAsync(Stokes->eqn_p, c->e.eqn_p, nc * 4, hipMemcpyDeviceToHost, c->stream);
    dropin_check(sync(c));
    Stokes->neq_mom = c->e.neq_mom;
    Stokes->neq_cont = c->e.neq_cont;
    Stokes->neq = c->e.neq_mom + c->e.neq_cont;
}

/* uploads what the assembly / residual rows read, and the caller's numbering */
static int asm_upload(mdz_ctx *c, grid *mesh, const params *model, SparseMat *Stokes, double *p_corr, double *p,
                      double *u, double *v, int kind) {
    int rc;
    if ((rc = validate_tags(mesh))) return rc;
    if ((rc = up_tags(c, mesh))) return rc;
    size_t nc = fam_len(MDZ_FAM_C, c->Nx, c->Nz), nu = fam_len(MDZ_FAM_U, c->Nx, c->Nz), nw = fam_len(MDZ_FAM_W, c->Nx, c->Nz);
    HIPCHK(hipMemcpyAsync(c->e.eqn_u, Stokes->eqn_u, nu * 4, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->e.eqn_v, Stokes->eqn_v, nw * 4, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->e.eqn_p, Stokes->eqn_p, nc * 4, hipMemcpyHostToDevice, c->stream));
    c->e.neq_mom = Stokes->neq_mom;
    c->e.neq_cont = Stokes->neq_cont;
    int n = (int)(nu + nw + nc);
    hipLaunchKernelGGL(k_nodes_from_eqn, dim3(mdz_div_up(n, 256)), dim3(256), 0, c->stream, c->g, c->e);
    /* iterate arrays as passed (the reference passes mesh->u_in etc.) */
    HIPCHK(hipMemcpyAsync(c->g.u_in, u, nu * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->g.v_in, v, nw * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->g.p_corr, p_corr, nc * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->g.p_in, p, nc * 8, hipMemcpyHostToDevice, c->stream));
    if ((rc = up_list(c, mesh, {FI_roger_x, FI_roger_z, FI_rhs_p, FI_eta_n, FI_eta_s, FI_rho_n, FI_gx, FI_gz, FI_bet_n}))) return rc;
    if (kind == 0) { if ((rc = up_list(c, mesh, {FI_D11_n, FI_D22_n, FI_D33_s}))) return rc; }
    else if ((rc = up_list(c, mesh, {DT_OUT}))) return rc;
    if (model->aniso == 1) { if ((rc = up_list(c, mesh, {FI_sxxd, FI_szzd, FI_sxz}))) return rc; }
    return MDZ_OK;
}

/* host CSR of one block: malloc()ed Ic/J/A/bbc; J/A NULL when empty
 * (what realloc(p, 0) leaves in the reference) */
static int download_block(mdz_ctx *c, DevBlock *b, SparseMat *M, int with_b) {
    M->neq = b->neq;
    M->nnz = b->nnz;
    M->Ic = (int *)malloc(((size_t)b->neq + 1) * sizeof(int));
    M->J = b->nnz ? (int *)malloc((size_t)b->nnz * sizeof(int)) : NULL;
    M->A = b->nnz ? (double *)malloc((size_t)b->nnz * sizeof(double)) : NULL;
    M->bbc = (double *)malloc(((size_t)b->neq + 1) * sizeof(double));
    if (!M->Ic || !M->bbc || (b->nnz && (!M->J || !M->A))) return set_err(MDZ_ENOMEM, "host CSR");
    HIPCHK(hipMemcpyAsync(M->Ic, b->Ic, ((size_t)b->neq + 1) * 4, hipMemcpyDeviceToHost, c->stream));
    if (b->nnz) {
        HIPCHK(hipMemcpyAsync(M->J, b->J, (size_t)b->nnz * 4, hipMemcpyDeviceToHost, c->stream));
        HIPCHK(hipMemcpyAsync(M->A, b->A, (size_t)b->nnz * 8, hipMemcpyDeviceToHost, c->stream));
    }
    HIPCHK(hipMemcpyAsync(M->bbc, b->bbc, (size_t)b->neq * 8, hipMemcpyDeviceToHost, c->stream));
    if (with_b && M->b) HIPCHK(hipMemcpyAsync(M->b, b->b, (size_t)b->neq * 8, hipMemcpyDeviceToHost, c->stream));
    return MDZ_OK;
}

static void build_operator_dropin(int kind, grid *mesh, params model, double *p_corr, double *p, double *u, double *v,
                                  SparseMat *Stokes, SparseMat *SA, SparseMat *SB, SparseMat *SC, SparseMat *SD,
                                  int Assemble) {
    mdz_ctx *c = dropin_ctx(mesh, model.Nb_phases > 0 ? model.Nb_phases : 1);
    if (!c) return;
    dropin_geometry(c, mesh);
    fill_params(c, &model, &c->scaling);
    int rc = asm_upload(c, mesh, &model, Stokes, p_corr, p, u, v, kind);
    if (rc) { dropin_check(rc); return; }
    SA->neq = Stokes->neq_mom; SB->neq = Stokes->neq_mom;
    SC->neq = Stokes->neq_cont; SC->neq_mom = Stokes->neq_mom;
    SD->neq = Stokes->neq_cont; SD->neq_mom = Stokes->neq_mom;
    rc = ensure_rows(c);
    if (rc) { dropin_check(rc); return; }
    DevBlock *A = &c->blk[4 * kind], *B = &c->blk[4 * kind + 1], *C = &c->blk[4 * kind + 2], *D = &c->blk[4 * kind + 3];
    DevAsm a = make_asm(c);
    if (Assemble == 1) {
        rc = build_pattern(c, kind);
        if (rc) { dropin_check(rc); return; }
        a = make_asm(c);
        mdz_launch_values(kind, a, A, B, C, D, kind == 0 ? c->shape.pic : c->shape.jac, c->stream);
        dropin_check(download_block(c, A, SA, 1));
        dropin_check(download_block(c, B, SB, 1));
        dropin_check(download_block(c, C, SC, 1));
        dropin_check(download_block(c, D, SD, 1));
        /* b of B and D equal those of A and C (already downloaded through with_b) */
        dropin_check(sync(c));
        if (model.write_debug == 1) {
            /* the debug dump of the assembled system (StokesAssemblyDecoupled.c:2041-2137, :4264-4360) */
            char fn[128];
            mdz_h5_dump_name(fn, sizeof(fn), kind, model.step, model.nit);
            printf("Writing %s matrix file: %s to disk...\n", kind ? "Jacobian" : "Stokes", fn);
            dropin_check(mdz_write_matrix_h5(fn, mesh, Stokes, SA, SB, SC, SD));
        }
    } else {
        /* residual: b from the right-hand sides; Neumann rows read the bbc
         * of the last assembly of this block */
        if (SA->bbc) {
            if (hipMemcpyAsync(A->bbc, SA->bbc, (size_t)SA->neq * 8, hipMemcpyHostToDevice, c->stream) != hipSuccess) {
                dropin_check(set_err(MDZ_EHIP, "bbc upload"));
                return;
            }
        } else {
            hipMemsetAsync(A->bbc, 0, (size_t)SA->neq * 8, c->stream);
        }
        /* the tags were uploaded again without a pattern build: the free-row
         * flags of the last build may not describe them, so every row takes
         * the general kernel here */
        if (A->free_row) hipMemsetAsync(A->free_row, 0, (size_t)A->neq, c->stream);
        mdz_launch_residual(kind, a, A, C, D, c->stream);
        hipMemcpyAsync(SA->F, A->F, (size_t)SA->neq * 8, hipMemcpyDeviceToHost, c->stream);
        hipMemcpyAsync(SA->b, A->b, (size_t)SA->neq * 8, hipMemcpyDeviceToHost, c->stream);
        hipMemcpyAsync(SC->F, C->F, (size_t)SC->neq * 8, hipMemcpyDeviceToHost, c->stream);
        hipMemcpyAsync(SC->b, C->b, (size_t)SC->neq * 8, hipMemcpyDeviceToHost, c->stream);
        hipMemcpyAsync(SD->F, D->F, (size_t)SD->neq * 8, hipMemcpyDeviceToHost, c->stream);
        dropin_check(sync(c));
    }
}

extern "C" void BuildStokesOperatorDecoupled(grid *mesh, params model, int lev, double *p_corr, double *p, double *u,
                                             double *v, SparseMat *Stokes, SparseMat *StokesA, SparseMat *StokesB,
                                             SparseMat *StokesC, SparseMat *StokesD, int Assemble) {
    g_status = 0;
    (void)lev;
    build_operator_dropin(0, mesh, model, p_corr, p, u, v, Stokes, StokesA, StokesB, StokesC, StokesD, Assemble);
}

extern "C" void BuildJacobianOperatorDecoupled(grid *mesh, params model, int lev, double *p_corr, double *p, double *u,
                                               double *v, SparseMat *Stokes, SparseMat *StokesA, SparseMat *StokesB,
                                               SparseMat *StokesC, SparseMat *StokesD, int Assemble) {
    g_status = 0;
    (void)lev;
    build_operator_dropin(1, mesh, model, p_corr, p, u, v, Stokes, StokesA, StokesB, StokesC, StokesD, Assemble);
}

static void finish_norms(Nparams *Nmodel, const double *out6, scale scaling, int quiet) {
    Nmodel->resx = sqrt(out6[0] / out6[3]);
    Nmodel->resz = sqrt(out6[1] / out6[4]);
    Nmodel->resp = sqrt(out6[2] / out6[5]);
    if (Nmodel->nit == 0) {
        Nmodel->resx0 = Nmodel->resx;
        Nmodel->resz0 = Nmodel->resz;
        Nmodel->resp0 = Nmodel->resp;
    }
    if (quiet == 0) {
        printf("Fu abs. = %2.6e --- Fu rel. = %2.6e\n", Nmodel->resx, Nmodel->resx / Nmodel->resx0);
        printf("Fv abs. = %2.6e --- Fv rel. = %2.6e\n", Nmodel->resz, Nmodel->resz / Nmodel->resz0);
        printf("Fp abs. = %2.6e --- Fp rel. = %2.6e\n", Nmodel->resp, Nmodel->resp / Nmodel->resp0);
    }
    if (isnan(Nmodel->resx) || isnan(Nmodel->resz) || isnan(Nmodel->resp)) {
        printf("Fu = %2.6e\n", Nmodel->resx * scaling.S * scaling.L);
        printf("Fv = %2.6e\n", Nmodel->resz * scaling.S * scaling.L);
        printf("Fp = %2.6e\n", Nmodel->resp * scaling.E * scaling.L * scaling.L);
        dropin_fail(MDZ_ENAN, 122, "Solve went wrong - Nan residuals...\nExiting...\n");
    }
}

extern "C" void EvaluateStokesResidualDecoupled(SparseMat *Stokes, SparseMat *StokesA, SparseMat *StokesB,
                                                SparseMat *StokesC, SparseMat *StokesD, Nparams *Nmodel, grid *mesh,
                                                params model, scale scaling, int quiet) {
    g_status = 0;
    int kind = model.aniso == 1 ? 1 : 0;
    mdz_ctx *c = dropin_ctx(mesh, model.Nb_phases > 0 ? model.Nb_phases : 1);
    if (!c) return;
    c->scaling = scaling;
    build_operator_dropin(kind, mesh, model, mesh->p_corr, mesh->p_in, mesh->u_in, mesh->v_in, Stokes, StokesA,
                          StokesB, StokesC, StokesD, 0);
    if (g_status && !g_exit_on_error) return;
    DevBlock *A = &c->blk[4 * kind], *D = &c->blk[4 * kind + 3];
    /* ru/rv/rp are written on the degrees of freedom only; the other entries
     * keep the caller's values */
    dropin_check(up_list(c, mesh, {FI_ru, FI_rv, FI_rp}));
    /* residual scaling vectors d */
    hipMemcpyAsync(A->d, StokesA->d, (size_t)StokesA->neq * 8, hipMemcpyHostToDevice, c->stream);
    hipMemcpyAsync(D->d, StokesD->d, (size_t)StokesD->neq * 8, hipMemcpyHostToDevice, c->stream);
    c->d_scaled[kind] = 1;
    DevAsm a = make_asm(c);
    mdz_launch_norms(a, A, D, c->norm_partial, c->norm_out, c->stream);
    double out6[6];
    hipMemcpyAsync(out6, c->norm_out, 6 * 8, hipMemcpyDeviceToHost, c->stream);
    hipMemcpyAsync(StokesA->F, A->F, (size_t)StokesA->neq * 8, hipMemcpyDeviceToHost, c->stream);
    hipMemcpyAsync(StokesD->F, D->F, (size_t)StokesD->neq * 8, hipMemcpyDeviceToHost, c->stream);
    dropin_check(down_list(c, mesh, {FI_ru, FI_rv, FI_rp}));
    dropin_check(sync(c));
    finish_norms(Nmodel, out6, scaling, quiet);
}

/* ---- diagonal scaling drop-ins (host CSR in, host CSR out) ---- */
struct HostBlocks {
    DevBlock b[4];
    int rows[4];
};

static void tmp_blocks_free(HostBlocks &h) {
    for (int q = 0; q < 4; q++) {
        hipFree(h.b[q].Ic); hipFree(h.b[q].J); hipFree(h.b[q].A);
        hipFree(h.b[q].b); hipFree(h.b[q].F); hipFree(h.b[q].d);
    }
}

/* Device copies of the four blocks: rows of D are those of C, as in the
 * reference's loops. */
static int tmp_blocks_upload(SparseMat *M[4], HostBlocks &h, hipStream_t s) {
    memset(&h, 0, sizeof(h));
    h.rows[0] = M[0]->neq; h.rows[1] = M[1]->neq; h.rows[2] = M[2]->neq; h.rows[3] = M[2]->neq;
    for (int q = 0; q < 4; q++) {
        int n = h.rows[q];
        if (n <= 0) continue;
        if (!M[q]->Ic || !M[q]->d || !M[q]->b || !M[q]->F) return set_err(MDZ_EINVAL, "block %d: missing arrays", q);
        int nnz = M[q]->Ic[n];
        DevBlock &b = h.b[q];
        b.neq = n; b.nnz = nnz;
        HIPCHK(hipMalloc((void **)&b.Ic, ((size_t)n + 1) * sizeof(int)));
        HIPCHK(hipMalloc((void **)&b.d, (size_t)n * 8));
        HIPCHK(hipMalloc((void **)&b.b, (size_t)n * 8));
        HIPCHK(hipMalloc((void **)&b.F, (size_t)n * 8));
        HIPCHK(hipMemcpyAsync(b.Ic, M[q]->Ic, ((size_t)n + 1) * sizeof(int), hipMemcpyHostToDevice, s));
        HIPCHK(hipMemcpyAsync(b.d, M[q]->d, (size_t)n * 8, hipMemcpyHostToDevice, s));
        HIPCHK(hipMemcpyAsync(b.b, M[q]->b, (size_t)n * 8, hipMemcpyHostToDevice, s));
        HIPCHK(hipMemcpyAsync(b.F, M[q]->F, (size_t)n * 8, hipMemcpyHostToDevice, s));
        if (nnz > 0) {
            HIPCHK(hipMalloc((void **)&b.J, (size_t)nnz * sizeof(int)));
            HIPCHK(hipMalloc((void **)&b.A, (size_t)nnz * 8));
            HIPCHK(hipMemcpyAsync(b.J, M[q]->J, (size_t)nnz * sizeof(int), hipMemcpyHostToDevice, s));
            HIPCHK(hipMemcpyAsync(b.A, M[q]->A, (size_t)nnz * 8, hipMemcpyHostToDevice, s));
        }
    }
    return MDZ_OK;
}

static int diag_dropin(SparseMat *SA, SparseMat *SB, SparseMat *SC, SparseMat *SD, int scale) {
    if (!SA || !SB || !SC || !SD) return set_err(MDZ_EINVAL, "NULL block");
    SparseMat *M[4] = {SA, SB, SC, SD};
    hipStream_t s;
    HIPCHK(hipStreamCreate(&s));
    HostBlocks h;
    int rc = tmp_blocks_upload(M, h, s);
    if (rc == MDZ_OK) {
        if (scale) mdz_launch_scale_matrix(&h.b[0], &h.b[1], &h.b[2], &h.b[3], s);
        else mdz_launch_extract_diagonal(&h.b[0], &h.b[1], &h.b[2], &h.b[3], s);
        for (int q = 0; q < 4 && rc == MDZ_OK; q++) {
            int n = h.rows[q];
            if (n <= 0) continue;
            if (!scale) {
                if (hipMemcpyAsync(M[q]->d, h.b[q].d, (size_t)n * 8, hipMemcpyDeviceToHost, s) != hipSuccess) rc = MDZ_EHIP;
                continue;
            }
            if (hipMemcpyAsync(M[q]->b, h.b[q].b, (size_t)n * 8, hipMemcpyDeviceToHost, s) != hipSuccess) rc = MDZ_EHIP;
            if (hipMemcpyAsync(M[q]->F, h.b[q].F, (size_t)n * 8, hipMemcpyDeviceToHost, s) != hipSuccess) rc = MDZ_EHIP;
            if (h.b[q].nnz > 0 &&
                hipMemcpyAsync(M[q]->A, h.b[q].A, (size_t)h.b[q].nnz * 8, hipMemcpyDeviceToHost, s) != hipSuccess)
                rc = MDZ_EHIP;
        }
        if (hipStreamSynchronize(s) != hipSuccess || hipGetLastError() != hipSuccess) rc = MDZ_EHIP;
        if (rc) set_err(rc, "diagonal scaling: HIP error");
    }
    tmp_blocks_free(h);
    hipStreamDestroy(s);
    return rc;
}

extern "C" void ExtractDiagonalScale(SparseMat *StokesA, SparseMat *StokesB, SparseMat *StokesC, SparseMat *StokesD) {
    g_status = 0;
    dropin_check(diag_dropin(StokesA, StokesB, StokesC, StokesD, 0));
}

extern "C" void ScaleMatrix(SparseMat *StokesA, SparseMat *StokesB, SparseMat *StokesC, SparseMat *StokesD) {
    g_status = 0;
    dropin_check(diag_dropin(StokesA, StokesB, StokesC, StokesD, 1));
}

/* StokesAssemblyCoupled.c:47 -- append a coefficient, or fold a Dirichlet /
 * surface-pressure / non-conforming / matching-Neumann neighbour into the
 * right-hand side.  Host bookkeeping helper of the assembly interface. */
extern "C" void AddCoeff2(int *J, double *A, int eqn, int jeq, int *nnzc, double coeff, int NODE_TYPE, double NODE_VAL,
                          double *RHS) {
    if (NODE_TYPE == 0 || NODE_TYPE == 31 || NODE_TYPE == 11 || NODE_TYPE == 13) {
        RHS[eqn] -= coeff * NODE_VAL;
    } else {
        J[*nnzc] = jeq;
        A[*nnzc] = coeff;
        (*nnzc)++;
    }
}

/* Pointwise Viscosity: evaluated by one GPU lane. */
struct ViscArgs {
    int phase;
    double G, T, P, d, phi, X0, Exx, Ezz, Exz, Gxx, Gzz, Gxz, Txx0, Tzz0, Txz0, dil, fric, C, P0, beta;
};
__global__ void k_viscosity_point(ViscArgs a, const mat_prop *mt, DevParams prm, VOut *out) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    VGuess gs;
    gs.mode = MDZ_RHEO_FP64;
    gs.factor = 0.0;
    gs.gdot = 0.0;
    VOut o;
    mdz_viscosity(a.phase, a.G, a.T, a.P, a.d, a.phi, a.X0, a.Exx, a.Ezz, a.Exz, a.Gxx, a.Gzz, a.Gxz, a.Txx0, a.Tzz0,
                  a.Txz0, mt, prm, a.dil, a.fric, a.C, a.P0, a.beta, gs, o);
    *out = o;
}

static mdz_ctx *g_point_ctx = nullptr;
static VOut *g_point_out = nullptr;

extern "C" double Viscosity(int phase, double G, double T, double P, double d, double phi, double X0, double Exx,
                            double Ezz, double Exz, double Gxx, double Gzz, double Gxz, double Txx0, double Tzz0,
                            double Txz0, mat_prop *materials, params *model, scale *scaling, double *txxn,
                            double *tzzn, double *txzn, double *etaVE, double *VEcoeff, double *Eii_el, double *Eii_pl,
                            double *Eii_pwl, double *Eii_exp, double *Eii_lin, double *Eii_gbs, double *Eii_cst,
                            double *Exx_el, double *Ezz_el, double *Exz_el, double *Exx_diss, double *Ezz_diss,
                            double *Exz_diss, double *d1, double strain_acc, double dil, double fric, double C,
                            double *detadexx, double *detadezz, double *detadexz, double *detadp, double P0, double *X1,
                            double *OverS, double *ddivpdexx, double *ddivpdezz, double *ddivpdexz, double *ddivpdp,
                            double *Pcorr, double *drhodp, double *rho, double beta, double div, double *div_el,
                            double *div_pl, double *div_r) {
    g_status = 0;
    (void)strain_acc; (void)div;
    if (!g_point_ctx) {
        if (ctx_alloc(&g_point_ctx, 4, 4, 1)) { dropin_check(g_status); return 0.0; }
        if (hipMalloc((void **)&g_point_out, sizeof(VOut)) != hipSuccess) { dropin_check(set_err(MDZ_ENOMEM, "point")); return 0.0; }
    }
    mdz_ctx *c = g_point_ctx;
    fill_params(c, model, scaling);
    if (check_supported(model, materials)) { dropin_check(g_status); return 0.0; }
    up_materials(c, materials);
    ViscArgs a = {phase, G, T, P, d, phi, X0, Exx, Ezz, Exz, Gxx, Gzz, Gxz, Txx0, Tzz0, Txz0, dil, fric, C, P0, beta};
    hipLaunchKernelGGL(k_viscosity_point, dim3(1), dim3(64), 0, c->stream, a, (const mat_prop *)c->d_mat, c->prm, g_point_out);
    VOut o;
    hipMemcpyAsync(&o, g_point_out, sizeof(VOut), hipMemcpyDeviceToHost, c->stream);
    dropin_check(sync(c));
    *txxn = o.txx; *tzzn = o.tzz; *txzn = o.txz; *etaVE = o.etaVE; *VEcoeff = o.VEcoeff;
    *Eii_el = o.Eii_el; *Eii_pl = o.Eii_pl; *Eii_pwl = o.Eii_pwl; *Eii_exp = o.Eii_exp; *Eii_lin = o.Eii_lin;
    *Eii_gbs = o.Eii_gbs; *Eii_cst = o.Eii_cst; *Exx_el = o.Exx_el; *Ezz_el = o.Ezz_el; *Exz_el = o.Exz_el;
    *Exx_diss = o.Exx_diss; *Ezz_diss = o.Ezz_diss; *Exz_diss = o.Exz_diss; *d1 = o.d1;
    *detadexx = o.detadexx; *detadezz = o.detadezz; *detadexz = o.detadexz; *detadp = o.detadp; *X1 = o.X1;
    *OverS = o.OverS; *ddivpdexx = o.ddivpdexx; *ddivpdezz = o.ddivpdezz; *ddivpdexz = o.ddivpdexz;
    *ddivpdp = o.ddivpdp; *Pcorr = o.Pcorr; *drhodp = o.drhodp; *rho = o.rho; *div_el = o.div_el;
    *div_pl = o.div_pl; *div_r = o.div_r;
    return o.eta;
}

/* ------------------------------------------------------------------ */
/* device-resident interface                                            */
/* ------------------------------------------------------------------ */
extern "C" int mdz_ctx_create(mdz_ctx **out, const grid *mesh, const mat_prop *materials, const params *model,
                              const scale *scaling) {
    g_status = 0;
    if (!out || !mesh || !materials || !model || !scaling) return set_err(MDZ_EINVAL, "NULL argument");
    int rc = check_supported(model, materials);
    if (rc) return rc;
    if ((rc = validate_tags(mesh))) return rc;
    mdz_ctx *c = nullptr;
    if ((rc = ctx_alloc(&c, mesh->Nx, mesh->Nz, model->Nb_phases))) return rc;
    c->g.dx = mesh->dx; c->g.dz = mesh->dz;
    fill_params(c, model, scaling);
    c->prm.rheo_mode = MDZ_RHEO_FP64;
    if ((rc = up_tags(c, mesh)) || (rc = up_coords(c, mesh)) || (rc = up_phases(c, mesh, model->Nb_phases)) ||
        (rc = up_materials(c, materials))) { ctx_release(c); return rc; }
    for (int i = 0; i < FI_COUNT; i++)
        if ((rc = up(c, mesh, i))) { ctx_release(c); return rc; }
    if ((rc = mdz_number_equations(c->g, c->e, c->scratch, c->scratch_len, c->stream))) { ctx_release(c); return rc; }
    if ((rc = build_pattern(c, 0)) || (rc = build_pattern(c, 1))) { ctx_release(c); return rc; }
    *out = c;
    return MDZ_OK;
}

extern "C" void mdz_ctx_destroy(mdz_ctx *ctx) { ctx_release(ctx); }

extern "C" void *mdz_ctx_stream(mdz_ctx *ctx) { return ctx ? (void *)ctx->stream : nullptr; }

extern "C" int mdz_ctx_upload_step_fields(mdz_ctx *c, const grid *mesh) {
    if (!c || !mesh) return set_err(MDZ_EINVAL, "NULL argument");
    int rc;
    if ((rc = flush_diagnostics(c))) return rc;
    for (int i = 0; i < FI_COUNT; i++)
        if (FREF[i].role == MDZ_ROLE_I && i != FI_u_in && i != FI_v_in && i != FI_p_in)
            if ((rc = up(c, mesh, i))) return rc;
    if ((rc = up_phases(c, mesh, c->nph))) return rc;
    return sync(c);
}

extern "C" int mdz_ctx_update_step(mdz_ctx *c, const grid *mesh, const mat_prop *materials, const params *model,
                                   const scale *scaling) {
    g_status = 0;
    if (!c || !mesh || !materials || !model || !scaling) return set_err(MDZ_EINVAL, "NULL argument");
    if (mesh->Nx != c->Nx || mesh->Nz != c->Nz || model->Nb_phases != c->nph)
        return set_err(MDZ_EINVAL, "time-step update: grid %d x %d with %d phases, context %d x %d with %d", mesh->Nx,
                       mesh->Nz, model->Nb_phases, c->Nx, c->Nz, c->nph);
    int rc = check_supported(model, materials);
    if (rc) return rc;
    if ((rc = validate_tags(mesh))) return rc;
    if ((rc = sync(c))) return rc;
    c->g.dx = mesh->dx; c->g.dz = mesh->dz;
    fill_params(c, model, scaling);
    if ((rc = up_tags(c, mesh)) || (rc = up_coords(c, mesh)) || (rc = up_phases(c, mesh, c->nph)) ||
        (rc = up_materials(c, materials)))
        return rc;
    for (int i = 0; i < FI_COUNT; i++)
        if ((rc = up(c, mesh, i))) return rc;
    /* every output field is now the host's: nothing deferred, no snapshot, J = 0 layout */
    c->diag_stale = 0;
    c->p_snapped = 0;
    c->d_jac = 0;
    if ((rc = mdz_number_equations(c->g, c->e, c->scratch, c->scratch_len, c->stream))) return rc;
    if ((rc = build_pattern(c, 0)) || (rc = build_pattern(c, 1))) return rc;
    c->version++;
    return sync(c);
}

extern "C" int mdz_ctx_upload_solution(mdz_ctx *c, const double *u, const double *v, const double *p) {
    if (!c || !u || !v || !p) return set_err(MDZ_EINVAL, "NULL argument");
    int rc;
    if ((rc = snapshot_p(c, c->stream))) return rc;
    HIPCHK(hipMemcpyAsync(c->g.u_in, u, fam_len(MDZ_FAM_U, c->Nx, c->Nz) * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->g.v_in, v, fam_len(MDZ_FAM_W, c->Nx, c->Nz) * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->g.p_in, p, fam_len(MDZ_FAM_C, c->Nx, c->Nz) * 8, hipMemcpyHostToDevice, c->stream));
    return sync(c);
}

extern "C" int mdz_ctx_download_solution(mdz_ctx *c, double *u, double *v, double *p) {
    if (!c || !u || !v || !p) return set_err(MDZ_EINVAL, "NULL argument");
    HIPCHK(hipMemcpyAsync(u, c->g.u_in, fam_len(MDZ_FAM_U, c->Nx, c->Nz) * 8, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipMemcpyAsync(v, c->g.v_in, fam_len(MDZ_FAM_W, c->Nx, c->Nz) * 8, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipMemcpyAsync(p, c->g.p_in, fam_len(MDZ_FAM_C, c->Nx, c->Nz) * 8, hipMemcpyDeviceToHost, c->stream));
    return sync(c);
}

extern "C" int mdz_ctx_download_grid(mdz_ctx *c, grid *mesh) {
    if (!c || !mesh) return set_err(MDZ_EINVAL, "NULL argument");
    int rc;
    if ((rc = flush_diagnostics(c))) return rc;
    /* the grid after a unit holds the J = 0 tensor, as the reference's does
     * (RheologicalOperators(..., 0) before the residual) */
    if (c->d_jac) {
        mdz_launch_dtensor(c->g, c->prm, 0, c->status, c->stream);
        c->d_jac = 0;
    }
    for (int i = 0; i < FI_COUNT; i++)
        if (FREF[i].role & MDZ_ROLE_O)
            if ((rc = down(c, mesh, i))) return rc;
    return sync(c);
}

extern "C" int mdz_ctx_fuse_guess(mdz_ctx *c, int on) {
    if (!c) return set_err(MDZ_EINVAL, "NULL context");
    int rc;
    if ((rc = flush_diagnostics(c))) return rc;
    c->guess_fused = on != 0;
    c->version++;
    return MDZ_OK;
}

extern "C" int mdz_ctx_defer_diagnostics(mdz_ctx *c, int on) {
    if (!c) return set_err(MDZ_EINVAL, "NULL context");
    c->defer_diag = on != 0;
    c->version++;
    return MDZ_OK;
}

extern "C" int mdz_ctx_set_rheology_mode(mdz_ctx *c, int mode) {
    if (!c || mode < MDZ_RHEO_FP64 || mode > MDZ_RHEO_LEARNED) return set_err(MDZ_EINVAL, "rheology mode %d", mode);
    if (mode == MDZ_RHEO_LEARNED && !c->d_net) return set_err(MDZ_EINVAL, "learned mode needs mdz_ctx_set_network first");
    int rc;
    if ((rc = flush_diagnostics(c))) return rc;
    c->prm.rheo_mode = mode;
    c->version++;
    return MDZ_OK;
}

/* residual rows of block family `kind` and their norms into c->norm_out
 * (and copy6, see mdz_launch_residual_norms) */
static int residual_norms(mdz_ctx *c, int kind, const DevAsm &a, hipStream_t s, double *copy6 = nullptr) {
    int rc = mdz_launch_residual_norms(kind, a, &c->blk[4 * kind], &c->blk[4 * kind + 2], &c->blk[4 * kind + 3],
                                       c->norm_partial, c->norm_partial_len, c->norm_out, s, c->d_scaled[kind], copy6);
    return rc ? set_err(rc, "residual norms") : MDZ_OK;
}

/* One Newton-iteration unit of a context, enqueued on stream s with no
 * allocation, memset, host synchronisation or copy: safe to capture into a
 * graph.  The norms stay in c->norm_out (six doubles); copy6 (optional,
 * pinned) receives them too. */
static int enqueue_unit(mdz_ctx *c, hipStream_t s, double *copy6 = nullptr) {
    DevAsm a = make_asm(c), ap = picard_asm(c);
    mdz_launch_strain_interp5(c->g, c->prm, s);
    int rc = rheology_pass(c, c->prm.rheo_mode == MDZ_RHEO_LEARNED, s, true);
    if (rc) return rc;
    const int kind = c->model.aniso == 1 ? 1 : 0;
    if (fused_dtensor(c)) {
        mdz_launch_rhs_dtensor(c->g, c->prm, 2, c->xg, c->zvx, c->xvz, c->zg, c->status, s, c->dpic_n, c->dpic_s);
        const bool pair = mdz_launch_values_pair(ap, &c->blk[0], &c->blk[4], c->shape, s);
        if (!pair) mdz_launch_values(0, ap, &c->blk[0], &c->blk[1], &c->blk[2], &c->blk[3], c->shape.pic, s);
        if ((rc = residual_norms(c, 0, ap, s, copy6))) return rc;
        if (!pair) mdz_launch_values(1, a, &c->blk[4], &c->blk[5], &c->blk[6], &c->blk[7], c->shape.jac, s);
        c->d_jac = 1;
        return MDZ_OK;
    }
    mdz_launch_rhs_dtensor(c->g, c->prm, 0, c->xg, c->zvx, c->xvz, c->zg, c->status, s);
    mdz_launch_values(0, a, &c->blk[0], &c->blk[1], &c->blk[2], &c->blk[3], c->shape.pic, s);
    mdz_launch_dtensor(c->g, c->prm, 1, c->status, s);
    mdz_launch_values(1, a, &c->blk[4], &c->blk[5], &c->blk[6], &c->blk[7], c->shape.jac, s);
    mdz_launch_dtensor(c->g, c->prm, 0, c->status, s);
    return residual_norms(c, kind, a, s, copy6);
}

/* resx, resz, resp from the six sums of the norm kernels */
static int norms_to_res(const double *out6, double *res3) {
    res3[0] = sqrt(out6[0] / out6[3]);
    res3[1] = sqrt(out6[1] / out6[4]);
    res3[2] = sqrt(out6[2] / out6[5]);
    if (isnan(res3[0]) || isnan(res3[1]) || isnan(res3[2])) return set_err(MDZ_ENAN, "NaN residual");
    return MDZ_OK;
}

extern "C" int mdz_ctx_newton_unit(mdz_ctx *c, double *res3) {
    if (!c) return set_err(MDZ_EINVAL, "NULL context");
    g_status = 0;
    int rc = enqueue_unit(c, c->stream, res3 ? c->norm_host : nullptr);
    if (rc) return rc;
    if (res3) {
        if ((rc = sync(c))) return rc;
        if ((rc = norms_to_res(c->norm_host, res3))) return rc;
    }
    HIPCHK(hipGetLastError());
    return MDZ_OK;
}

extern "C" int mdz_ctx_block_info(mdz_ctx *c, int which, int *neq, int *nnz) {
    if (!c || which < 0 || which > 7) return set_err(MDZ_EINVAL, "block %d", which);
    if (neq) *neq = c->blk[which].neq;
    if (nnz) *nnz = c->blk[which].nnz;
    return MDZ_OK;
}

extern "C" int mdz_ctx_download_block(mdz_ctx *c, int which, int *Ic, int *J, double *A, double *b, double *bbc) {
    if (!c || which < 0 || which > 7) return set_err(MDZ_EINVAL, "block %d", which);
    DevBlock *k = &c->blk[which];
    if (Ic) HIPCHK(hipMemcpyAsync(Ic, k->Ic, ((size_t)k->neq + 1) * 4, hipMemcpyDeviceToHost, c->stream));
    if (J && k->nnz) HIPCHK(hipMemcpyAsync(J, k->J, (size_t)k->nnz * 4, hipMemcpyDeviceToHost, c->stream));
    if (A && k->nnz) HIPCHK(hipMemcpyAsync(A, k->A, (size_t)k->nnz * 8, hipMemcpyDeviceToHost, c->stream));
    if (b) HIPCHK(hipMemcpyAsync(b, k->b, (size_t)k->neq * 8, hipMemcpyDeviceToHost, c->stream));
    if (bbc) HIPCHK(hipMemcpyAsync(bbc, k->bbc, (size_t)k->neq * 8, hipMemcpyDeviceToHost, c->stream));
    return sync(c);
}

extern "C" int mdz_ctx_download_residual(mdz_ctx *c, double *Fmom, double *Fcont) {
    if (!c) return set_err(MDZ_EINVAL, "NULL context");
    int kind = c->model.aniso == 1 ? 1 : 0;
    if (Fmom) HIPCHK(hipMemcpyAsync(Fmom, c->blk[4 * kind].F, (size_t)c->e.neq_mom * 8, hipMemcpyDeviceToHost, c->stream));
    if (Fcont) HIPCHK(hipMemcpyAsync(Fcont, c->blk[4 * kind + 3].F, (size_t)c->e.neq_cont * 8, hipMemcpyDeviceToHost, c->stream));
    return sync(c);
}

/* ------------------------------------------------------------------ */
/* marker -> grid                                                       */
/* ------------------------------------------------------------------ */
static int ensure_mstore(mdz_ctx *c) {
    if (c->ms) return MDZ_OK;
    return mdz_mstore_create(&c->ms, c->Nx, c->Nz);
}

/* family slot of P2Mastah's `centroid` (1 centroids, 0 vertices, -1 Vx, -2 Vz nodes) */
static int p2g_family(int centroid) {
    switch (centroid) {
    case 1: return 0;
    case 0: return 1;
    case -1: return 2;
    case -2: return 3;
    default: return -1;
    }
}

extern "C" void P2Mastah(params *model, markers particles, DoodzFP *mat_prop, grid *mesh, double *NodeField,
                         char *NodeType, int flag, int avg, int prop, int centroid, int itp_stencil) {
    g_status = 0;
    const int fam = p2g_family(centroid);
    if (!model || !mesh || !NodeType || fam < 0 || (itp_stencil != 1 && itp_stencil != 9) || flag < 0 || flag > 1 ||
        avg < 0 || avg > 2 || (prop == 0 && (!mat_prop || !NodeField))) {
        dropin_check(set_err(MDZ_EINVAL, "P2Mastah: bad arguments"));
        return;
    }
    const int nph = model->Nb_phases > 0 ? model->Nb_phases : 1;
    mdz_ctx *c = dropin_ctx(mesh, nph);
    if (!c) return;
    int rc = ensure_mstore(c);
    int nx, nz;
    mdz_family_dims(fam, mesh->Nx, mesh->Nz, &nx, &nz);
    const size_t n = (size_t)nx * nz;
    NodeAxes a;
    if (!rc) rc = mdz_mstore_axes(c->ms, fam, mesh, nullptr, nullptr, model->isperiodic_x == 1, c->stream, &a);
    if (!rc) rc = mdz_mstore_upload(c->ms, &particles, prop == 0 && flag == 1 ? mat_prop : nullptr, nph, c->stream);
    if (!rc) rc = mdz_mstore_bin(c->ms, fam, a, c->stream);
    if (rc) { dropin_check(rc); return; }
    int8_t *ntype = mdz_mstore_node_types(c->ms);
    double *field = mdz_mstore_node_field(c->ms), *pval = mdz_mstore_phase_values(c->ms);
    double **perc = centroid == 0 ? mesh->phase_perc_s : centroid == 1 ? mesh->phase_perc_n : nullptr;
    double *dperc = centroid == 0 ? c->g.phase_s : c->g.phase_n;
    const int np = nph < c->nph ? nph : c->nph;
    if (hipMemcpyAsync(ntype, NodeType, n, hipMemcpyHostToDevice, c->stream) != hipSuccess ||
        (prop == 0 && hipMemcpyAsync(field, NodeField, n * 8, hipMemcpyHostToDevice, c->stream) != hipSuccess) ||
        (prop == 0 && flag == 0 &&
         hipMemcpyAsync(pval, mat_prop, (size_t)nph * 8, hipMemcpyHostToDevice, c->stream) != hipSuccess)) {
        dropin_check(set_err(MDZ_EHIP, "P2Mastah: upload"));
        return;
    }
    if (prop == 1 && !perc) return; /* Vx / Vz nodes hold no phase fractions: nothing to write */
    P2GArgs g{flag, avg, np, mdz_mstore_dev(c->ms).val, pval, ntype, field, dperc};
    mdz_launch_p2mastah(mdz_mstore_dev(c->ms), fam, a, prop, itp_stencil, g, c->stream);
    if (prop == 0) {
        if (hipMemcpyAsync(NodeField, field, n * 8, hipMemcpyDeviceToHost, c->stream) != hipSuccess) {
            dropin_check(set_err(MDZ_EHIP, "P2Mastah: download"));
            return;
        }
    } else {
        for (int p = 0; p < np; p++)
            if (hipMemcpyAsync(perc[p], dperc + (size_t)p * n, n * 8, hipMemcpyDeviceToHost, c->stream) != hipSuccess) {
                dropin_check(set_err(MDZ_EHIP, "P2Mastah: download"));
                return;
            }
    }
    dropin_check(sync(c));
}

extern "C" void Interp_P2N(markers particles, DoodzFP *mat_prop, grid *mesh, double *NodeField, double *X_vect,
                           double *Z_vect, int flag, int itp_type, params *model) {
    g_status = 0;
    if (!model || !mesh || !mat_prop || !NodeField || !X_vect || !Z_vect || flag < 0 || flag > 1 || itp_type < 0 ||
        itp_type > 2) {
        dropin_check(set_err(MDZ_EINVAL, "Interp_P2N: bad arguments"));
        return;
    }
    const int nph = model->Nb_phases > 0 ? model->Nb_phases : 1;
    mdz_ctx *c = dropin_ctx(mesh, nph);
    if (!c) return;
    /* the grid's own vertex axes share the vertex bins; other axes get slot 4 */
    const int fam = X_vect == mesh->xg_coord && Z_vect == mesh->zg_coord ? 1 : 4;
    int rc = ensure_mstore(c);
    const size_t n = (size_t)mesh->Nx * mesh->Nz;
    NodeAxes a;
    if (!rc) rc = mdz_mstore_axes(c->ms, fam, mesh, X_vect, Z_vect, model->isperiodic_x == 1, c->stream, &a);
    if (!rc) rc = mdz_mstore_upload(c->ms, &particles, flag == 1 ? mat_prop : nullptr, nph, c->stream);
    if (!rc) rc = mdz_mstore_bin(c->ms, fam, a, c->stream);
    if (rc) { dropin_check(rc); return; }
    int8_t *ntype = mdz_mstore_node_types(c->ms);
    double *field = mdz_mstore_node_field(c->ms), *pval = mdz_mstore_phase_values(c->ms);
    if (hipMemcpyAsync(ntype, mesh->BCg.type, n, hipMemcpyHostToDevice, c->stream) != hipSuccess ||
        hipMemcpyAsync(field, NodeField, n * 8, hipMemcpyHostToDevice, c->stream) != hipSuccess ||
        (flag == 0 && hipMemcpyAsync(pval, mat_prop, (size_t)nph * 8, hipMemcpyHostToDevice, c->stream) != hipSuccess)) {
        dropin_check(set_err(MDZ_EHIP, "Interp_P2N: upload"));
        return;
    }
    P2GArgs g{flag, itp_type, nph, mdz_mstore_dev(c->ms).val, pval, ntype, field, nullptr};
    mdz_launch_interp_p2n(mdz_mstore_dev(c->ms), fam, a, g, c->stream);
    if (hipMemcpyAsync(NodeField, field, n * 8, hipMemcpyDeviceToHost, c->stream) != hipSuccess) {
        dropin_check(set_err(MDZ_EHIP, "Interp_P2N: download"));
        return;
    }
    dropin_check(sync(c));
}

/* the marker-to-grid strength parameters on a context's device-resident
 * phase fractions and tags, into its C / fric / dil fields */
static int cfd_on_ctx(mdz_ctx *c, const grid *mesh, const mat_prop *materials, const params *model) {
    NodeAxes ac, av;
    int rc = mdz_mstore_axes(c->ms, 0, mesh, nullptr, nullptr, model->isperiodic_x == 1, c->stream, &ac);
    if (!rc) rc = mdz_mstore_axes(c->ms, 1, mesh, nullptr, nullptr, model->isperiodic_x == 1, c->stream, &av);
    if (rc) return rc;
    const SoftK sk = mdz_soft_constants(materials, model->Nb_phases < c->nph ? model->Nb_phases : c->nph);
    return mdz_mstore_cfd(c->ms, ac, av, model->itp_stencil, sk, c->g.phase_n, c->g.phase_s, c->g.BCp, c->g.BCg,
                          c->g.fric_n, c->g.dil_n, c->g.C_n, c->g.fric_s, c->g.dil_s, c->g.C_s, c->stream);
}

extern "C" void CohesionFrictionDilationGrid(grid *mesh, markers *particles, mat_prop materials, params model,
                                             scale scaling) {
    g_status = 0;
    (void)scaling;
    if (!mesh || !particles || !particles->strain_pl || (model.itp_stencil != 1 && model.itp_stencil != 9)) {
        dropin_check(set_err(MDZ_EINVAL, "CohesionFrictionDilationGrid: bad arguments"));
        return;
    }
    const int nph = model.Nb_phases > 0 ? model.Nb_phases : 1;
    mdz_ctx *c = dropin_ctx(mesh, nph);
    if (!c) return;
    int rc = ensure_mstore(c);
    const size_t nc = fam_len(MDZ_FAM_C, c->Nx, c->Nz), nv = fam_len(MDZ_FAM_V, c->Nx, c->Nz);
    if (!rc && (hipMemcpyAsync(c->g.BCp, mesh->BCp.type, nc, hipMemcpyHostToDevice, c->stream) != hipSuccess ||
                hipMemcpyAsync(c->g.BCg, mesh->BCg.type, nv, hipMemcpyHostToDevice, c->stream) != hipSuccess))
        rc = set_err(MDZ_EHIP, "CohesionFrictionDilationGrid: tags");
    if (!rc) rc = up_phases(c, mesh, nph);
    if (!rc) rc = mdz_mstore_upload(c->ms, particles, particles->strain_pl, nph, c->stream);
    if (!rc) rc = cfd_on_ctx(c, mesh, &materials, &model);
    if (rc) { dropin_check(rc); return; }
    dropin_check(down_list(c, mesh, {FI_fric_n, FI_dil_n, FI_C_n, FI_fric_s, FI_dil_s, FI_C_s}));
    dropin_check(sync(c));
}

/* Device-resident marker-to-grid step of a context: the markers (x, z,
 * phase, strain_pl) go to the device, then the phase fractions at the
 * centroids and vertices (CountPartCell's P2Mastah calls,
 * ParticleRoutines.c:3566-3567) and the strength parameters
 * (CohesionFrictionDilationGrid) are computed into the context's fields,
 * where the next unit reads them. */
extern "C" int mdz_ctx_markers_to_grid(mdz_ctx *c, grid *mesh, const markers *m, int download) {
    g_status = 0;
    if (!c || !mesh) return set_err(MDZ_EINVAL, "NULL argument");
    if (mesh->Nx != c->Nx || mesh->Nz != c->Nz) return set_err(MDZ_EINVAL, "markers: grid size differs from the context's");
    if (m && !m->strain_pl && m->Nb_part > 0) return set_err(MDZ_EINVAL, "markers: strain_pl missing");
    if (!m && !c->ms) return set_err(MDZ_EINVAL, "markers: none on the device yet");
    int rc = flush_diagnostics(c);
    if (!rc) rc = ensure_mstore(c);
    if (!rc && m) rc = mdz_mstore_upload(c->ms, m, m->strain_pl, c->model.Nb_phases, c->stream);
    /* markers already on the device: bin them again (they may have moved) */
    if (!rc && !m) mdz_mstore_rebin(c->ms);
    const int periodic = c->model.isperiodic_x == 1;
    NodeAxes ac, av;
    if (!rc) rc = mdz_mstore_axes(c->ms, 0, mesh, nullptr, nullptr, periodic, c->stream, &ac);
    if (!rc) rc = mdz_mstore_axes(c->ms, 1, mesh, nullptr, nullptr, periodic, c->stream, &av);
    if (rc) return rc;
    const int np = c->model.Nb_phases < c->nph ? c->model.Nb_phases : c->nph;
    const int itp = c->model.itp_stencil == 9 ? 9 : 1;
    /* the 1-node stencil takes one binning by quarter cell for both families
     * where the centroids lie between the vertices, as on any grid of the
     * reference */
    const double sx = (mesh->xc_coord[0] - mesh->xg_coord[0]) / mesh->dx;
    const double sz = (mesh->zc_coord[0] - mesh->zg_coord[0]) / mesh->dz;
    if (itp == 1 && sx > 0.25 && sx < 0.75 && sz > 0.25 && sz < 0.75) {
        const SoftK sk = mdz_soft_constants(&c->materials, np);
        if ((rc = mdz_mstore_step(c->ms, ac, av, sk, c->g.phase_n, c->g.phase_s, c->g.BCp, c->g.BCg, c->g.fric_n,
                                  c->g.dil_n, c->g.C_n, c->g.fric_s, c->g.dil_s, c->g.C_s, c->stream)))
            return rc;
    } else {
        if ((rc = mdz_mstore_bin(c->ms, 0, ac, c->stream)) || (rc = mdz_mstore_bin(c->ms, 1, av, c->stream))) return rc;
        const MarkerDev &md = mdz_mstore_dev(c->ms);
        mdz_launch_p2mastah(md, 0, ac, 1, itp, P2GArgs{0, 0, np, nullptr, nullptr, c->g.BCp, nullptr, c->g.phase_n},
                            c->stream);
        mdz_launch_p2mastah(md, 1, av, 1, itp, P2GArgs{0, 0, np, nullptr, nullptr, c->g.BCg, nullptr, c->g.phase_s},
                            c->stream);
        if ((rc = cfd_on_ctx(c, mesh, &c->materials, &c->model))) return rc;
    }
    HIPCHK(hipGetLastError());
    if (download) {
        const size_t nc = fam_len(MDZ_FAM_C, c->Nx, c->Nz), nv = fam_len(MDZ_FAM_V, c->Nx, c->Nz);
        for (int p = 0; p < np; p++) {
            HIPCHK(hipMemcpyAsync(mesh->phase_perc_n[p], c->g.phase_n + p * nc, nc * 8, hipMemcpyDeviceToHost, c->stream));
            HIPCHK(hipMemcpyAsync(mesh->phase_perc_s[p], c->g.phase_s + p * nv, nv * 8, hipMemcpyDeviceToHost, c->stream));
        }
        if ((rc = down_list(c, mesh, {FI_fric_n, FI_dil_n, FI_C_n, FI_fric_s, FI_dil_s, FI_C_s}))) return rc;
    }
    return sync(c);
}

/* The HDF5 dump of the blocks of the last unit (kind 0 Picard, 1 Jacobian);
 * the right-hand sides are those of that kind's assembly, the residuals
 * those of the unit's residual evaluation. */
extern "C" int mdz_ctx_write_matrix_h5(mdz_ctx *c, int kind, const char *filename) {
    if (!c || kind < 0 || kind > 1 || !filename) return set_err(MDZ_EINVAL, "matrix dump: bad argument");
    if (!c->pattern_ready[kind]) return set_err(MDZ_EINVAL, "matrix dump before the blocks are assembled");
    const size_t nx = c->Nx, nz = c->Nz, nu = nx * (nz + 1), nw = (nx + 1) * nz, nc = (nx - 1) * (nz - 1), nv = nx * nz;
    std::vector<int> eu(nu), ev(nw), ep(nc);
    std::vector<double> eta_n(nc), eta_s(nv);
    std::vector<char> ts(nv), tn(nc), tu(nu), tv(nw);
    HIPCHK(hipMemcpyAsync(eu.data(), c->e.eqn_u, nu * 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipMemcpyAsync(ev.data(), c->e.eqn_v, nw * 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipMemcpyAsync(ep.data(), c->e.eqn_p, nc * 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipMemcpyAsync(eta_n.data(), c->g.eta_n, nc * 8, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipMemcpyAsync(eta_s.data(), c->g.eta_s, nv * 8, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipMemcpyAsync(ts.data(), c->g.BCg, nv, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipMemcpyAsync(tn.data(), c->g.BCp, nc, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipMemcpyAsync(tu.data(), c->g.BCu, nu, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipMemcpyAsync(tv.data(), c->g.BCv, nw, hipMemcpyDeviceToHost, c->stream));
    std::vector<int> Ic[4], J[4];
    std::vector<double> V[4];
    for (int b = 0; b < 4; b++) {
        const DevBlock &k = c->blk[4 * kind + b];
        Ic[b].resize((size_t)k.neq + 1);
        J[b].resize(k.nnz);
        V[b].resize(k.nnz);
        HIPCHK(hipMemcpyAsync(Ic[b].data(), k.Ic, ((size_t)k.neq + 1) * 4, hipMemcpyDeviceToHost, c->stream));
        if (k.nnz) {
            HIPCHK(hipMemcpyAsync(J[b].data(), k.J, (size_t)k.nnz * 4, hipMemcpyDeviceToHost, c->stream));
            HIPCHK(hipMemcpyAsync(V[b].data(), k.A, (size_t)k.nnz * 8, hipMemcpyDeviceToHost, c->stream));
        }
    }
    const int rk = c->model.aniso == 1 ? 1 : 0;
    const DevBlock &A = c->blk[4 * kind], &C = c->blk[4 * kind + 2];
    std::vector<double> bm(A.neq), bc(C.neq), Fm(A.neq), Fc(C.neq);
    HIPCHK(hipMemcpyAsync(bm.data(), A.b, (size_t)A.neq * 8, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipMemcpyAsync(bc.data(), C.b, (size_t)C.neq * 8, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipMemcpyAsync(Fm.data(), c->blk[4 * rk].F, (size_t)A.neq * 8, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipMemcpyAsync(Fc.data(), c->blk[4 * rk + 2].F, (size_t)C.neq * 8, hipMemcpyDeviceToHost, c->stream));
    int rc = sync(c);
    if (rc) return rc;
    MdzMatrixDump d;
    d.nx = c->Nx; d.nz = c->Nz; d.dx = c->g.dx; d.dz = c->g.dz;
    d.eqn_u = eu.data(); d.eqn_v = ev.data(); d.eqn_p = ep.data();
    d.eta_n = eta_n.data(); d.eta_s = eta_s.data();
    d.tag_s = ts.data(); d.tag_n = tn.data(); d.tag_u = tu.data(); d.tag_v = tv.data();
    for (int b = 0; b < 4; b++) {
        d.neq[b] = c->blk[4 * kind + b].neq; d.nnz[b] = c->blk[4 * kind + b].nnz;
        d.Ic[b] = Ic[b].data(); d.J[b] = J[b].data(); d.V[b] = V[b].data();
    }
    d.rhs_mom = bm.data(); d.rhs_cont = bc.data(); d.F_mom = Fm.data(); d.F_cont = Fc.data();
    return mdz_h5_write_dump(filename, d);
}

extern "C" int mdz_ctx_diagonal_scaling(mdz_ctx *c, int kind) {
    if (!c || kind < 0 || kind > 1) return set_err(MDZ_EINVAL, "diagonal scaling kind %d", kind);
    if (!c->pattern_ready[kind]) return set_err(MDZ_EINVAL, "diagonal scaling before the blocks are assembled");
    DevBlock *b = &c->blk[4 * kind];
    mdz_launch_extract_diagonal(&b[0], &b[1], &b[2], &b[3], c->stream);
    mdz_launch_scale_matrix(&b[0], &b[1], &b[2], &b[3], c->stream);
    c->d_scaled[kind] = 1;
    HIPCHK(hipGetLastError());
    return MDZ_OK;
}

extern "C" int mdz_ctx_collect_histogram(mdz_ctx *c, int on) {
    if (!c) return set_err(MDZ_EINVAL, "NULL context");
    c->hist_on = on != 0;
    c->version++;
    return MDZ_OK;
}

extern "C" int mdz_ctx_iteration_histogram(mdz_ctx *c, long long *hist) {
    if (!c || !hist) return set_err(MDZ_EINVAL, "NULL argument");
    HIPCHK(hipMemcpyAsync(hist, c->hist, 3 * MDZ_HIST_BINS * 8, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipMemsetAsync(c->hist, 0, 3 * MDZ_HIST_BINS * 8, c->stream));
    return sync(c);
}

extern "C" int mdz_ctx_set_network(mdz_ctx *c, const float *w, size_t n) {
    if (!c || !w) return set_err(MDZ_EINVAL, "network weights");
    if (n != MLP_NPARAMS) return set_err(MDZ_EINVAL, "network weights: %zu floats, expected %d", n, MLP_NPARAMS);
    if (c->nph > 3 || c->prm.Nb_phases > 3) return set_err(MDZ_EUNSUPPORTED, "the network encodes three phases");
    if (!c->d_net) {
        HIPCHK(hipMalloc((void **)&c->d_net, n * sizeof(float)));
        HIPCHK(hipMalloc((void **)&c->net_wp, MLI_TOTAL * sizeof(unsigned short)));
        HIPCHK(hipMalloc((void **)&c->net_bp, MLI_B_TOTAL * sizeof(float)));
    }
    if (!c->guess_n) {
        /* per phase: the eta_ve factor, then the plastic multiplier */
        HIPCHK(hipMalloc((void **)&c->guess_n, 2 * (size_t)c->nph * (c->Nx - 1) * (c->Nz - 1) * sizeof(float)));
        HIPCHK(hipMalloc((void **)&c->guess_s, 2 * (size_t)c->nph * c->Nx * c->Nz * sizeof(float)));
        HIPCHK(hipMalloc((void **)&c->cellnet, (size_t)(c->Nx - 1) * (c->Nz - 1) * sizeof(CellNet)));
    }
    HIPCHK(hipMemcpyAsync(c->d_net, w, n * sizeof(float), hipMemcpyHostToDevice, c->stream));
    mdz_mlp_pack_inference(c->d_net, c->net_wp, c->net_bp, c->stream);
    HIPCHK(hipStreamSynchronize(c->stream));
    HIPCHK(hipGetLastError());
    c->net_floats = n;
    c->version++;
    return MDZ_OK;
}

/* ------------------------------------------------------------------ */
/* timing                                                               */
/* ------------------------------------------------------------------ */
/* Runs `reps` Newton units with HIP events around each stage on the
 * context's stream; ms[0..8] = mean milliseconds of the stages
 * (strain rates, rheology, rhs, D(0), Picard values, D(1), Jacobian values,
 * D(0), residual + norms), ms[9] = mean total per unit. */
extern "C" int mdz_ctx_stage_times(mdz_ctx *c, int reps, double *ms) {
    if (!c || reps < 1 || !ms) return set_err(MDZ_EINVAL, "stage times");
    const int NS = 10;
    /* begin / end event of each stage, recorded in execution order; a stage
     * that does not run (the second J = 0 tensor of a fused unit) has both
     * at the same point */
    hipEvent_t eb[NS], ee[NS];
    for (int i = 0; i < NS; i++) { HIPCHK(hipEventCreate(&eb[i])); HIPCHK(hipEventCreate(&ee[i])); }
    double acc[NS + 1] = {0};
    DevAsm a = make_asm(c), ap = picard_asm(c);
    int kind = c->model.aniso == 1 ? 1 : 0;
    const bool fused = fused_dtensor(c);
    const int learned = c->prm.rheo_mode == MDZ_RHEO_LEARNED;
    hipStream_t s = c->stream;
    auto run = [&]() -> int {
        for (int r = 0; r < reps; r++) {
            int rc;
#define STAGE(i, body) do { HIPCHK(hipEventRecord(eb[i], s)); body; HIPCHK(hipEventRecord(ee[i], s)); } while (0)
            STAGE(0, mdz_launch_strain_interp5(c->g, c->prm, s));
            STAGE(1, if ((rc = rheology_prep(c, learned, s, true))) return rc);
            STAGE(2, if ((rc = rheology_kernels(c, learned, s))) return rc);
            STAGE(3, mdz_launch_rhs(c->g, c->prm, c->xg, c->zvx, c->xvz, c->zg, s));
            if (fused) {
                /* J = 1 tensor with the J = 0 Picard components, Picard
                 * values, residual, Jacobian values */
                STAGE(6, mdz_launch_dtensor(c->g, c->prm, 2, c->status, s, c->dpic_n, c->dpic_s));
                STAGE(4, (void)0);
                STAGE(5, mdz_launch_values(0, ap, &c->blk[0], &c->blk[1], &c->blk[2], &c->blk[3], c->shape.pic, s));
                STAGE(9, if ((rc = residual_norms(c, 0, ap, s))) return rc);
                STAGE(7, mdz_launch_values(1, a, &c->blk[4], &c->blk[5], &c->blk[6], &c->blk[7], c->shape.jac, s));
                STAGE(8, (void)0);
                c->d_jac = 1;
            } else {
                STAGE(4, mdz_launch_dtensor(c->g, c->prm, 0, c->status, s));
                STAGE(5, mdz_launch_values(0, a, &c->blk[0], &c->blk[1], &c->blk[2], &c->blk[3], c->shape.pic, s));
                STAGE(6, mdz_launch_dtensor(c->g, c->prm, 1, c->status, s));
                STAGE(7, mdz_launch_values(1, a, &c->blk[4], &c->blk[5], &c->blk[6], &c->blk[7], c->shape.jac, s));
                STAGE(8, mdz_launch_dtensor(c->g, c->prm, 0, c->status, s));
                STAGE(9, if ((rc = residual_norms(c, kind, a, s))) return rc);
            }
#undef STAGE
            hipEvent_t last = fused ? ee[8] : ee[9];
            HIPCHK(hipEventSynchronize(last));
            for (int i = 0; i < NS; i++) {
                float t = 0;
                HIPCHK(hipEventElapsedTime(&t, eb[i], ee[i]));
                acc[i] += t;
            }
            float tt = 0;
            HIPCHK(hipEventElapsedTime(&tt, eb[0], last));
            acc[NS] += tt;
        }
        return MDZ_OK;
    };
    int rc = run();
    for (int i = 0; i < NS; i++) { hipEventDestroy(eb[i]); hipEventDestroy(ee[i]); }
    if (rc) return rc;
    for (int i = 0; i <= NS; i++) ms[i] = acc[i] / reps;
    HIPCHK(hipGetLastError());
    return MDZ_OK;
}

/* Streaming copy of n doubles (8-byte loads and stores, grid-stride): the
 * reference kernel for achievable HBM bandwidth and for scaling the
 * FETCH_SIZE / WRITE_SIZE counters. */
/* HBM copy probe: 16-byte non-temporal loads and stores, U of them in
 * flight per lane, one pass over the arrays (no grid-stride loop), so that
 * a launch holds enough waves and bytes in flight to reach the copy rate
 * the memory system sustains. */
typedef double mdz_d2 __attribute__((ext_vector_type(2)));
template <int U, bool NT>
__global__ void __launch_bounds__(256) k_copy_probe(const mdz_d2 *__restrict__ src, mdz_d2 *__restrict__ dst, size_t n) {
    const size_t base = (size_t)blockIdx.x * 256 * U + threadIdx.x;
    mdz_d2 v[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const size_t i = base + (size_t)u * 256;
        if (i < n) v[u] = NT ? __builtin_nontemporal_load(src + i) : src[i];
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        const size_t i = base + (size_t)u * 256;
        if (i < n) {
            if (NT) __builtin_nontemporal_store(v[u], dst + i);
            else dst[i] = v[u];
        }
    }
}

template <int U, bool NT>
static int time_copy(const mdz_d2 *a, mdz_d2 *b, size_t n, int reps, hipStream_t s, float *ms) {
    const unsigned blocks = (unsigned)((n + 256 * U - 1) / (256 * U));
    hipLaunchKernelGGL((k_copy_probe<U, NT>), dim3(blocks), dim3(256), 0, s, a, b, n);
    hipEvent_t e0, e1;
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    HIPCHK(hipEventRecord(e0, s));
    for (int r = 0; r < reps; r++) hipLaunchKernelGGL((k_copy_probe<U, NT>), dim3(blocks), dim3(256), 0, s, a, b, n);
    HIPCHK(hipEventRecord(e1, s));
    HIPCHK(hipEventSynchronize(e1));
    HIPCHK(hipEventElapsedTime(ms, e0, e1));
    *ms /= reps;
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    return MDZ_OK;
}

/* Copy rate of the best of three probe shapes (bytes read + written per
 * second, GB/s); bytes = size of each of the two arrays. */
extern "C" int mdz_copy_probe(size_t bytes, int reps, double *gbs) {
    if (bytes < 1024 || reps < 1 || !gbs) return set_err(MDZ_EINVAL, "copy probe");
    size_t n = bytes / sizeof(mdz_d2);
    mdz_d2 *a = nullptr, *b = nullptr;
    hipStream_t s;
    HIPCHK(hipStreamCreate(&s));
    if (hipMalloc((void **)&a, n * sizeof(mdz_d2)) != hipSuccess) return set_err(MDZ_ENOMEM, "copy probe");
    if (hipMalloc((void **)&b, n * sizeof(mdz_d2)) != hipSuccess) { hipFree(a); return set_err(MDZ_ENOMEM, "copy probe"); }
    HIPCHK(hipMemsetAsync(a, 0, n * sizeof(mdz_d2), s));
    float t[3] = {0, 0, 0};
    int rc = time_copy<4, true>(a, b, n, reps, s, &t[0]);
    if (!rc) rc = time_copy<8, true>(a, b, n, reps, s, &t[1]);
    if (!rc) rc = time_copy<4, false>(a, b, n, reps, s, &t[2]);
    hipFree(a);
    hipFree(b);
    hipStreamDestroy(s);
    if (rc) return rc;
    const float best = fminf(t[0], fminf(t[1], t[2]));
    *gbs = 2.0 * (double)(n * sizeof(mdz_d2)) / (best * 1e-3) / 1e9;
    return MDZ_OK;
}

/* Times `reps` back-to-back Newton units (no host synchronisation inside)
 * between two events; returns the mean milliseconds per unit. */
extern "C" int mdz_ctx_time_units(mdz_ctx *c, int reps, double *ms_per_unit) {
    if (!c || reps < 1 || !ms_per_unit) return set_err(MDZ_EINVAL, "time units");
    hipEvent_t e0, e1;
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    HIPCHK(hipEventRecord(e0, c->stream));
    for (int r = 0; r < reps; r++) {
        int rc = mdz_ctx_newton_unit(c, nullptr);
        if (rc) return rc;
    }
    HIPCHK(hipEventRecord(e1, c->stream));
    HIPCHK(hipEventSynchronize(e1));
    float t = 0;
    HIPCHK(hipEventElapsedTime(&t, e0, e1));
    *ms_per_unit = t / reps;
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    return MDZ_OK;
}

/* ------------------------------------------------------------------ */
/* line search of the Newton step as one graph launch                   */
/* ------------------------------------------------------------------ */
#define MDZ_LS_MAX 16

/* iterate = saved iterate + alpha[k] * dx on every node with an equation
 * (StokesRoutines.c:468-485); k_apply_bc then sets the ghost nodes
 * (StokesRoutines.c:491).  k < 0 restores the saved iterate. */
__global__ void k_line_step(DevEqn e, int nu, int nw, int nc, const double *__restrict__ base,
                            const double *__restrict__ dx, const double *__restrict__ alpha, int k, double *u,
                            double *v, double *p) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nu + nw + nc) return;
    const double a = k >= 0 ? alpha[k] : 0.0;
    int eq;
    double *dst;
    if (i < nu) { eq = e.eqn_u[i]; dst = u + i; }
    else if (i < nu + nw) { eq = e.eqn_v[i - nu]; dst = v + (i - nu); }
    else { eq = e.eqn_p[i - nu - nw]; dst = p + (i - nu - nw); }
    *dst = (k >= 0 && eq >= 0) ? base[i] + a * dx[eq] : base[i];
}

/* ghost velocities after a trial step, as ApplyBC sets them
 * (StokesRoutines.c:51-129): type 13 copies the inner neighbour, type 11
 * mirrors it about the wall value, type -12 copies the periodic twin.  The
 * south/north Vx rows and the west/east Vz columns read only nodes that no
 * rule writes; the Vx periodic column copies column 0 after those rows are
 * set, and the corner rules read its pre-copy values, as the reference's
 * sequence does.  So one workgroup runs the two phases with a barrier
 * between them (a few thousand ghost nodes). */
__global__ void __launch_bounds__(1024) k_apply_bc(DevGrid g) {
    const int nx = g.Nx, nz = g.Nz, nzvx = nz + 1, nxvz = nx + 1;
    double *u = g.u_in, *v = g.v_in;
    const int8_t *tu = g.BCu, *tv = g.BCv;
    const double *bu = g.BCu_val, *bv = g.BCv_val;
    for (int t = threadIdx.x; t < nx + nz; t += blockDim.x) {
        if (t < nx) {
            const int s = t, n = t + (nzvx - 1) * nx;
            if (tu[s] == 13) u[s] = u[s + nx];
            else if (tu[s] == 11) u[s] = 2.0 * bu[s] - u[s + nx];
            if (tu[n] == 13) u[n] = u[n - nx];
            else if (tu[n] == 11) u[n] = 2.0 * bu[n] - u[n - nx];
        } else {
            const int j = t - nx, w = j * nxvz, e = j * nxvz + nxvz - 1;
            if (tv[w] == 13) v[w] = v[w + 1];
            else if (tv[w] == 11) v[w] = 2.0 * bv[w] - v[w + 1];
            else if (tv[w] == -12) v[w] = v[e - 1];
            if (tv[e] == 13) v[e] = v[e - 1];
            else if (tv[e] == 11) v[e] = 2.0 * bv[e] - v[e - 1];
            else if (tv[e] == -12) v[e] = v[w + 1];
        }
    }
    __syncthreads();
    for (int j = threadIdx.x; j < nzvx; j += blockDim.x)
        if (tu[j * nx + nx - 1] == -12) u[j * nx + nx - 1] = u[j * nx];
}

/* Device buffers of a line search: the saved iterate (u, v, p), the
 * correction by equation number, the step lengths and six norm sums per
 * trial. */
struct LsBufs {
    const double *base, *dx, *alpha;
    double *res;
};

/* one trial: UpdateNonLinearity (StokesRoutines.c:137-157) then the residual
 * and its norms (EvaluateStokesResidualDecoupled), norms into res[6k..] */
static int enqueue_trial(mdz_ctx *c, const LsBufs &lb, int k, hipStream_t s) {
    const int nu = c->Nx * (c->Nz + 1), nw = (c->Nx + 1) * c->Nz, nc = (c->Nx - 1) * (c->Nz - 1);
    if (k < 0) {
        int rc = snapshot_p(c, s); /* the restore changes p_in under the last trial's rheology */
        if (rc) return rc;
    }
    hipLaunchKernelGGL(k_line_step, dim3(mdz_div_up(nu + nw + nc, 256)), dim3(256), 0, s, c->e, nu, nw, nc,
                       lb.base, lb.dx, lb.alpha, k, c->g.u_in, c->g.v_in, c->g.p_in);
    if (k < 0) return MDZ_OK;
    hipLaunchKernelGGL(k_apply_bc, dim3(1), dim3(1024), 0, s, c->g);
    DevAsm a = make_asm(c);
    mdz_launch_strain_interp5(c->g, c->prm, s);
    int rc = rheology_pass(c, c->prm.rheo_mode == MDZ_RHEO_LEARNED, s, true);
    if (rc) return rc;
    int kind = c->model.aniso == 1 ? 1 : 0;
    const bool fused = fused_dtensor(c);
    if (fused) a = picard_asm(c);
    mdz_launch_rhs_dtensor(c->g, c->prm, fused ? 3 : 0, c->xg, c->zvx, c->xvz, c->zg, c->status, s,
                           fused ? c->dpic_n : nullptr, fused ? c->dpic_s : nullptr);
    return residual_norms(c, kind, a, s, lb.res + 6 * k);
}

extern "C" int mdz_ctx_line_search(mdz_ctx *c, const double *dx, int ntry, const double *alpha, double *res3n) {
    if (!c || !alpha || !res3n || ntry < 1 || ntry > MDZ_LS_MAX)
        return set_err(MDZ_EINVAL, "line search: %d trials (1..%d)", ntry, MDZ_LS_MAX);
    if (!dx && !c->sol_ready) return set_err(MDZ_EINVAL, "line search without a correction (no mdz_ctx_solve)");
    if (!c->pattern_ready[c->model.aniso == 1 ? 1 : 0])
        return set_err(MDZ_EINVAL, "line search before the blocks are assembled");
    g_status = 0;
    const size_t nu = (size_t)c->Nx * (c->Nz + 1), nw = (size_t)(c->Nx + 1) * c->Nz, nc = (size_t)(c->Nx - 1) * (c->Nz - 1);
    const size_t neq = (size_t)c->e.neq_mom + c->e.neq_cont;
    if (!c->ls_base) {
        HIPCHK(hipMalloc((void **)&c->ls_base, (nu + nw + nc) * sizeof(double)));
        HIPCHK(hipMalloc((void **)&c->ls_dx, (neq > 0 ? neq : 1) * sizeof(double)));
        HIPCHK(hipMalloc((void **)&c->ls_alpha, MDZ_LS_MAX * sizeof(double)));
        HIPCHK(hipMalloc((void **)&c->ls_res, 6 * MDZ_LS_MAX * sizeof(double)));
    }
    hipStream_t s = c->stream;
    HIPCHK(hipMemcpyAsync(c->ls_base, c->g.u_in, nu * 8, hipMemcpyDeviceToDevice, s));
    HIPCHK(hipMemcpyAsync(c->ls_base + nu, c->g.v_in, nw * 8, hipMemcpyDeviceToDevice, s));
    HIPCHK(hipMemcpyAsync(c->ls_base + nu + nw, c->g.p_in, nc * 8, hipMemcpyDeviceToDevice, s));
    if (dx) HIPCHK(hipMemcpyAsync(c->ls_dx, dx, neq * 8, hipMemcpyHostToDevice, s));
    else HIPCHK(hipMemcpyAsync(c->ls_dx, c->sol, neq * 8, hipMemcpyDeviceToDevice, s));
    HIPCHK(hipMemcpyAsync(c->ls_alpha, alpha, ntry * sizeof(double), hipMemcpyHostToDevice, s));
    if (!c->ls_exec || c->ls_ntry != ntry || c->ls_version != c->version || c->ls_kernel != g_rheo_kernel) {
        if (c->ls_exec) hipGraphExecDestroy(c->ls_exec);
        if (c->ls_graph) hipGraphDestroy(c->ls_graph);
        c->ls_exec = nullptr;
        c->ls_graph = nullptr;
        HIPCHK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        int rc = MDZ_OK;
        const LsBufs lb{c->ls_base, c->ls_dx, c->ls_alpha, c->ls_res};
        for (int k = 0; k < ntry && !rc; k++) rc = enqueue_trial(c, lb, k, s);
        if (!rc) rc = enqueue_trial(c, lb, -1, s);
        hipGraph_t gr = nullptr;
        hipError_t he = hipStreamEndCapture(s, &gr);
        if (rc) { if (gr) hipGraphDestroy(gr); return rc; }
        if (he != hipSuccess) return set_err(MDZ_EHIP, "line search capture: %s", hipGetErrorString(he));
        c->ls_graph = gr;
        HIPCHK(hipGraphInstantiate(&c->ls_exec, c->ls_graph, nullptr, nullptr, 0));
        c->ls_ntry = ntry;
        c->ls_version = c->version;
        c->ls_kernel = g_rheo_kernel;
        c->ls_stale = c->diag_stale;
        c->ls_snapped = c->p_snapped;
    }
    HIPCHK(hipGraphLaunch(c->ls_exec, s));
    /* the graph leaves the deferred-diagnostics state its capture left */
    c->diag_stale = c->ls_stale;
    c->p_snapped = c->ls_snapped;
    std::vector<double> h(6 * (size_t)ntry);
    HIPCHK(hipMemcpyAsync(h.data(), c->ls_res, h.size() * 8, hipMemcpyDeviceToHost, s));
    int rc = sync(c);
    if (rc) return rc;
    for (int k = 0; k < ntry; k++) {
        int r = norms_to_res(&h[6 * (size_t)k], res3n + 3 * (size_t)k);
        if (r && !rc) rc = r;
    }
    return rc;
}

/* ------------------------------------------------------------------ */
/* the line search without allocation                                    */
/* ------------------------------------------------------------------ */
/* Scratch of mdz_ctx_line_search_noalloc: the saved iterate, the correction,
 * the step lengths and the trial norms (nu + nw + nc + neq + 7 MDZ_LS_MAX
 * doubles; 16 Mi doubles = 128 MiB per GPU, enough for grids of about
 * 2.7 M cells).  Every GPU the library runs on holds its own copy until the
 * process ends.  In host code `scratch` only names the array: its address
 * on a device comes from hipGetSymbolAddress (scratch_on_device). */
#define MDZ_NOALLOC_MAX_DOUBLES ((size_t)16 << 20)
static __device__ __align__(256) double scratch[MDZ_NOALLOC_MAX_DOUBLES];

#define MDZ_MAX_DEVICES 64
static double *g_scratch_ptr[MDZ_MAX_DEVICES];
static std::mutex g_scratch_mu;

/* the current device's address of `scratch`, looked up once per device */
static int scratch_on_device(double **out) {
    int dev = 0;
    HIPCHK(hipGetDevice(&dev));
    if (dev < 0 || dev >= MDZ_MAX_DEVICES) return set_err(MDZ_EINVAL, "device %d", dev);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        double *p = nullptr;
        hipError_t e = hipGetSymbolAddress((void **)&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return set_err(MDZ_EHIP, "address of the line-search scratch on device %d: %s", dev, hipGetErrorString(e));
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return MDZ_OK;
}

extern "C" int mdz_ctx_line_search_noalloc(mdz_ctx *c, const double *dx, int ntry, const double *alpha,
                                           double *res3n) {
    if (!c || !dx || !alpha || !res3n || ntry < 1 || ntry > MDZ_LS_MAX)
        return set_err(MDZ_EINVAL, "line search: %d trials (1..%d)", ntry, MDZ_LS_MAX);
    if (!c->pattern_ready[c->model.aniso == 1 ? 1 : 0])
        return set_err(MDZ_EINVAL, "line search before the blocks are assembled");
    g_status = 0;
    const size_t nu = (size_t)c->Nx * (c->Nz + 1), nw = (size_t)(c->Nx + 1) * c->Nz, nc = (size_t)(c->Nx - 1) * (c->Nz - 1);
    const size_t neq = (size_t)c->e.neq_mom + c->e.neq_cont;
    const size_t need = nu + nw + nc + neq + 7 * (size_t)MDZ_LS_MAX;
    if (need > MDZ_NOALLOC_MAX_DOUBLES)
        return set_err(MDZ_EINVAL, "allocation-free line search: a %d x %d grid needs %zu doubles of scratch, the "
                                   "maximum is %zu (use mdz_ctx_line_search)", c->Nx, c->Nz, need,
                       MDZ_NOALLOC_MAX_DOUBLES);
    double *sp = nullptr;
    int rc = scratch_on_device(&sp);
    if (rc) return rc;
    /* every scratch element a trial reads is written first: nothing to clear */
    double *base = sp, *d_dx = sp + nu + nw + nc, *d_alpha = d_dx + neq, *d_res = d_alpha + MDZ_LS_MAX;
    hipStream_t s = c->stream;
    HIPCHK(hipMemcpyAsync(base, c->g.u_in, nu * 8, hipMemcpyDeviceToDevice, s));
    HIPCHK(hipMemcpyAsync(base + nu, c->g.v_in, nw * 8, hipMemcpyDeviceToDevice, s));
    HIPCHK(hipMemcpyAsync(base + nu + nw, c->g.p_in, nc * 8, hipMemcpyDeviceToDevice, s));
    HIPCHK(hipMemcpyAsync(d_dx, dx, neq * 8, hipMemcpyHostToDevice, s));
    HIPCHK(hipMemcpyAsync(d_alpha, alpha, ntry * sizeof(double), hipMemcpyHostToDevice, s));
    const LsBufs lb{base, d_dx, d_alpha, d_res};
    for (int k = 0; k < ntry && !rc; k++) rc = enqueue_trial(c, lb, k, s);
    if (!rc) rc = enqueue_trial(c, lb, -1, s);
    if (rc) return rc;
    double h[6 * MDZ_LS_MAX];
    HIPCHK(hipMemcpyAsync(h, d_res, 6 * (size_t)ntry * 8, hipMemcpyDeviceToHost, s));
    if ((rc = sync(c))) return rc;
    for (int k = 0; k < ntry; k++) {
        int r = norms_to_res(&h[6 * k], res3n + 3 * (size_t)k);
        if (r && !rc) rc = r;
    }
    return rc;
}

/* ------------------------------------------------------------------ */
/* ensembles: many independent models, one graph launch per Newton      */
/* iteration                                                            */
/* ------------------------------------------------------------------ */
/* ------------------------------------------------------------------ */
/* device solve (KillerSolver)                                          */
/* ------------------------------------------------------------------ */
/* penalty and tolerances: the context's params, the reference's input
 * defaults (InputOutput.c:1063-1069, :1499) where they are 0 */
static void solver_settings(const params &m, SolverInput &in) {
    in.pc_type = m.pc_type;
    in.noisy = m.noisy;
    in.rel_tol_KSP = m.rel_tol_KSP > 0.0 ? m.rel_tol_KSP : 1e-4;
    in.abs_tol_div = m.abs_tol_div > 0.0 ? m.abs_tol_div : 1e-14;
    in.rel_tol_div = m.rel_tol_div > 0.0 ? m.rel_tol_div : 1e-5;
}
static double solver_penalty(const params &m) { return m.penalty > 0.0 ? m.penalty : 1e10; }

static SolverCsr csr_of(const DevBlock &b) { return SolverCsr{b.neq, b.Ic, b.J, b.A}; }

static int pattern_to_host(mdz_ctx *c, const DevBlock &b, std::vector<int> &Ic, std::vector<int> &J) {
    Ic.resize((size_t)b.neq + 1);
    J.resize((size_t)std::max(b.nnz, 1));
    HIPCHK(hipMemcpyAsync(Ic.data(), b.Ic, Ic.size() * sizeof(int), hipMemcpyDeviceToHost, c->stream));
    if (b.nnz > 0) HIPCHK(hipMemcpyAsync(J.data(), b.J, (size_t)b.nnz * sizeof(int), hipMemcpyDeviceToHost, c->stream));
    return MDZ_OK;
}

/* x[i] *= dA[i] (momentum), x[nu + k] *= dD[k] (continuity):
 * ScaleVelocitiesRHSBack, StokesRoutines.c:1348 */
__global__ void k_scale_back(int nu, int np, const double *dA, const double *dD, double *x) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nu) x[i] *= dA[i];
    else if (i < nu + np) x[i] *= dD[i - nu];
}

extern "C" int mdz_ctx_solve(mdz_ctx *c, int nb, double *dx, mdz_solve_info *info) {
    g_status = 0;
    if (!c) return set_err(MDZ_EINVAL, "NULL context");
    if (!c->pattern_ready[0] || !c->pattern_ready[1])
        return set_err(MDZ_EINVAL, "solve before a Newton unit assembled the blocks");
    int rc;
    if ((rc = sync(c))) return rc;
    const int nu = c->e.neq_mom, np = c->e.neq_cont;
    if (nu < 1 || np < 1) return set_err(MDZ_EINVAL, "solve: %d momentum and %d continuity equations", nu, np);
    hipStream_t s = c->stream;
    if (!c->sv && (rc = mdz_solver_create(&c->sv, s))) return rc;
    SolverInput in;
    memset(&in, 0, sizeof(in));
    solver_settings(c->model, in);
    if (in.pc_type != 0 && in.pc_type != 1) return set_err(MDZ_EUNSUPPORTED, "pc_type = %d", in.pc_type);
    const DevBlock &A = c->blk[0], &B = c->blk[1], &Cb = c->blk[2], &D = c->blk[3];
    const DevBlock &AJ = c->blk[4], &BJ = c->blk[5], &CJ = c->blk[6];
    const unsigned gen = c->pattern_gen * 2u + (unsigned)in.pc_type;
    c->sol_ready = 0;
    if (c->sv_gen != gen || c->sv_nb != nb || !c->sol) {
        std::vector<int> mom((size_t)nu), hI[5], hJ[5];
        const DevBlock *src[5] = {&A, &B, &Cb, &AJ, &BJ};
        HIPCHK(hipMemcpyAsync(mom.data(), c->e.mom_node, (size_t)nu * sizeof(int), hipMemcpyDeviceToHost, s));
        for (int q = 0; q < 5; q++)
            if ((rc = pattern_to_host(c, *src[q], hI[q], hJ[q]))) return rc;
        if ((rc = sync(c))) return rc;
        SolverPattern pt[5];
        for (int q = 0; q < 5; q++) pt[q] = SolverPattern{hI[q].data(), hJ[q].data()};
        if ((rc = mdz_solver_order(c->sv, c->Nx, c->Nz, nu, np, mom.data(), pt[0], pt[1], pt[2], pt[3], pt[4],
                                   in.pc_type, nb)))
            return rc;
        hipFree(c->sv_pd); hipFree(c->sol);
        c->sv_pd = c->sol = nullptr;
        HIPCHK(hipMalloc((void **)&c->sv_pd, 3 * (size_t)np * sizeof(double)));
        HIPCHK(hipMalloc((void **)&c->sol, ((size_t)nu + np) * sizeof(double)));
        c->sv_gen = gen;
        c->sv_nb = nb;
    }
    double *Dpen = c->sv_pd, *D1 = Dpen + np, *inc = D1 + np;
    double celvol = c->model.dx * c->model.dz;
    if (!(celvol > 0.0)) celvol = c->g.dx * c->g.dz;
    mdz_solver_pdiag(np, c->e.cont_node, c->g.comp_cells, c->g.bet_n, D.d, solver_penalty(c->model), celvol,
                     c->model.dt, Dpen, D1, inc, s);
    in.nu = nu;
    in.np = np;
    in.A = csr_of(A); in.B = csr_of(B); in.C = csr_of(Cb);
    in.AJ = csr_of(AJ); in.BJ = csr_of(BJ); in.CJ = csr_of(CJ);
    in.Dpen = Dpen; in.D1 = D1; in.incomp = inc;
    in.bu = A.F;
    in.bp = D.F;
    if ((rc = mdz_solver_solve(c->sv, in, c->sol, c->sol + nu, info))) return rc;
    if (c->d_scaled[0])
        hipLaunchKernelGGL(k_scale_back, dim3(mdz_div_up(nu + np, 256)), dim3(256), 0, s, nu, np,
                           (const double *)A.d, (const double *)D.d, c->sol);
    if (dx) HIPCHK(hipMemcpyAsync(dx, c->sol, ((size_t)nu + np) * sizeof(double), hipMemcpyDeviceToHost, s));
    if ((rc = sync(c))) return rc;
    c->sol_ready = 1;
    return MDZ_OK;
}

/* KillerSolver drop-in: the host blocks go to the device for one solve. */
static int killer_solver(SparseMat *mA, SparseMat *mB, SparseMat *mC, SparseMat *mD, const double *rhs_mom,
                         const double *rhs_cont, double *sol, const params &model, const grid *mesh,
                         const SparseMat *Stokes, SparseMat *JA, SparseMat *JB, SparseMat *JC, mdz_solve_info *info) {
    if (!mA || !mB || !mC || !mD || !rhs_mom || !rhs_cont || !sol || !mesh || !Stokes || !JA || !JB || !JC)
        return set_err(MDZ_EINVAL, "KillerSolver: NULL argument");
    const int nu = mA->neq, np = mC->neq, Nx = mesh->Nx, Nz = mesh->Nz;
    if (nu < 1 || np < 1 || mB->neq != nu || JA->neq != nu || JB->neq != nu || JC->neq != np || mD->neq != np)
        return set_err(MDZ_EINVAL, "KillerSolver: block sizes (%d, %d)", nu, np);
    if (!Stokes->eqn_u || !Stokes->eqn_v || !Stokes->eqn_p || !mesh->BCu.type || !mesh->BCv.type || !mesh->BCp.type)
        return set_err(MDZ_EINVAL, "KillerSolver: equation numbering or tags missing");
    /* node of each momentum row, continuity diagonals (Solvers.c:2278-2297) */
    auto has_row = [](int t) { return t != 0 && t != 30 && t != 13 && t != 11 && t != -12; };
    std::vector<int> mom((size_t)nu, -1);
    const long long nun = (long long)Nx * (Nz + 1), nvn = (long long)(Nx + 1) * Nz;
    for (long long kk = 0; kk < nun; kk++) {
        const int eq = Stokes->eqn_u[kk];
        if (has_row(mesh->BCu.type[kk]) && eq >= 0 && eq < nu) mom[eq] = (int)kk;
    }
    for (long long kk = 0; kk < nvn; kk++) {
        const int eq = Stokes->eqn_v[kk];
        if (has_row(mesh->BCv.type[kk]) && eq >= 0 && eq < nu) mom[eq] = (int)(nun + kk);
    }
    for (int i = 0; i < nu; i++)
        if (mom[i] < 0) return set_err(MDZ_EINVAL, "KillerSolver: momentum equation %d has no node", i);
    const double celvol = model.dx * model.dz, penalty = solver_penalty(model) / celvol;
    std::vector<double> pd(3 * (size_t)np, 0.0);
    double *Dpen = pd.data(), *D1 = Dpen + np, *inc = D1 + np;
    for (int k = 0; k < np; k++) { Dpen[k] = 1.0; D1[k] = 1.0; inc[k] = 1.0; }
    const long long nc = (long long)(Nx - 1) * (Nz - 1);
    for (long long kk = 0; kk < nc; kk++) {
        if (mesh->BCp.type[kk] == 30 || mesh->BCp.type[kk] == 31) continue;
        const int i = Stokes->eqn_p[kk] - nu;
        if (i < 0 || i >= np) return set_err(MDZ_EINVAL, "KillerSolver: pressure equation of cell %lld", kk);
        const int comp = mesh->comp_cells ? mesh->comp_cells[kk] : 0;
        if (comp == 1 && model.VolChangeReac == 1) return set_err(MDZ_EUNSUPPORTED, "VolChangeReac = 1");
        if (comp == 0) { D1[i] = 0.0; Dpen[i] = penalty; }
        if (comp == 1) {
            const double d = mD->d ? mD->d[i] : 1.0;
            D1[i] = mesh->bet_n[kk] / model.dt * celvol * d * d;
            Dpen[i] = 1.0 / D1[i];
            inc[i] = 0.0;
        }
    }
    SolverInput in;
    memset(&in, 0, sizeof(in));
    solver_settings(model, in);
    in.noisy = 1; /* KillerSolver prints its iterations whatever model.noisy (Solvers.c:2232) */
    if (in.pc_type != 0 && in.pc_type != 1) return set_err(MDZ_EUNSUPPORTED, "pc_type = %d", in.pc_type);
    SparseMat *blocks[6] = {mA, mB, mC, JA, JB, JC};
    const int ncols[6] = {nu, np, nu, nu, np, nu};
    size_t bytes = 0;
    for (int q = 0; q < 6; q++) {
        const SparseMat *b = blocks[q];
        if (!b->Ic || (b->nnz > 0 && (!b->J || !b->A))) return set_err(MDZ_EINVAL, "KillerSolver: empty block");
        if (b->Ic[0] != 0 || b->Ic[b->neq] != b->nnz) return set_err(MDZ_EINVAL, "KillerSolver: row pointers of block %d", q);
        for (int r = 0; r < b->neq; r++)
            if (b->Ic[r + 1] < b->Ic[r]) return set_err(MDZ_EINVAL, "KillerSolver: row pointers of block %d", q);
        for (int e = 0; e < b->nnz; e++)
            if (b->J[e] < 0 || b->J[e] >= ncols[q]) return set_err(MDZ_EINVAL, "KillerSolver: column of block %d", q);
        bytes += align256(((size_t)b->neq + 1) * 4) + align256((size_t)b->nnz * 4) + align256((size_t)b->nnz * 8);
    }
    bytes += align256(pd.size() * 8) + align256((size_t)nu * 8) + align256((size_t)np * 8) +
             align256(((size_t)nu + np) * 8);
    hipStream_t s;
    HIPCHK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    char *slab = nullptr;
    MdzSolver *sv = nullptr;
    int rc = MDZ_OK;
    do {
        if (hipMalloc((void **)&slab, bytes) != hipSuccess) { rc = set_err(MDZ_ENOMEM, "KillerSolver: %zu bytes", bytes); break; }
        char *p = slab;
        auto take = [&](size_t n) { char *q = p; p += align256(n); return q; };
        SolverCsr csr[6];
        for (int q = 0; q < 6 && !rc; q++) {
            SparseMat *b = blocks[q];
            int *Ic = (int *)take(((size_t)b->neq + 1) * 4), *J = (int *)take((size_t)b->nnz * 4);
            double *A = (double *)take((size_t)b->nnz * 8);
            if (hipMemcpyAsync(Ic, b->Ic, ((size_t)b->neq + 1) * 4, hipMemcpyHostToDevice, s) != hipSuccess ||
                (b->nnz > 0 && (hipMemcpyAsync(J, b->J, (size_t)b->nnz * 4, hipMemcpyHostToDevice, s) != hipSuccess ||
                                hipMemcpyAsync(A, b->A, (size_t)b->nnz * 8, hipMemcpyHostToDevice, s) != hipSuccess)))
                rc = set_err(MDZ_EHIP, "KillerSolver: upload");
            csr[q] = SolverCsr{b->neq, Ic, J, A};
        }
        if (rc) break;
        double *dpd = (double *)take(pd.size() * 8), *bu = (double *)take((size_t)nu * 8), *bp = (double *)take((size_t)np * 8);
        double *x = (double *)take(((size_t)nu + np) * 8);
        if (hipMemcpyAsync(dpd, pd.data(), pd.size() * 8, hipMemcpyHostToDevice, s) != hipSuccess ||
            hipMemcpyAsync(bu, rhs_mom, (size_t)nu * 8, hipMemcpyHostToDevice, s) != hipSuccess ||
            hipMemcpyAsync(bp, rhs_cont, (size_t)np * 8, hipMemcpyHostToDevice, s) != hipSuccess) {
            rc = set_err(MDZ_EHIP, "KillerSolver: upload");
            break;
        }
        if ((rc = mdz_solver_create(&sv, s))) break;
        if ((rc = mdz_solver_order(sv, Nx, Nz, nu, np, mom.data(), SolverPattern{mA->Ic, mA->J},
                                   SolverPattern{mB->Ic, mB->J}, SolverPattern{mC->Ic, mC->J},
                                   SolverPattern{JA->Ic, JA->J}, SolverPattern{JB->Ic, JB->J}, in.pc_type, 0)))
            break;
        in.nu = nu; in.np = np;
        in.A = csr[0]; in.B = csr[1]; in.C = csr[2]; in.AJ = csr[3]; in.BJ = csr[4]; in.CJ = csr[5];
        in.Dpen = dpd; in.D1 = dpd + np; in.incomp = dpd + 2 * (size_t)np;
        in.bu = bu; in.bp = bp;
        const int rs = mdz_solver_solve(sv, in, x, x + nu, info);
        if (rs && rs != MDZ_ESOLVE) { rc = rs; break; }
        if (hipMemcpyAsync(sol, x, ((size_t)nu + np) * 8, hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess) {
            rc = set_err(MDZ_EHIP, "KillerSolver: download");
            break;
        }
        rc = rs;
    } while (0);
    mdz_solver_destroy(sv);
    hipStreamSynchronize(s);
    hipFree(slab);
    hipStreamDestroy(s);
    return rc;
}

extern "C" void KillerSolver(SparseMat *matA, SparseMat *matB, SparseMat *matC, SparseMat *matD, DirectSolver *pardi,
                             double *rhs_mom, double *rhs_cont, double *sol, params model, grid *mesh, scale scaling,
                             SparseMat *Stokes, SparseMat *Jacobian, SparseMat *JmatA, SparseMat *JmatB,
                             SparseMat *JmatC) {
    (void)pardi; (void)scaling; (void)Jacobian;
    g_status = 0;
    mdz_solve_info info;
    memset(&info, 0, sizeof(info));
    const int rc = killer_solver(matA, matB, matC, matD, rhs_mom, rhs_cont, sol, model, mesh, Stokes, JmatA, JmatB,
                                 JmatC, &info);
    if (rc == MDZ_ESOLVE) {
        char msg[600];
        snprintf(msg, sizeof(msg), "%s\n", g_err);
        dropin_fail(MDZ_ESOLVE, 1, msg);
        return;
    }
    dropin_check(rc);
}

extern "C" int mdz_ctx_set_launch_shape(mdz_ctx *c, int rheo, int pic, int jac) {
    if (!c) return set_err(MDZ_EINVAL, "NULL context");
    LaunchShape sh{rheo, pic, jac, true};
    if (!mdz_shape_valid(sh))
        return set_err(MDZ_EINVAL, "launch shape (%d, %d, %d): rheology 64/128/256, Picard 0/64/128/256, Jacobian 0/64/128",
                       rheo, pic, jac);
    c->shape = sh;
    c->version++;
    return MDZ_OK;
}

extern "C" int mdz_ctx_get_launch_shape(mdz_ctx *c, int *shape3) {
    if (!c || !shape3) return set_err(MDZ_EINVAL, "NULL argument");
    shape3[0] = c->shape.rheo;
    shape3[1] = c->shape.pic;
    shape3[2] = c->shape.jac;
    return MDZ_OK;
}

#define MDZ_MAX_BRANCHES 8

struct mdz_ensemble {
    int n;
    std::vector<mdz_ctx *> ctx;
    int branches;                 /* concurrent chains of the captured graph */
    hipStream_t st[MDZ_MAX_BRANCHES];
    hipEvent_t fork, join[MDZ_MAX_BRANCHES];
    hipGraph_t graph;
    hipGraphExec_t exec;
    std::vector<unsigned> captured_version;
    int captured_kernel;          /* rheology kernel selection at capture */
    double **d_src;               /* per model: its norm_out */
    double *d_res;                /* gathered norm sums, 6 per model */
    std::vector<int> branch_of;   /* model -> chain */
};

/* norm sums of every model into one array (one copy to the host after the graph) */
__global__ void k_gather_norms(const double *const *__restrict__ src, double *__restrict__ dst, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < 6 * n) dst[i] = src[i / 6][i % 6];
}

static size_t ctx_cells(const mdz_ctx *c) { return (size_t)(c->Nx - 1) * (c->Nz - 1); }

/* Chains balanced by cell count: largest model first onto the least loaded
 * chain (longest-processing-time rule). */
static void assign_branches(mdz_ensemble *e) {
    std::vector<int> order(e->n);
    for (int i = 0; i < e->n; i++) order[i] = i;
    std::sort(order.begin(), order.end(), [e](int a, int b) {
        size_t ca = ctx_cells(e->ctx[a]), cb = ctx_cells(e->ctx[b]);
        return ca != cb ? ca > cb : a < b;
    });
    std::vector<double> load(e->branches, 0.0);
    e->branch_of.assign(e->n, 0);
    for (int m : order) {
        int best = 0;
        for (int b = 1; b < e->branches; b++)
            if (load[b] < load[best]) best = b;
        e->branch_of[m] = best;
        load[best] += (double)ctx_cells(e->ctx[m]);
    }
}

static void drop_graph(mdz_ensemble *e) {
    if (e->exec) hipGraphExecDestroy(e->exec);
    if (e->graph) hipGraphDestroy(e->graph);
    e->exec = nullptr;
    e->graph = nullptr;
}

/* Captures one Newton unit of every model: a fork into `branches` chains,
 * the units of each chain in order of decreasing size, a join, and the
 * gather of the norm sums.  Nothing captured allocates, clears memory with
 * a memset node or synchronises with the host. */
static int capture(mdz_ensemble *e) {
    drop_graph(e);
    assign_branches(e);
    hipStream_t s0 = e->st[0];
    HIPCHK(hipStreamBeginCapture(s0, hipStreamCaptureModeThreadLocal));
    int rc = MDZ_OK;
    hipError_t he = hipEventRecord(e->fork, s0);
    for (int b = 1; b < e->branches && he == hipSuccess; b++) he = hipStreamWaitEvent(e->st[b], e->fork, 0);
    std::vector<int> order(e->n);
    for (int i = 0; i < e->n; i++) order[i] = i;
    std::stable_sort(order.begin(), order.end(),
                     [e](int a, int b) { return ctx_cells(e->ctx[a]) > ctx_cells(e->ctx[b]); });
    for (int k = 0; k < e->n && he == hipSuccess && rc == MDZ_OK; k++) {
        int m = order[k];
        rc = enqueue_unit(e->ctx[m], e->st[e->branch_of[m]]);
    }
    for (int b = 1; b < e->branches && he == hipSuccess; b++) {
        he = hipEventRecord(e->join[b], e->st[b]);
        if (he == hipSuccess) he = hipStreamWaitEvent(s0, e->join[b], 0);
    }
    if (he == hipSuccess)
        hipLaunchKernelGGL(k_gather_norms, dim3(mdz_div_up(6 * e->n, 256)), dim3(256), 0, s0,
                           (const double *const *)e->d_src, e->d_res, e->n);
    hipGraph_t gr = nullptr;
    hipError_t he2 = hipStreamEndCapture(s0, &gr);
    if (rc) { if (gr) hipGraphDestroy(gr); return rc; }
    if (he != hipSuccess) { if (gr) hipGraphDestroy(gr); return set_err(MDZ_EHIP, "ensemble capture: %s", hipGetErrorString(he)); }
    if (he2 != hipSuccess) return set_err(MDZ_EHIP, "hipStreamEndCapture: %s", hipGetErrorString(he2));
    e->graph = gr;
    HIPCHK(hipGraphInstantiate(&e->exec, e->graph, nullptr, nullptr, 0));
    e->captured_version.resize(e->n);
    for (int i = 0; i < e->n; i++) e->captured_version[i] = e->ctx[i]->version;
    e->captured_kernel = g_rheo_kernel;
    return MDZ_OK;
}

static bool graph_current(const mdz_ensemble *e) {
    if (!e->exec || e->captured_kernel != g_rheo_kernel) return false;
    for (int i = 0; i < e->n; i++)
        if (e->captured_version[i] != e->ctx[i]->version) return false;
    return true;
}

extern "C" void mdz_ensemble_destroy(mdz_ensemble *e) {
    if (!e) return;
    if (e->st[0]) hipStreamSynchronize(e->st[0]);
    drop_graph(e);
    for (int b = 0; b < MDZ_MAX_BRANCHES; b++) {
        if (e->st[b]) hipStreamDestroy(e->st[b]);
        if (e->join[b]) hipEventDestroy(e->join[b]);
    }
    if (e->fork) hipEventDestroy(e->fork);
    hipFree(e->d_src);
    hipFree(e->d_res);
    delete e;
}

extern "C" int mdz_ensemble_create(mdz_ensemble **out, mdz_ctx *const *ctx, int n) {
    g_status = 0;
    if (!out || !ctx || n < 1) return set_err(MDZ_EINVAL, "ensemble of %d contexts", n);
    for (int i = 0; i < n; i++) {
        if (!ctx[i]) return set_err(MDZ_EINVAL, "ensemble: context %d is NULL", i);
        for (int j = 0; j < i; j++)
            if (ctx[j] == ctx[i]) return set_err(MDZ_EINVAL, "ensemble: context %d repeats context %d", i, j);
    }
    mdz_ensemble *e = new mdz_ensemble();
    e->n = n;
    e->ctx.assign(ctx, ctx + n);
    e->branches = 4;
    int rc = MDZ_OK;
    for (int b = 0; b < MDZ_MAX_BRANCHES && !rc; b++) {
        if (hipStreamCreate(&e->st[b]) != hipSuccess || hipEventCreateWithFlags(&e->join[b], hipEventDisableTiming) != hipSuccess)
            rc = set_err(MDZ_EHIP, "ensemble streams");
    }
    if (!rc && hipEventCreateWithFlags(&e->fork, hipEventDisableTiming) != hipSuccess) rc = set_err(MDZ_EHIP, "ensemble event");
    if (!rc && (hipMalloc((void **)&e->d_src, n * sizeof(double *)) != hipSuccess ||
                hipMalloc((void **)&e->d_res, 6 * (size_t)n * sizeof(double)) != hipSuccess))
        rc = set_err(MDZ_ENOMEM, "ensemble buffers");
    if (!rc) {
        std::vector<double *> src(n);
        for (int i = 0; i < n; i++) {
            src[i] = ctx[i]->norm_out;
            if (hipStreamSynchronize(ctx[i]->stream) != hipSuccess) rc = set_err(MDZ_EHIP, "context %d stream", i);
        }
        if (!rc && hipMemcpy(e->d_src, src.data(), n * sizeof(double *), hipMemcpyHostToDevice) != hipSuccess)
            rc = set_err(MDZ_EHIP, "ensemble pointer table");
    }
    if (rc) { mdz_ensemble_destroy(e); return rc; }
    *out = e;
    return MDZ_OK;
}

extern "C" int mdz_ensemble_set_branches(mdz_ensemble *e, int branches) {
    if (!e || branches < 1 || branches > MDZ_MAX_BRANCHES)
        return set_err(MDZ_EINVAL, "ensemble branches %d (1..%d)", branches, MDZ_MAX_BRANCHES);
    if (e->branches != branches) {
        e->branches = branches;
        drop_graph(e);
    }
    return MDZ_OK;
}

extern "C" int mdz_ensemble_launch(mdz_ensemble *e) {
    if (!e) return set_err(MDZ_EINVAL, "NULL ensemble");
    g_status = 0;
    if (!graph_current(e)) {
        int rc = capture(e);
        if (rc) return rc;
    }
    HIPCHK(hipGraphLaunch(e->exec, e->st[0]));
    /* each unit's rheology pass leaves the deferred-diagnostics state of a
     * fresh pass (as the capture left it) */
    for (mdz_ctx *c : e->ctx) {
        c->p_snapped = 0;
        c->diag_stale = c->defer_diag && g_rheo_kernel == 0 && mdz_rheo_fast_eligible(c->prm, &c->materials);
    }
    return MDZ_OK;
}

extern "C" int mdz_ensemble_synchronize(mdz_ensemble *e) {
    if (!e) return set_err(MDZ_EINVAL, "NULL ensemble");
    HIPCHK(hipStreamSynchronize(e->st[0]));
    HIPCHK(hipGetLastError());
    return MDZ_OK;
}

extern "C" int mdz_ensemble_residuals(mdz_ensemble *e, double *res) {
    if (!e || !res) return set_err(MDZ_EINVAL, "NULL argument");
    std::vector<double> h(6 * (size_t)e->n);
    HIPCHK(hipMemcpyAsync(h.data(), e->d_res, h.size() * sizeof(double), hipMemcpyDeviceToHost, e->st[0]));
    HIPCHK(hipStreamSynchronize(e->st[0]));
    int rc = MDZ_OK;
    for (int i = 0; i < e->n; i++) {
        int r = norms_to_res(&h[6 * (size_t)i], res + 3 * (size_t)i);
        if (r && !rc) rc = set_err(MDZ_ENAN, "NaN residual in model %d", i);
    }
    return rc;
}

extern "C" int mdz_ensemble_time(mdz_ensemble *e, int reps, double *ms_per_launch) {
    if (!e || reps < 1 || !ms_per_launch) return set_err(MDZ_EINVAL, "ensemble time");
    int rc = mdz_ensemble_launch(e); /* captures if needed; warm-up */
    if (rc) return rc;
    hipEvent_t e0, e1;
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    HIPCHK(hipEventRecord(e0, e->st[0]));
    for (int r = 0; r < reps && !rc; r++) rc = mdz_ensemble_launch(e);
    HIPCHK(hipEventRecord(e1, e->st[0]));
    HIPCHK(hipEventSynchronize(e1));
    float t = 0;
    HIPCHK(hipEventElapsedTime(&t, e0, e1));
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    if (rc) return rc;
    *ms_per_launch = t / reps;
    return MDZ_OK;
}

/* ---- autotuner ---- */
/* Mean milliseconds of one tunable stage of context c on stream s, over
 * `reps` launches after one untimed launch: 0 = rheology (interpolation,
 * guess and local iterations), 1 = Picard values, 2 = Jacobian values (the
 * D tensor of its kind is put in place first; after the Jacobian values the
 * J = 0 tensor of the residual is restored, or, for a fused model, the
 * J = 1 tensor is recorded as present, as after a unit). */
static int time_stage(mdz_ctx *c, int stage, hipStream_t s, int reps, hipEvent_t e0, hipEvent_t e1, float *ms) {
    DevAsm a = make_asm(c), ap = picard_asm(c);
    const bool fused = fused_dtensor(c);
    if (stage == 1 && fused) mdz_launch_dtensor(c->g, c->prm, 3, c->status, s, c->dpic_n, c->dpic_s);
    if (stage == 2) mdz_launch_dtensor(c->g, c->prm, 1, c->status, s);
    float t = 0;
    for (int r = 0; r <= reps; r++) {
        if (r == 1) HIPCHK(hipEventRecord(e0, s));
        if (stage == 0) {
            int rc = rheology_pass(c, c->prm.rheo_mode == MDZ_RHEO_LEARNED, s);
            if (rc) return rc;
        } else if (stage == 1) {
            mdz_launch_values(0, ap, &c->blk[0], &c->blk[1], &c->blk[2], &c->blk[3], c->shape.pic, s);
        } else {
            mdz_launch_values(1, a, &c->blk[4], &c->blk[5], &c->blk[6], &c->blk[7], c->shape.jac, s);
        }
    }
    HIPCHK(hipEventRecord(e1, s));
    HIPCHK(hipEventSynchronize(e1));
    HIPCHK(hipEventElapsedTime(&t, e0, e1));
    if (stage == 2) {
        if (fused) c->d_jac = 1;
        else mdz_launch_dtensor(c->g, c->prm, 0, c->status, s);
    }
    HIPCHK(hipGetLastError());
    *ms = t / reps;
    return MDZ_OK;
}

/* Picks, for every size class of the ensemble (models whose cell counts
 * share a power of two), the block shape of each tunable stage by timing
 * the candidates on the largest model of the class, applies it to the
 * class, then picks the number of graph chains (1, 2, 4, 8) by timing the
 * captured ensemble.  report (optional, n * 3 ints) receives the chosen
 * shape of each model; *branches (optional) the chosen chain count. */
extern "C" int mdz_ensemble_autotune(mdz_ensemble *e, int reps, int *report, int *branches) {
    if (!e || reps < 1) return set_err(MDZ_EINVAL, "autotune");
    g_status = 0;
    hipStream_t s = e->st[0];
    hipEvent_t e0, e1;
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    static const int cand_rheo[] = {64, 128, 256}, cand_pic[] = {0, 64, 128, 256}, cand_jac[] = {0, 64, 128};
    const int *cand[3] = {cand_rheo, cand_pic, cand_jac};
    const int ncand[3] = {3, 4, 3};
    int rc = MDZ_OK;
    std::vector<int> done(e->n, 0);
    for (int i = 0; i < e->n && !rc; i++) {
        if (done[i]) continue;
        int cls = 0;
        for (size_t v = ctx_cells(e->ctx[i]); v > 1; v >>= 1) cls++;
        int rep = i;
        std::vector<int> members;
        for (int j = i; j < e->n; j++) {
            int cj = 0;
            for (size_t v = ctx_cells(e->ctx[j]); v > 1; v >>= 1) cj++;
            if (cj != cls || done[j]) continue;
            members.push_back(j);
            if (ctx_cells(e->ctx[j]) > ctx_cells(e->ctx[rep])) rep = j;
        }
        mdz_ctx *c = e->ctx[rep];
        LaunchShape best = c->shape;
        best.asked = false;
        for (int stage = 0; stage < 3 && !rc; stage++) {
            /* two rounds over the candidates, the second in reverse order,
             * and each candidate's faster round: a candidate timed while the
             * clocks still ramp up, or next to a slow neighbour, is not
             * picked or dropped on that alone */
            float tmin[4] = {1e30f, 1e30f, 1e30f, 1e30f};
            for (int round = 0; round < 2 && !rc; round++) {
                for (int q = 0; q < ncand[stage] && !rc; q++) {
                    const int k = round == 0 ? q : ncand[stage] - 1 - q;
                    LaunchShape sh = best;
                    (stage == 0 ? sh.rheo : stage == 1 ? sh.pic : sh.jac) = cand[stage][k];
                    c->shape = sh;
                    float t = 0;
                    rc = time_stage(c, stage, s, reps, e0, e1, &t);
                    if (!rc && t < tmin[k]) tmin[k] = t;
                }
            }
            int kbest = 0;
            for (int k = 1; k < ncand[stage]; k++)
                if (tmin[k] < tmin[kbest]) kbest = k;
            (stage == 0 ? best.rheo : stage == 1 ? best.pic : best.jac) = cand[stage][kbest];
        }
        for (int j : members) {
            e->ctx[j]->shape = best;
            e->ctx[j]->version++;
            done[j] = 1;
        }
    }
    int bbest = e->branches;
    if (!rc) {
        double tb = 1e30;
        for (int b = 1; b <= MDZ_MAX_BRANCHES && !rc; b *= 2) {
            if ((rc = mdz_ensemble_set_branches(e, b))) break;
            double t = 0;
            rc = mdz_ensemble_time(e, reps, &t);
            if (!rc && t < tb) { tb = t; bbest = b; }
        }
    }
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    if (rc) return rc;
    if ((rc = mdz_ensemble_set_branches(e, bbest))) return rc;
    if (report)
        for (int i = 0; i < e->n; i++) {
            report[3 * i] = e->ctx[i]->shape.rheo;
            report[3 * i + 1] = e->ctx[i]->shape.pic;
            report[3 * i + 2] = e->ctx[i]->shape.jac;
        }
    if (branches) *branches = bbest;
    return MDZ_OK;
}
