/*
 * mdoodz_hot.h -- C ABI of the MI355X (gfx950) implementation of the MDOODZ 6.0
 * per-Newton-iteration grid path: rheology, Stokes residual, decoupled
 * Picard/Jacobian CSR assembly.
 *
 * Two layers are declared here:
 *
 *  1. Drop-in entry points with the reference's own names and prototypes
 *     (SOURCE/header_MDOODZ.h).  A host driver that links libmdz_hot.so in
 *     place of RheologyDensity.o / StokesAssemblyDecoupled.o / the hot part
 *     of StokesRoutines.o gets GPU execution with host-resident structs:
 *     every call uploads the fields it reads and downloads the fields it
 *     writes.  CSR blocks are returned in malloc() buffers that the caller
 *     releases with free(), exactly as SOURCE/MemoryAllocFree.c:113 FreeMat.
 *
 *  2. A device-resident interface (mdz_*): the grid lives in HBM between
 *     calls, the CSR sparsity pattern is built once per boundary-condition
 *     set and only values are rewritten per Newton iteration.
 *
 * The struct layouts below are the reference's (field order and types are
 * the ABI and must not change); they follow SOURCE/header_MDOODZ.h:25-219.
 */
#ifndef MDOODZ_HOT_H
#define MDOODZ_HOT_H

#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

#define DoodzFP double

/* ---------------------------------------------------------------------- */
/* Reference data model (ABI).  SOURCE/header_MDOODZ.h:25-219              */
/* ---------------------------------------------------------------------- */

/* header_MDOODZ.h:25 */
typedef struct _scale scale;
struct _scale {
    double eta, L, V, T, t, a, E, S, m, rho, F, J, W, Cv, rhoE, k;
};

/* header_MDOODZ.h:31 -- only passed through by UpdateNonLinearity */
typedef struct _surface surface;
/* header_MDOODZ.h:66-78 -- the markers (particles); the marker-to-grid
 * drop-ins read x, z, phase and the interpolated property arrays */
typedef struct _p_markers markers;
struct _p_markers {
    int      Nx_part, Nz_part, Nb_part, Nb_part_max, min_part_cell, Nb_part_ini;
    DoodzFP *x, *z, *Vx, *Vz, *P, *sxxd, *szzd, *sxz, *progress, *rho, *T, *d, *phi, *X, *syy, *dsyy;
    DoodzFP *strain, *strain_el, *strain_pl, *strain_pwl, *strain_exp, *strain_lin, *strain_gbs;
    int     *phase, *generation;
    markers *marker_chain;
    int     *intag;
    double  *Fxx, *Fxz, *Fzx, *Fzz, *dnx, *dnz, *nx, *nz;
    double  *T0, *P0, *x0, *z0, *Tmax, *Pmax, *divth;
    double  *dsxxd, *dszzd, *dsxz;
};

/* header_MDOODZ.h:46 */
typedef struct _mat_prop mat_prop;
struct _mat_prop {
    int     Nb_phases;
    DoodzFP R;
    DoodzFP eta0[20], rho[20], mu[20], Cv[20], k[20], Qr[20], C[20], phi[20], psi[20], Slim[20],
            n[20], A[20], Ea[20], Va[20], alp[20], bet[20], Qm[20], T0[20], P0[20], drho[20], k_eff[20];
    DoodzFP tpwl[20], Qpwl[20], Vpwl[20], npwl[20], mpwl[20], Apwl[20], apwl[20], fpwl[20], rpwl[20],
            Fpwl[20], pref_pwl[20];
    DoodzFP texp[20], Qexp[20], Vexp[20], Sexp[20], Eexp[20], Gexp[20], aexp[20], fexp[20], rexp[20],
            qexp[20], nexp[20];
    DoodzFP tlin[20], Qlin[20], Vlin[20], nlin[20], mlin[20], Alin[20], alin[20], flin[20], rlin[20],
            Flin[20];
    DoodzFP tgbs[20], Qgbs[20], Vgbs[20], ngbs[20], mgbs[20], Agbs[20], agbs[20], fgbs[20], rgbs[20],
            Fgbs[20];
    DoodzFP ppzm[20], Kpzm[20], Qpzm[20], Vpzm[20], Gpzm[20], cpzm[20], Lpzm[20], gs_ref[20];
    int     gs[20], cstv[20], pwlv[20], linv[20], expv[20], gbsv[20], phase_diagram[20], density_model[20];
    DoodzFP C_end[20], phi_end[20], psi_end[20], pls_start[20], pls_end[20], eta_vp[20], n_vp[20];
    int     phi_soft[20], psi_soft[20], coh_soft[20], is_tensile[20];
    DoodzFP Pr[20], tau_kin[20], dPr[20], k_chem[20];
    int     reac_soft[20], reac_phase[20];
    int     phase_mix[20], phase_two[20];
    double  aniso_factor[20], aniso_angle[20];
};

/* header_MDOODZ.h:81 -- mechanical boundary tags and values */
typedef struct _BC BC;
struct _BC {
    char   *type;
    double *val;
};

/* header_MDOODZ.h:88 -- thermal-style boundary record (BCg is one) */
typedef struct _BCT BCT;
struct _BCT {
    char   *type, *typW, *typE, *typS, *typN;
    double *val, *valW, *valE, *valS, *valN;
};

/* header_MDOODZ.h:95 -- one CSR block plus its vectors */
typedef struct _SparseMat SparseMat;
struct _SparseMat {
    double *A, *x, *b, *F, *d, *bbc;
    int    *Ic, *J, neq;
    int    *eqn_u, *eqn_v, *eqn_p;
    int     nnz, neq_mom, neq_cont;
};

/* header_MDOODZ.h:104 */
typedef struct _params params;
struct _params {
    double xmin, zmin, xmax, zmax, time, dx, dz, dt, dt0, dt_start, dt_max, L0, dt_min;
    double xmin0, zmin0, xmax0, zmax0;
    double gx, gz;
    int    Nx, Nz, Nt, step, nit, Newton, noisy;
    int    eta_avg, itp_stencil;
    double nexp_radial_basis;
    int    ismechanical, isperiodic_x, isinertial, iselastic, isnonnewtonian, isthermal, ispureshear_ale,
           free_surf, eqn_state, write_markers, write_debug, write_energies, no_markers;
    double free_surf_stab;
    int    dt_constant, RK, line_search, thermal_eq, subgrid_diff, adiab_heat, shear_heat, advection,
           fstrain, ConservInterp;
    int    surf_processes, cpc, surf_remesh, loc_iter, therm_pert, surf_ised1, surf_ised2, MantleID,
           topografix, Reseed, SmoothSoftening;
    double EpsBG, user0, user1, user2, user3, user4, user5, user6, user7, user8;
    char  *input_file;
    int    Nb_phases;
    int    ncont;
    double Courant, mineta, maxeta;
    int    initial_noise, initial_part;
    int    decoupled_solve, lsolver, diag_scaling, pc_type;
    double penalty, abs_tol_div, rel_tol_div, auto_penalty, compressible, rel_tol_KSP;
    double line_search_min, safe_dt_div;
    int    safe_mode, nstagmax;
    int    nT, nE, nd, def_maps;
    double Pn, Tmin, Tmax, Emin, Emax, dmin, dmax, PrBG;
    double surf_diff, surf_sedirate, surf_baselev, surf_Winc, surf_Vinc;
    double therm_pert_x0, therm_pert_z0, therm_pert_dT, therm_pert_rad, cooling_time;
    int    force_act_vol_ast;
    double act_vol_dis_ast, act_vol_dif_ast;
    int    isPD, num_PD, *PDMnT, *PDMnP;
    double **PDMrho, *PDMTmin, *PDMTmax, *PDMPmin, *PDMPmax;
    int    rec_T_P_x_z, delete_breakpoints, GNUplot_residuals;
    int    BC_setup_type, shear_style, polar;
    int    StressRotation, StressUpdate, DirectNeighbour;
    int    diffuse_X, diffuse_avg;
    double diffusion_length;
    int    ProgReac, NoReturn, VolChangeReac, Plith_trick, UnsplitDiffReac;
    int    aniso, aniso_fstrain;
};

/* header_MDOODZ.h:157 */
typedef struct _n_params Nparams;
struct _n_params {
    int    nit, nit_max, stagnated;
    double abs_tol_u, rel_tol_u, abs_tol_p, rel_tol_p;
    double resx, resz, resp, rest;
    double resx0, resz0, resp0;
    double resx_f, resz_f, resp_f;
    double vrlx, prlx, trlx;
    int    Picard2Newton, let_res_grow, nit_Pic_max;
    double Pic2NewtCond;
};

/* header_MDOODZ.h:170 -- every array is a separate host allocation; index
 * k + l*row_length, row-major in x.  Centroids (Nx-1)(Nz-1), vertices Nx*Nz,
 * Vx nodes Nx(Nz+1), Vz nodes (Nx+1)Nz. */
typedef struct _grid grid;
struct _grid {
    int    Nx, Nz, NN, NC;
    double dx, dz;
    double *roger_x, *roger_z, *div_u, *div_u_s, *div_u_el, *div_u_pl, *div_u_r, *u_in, *v_in, *p_in,
           *p_corr, *sxxd, *szzd, *sxz, *exxd, *ezzd, *exz, *VE_s, *VE_n, *sxxd0, *szzd0, *sxz0, *mu_s,
           *mu_n, *u_adv, *v_adv, *eta_phys_n, *kx, *kz, *Cv, *Qr, *eta_phys_s, *u_start, *v_start,
           *p_start, *divth0_n, *T0_n;
    int    *iter_smooth;
    int    *nb_part_cell, *nb_part_vert;
    BC      BCu, BCv, BCp, BCp_exp;
    BCT     BCt, BCg, BCc;
    double *xg_coord, *zg_coord, *xc_coord, *zc_coord, *xvz_coord, *zvx_coord, *xg_coord0, *zg_coord0,
           *xg_coord_ext, *zg_coord_ext;
    double *eta_s, *eta_n, *rho_s, *rho_n;
    double *X_s, *X_n, *X0_s, *X0_n, *p0_n, *p0_s;
    double *OverS_n, *OverS_s;
    double *strain_n, *strain_s;
    double *u, *v, *p;
    double *ru, *rv, *rp;
    double *rhs_u, *rhs_v, *rhs_p, *rhs_t, *gx, *gz;
    double  p_scale;
    double *alp, *bet_n, *bet_s, *p_lith, *p_lith0, *dp, *Qrho;
    double *VxVz, *VzVx;
    int    *P2N, *P2C;
    int    *kvx, *lvx, *kvz, *lvz, *kp, *lp, *kn, *ln;
    double **phase_perc_n, **phase_perc_s;
    double *sxxd0_s, *szzd0_s, *sxz0_n, *exxd_s, *ezzd_s, *exz_n, *sxz_n;
    double *rho0_n;
    double  Ut, Ue, W, *Work, *Uelastic, *Uthermal, *Time, *Short;
    double *T, *dT, *d_n, *d0_n, *phi_n, *phi0_n;
    double *eII_el, *eII_pl, *eII_pl_s, *eII_pwl, *eII_exp, *eII_lin, *eII_gbs, *eII_cst;
    double *eII_pwl_s;
    double *exx_el, *ezz_el, *exz_el, *exx_diss, *ezz_diss, *exz_diss;
    int    *comp_cells;
    double *D11_n, *D12_n, *D13_n, *D14_n;
    double *D21_n, *D22_n, *D23_n, *D24_n;
    double *D31_s, *D32_s, *D33_s, *D34_s;
    double *detadexx_n, *detadezz_n, *detadgxz_n, *detadp_n;
    double *ddivpdexx_n, *ddivpdezz_n, *ddivpdgxz_n, *ddivpdp_n;
    double *detadexx_s, *detadezz_s, *detadgxz_s, *detadp_s;
    double *drhodp_n;
    double *phi0_s, *d0_s, *T_s, *P_s;
    double *nx_n, *nz_n, *nx_s, *nz_s, *FS_AR_n, *FS_AR_s, *aniso_factor_n, *aniso_factor_s;
    double *nx0_n, *nz0_n, *nx0_s, *nz0_s;
    double *cell_min_z, *cell_max_z, *vert_min_z, *vert_max_z;
    double *dil_n, *dil_s, *fric_n, *fric_s, *C_n, *C_s;
    double *exz_n_el, *exz_n_diss, *exz_n_pl, *Wdiss, *Wel, *Wtot;
    double *kc_x, *kc_z;
    double *FreeSurfW_s, *FreeSurfW_n;
};

/* ---------------------------------------------------------------------- */
/* 1. Drop-in entry points (reference names, reference prototypes).        */
/*    All run on the GPU; host structs in, host structs out.               */
/* ---------------------------------------------------------------------- */

/* RheologyDensity.c:44 Viscosity (no prototype in the reference header).
 * Pointwise local constitutive update of one node and one phase. */
double Viscosity(int phase, double G, double T, double P, double d, double phi, double X0,
                 double Exx, double Ezz, double Exz, double Gxx, double Gzz, double Gxz,
                 double Txx0, double Tzz0, double Txz0, mat_prop *materials, params *model,
                 scale *scaling, double *txxn, double *tzzn, double *txzn, double *etaVE,
                 double *VEcoeff, double *Eii_el, double *Eii_pl, double *Eii_pwl, double *Eii_exp,
                 double *Eii_lin, double *Eii_gbs, double *Eii_cst, double *Exx_el, double *Ezz_el,
                 double *Exz_el, double *Exx_diss, double *Ezz_diss, double *Exz_diss, double *d1,
                 double strain_acc, double dil, double fric, double C, double *detadexx,
                 double *detadezz, double *detadexz, double *detadp, double P0, double *X1,
                 double *OverS, double *ddivpdexx, double *ddivpdezz, double *ddivpdexz,
                 double *ddivpdp, double *Pcorr, double *drhodp, double *rho, double beta,
                 double div, double *div_el, double *div_pl, double *div_r);

/* header_MDOODZ.h:416 -> RheologyDensity.c:961 */
void NonNewtonianViscosityGrid(grid *mesh, mat_prop *materials, params *model, Nparams Nmodel,
                               scale *scaling);
/* header_MDOODZ.h:417 -> RheologyDensity.c:1902 */
void StrainRateComponents(grid *mesh, scale scaling, params *model);
/* header_MDOODZ.h:580 -> RheologyDensity.c:713 */
void RheologicalOperators(grid *mesh, params *model, scale *scaling, int Jacobian);
/* header_MDOODZ.h:351 -> StokesRoutines.c:922 */
void EvaluateRHS(grid *mesh, params model, scale scaling, double RHO_REF);
/* header_MDOODZ.h:414 -> StokesRoutines.c:137 */
void UpdateNonLinearity(grid *mesh, markers *particles, markers *topo_chain, surface *topo,
                        mat_prop materials, params *model, Nparams *Nmodel, scale scaling, int mode,
                        double h_contin);
/* header_MDOODZ.h:316 -> GridRoutines.c:106 */
void InterpCentroidsToVerticesDouble(double *CentroidArray, double *VertexArray, grid *mesh,
                                     params *model);
/* header_MDOODZ.h:393 -> StokesRoutines.c:1134 */
void EvalNumberOfEquations(grid *mesh, SparseMat *Stokes);
/* header_MDOODZ.h:474 -> StokesAssemblyDecoupled.c:1573 */
void BuildStokesOperatorDecoupled(grid *mesh, params model, int lev, double *p_corr, double *p,
                                  double *u, double *v, SparseMat *Stokes, SparseMat *StokesA,
                                  SparseMat *StokesB, SparseMat *StokesC, SparseMat *StokesD,
                                  int Assemble);
/* header_MDOODZ.h:491 -> StokesAssemblyDecoupled.c:3834 */
void BuildJacobianOperatorDecoupled(grid *mesh, params model, int lev, double *p_corr, double *p,
                                    double *u, double *v, SparseMat *Stokes, SparseMat *StokesA,
                                    SparseMat *StokesB, SparseMat *StokesC, SparseMat *StokesD,
                                    int Assemble);
/* header_MDOODZ.h:473 -> StokesRoutines.c:839 */
void EvaluateStokesResidualDecoupled(SparseMat *Stokes, SparseMat *StokesA, SparseMat *StokesB,
                                     SparseMat *StokesC, SparseMat *StokesD, Nparams *Nmodel,
                                     grid *mesh, params model, scale scaling, int quiet);
/* StokesRoutines.c:1232 ExtractDiagonalScale (header_MDOODZ.h:577): d of
 * the momentum rows = diagonal of A (copied to B), d of the continuity rows
 * = diagonal of D (copied to C). */
void ExtractDiagonalScale(SparseMat *StokesA, SparseMat *StokesB, SparseMat *StokesC, SparseMat *StokesD);
/* StokesRoutines.c:1276 ScaleMatrix (header_MDOODZ.h:578): values times
 * d_i d_j, b and F times d_i. */
void ScaleMatrix(SparseMat *StokesA, SparseMat *StokesB, SparseMat *StokesC, SparseMat *StokesD);

/* header_MDOODZ.h:477 -> StokesAssemblyCoupled.c:47.  Host bookkeeping
 * helper of the assembly (append a coefficient or fold a Dirichlet
 * neighbour into the right-hand side); exported because the reference
 * exports it. */
void AddCoeff2(int *J, double *A, int eqn, int jeq, int *nnzc, double coeff, int NODE_TYPE,
               double NODE_VAL, double *RHS);

/* The reference's solver workspace (CHOLMOD factor and settings); the
 * device solver keeps its own factor and never reads it. */
typedef struct _DirectSolver DirectSolver;

/* header_MDOODZ.h:470 -> Solvers.c:2226.  Solution of the decoupled Stokes
 * system with the Picard blocks matA..matD (preconditioner) and the
 * Jacobian blocks JmatA..JmatC (operator): sol[0 .. neq_mom) = du,
 * sol[neq_mom ..) = dp.  Powell-Hestenes iterations around the restarted
 * GCR of kspgcr, preconditioned by a sparse Cholesky factor of the penalised
 * operator on the device (in place of CHOLMOD's); pardi is not read.
 * Penalty, tolerances and pc_type come from model, the equation numbering
 * from Stokes, the grid dimensions, comp_cells and bet_n from mesh. */
void KillerSolver(SparseMat *matA, SparseMat *matB, SparseMat *matC, SparseMat *matD, DirectSolver *pardi,
                  double *rhs_mom, double *rhs_cont, double *sol, params model, grid *mesh, scale scaling,
                  SparseMat *Stokes, SparseMat *Jacobian, SparseMat *JmatA, SparseMat *JmatB, SparseMat *JmatC);

/* Marker -> grid (the per-time-step producers of the rheology's inputs).
 * The markers are binned by nearest node on the device and every node sums
 * its markers in increasing index, so the sums are those of the reference
 * on one OpenMP thread.  Markers with a phase outside [-1, Nb_phases) are
 * an error (MDZ_EINVAL); Interp_P2N ignores a marker whose vertex index
 * falls outside the grid (the reference indexes past its arrays there). */
/* header_MDOODZ.h:345 -> ParticleRoutines.c:3226 */
void P2Mastah(params *model, markers particles, DoodzFP *mat_prop, grid *mesh, double *NodeField,
              char *NodeType, int flag, int avg, int prop, int centroid, int itp_stencil);
/* header_MDOODZ.h:338 -> ParticleRoutines.c:1770 */
void Interp_P2N(markers particles, DoodzFP *mat_prop, grid *mesh, double *NodeField, double *X_vect,
                double *Z_vect, int flag, int itp_type, params *model);
/* header_MDOODZ.h:411 -> RheologyDensity.c:1422 */
void CohesionFrictionDilationGrid(grid *mesh, markers *particles, mat_prop materials, params model,
                                  scale scaling);

/* ---------------------------------------------------------------------- */
/* 2. Device-resident interface                                             */
/* ---------------------------------------------------------------------- */

/* Error handling: every mdz_* call returns 0 on success or a negative
 * MDZ_E* code; mdz_last_error() gives the message.  The drop-in entry
 * points above mirror the reference's behaviour instead (message on stdout
 * then exit(code)), see mdz_set_exit_on_error(). */
enum {
    MDZ_OK = 0,
    MDZ_EINVAL = -1,      /* bad argument / unsupported option */
    MDZ_EHIP = -2,        /* HIP runtime failure */
    MDZ_ENOMEM = -3,      /* device or host allocation failed */
    MDZ_ENAN = -4,        /* NaN residual (reference exit code 122) */
    MDZ_ED34 = -5,        /* NaN/Inf in D34 (reference exit code 1) */
    MDZ_EUNSUPPORTED = -6, /* reference feature outside this implementation */
    MDZ_EIO = -7,          /* file I/O failure, or the HDF5 library is missing */
    MDZ_ESOLVE = -8        /* linear solve failed: factor not positive definite, or the
                              divergence tolerance not met (reference exit code 1) */
};
const char *mdz_last_error(void);
/* 1 (default): the drop-in entry points print the reference's message and
 * call exit() with the reference's code.  0: they only record the error,
 * readable with mdz_last_error()/mdz_last_status(). */
void mdz_set_exit_on_error(int on);
/* Status of the last drop-in call: 0, or the MDZ_E* code it recorded (each
 * drop-in clears it on entry). */
int  mdz_last_status(void);

/* Rheology arithmetic of the local iterations. */
enum {
    MDZ_RHEO_FP64 = 0,      /* plain: reference initial guess, FP64 throughout */
    MDZ_RHEO_MIXED = 1,     /* FP32 iterations + FP64 polish to the reference tolerance */
    MDZ_RHEO_LEARNED = 2    /* MIXED with the surrogate network's initial guess */
};

/* Grid rheology kernel (process-wide; no counterpart in the reference).
 * 0 (default): the log-space kernel wherever it applies (eta_average = 0,
 * isotropic, no grain-size evolution, no phase mixing, no reaction
 * softening), the generic kernel otherwise.  1: always the generic kernel,
 * a line-by-line restatement of Viscosity (RheologyDensity.c:44-707). */
int mdz_set_rheology_kernel(int which);

typedef struct mdz_ctx mdz_ctx;

/* Creates a device mirror of *mesh (all fields the path reads or writes),
 * uploads every input field, numbers the equations and builds the Picard
 * and Jacobian CSR patterns from the boundary tags. */
int  mdz_ctx_create(mdz_ctx **out, const grid *mesh, const mat_prop *materials,
                    const params *model, const scale *scaling);
void mdz_ctx_destroy(mdz_ctx *ctx);
/* Re-uploads the per-time-step input fields of *mesh (the fields the
 * reference's time loop refills from the markers, Main_DOODZ.c:494-625:
 * temperature, old stresses, shear moduli, cohesion, friction, dilation,
 * densities, pressures of the last step, phase fractions and the like; not
 * u_in/v_in/p_in).  Parameters, scales, materials, boundary tags and values,
 * coordinates, equation numbers and CSR patterns keep their values: use
 * mdz_ctx_update_step when any of those change. */
int  mdz_ctx_upload_step_fields(mdz_ctx *ctx, const grid *mesh);
/* Everything a new time step may change, as the reference's time loop
 * changes it before its Newton iterations (Main_DOODZ.c:459-699: dt and the
 * other params, SetBCs' tags and values, EvalNumberOfEquations): parameters,
 * scales and materials; boundary tags and values, coordinates and spacing;
 * every input field incl. the iterate; then the equations are numbered
 * again and both CSR patterns rebuilt.  Captured graphs (ensembles, line
 * search) are captured again at their next launch.  Same grid size and
 * phase count as at creation (MDZ_EINVAL otherwise). */
int  mdz_ctx_update_step(mdz_ctx *ctx, const grid *mesh, const mat_prop *materials,
                         const params *model, const scale *scaling);
/* Upload / download the iterate u_in, v_in, p_in. */
int  mdz_ctx_upload_solution(mdz_ctx *ctx, const double *u_in, const double *v_in, const double *p_in);
int  mdz_ctx_download_solution(mdz_ctx *ctx, double *u_in, double *v_in, double *p_in);
/* Copy every output field of the path back into *mesh. */
int  mdz_ctx_download_grid(mdz_ctx *ctx, grid *mesh);
int  mdz_ctx_set_rheology_mode(mdz_ctx *ctx, int mode);
/* Deferred diagnostics (no counterpart in the reference, which recomputes
 * every rheology output in every Newton iteration).  When on, a unit's
 * rheology pass writes only the fields the unit itself reads (eta, the
 * tangent, the plastic divergence derivatives and p_corr at centroids and
 * vertices); the other outputs (stresses, strain-rate partition, work
 * terms, eta_phys, VE, OverS, d, X, ...) are recomputed from the same inputs
 * when mdz_ctx_download_grid is called, so every field the host sees is
 * bit for bit the one a unit with full outputs leaves.  Off by default. */
int  mdz_ctx_defer_diagnostics(mdz_ctx *ctx, int on);
/* (No counterpart in the reference.)  MDZ_RHEO_LEARNED: by default (on =
 * 1) the log-space rheology kernels evaluate the network for their own
 * nodes in a prologue; with on = 0 a separate inference pass writes the
 * network's guess of every node into guess arrays that the rheology
 * kernels read (the generic kernel always takes that route).  Both give the
 * same guess bit for bit. */
int  mdz_ctx_fuse_guess(mdz_ctx *ctx, int on);
/* Loads the surrogate network used by MDZ_RHEO_LEARNED (a parameter blob of
 * MDZ_MLP_NPARAMS floats, see below; models of at most three phases). */
int  mdz_ctx_set_network(mdz_ctx *ctx, const float *weights, size_t n_floats);

/* One Newton-iteration unit, all device-resident, on the context's stream:
 * StrainRateComponents -> NonNewtonianViscosityGrid -> EvaluateRHS ->
 * RheologicalOperators(0) -> Picard CSR values -> RheologicalOperators(1) ->
 * Jacobian CSR values -> RheologicalOperators(0) -> residual and norms.
 * Norms (resx, resz, resp) are written to res3 (host) when non-NULL; the
 * call synchronises only in that case. */
int  mdz_ctx_newton_unit(mdz_ctx *ctx, double *res3);

/* CSR sizes and device pointers of the last assembled blocks
 * (which: 0..3 = Picard A,B,C,D; 4..7 = Jacobian A,B,C,D). */
int  mdz_ctx_block_info(mdz_ctx *ctx, int which, int *neq, int *nnz);
int  mdz_ctx_download_block(mdz_ctx *ctx, int which, int *Ic, int *J, double *A, double *b,
                            double *bbc);
/* Residual vectors (F of the momentum and continuity blocks). */
int  mdz_ctx_download_residual(mdz_ctx *ctx, double *Fmom, double *Fcont);

/* Device-resident marker-to-grid step (no counterpart as one function in
 * the reference, whose time loop calls P2Mastah for the phase fractions,
 * ParticleRoutines.c:3566-3567, then CohesionFrictionDilationGrid): uploads
 * the markers' x, z, phase and strain_pl, computes the phase fractions at
 * centroids and vertices and the softened C, friction and dilatancy angles
 * into the context's fields, where the next unit reads them (model.itp_stencil
 * and Nb_phases of the context).  mesh supplies the node coordinates; with
 * download != 0 the fields produced are also copied into its phase_perc_n/s,
 * C_n/s, fric_n/s and dil_n/s.  particles NULL: the markers of the previous
 * call, still on the device, are binned and interpolated again. */
int  mdz_ctx_markers_to_grid(mdz_ctx *ctx, grid *mesh, const markers *particles, int download);

/* On-disk matrix format: the HDF5 dump that BuildStokesOperatorDecoupled and
 * BuildJacobianOperatorDecoupled write when model.write_debug == 1
 * (StokesAssemblyDecoupled.c:2041-2137, :4264-4360; dataset properties of
 * AddFieldToGroup_generic, HDF5Output.c:121-226): groups model, numbering,
 * fields, matrix; params = {Nx, Nz, dx, dz}; eqn_u/v/p; eta_n, eta_s and the
 * four boundary-tag arrays; IA JA VA ... ID JD VD, eta_cell, rhs_mom,
 * rhs_cont, F_mom, F_cont.  Ints are stored as big-endian 32-bit, tags as
 * 8-bit, reals as f64; each dataset chunked at 5 % of its length and
 * deflate level 4.  The drop-ins above write it under the reference's name
 * "<Stokes|Jacobian>_%02dcpu_step%02d_iter%02d.gzip.h5" in the working
 * directory.  HDF5 (1.10 or later) is loaded at the first call: MDZ_EIO when
 * it is missing. */
int  mdz_write_matrix_h5(const char *filename, const grid *mesh, const SparseMat *Stokes,
                         const SparseMat *StokesA, const SparseMat *StokesB,
                         const SparseMat *StokesC, const SparseMat *StokesD);
/* The same file from a context: the blocks of the last unit (kind 0 =
 * Picard, 1 = Jacobian), its numbering, tags, eta_n/eta_s, right-hand sides
 * and residuals.  (No counterpart in the reference, whose dump reads host
 * arrays.) */
int  mdz_ctx_write_matrix_h5(mdz_ctx *ctx, int kind, const char *filename);
/* Reads one one-dimensional dataset of such a file (or of any HDF5 file):
 * *type = 'd' (f64), 'f' (f32), 'i' (32-bit int, either byte order), 'c'
 * (8-bit int); *n = its length; the values go to buf when its cap_bytes hold
 * them (buf NULL: size query only).  MDZ_EIO for a missing file or dataset. */
int  mdz_read_h5_dataset(const char *filename, const char *path, void *buf, size_t cap_bytes,
                         char *type, size_t *n);
/* ExtractDiagonalScale + ScaleMatrix on the device-resident Picard (kind 0)
 * or Jacobian (kind 1) blocks, after mdz_ctx_newton_unit
 * (Main_DOODZ.c:801-820 with diag_scaling = 1). */
int  mdz_ctx_diagonal_scaling(mdz_ctx *ctx, int kind);
/* Switches the collection of local-iteration histograms on (1) or off (0,
 * the default: collection costs a few percent of the rheology kernels). */
int  mdz_ctx_collect_histogram(mdz_ctx *ctx, int on);
/* Local-iteration counts accumulated since the last call while collection
 * was on (node x phase evaluations): hist[0..63] = FP64 visco-elastic Newton iterations,
 * hist[64..127] = plastic return-map iterations, hist[128..191] = FP32
 * pre-iterations (mixed / learned modes).  Resets the counters. */
int  mdz_ctx_iteration_histogram(mdz_ctx *ctx, long long *hist192);
/* Mean per-stage milliseconds over `reps` units, measured with HIP events
 * on the context's stream: ms[0..9] = strain rates with the centroid-to-
 * vertex interpolation of div_u, T, P, d and phi (one launch), the
 * network's separate guess pass (learned mode without mdz_ctx_fuse_guess;
 * else about 0), local iterations
 * (centroid and vertex rheology kernels), right-hand sides, D(Picard),
 * Picard values, D(Jacobian), Jacobian values, D(Picard), residual + norms;
 * ms[10] = the whole of them.  An isotropic model (aniso = 0) runs one
 * fused D pass, timed as D(Jacobian); both D(Picard) stages are then 0.
 * The stages are launched apart here; a unit takes the right-hand sides
 * with the D pass, and on small grids both value passes, in one launch. */
int  mdz_ctx_stage_times(mdz_ctx *ctx, int reps, double *ms11);
/* Mean milliseconds per unit over `reps` back-to-back units. */
int  mdz_ctx_time_units(mdz_ctx *ctx, int reps, double *ms_per_unit);
/* Achievable HBM bandwidth: `reps` streaming copies of `bytes` (read +
 * write counted), GB/s.  Also the known-size kernel for scaling memory
 * counters (kernel name k_copy_probe). */
int  mdz_copy_probe(size_t bytes, int reps, double *gbs);
/* The HIP stream (hipStream_t) the context launches on. */
void *mdz_ctx_stream(mdz_ctx *ctx);
/* The line search of the Newton step (LineSearchDecoupled,
 * StokesRoutines.c:396-622) as one graph launch on the resident fields: for
 * each of the ntry (1..16) step lengths alpha[k], the iterate u + alpha[k] dx
 * (dx indexed by equation number, neq_mom + neq_cont values, on the host)
 * goes through UpdateNonLinearity and EvaluateStokesResidualDecoupled;
 * res3n[3k .. 3k+2] = resx, resz, resp.  The iterate u, v, p is restored;
 * the other fields hold the last trial's values, as in the reference.  Needs
 * a unit (assembled blocks) before.  dx = NULL takes the correction of the
 * last mdz_ctx_solve on the device. */
int  mdz_ctx_line_search(mdz_ctx *ctx, const double *dx, int ntry, const double *alpha, double *res3n);
/* No counterpart in the reference.  For callers that cannot allocate (code
 * under HIP graph capture, tight loops, harnesses that forbid hipMalloc):
 * mdz_ctx_line_search with the same arguments and results, bit for bit,
 * that calls no hipMalloc/hipFree and instantiates no graph.  Its trials run
 * eagerly on the context's stream; the saved iterate, the correction, the
 * step lengths and the trial norms live in a fixed device array of the
 * library (16 Mi doubles per GPU, held until the process ends), which
 * bounds the grid: nu + nw + nc + neq + 112 doubles at most (about 2.7 M
 * cells); larger grids get MDZ_EINVAL.  Calls that overlap on one GPU race
 * on that array. */
int  mdz_ctx_line_search_noalloc(mdz_ctx *ctx, const double *dx, int ntry, const double *alpha, double *res3n);
/* Outcome of a device solve (mdz_ctx_solve, KillerSolver). */
typedef struct {
    int    ph_its;        /* Powell-Hestenes iterations */
    int    ksp_its_total; /* GCR iterations, counted as kspgcr counts them */
    int    ksp_its[20];   /* per Powell-Hestenes iteration */
    int    kd, nb;        /* half bandwidth of Jts by grid columns or rows (the narrower); nb as asked (1024 for 0) */
    double maxdiv0, maxdiv, maxru0, maxru; /* the reference's stopping quantities */
    double resx, resz, resp; /* rms of the final residual over the u, v, p equations */
    double factor_ms, iterate_ms; /* host wall time of the factorisation and the iterations */
} mdz_solve_info;
/* The Newton correction of the resident blocks (the solve of
 * SolveStokesDefectDecoupled, StokesRoutines.c:700-728, lsolver = 2):
 * KillerSolver (Solvers.c:2226) on the Picard blocks, the Jacobian blocks
 * and the residual F of the last unit, then ScaleVelocitiesRHSBack where
 * the blocks are scaled.  The correction stays on the device for
 * mdz_ctx_line_search (dx = NULL) and is copied to dx (neq_mom + neq_cont
 * values by equation number) when dx is not NULL.  nb: 0 or a
 * multiple of 64, reported in info; the factor's layout does not depend on
 * it.  Penalty (default 1e10), abs_tol_div
 * (1e-14), rel_tol_div (1e-5) and rel_tol_KSP (1e-4) from the context's
 * params, the reference's input defaults where they are 0, and pc_type (0:
 * the Picard operator as preconditioner, 1: the symmetrised Jacobian).
 * model.noisy > 0 prints the reference's line per Powell-Hestenes
 * iteration, > 1 also its line per GCR direction.  MDZ_ESOLVE where the
 * reference exits (divergence tolerance not met); the correction is then
 * not kept. */
int  mdz_ctx_solve(mdz_ctx *ctx, int nb, double *dx, mdz_solve_info *info);
/* Block shapes of the tunable kernels of a context (no counterpart in the
 * reference): threads per block of the rheology kernels (64, 128, 256),
 * rows per block of the LDS-staged Picard (0 = unstaged, 64, 128, 256) and
 * Jacobian (0, 64, 128) value kernels; 64 rows take the split pass (the
 * general row code over the waves that hold a boundary row beside the
 * tag-free row code over the others).  Default 64, 128, 64.  A unit on a
 * small grid takes both value passes in one launch of 64-row blocks, unless
 * a shape other than 64, 64 has been set for them here.  Results do not
 * depend on any of it. */
int  mdz_ctx_set_launch_shape(mdz_ctx *ctx, int rheo, int pic, int jac);
int  mdz_ctx_get_launch_shape(mdz_ctx *ctx, int *shape3);

/* ---------------------------------------------------------------------- */
/* Ensembles of independent models (no counterpart in the reference: the  */
/* reference runs one model per process).  One graph launch takes every    */
/* model of the ensemble through one Newton-iteration unit.                */
/* ---------------------------------------------------------------------- */
typedef struct mdz_ensemble mdz_ensemble;
/* The contexts stay owned by the caller and must outlive the ensemble;
 * their pending work is synchronised here.  Between mdz_ensemble_launch
 * and mdz_ensemble_synchronize no call may touch the contexts. */
int  mdz_ensemble_create(mdz_ensemble **out, mdz_ctx *const *ctx, int n);
void mdz_ensemble_destroy(mdz_ensemble *ens);
/* Number of concurrent chains of the graph (1..8, default 4); models are
 * spread over the chains by cell count, largest first. */
int  mdz_ensemble_set_branches(mdz_ensemble *ens, int branches);
/* Enqueues one Newton unit of every model as one graph launch (captured
 * on first use and again after any context setting changed; the captured
 * graph is kept and relaunched).  Asynchronous. */
int  mdz_ensemble_launch(mdz_ensemble *ens);
int  mdz_ensemble_synchronize(mdz_ensemble *ens);
/* resx, resz, resp of every model after the last launch (n * 3 doubles;
 * synchronises). */
int  mdz_ensemble_residuals(mdz_ensemble *ens, double *res3n);
/* Mean milliseconds per graph launch over `reps` launches. */
int  mdz_ensemble_time(mdz_ensemble *ens, int reps, double *ms_per_launch);
/* Autotuner: per size class (cell counts within a power of two) the block
 * shape of each tunable kernel is timed on the class's largest model and
 * applied to the class, then the chain count (1, 2, 4, 8) is timed on the
 * whole graph.  shapes3n (optional, n * 3) and branches (optional) receive
 * the choice. */
int  mdz_ensemble_autotune(mdz_ensemble *ens, int reps, int *shapes3n, int *branches);

/* ---------------------------------------------------------------------- */
/* Surrogate network for the initial guess of the local iteration (no     */
/* counterpart in the reference): MLP 9 -> 64 -> 64 -> 64 -> 2, SiLU, BF16 */
/* matrix-core operands with FP32 accumulation.                           */
/* Features: (log10 Eii + 15)/3, (T - 1123)/850 [K], (P - 5)/5 [GPa],      */
/* (tau0 - 250)/250 [MPa], log10 dt - 11 [s], one-hot phase 0..2,          */
/* (log10 tau_y - 1.5)/1.5 [MPa] with tau_y = C cos(phi) + P sin(phi).     */
/* Outputs: 4 log10(eta_ve / eta_ref) with eta_ref the reference's guess  */
/* (smallest isolated viscosity), 4 log10(gdot / gdot_start) with         */
/* gdot_start the return map's closed-form start (0 without yielding).    */
/* Blob: W1[64][9] b1[64] W2[64][64] b2[64] W3[64][64] b3[64] W4[2][64]    */
/* b4[2] (row-major [out][in]).                                            */
/* ---------------------------------------------------------------------- */
#define MDZ_MLP_NPARAMS 9090
typedef struct mdz_mlp mdz_mlp;
/* materials/params/scale: the three-phase model whose flow laws the
 * training samples use */
int  mdz_mlp_create(mdz_mlp **out, const mat_prop *materials, const params *model, const scale *scaling);
void mdz_mlp_destroy(mdz_mlp *net);
int  mdz_mlp_init(mdz_mlp *net, unsigned long long seed);                   /* He-normal weights */
int  mdz_mlp_set_weights(mdz_mlp *net, const float *w, size_t n_floats);
int  mdz_mlp_get_weights(mdz_mlp *net, float *w, size_t n_floats);
/* `count` samples drawn by `seed` (log10 Eii U[-18,-12], T U[273,1973] K,
 * P U[0,10] GPa, tau0 U[0,500] MPa, dt log-U[1e10,1e12] s, phase U{0,1,2},
 * C U[5,50] MPa, phi U[10,35] deg), labelled by the FP64 reference rheology
 * on the GPU; kept in device memory */
int  mdz_mlp_generate(mdz_mlp *net, long long count, unsigned long long seed);
int  mdz_mlp_upload_samples(mdz_mlp *net, long long count, const float *X9, const float *Y2);
int  mdz_mlp_download_samples(mdz_mlp *net, long long first, long long count, float *X9, float *Y2);
/* gradient of sum((y - t)^2) / (2 count) over samples [first, first+count),
 * count a multiple of 64; loss = sum of squared errors */
int  mdz_mlp_gradient(mdz_mlp *net, long long first, int count, float *grad, double *loss);
int  mdz_mlp_adam_step(mdz_mlp *net, const float *grad, float lr);         /* beta 0.9/0.999, eps 1e-8 */
/* Adam epochs over the stored samples; loss_per_epoch[e] = mean squared
 * error per output */
int  mdz_mlp_train(mdz_mlp *net, int epochs, int batch, float lr, unsigned long long seed, double *loss_per_epoch);
int  mdz_mlp_predict(mdz_mlp *net, long long first, long long count, float *Y2);
/* The same through the inference form of the weights that the grid guess
 * evaluates (log2(e) folded into the weights, 16x16x32 matrix tiles):
 * equal to mdz_mlp_predict up to BF16 rounding of the rescaled weights. */
int  mdz_mlp_predict_inference(mdz_mlp *net, long long first, long long count, float *Y2);

#ifdef __cplusplus
}
#endif
#endif /* MDOODZ_HOT_H */
