/*
 * mdz_kernels.h -- host-side launch interface of the gfx950 kernels.
 */
#pragma once

#include "mdz_device.h"

/* records an error for mdz_last_error() / mdz_last_status(); returns code */
int mdz_error(int code, const char *msg);

/* rheology half (mdz_rheology.hip) */
void mdz_launch_strain_rates(const DevGrid &g, const DevParams &prm, hipStream_t s);
/* the strain rates and mdz_launch_interp5 in one launch (the vertex values
 * of div_u from the strain rates of the same launch) */
void mdz_launch_strain_interp5(const DevGrid &g, const DevParams &prm, hipStream_t s);
void mdz_launch_interp(const DevGrid &g, const DevParams &prm, const double *src, double *dst, hipStream_t s);
/* grid rheology (the vertex fields of mdz_launch_interp5 must be in place) */
void mdz_launch_rheology(const DevGrid &g, const DevParams &prm, const mat_prop *mt, const float *guess_n,
                         const float *guess_s, unsigned long long *hist, hipStream_t s);
/* div_u, T, P, d, phi from centroids to vertices (input of the vertex rheology) */
void mdz_launch_interp5(const DevGrid &g, const DevParams &prm, hipStream_t s);

/* log-space rheology for eta_average = 0, isotropic, no grain-size evolution
 * or phase mixing (mdz_rheo_fast.hip); per-phase constants precomputed */
#define MDZ_MAX_PHASES 20
int mdz_rheo_fast_eligible(const DevParams &prm, const mat_prop *host_mt);
size_t mdz_phasek_bytes(void);
void mdz_launch_phase_constants(const mat_prop *d_mt, int nph, void *d_pk, hipStream_t s);
/* nt: threads per block, 64, 128 or 256 (anything else is MDZ_EINVAL);
 * diag != 0 writes every output field, diag == 0 only those the rest of a
 * Newton-iteration unit reads (eta, tangent, plastic divergence
 * derivatives, p_corr): the same values, bit for bit.  The initial guess comes from guess_n / guess_s
 * (k_mlp_guess), or with net != nullptr from the network evaluated in the
 * kernels' prologue (the same guess, without the guess arrays). */
struct DevMLPI;
int mdz_launch_rheology_fast(const DevGrid &g, const DevParams &prm, const void *d_pk, double R, const float *guess_n,
                             const float *guess_s, unsigned long long *hist, int nt, int diag, hipStream_t s,
                             const DevMLPI *net = nullptr);
/* D tensor.  mode 0: the J = 0 tensor into D11_n..D34_s; 1: the J = 1
 * tensor; 2: the J = 1 tensor, and the J = 0 values of D11 (= D22) at the
 * centroids and D33 at the vertices into dp_n / dp_s; 3: only those two. */
void mdz_launch_dtensor(const DevGrid &g, const DevParams &prm, int mode, int *status, hipStream_t s,
                        double *dp_n = nullptr, double *dp_s = nullptr);
void mdz_launch_rhs(const DevGrid &g, const DevParams &prm, const double *xg, const double *zvx,
                    const double *xvz, const double *zg, hipStream_t s);
/* both in one launch (neither reads what the other writes) */
void mdz_launch_rhs_dtensor(const DevGrid &g, const DevParams &prm, int mode, const double *xg, const double *zvx,
                            const double *xvz, const double *zg, int *status, hipStream_t s, double *dp_n = nullptr,
                            double *dp_s = nullptr);

/* assembly half (mdz_assembly.hip) */
struct DevAsm {
    DevGrid g;
    DevEqn e;
    double celvol, one_dx, one_dz, one_dx_dx, one_dz_dz, one_dx_dz, om, dt, gz_model;
    /* Jacobian stencil factors (1 - 1/3)/dx, (1 - 1/3)/dz, (1/3)/dx, (1/3)/dz,
     * computed once per grid instead of per row */
    double jk_e1x, jk_e1z, jk_e3x, jk_e3z;
    int stab, comp_model, periodic, Nz_model;
    const double *u, *v, *p_mom, *p_cont; /* iterate: p_corr for momentum rows, p_in for continuity */
    const double *d11p, *d22p, *d33p;     /* D11, D22 (centroids) and D33 (vertices) of the J = 0 tensor,
                                             the only components the Picard rows read */
};

/* numbering: flags -> exclusive scan -> eqn_u/v/p, -12 copies, row->node maps */
int mdz_number_equations(const DevGrid &g, DevEqn &e, int *scratch_int, size_t scratch_len, hipStream_t s);
/* pattern of a block family: kind 0 = Picard, 1 = Jacobian; fills Ic/J and nnz */
int mdz_build_pattern(int kind, const DevAsm &a, DevBlock *A, DevBlock *B, DevBlock *C, int *scratch_int,
                      size_t scratch_len, hipStream_t s);
/* second half of the pattern build (after J is allocated to the nnz counts) */
void mdz_fill_pattern(int kind, const DevAsm &a, DevBlock *A, DevBlock *B, DevBlock *C, hipStream_t s);
/* Launch shape of the tunable kernels of one model: threads per block of
 * the log-space rheology kernels (64, 128, 256) and rows per block of the
 * LDS-staged momentum value kernels, Picard (64, 128, 256) and Jacobian
 * (64, 128); 0 selects the unstaged value kernel.  Every shape computes the
 * same values bit for bit: the per-row arithmetic does not depend on it. */
struct LaunchShape {
    int rheo, pic, jac;
    bool asked = false; /* by a caller, who gets this shape and no other */
};
/* the shape the autotuner picks at 2049 x 1025 (64-row value blocks take
 * the split pass: tag-free waves, then the listed general waves) */
#define MDZ_SHAPE_DEFAULT LaunchShape{64, 128, 64}
int mdz_shape_valid(const LaunchShape &sh);
/* values of the assembled blocks (Assemble = 1); vblk = rows per block of
 * the staged momentum kernel (0 = unstaged; a pattern whose rows do not fit
 * the LDS slots always takes the unstaged kernel) */
void mdz_launch_values(int kind, const DevAsm &a, DevBlock *A, DevBlock *B, DevBlock *C, DevBlock *D, int vblk,
                       hipStream_t s);
/* free-row flags of the momentum rows of a block family (after the
 * pattern; A->free_row allocated with neq_mom bytes) */
int mdz_launch_free_rows(int kind, const DevAsm &a, DevBlock *A, DevBlock *B, hipStream_t s);
/* residual rows (Assemble = 0) through the Picard (kind 0) or Jacobian (kind 1) stencils;
 * A/C carry b, F, bbc; D carries F and d */
void mdz_launch_residual(int kind, const DevAsm &a, DevBlock *A, DevBlock *C, DevBlock *D, hipStream_t s);
/* norms: sums of F^2 over the u, v, p DOF nodes, ru/rv/rp, F *= d.
 * partial: device buffer of at least mdz_norm_partials(g) doubles; out3: device double[6]
 * (sum_x, sum_z, sum_p, ndof_x, ndof_z, ndof_p) */
size_t mdz_norm_partials(const DevGrid &g);
void mdz_launch_norms(const DevAsm &a, DevBlock *A, DevBlock *D, double *partial, double *out6, hipStream_t s);
/* the value passes of both families (P Picard, J Jacobian) in one launch;
 * false, with nothing enqueued, where they are better apart, one of them
 * cannot take the split pass, or a caller asked for another shape */
bool mdz_launch_values_pair(const DevAsm &a, DevBlock *P, DevBlock *J, const LaunchShape &shape, hipStream_t s);
/* the waves of A that are not all free rows, into A->gen_waves / A->n_gen
 * (after the free-row flags; A->gen_waves holds 2 * (neq_mom / 64 + 2)
 * ints: the list, then the flags and their scan; synchronises s to read
 * the count) */
int mdz_build_general_waves(DevBlock *A, int neq_mom, int *scratch, size_t scratch_len, hipStream_t s);
/* residual rows and their norms in one pass (the sums of k_norms, over the
 * equations instead of the nodes): b, F, ru/rv/rp, F *= d, out6 as for
 * mdz_launch_norms.  partial: at least mdz_residual_norm_partials(...)
 * doubles (MDZ_ENOMEM when partial_len is smaller).  For kind 0 with the
 * free-node flags built, the free momentum rows and the continuity rows
 * run in LDS tiles (k_residual_tile), whose first blocks take the other rows
 * of the listed waves.  d_scaled = 0: every d is 1 (F *= d is skipped, with
 * the same result).  copy6 (optional, device or pinned host memory): the
 * six sums again; on the host readable once the stream has been
 * synchronised. */
size_t mdz_residual_norm_partials(int neq_mom, int n_gen, int neq_cont);
int mdz_launch_residual_norms(int kind, const DevAsm &a, DevBlock *A, DevBlock *C, DevBlock *D, double *partial,
                              size_t partial_len, double *out6, hipStream_t s, int d_scaled = 1,
                              double *copy6 = nullptr);

/* diagonal scaling: d from the diagonals of A and D (ExtractDiagonalScale),
 * then A_ij d_i d_j with b, F scaled by d (ScaleMatrix) */
void mdz_launch_extract_diagonal(DevBlock *A, DevBlock *B, DevBlock *C, DevBlock *D, hipStream_t s);
void mdz_launch_scale_matrix(DevBlock *A, DevBlock *B, DevBlock *C, DevBlock *D, hipStream_t s);

/* device-wide exclusive scan of n ints (in place), returns the total on the host (synchronises) */
int mdz_scan_exclusive(int *data, int n, int *scratch, size_t scratch_len, hipStream_t s, int *total);

/* ------------------------------------------------------------------ */
/* marker -> grid (mdz_markers.hip)                                     */
/* ------------------------------------------------------------------ */
struct MarkerSet {
    int n;
    const double *x, *z;
    const int *phase;
};

/* node axes of one node family: Nx x Nz nodes at X[i], Z[j] */
struct NodeAxes {
    int Nx, Nz;
    const double *X, *Z;
    double dx, dz;
    int periodic;
};

/* One marker as the gathers read it: position, the value of the current
 * interpolation, phase, and its index (the order of the reference's loop). */
struct MarkerRec {
    double x, z, val;
    int phase, k;
};

/* Markers on the device and their bins by nearest node, per node family
 * (slot 0 centroids, 1 vertices, 2 Vx nodes, 3 Vz nodes, 4 the axes a
 * caller of Interp_P2N passes, 5 the quarter cells): rec[f] holds the marker records bin by bin,
 * increasing marker index within a bin; start[f][b] ..
 * start[f][b + 1] is bin b. */
#define MDZ_MARKER_FAMS 6
#define MDZ_FAM_QUARTER 5
struct MarkerDev {
    int n, cap;
    double *x, *z;
    int *phase;
    double *val;                   /* per-marker values of the current interpolation */
    int *key, *key_out;            /* rank of each marker in its bin, or sort keys */
    MarkerRec *rec_in;             /* records bin by bin in any order, or the sort's input */
    MarkerRec *rec[MDZ_MARKER_FAMS];
    int *start[MDZ_MARKER_FAMS];
    size_t start_cap[MDZ_MARKER_FAMS];
    int binned[MDZ_MARKER_FAMS];   /* node count of the last binning, 0 = none */
    void *tmp;
    size_t tmp_bytes;
    int *scan;                     /* scratch of the bins' scan, then the flag of a long bin */
    size_t scan_len;
    int *long_bin;                 /* pinned copy of the flag */
    __host__ __device__ MarkerSet set() const { return MarkerSet{n, x, z, phase}; }
};

/* arguments of one interpolation: per-marker (flag 1: the records' val) or
 * per-phase (flag 0, pval) values, average 0 / 1 / 2 (arithmetic, harmonic,
 * geometric), node types (30 / 31 skipped), the output field, or with prop
 * = 1 the phase fractions perc[p][node] (nph phases) */
struct P2GArgs {
    int flag, avg, nph;
    const double *mval, *pval;
    const int8_t *ntype;
    double *field, *perc;
};

/* per-phase strength parameters and their strain softening */
struct SoftK {
    int nph;
    double phi[MDZ_MAX_PHASES], psi[MDZ_MAX_PHASES], C[MDZ_MAX_PHASES];
    double phi_end[MDZ_MAX_PHASES], psi_end[MDZ_MAX_PHASES], C_end[MDZ_MAX_PHASES];
    double pls_start[MDZ_MAX_PHASES], pls_end[MDZ_MAX_PHASES];
    int phi_soft[MDZ_MAX_PHASES], psi_soft[MDZ_MAX_PHASES], coh_soft[MDZ_MAX_PHASES];
};

/* bins of family slot fam on axes a, or (fam = MDZ_FAM_QUARTER) of the
 * quarter cells of centroid axes a and vertex axes *v (needs start_cap[fam]
 * >= bins + 1 and tmp_bytes >= mdz_markers_sort_bytes); synchronises */
int mdz_markers_bin(MarkerDev &md, int fam, const NodeAxes &a, const NodeAxes *v, hipStream_t s);
size_t mdz_markers_sort_bytes(int n, int nodes);
void mdz_launch_p2mastah(const MarkerDev &md, int fam, const NodeAxes &a, int prop, int itp_stencil,
                         const P2GArgs &g, hipStream_t s);
void mdz_launch_interp_p2n(const MarkerDev &md, int fam, const NodeAxes &a, const P2GArgs &g, hipStream_t s);
void mdz_launch_cfd_nodes(int n, const double *strain, const double *perc, const int8_t *tag, int cells,
                          const SoftK &sk, double *fric, double *dil, double *C, hipStream_t s);

/* The marker store of a context: device markers, their bins, node axes and
 * node buffers of an Nx x Nz vertex grid (host side in mdz_markers.hip). */
struct MarkerStore;
int mdz_mstore_create(MarkerStore **out, int Nx, int Nz);
void mdz_mstore_destroy(MarkerStore *s);
void mdz_family_dims(int fam, int Nx, int Nz, int *nx, int *nz);
/* axes of family slot fam: the grid's coordinates of that family, or Xh / Zh when given */
int mdz_mstore_axes(MarkerStore *s, int fam, const grid *mesh, const double *Xh, const double *Zh, int periodic,
                    hipStream_t st, NodeAxes *a);
int mdz_mstore_upload(MarkerStore *s, const markers *m, const double *mval, int nph, hipStream_t st);
int mdz_mstore_values(MarkerStore *s, const double *mval, hipStream_t st);
int mdz_mstore_bin(MarkerStore *s, int fam, const NodeAxes &a, hipStream_t st);
/* phase fractions and strength parameters of centroids and vertices, 1-node
 * stencil, from the quarter cells' bins */
int mdz_mstore_step(MarkerStore *s, const NodeAxes &ac, const NodeAxes &av, const SoftK &sk, double *perc_n,
                    double *perc_s, const int8_t *BCp, const int8_t *BCg, double *fric_n, double *dil_n, double *C_n,
                    double *fric_s, double *dil_s, double *C_s, hipStream_t st);
void mdz_mstore_rebin(MarkerStore *s); /* the next binning of every family sorts again */
MarkerDev &mdz_mstore_dev(MarkerStore *s);
double *mdz_mstore_node_field(MarkerStore *s);
int8_t *mdz_mstore_node_types(MarkerStore *s);
double *mdz_mstore_phase_values(MarkerStore *s);
double *mdz_mstore_strain(MarkerStore *s, int cells);
SoftK mdz_soft_constants(const mat_prop *mt, int nph);
int mdz_mstore_cfd(MarkerStore *s, const NodeAxes &ac, const NodeAxes &av, int itp_stencil, const SoftK &sk,
                   const double *perc_n, const double *perc_s, const int8_t *BCp, const int8_t *BCg, double *fric_n,
                   double *dil_n, double *C_n, double *fric_s, double *dil_s, double *C_s, hipStream_t st);
