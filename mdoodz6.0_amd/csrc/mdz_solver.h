/*
 * mdz_solver.h -- device solve of the decoupled Stokes system of one Newton
 * iteration: the Powell-Hestenes iterations of KillerSolver
 * (Solvers.c:2226-2751) around the restarted GCR of kspgcr
 * (Solvers.c:100-227), preconditioned by a Cholesky factor of the penalised
 * momentum operator Jts = PC - B Dpen C (Solvers.c:2408-2480).
 *
 * Internal interface of mdz_solver.hip, used by the context and the
 * KillerSolver drop-in of mdz_api.hip.  Every pointer in SolverInput is a
 * device pointer.
 */
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/mdoodz_hot.h"

/* One CSR block as the solver reads it (row pointers Ic[neq + 1]). */
struct SolverCsr {
    int neq;
    const int *Ic, *J;
    const double *A;
};

struct SolverInput {
    int nu, np;                       /* momentum and continuity unknowns */
    SolverCsr A, B, C;                /* Picard blocks (preconditioner; C also in Js) */
    SolverCsr AJ, BJ, CJ;             /* Jacobian blocks (Js, residuals, pressure update) */
    const double *Dpen, *D1, *incomp; /* per continuity row: Dcm0, D1cm0, whos_incompressible */
    const double *bu, *bp;            /* right-hand sides */
    int pc_type;                      /* PC = A (0) or (AJ + AJ^T) / 2 (1), as ordered */
    double rel_tol_KSP, abs_tol_div, rel_tol_div;
    int noisy; /* 1: one line per Powell-Hestenes iteration on stdout, as the reference prints */
};

struct MdzSolver;

int  mdz_solver_create(MdzSolver **out, hipStream_t s);
void mdz_solver_destroy(MdzSolver *sv);

/* Host pattern of one block (row pointers and column indices). */
struct SolverPattern {
    const int *Ic, *J;
};

/* Analysis of the factor from the node of each momentum row (u node
 * k + l Nx, v node Nx (Nz + 1) + k + l (Nx + 1)), and the patterns of Jts and Js, from the host patterns of the Picard A, B, C and
 * Jacobian A, B blocks, for the preconditioner pc_type (0: PC = A; 1:
 * PC = (AJ + AJ^T) / 2); nb (0, or a multiple of 64) is
 * checked and reported only: the factor's tiles do not depend on it.  Kept
 * until the next call. */
int mdz_solver_order(MdzSolver *sv, int Nx, int Nz, int nu, int np, const int *mom_node, const SolverPattern &A,
                     const SolverPattern &B, const SolverPattern &C, const SolverPattern &AJ, const SolverPattern &BJ,
                     int pc_type, int nb);

/* Factorisation and iterations; du[nu], dp[np] are device outputs. */
int mdz_solver_solve(MdzSolver *sv, const SolverInput &in, double *du, double *dp, mdz_solve_info *info);

/* Per continuity row diagonals of KillerSolver (Solvers.c:2278-2297) from
 * the centroid of each row: Dpen = penalty / celvol, D1 = 0, incomp = 1
 * for incompressible cells; D1 = bet_n / dt celvol d^2, Dpen = 1 / D1,
 * incomp = 0 for compressible ones (comp_cells = 1).  d may be null (1). */
void mdz_solver_pdiag(int np, const int *cont_node, const int *comp_cells, const double *bet_n, const double *d,
                      double penalty, double celvol, double dt, double *Dpen, double *D1, double *incomp,
                      hipStream_t s);
