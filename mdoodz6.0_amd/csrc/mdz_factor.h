/*
 * mdz_factor.h -- sparse Cholesky factor of the penalised momentum operator
 * on the staggered grid, by nested dissection (internal interface of
 * mdz_factor.hip, used by mdz_solver.hip).
 */
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

struct MdzFactor;

int  mdz_factor_create(MdzFactor **out, hipStream_t s);
void mdz_factor_destroy(MdzFactor *F);

/* Elimination tree and layout of the factor, from the node of each unknown
 * (u node k + l Nx, v node Nx (Nz + 1) + k + l (Nx + 1)) and the matrix's
 * pattern: every entry the numeric phase will place has to be in it.  Kept
 * until the next call. */
int mdz_factor_analyse(MdzFactor *F, int Nx, int Nz, int n, const int *mom_node, const std::vector<int> &Ic,
                       const std::vector<int> &J);

/* Numeric factor of the symmetric matrix whose lower triangle (column <=
 * row, equation order) is that of the pattern (Ic, J), given on the device in
 * slices of 64 rows (entry e of row i at base[i / 64] + 64 e + i % 64, row
 * lengths from Ic); *bad = an
 * equation whose pivot is not positive, or -1.  Synchronises. */
int mdz_factor_numeric(MdzFactor *F, const int *base, const int *Ic, const int *J, const double *val, int *bad);

/* x = (L L^T)^-1 f in equation order, on device vectors; enqueues only */
void mdz_factor_apply(MdzFactor *F, const double *f, double *x);

/* changes whenever the launches of mdz_factor_apply do */
unsigned long long mdz_factor_version(const MdzFactor *F);
