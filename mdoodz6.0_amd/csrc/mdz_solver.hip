/*
 * mdz_solver.hip -- device solve of the decoupled Stokes system of one Newton
 * iteration (gfx950): the Powell-Hestenes iterations of KillerSolver
 * (Solvers.c:2226-2751) around the restarted GCR of kspgcr
 * (Solvers.c:100-227), preconditioned by a Cholesky factor of the penalised
 * momentum operator Jts = PC - B Dpen C (Solvers.c:2408-2480).
 *
 * Steps kept as the reference takes them: PC = A (pc_type 0) or
 * (AJ + AJ^T) / 2 (pc_type 1, Solvers.c:2398-2409); the factor is that
 * of the symmetric matrix whose lower triangle (row >= column in equation
 * order) is the lower triangle of Jts (cholmod_copy with stype -1,
 * Solvers.c:2459); the GCR operator is the assembled Js = AJ - BJ Dpen C
 * (Solvers.c:2427); GCR restarts every 25 directions, takes
 * at most 1000 iterations and stops at |f| < rel_tol_KSP |f0|; its
 * orthogonalisation subtracts val[0..i1] (val[i1] holding the value of the
 * previous cycle, Solvers.c:164-168); the Powell-Hestenes loop takes at most
 * 20 iterations with the reference's stopping test on the signed maxima of
 * the residuals (Solvers.c:2536-2560).
 *
 * MI355X design:
 *  - the factor replaces CHOLMOD's supernodal one by a sparse Cholesky on
 *    the matrix cores (mdz_factor.hip);
 *  - Jts and Js are assembled once per solve, by one value function on
 *    patterns built with the ordering: their penalty entries are about
 *    penalty / celvol times larger than the viscous ones, and a
 *    matrix-free Js (AJ s - BJ Dpen C s) rounds differently from the
 *    factor's matrix by more than GCR's tolerance (it stalls at the noise
 *    floor), while the assembled pair matches to the last bit where the
 *    Jacobian equals the Picard operator;
 *  - dot products and maxima reduce through fixed per-block slots in a
 *    fixed order (results independent of scheduling).
 */
#include <hip/hip_runtime.h>

#include <limits.h>
#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <chrono>
#include <mutex>
#include <new>
#include <vector>

#include "mdz_factor.h"
#include "mdz_host_parallel.h"
#include "mdz_solver.h"

int mdz_error(int code, const char *msg);

#define SV_RESTART 25
#define SV_MAXIT 1000
#define SV_NITMAX 20
#define SV_NB_DEFAULT 1024
#define SV_RED 512 /* blocks of the reduction kernels (fixed: deterministic sums) */
#define SV_BLK 256

static inline int mdz_div_up_sv(long long a, int b) { return (int)((a + b - 1) / b); }

static int sv_err(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));
static int sv_err(int code, const char *fmt, ...) {
    char buf[400];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    return mdz_error(code, buf);
}

#define SVHIP(x)                                                                                   \
    do {                                                                                           \
        hipError_t _e = (x);                                                                       \
        if (_e != hipSuccess) return sv_err(MDZ_EHIP, "%s: %s", #x, hipGetErrorString(_e));        \
    } while (0)
/* A sparse matrix in slices of 64 rows: entry e of row i at base[i / 64] +
 * 64 e + i % 64, so that a wave reads its rows' e-th entries side by side;
 * a slice is as wide as its longest row, rounded up to eight, and a shorter
 * row is padded with zeros at column i. */
struct SliceView {
    const int *base, *Ic, *J;
    double *A;
};
struct SlicedRows {
    int *base = nullptr, *Ic = nullptr, *J = nullptr;
    double *A = nullptr;
    int width = 0; /* of the widest slice */
    SliceView view() const { return SliceView{base, Ic, J, A}; }
};

struct MdzSolver {
    hipStream_t s = nullptr;
    int n = 0, np = 0, kd = 0, nb = 0, nequ = 0;
    MdzFactor *fac = nullptr; /* factor of Jts */
    bool ordered = false;
    /* patterns of Jts = A - B Dpen C and Js = AJ - BJ Dpen C (unique sorted
     * columns per row), their values */
    SlicedRows ts, js;
    /* pc_type 1: AJ's transpose (row i: the entries of AJ's column i, their rows) */
    int pc_type = 0;
    int *tr_Ic = nullptr, *tr_J = nullptr, *tr_src = nullptr;
    /* vectors */
    double *work = nullptr;
    size_t work_len = 0;
    double *udum, *f, *sv, *v, *fu, *pdum, *fp, *tc, *VV, *SS;
    size_t ldv = 0;
    /* captured preconditioner application (f -> sv), and what it was captured for */
    hipGraph_t pc_graph = nullptr;
    hipGraphExec_t pc_exec = nullptr;
    const void *pc_key[2] = {};
    unsigned long long pc_version = 0;
    double *partial = nullptr; /* SV_RED * 32 slots, twice */
    double *dscal = nullptr;   /* the orthogonalisation's dots of the last directions */
    double *hscal = nullptr;   /* pinned: sums the host reads, written by the device */
};

/* ------------------------------------------------------------------ */
/* reductions                                                           */
/* ------------------------------------------------------------------ */
__device__ __forceinline__ double wave_sum(double x) {
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    return x;
}
__device__ __forceinline__ double wave_max(double x) {
    for (int o = 32; o > 0; o >>= 1) x = fmax(x, __shfl_xor(x, o, 64));
    return x;
}

/* block (256 threads) sum / max of one value per thread, returned to thread 0 */
__device__ __forceinline__ double block_sum(double x, double *lds4) {
    x = wave_sum(x);
    const int w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) lds4[w] = x;
    __syncthreads();
    return (lds4[0] + lds4[1]) + (lds4[2] + lds4[3]);
}
__device__ __forceinline__ double block_max(double x, double *lds4) {
    x = wave_max(x);
    const int w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) lds4[w] = x;
    __syncthreads();
    return fmax(fmax(lds4[0], lds4[1]), fmax(lds4[2], lds4[3]));
}

/* out[q] = sum over the SV_RED slots partial[b * 32 + q], q < nq (the
 * maximum instead where bit q of max_mask is set) */
__global__ void __launch_bounds__(SV_BLK) k_final(const double *partial, int nq, int max_mask, double *out) {
    __shared__ double lds4[4];
    const int q = blockIdx.x;
    if (q >= nq) return;
    const bool is_max = (max_mask >> q) & 1;
    double x = is_max ? -INFINITY : 0.0;
    for (int b = threadIdx.x; b < SV_RED; b += SV_BLK) {
        const double p = partial[(size_t)b * 32 + q];
        x = is_max ? fmax(x, p) : x + p;
    }
    x = is_max ? block_max(x, lds4) : block_sum(x, lds4);
    if (threadIdx.x == 0) out[q] = x;
}

/* ------------------------------------------------------------------ */
/* the assembled operators                                              */
/* ------------------------------------------------------------------ */
struct CsrView {
    const int *Ic, *J;
    const double *A;
};
static CsrView view(const SolverCsr &c) { return CsrView{c.Ic, c.J, c.A}; }

/* Values of P - B Dpen C on its pattern (Ic, J; columns unique in a row):
 * the product terms B(i,k) (Dpen(k) C(k,j)) are summed first, in row order,
 * then P's entries are taken off and the sign flipped, so that the entry is
 * P(i,j) - sum_k B(i,k) Dpen(k) C(k,j) (Solvers.c:2421-2426, cs_add of PC
 * and -L1); with the transpose's pattern (TIc, TJ: row i lists the entries
 * Tsrc of P's column i, TJ their rows), P is (P + P^T) / 2 (pc_type 1,
 * Solvers.c:2404-2408, pscale = 1/2).  Jts and Js go through this one function: on a linear model
 * (AJ = A, BJ = B) they are the same numbers, and the factor of Jts is an
 * exact inverse of Js. */
template <bool LDS>
__global__ void __launch_bounds__(64) k_schur_values(int n, SliceView M, CsrView P, double pscale, const int *TIc,
                                                     const int *TJ, const int *Tsrc, CsrView B, CsrView C,
                                                     const double *Dpen) {
    extern __shared__ double sv_lds[];
    const int l = threadIdx.x, i = blockIdx.x * 64 + l;
    const int base = M.base[blockIdx.x], wide = (M.base[blockIdx.x + 1] - base) >> 6;
    /* the slice's columns and sums in LDS (they are searched and summed some
     * forty times a row); rows too wide for it work in place */
    double *val = LDS ? sv_lds : M.A + base;
    const int *col = M.J + base;
    if (LDS) {
        int *c = (int *)(sv_lds + wide * 64);
        for (int e = 0; e < wide; e++) c[e * 64 + l] = col[e * 64 + l];
        col = c;
    }
    for (int e = 0; e < wide; e++) val[e * 64 + l] = 0.0;
    if (i < n) {
        const int len = M.Ic[i + 1] - M.Ic[i];
        auto at = [&](int j) { /* the row's columns increase */
            int a = 0, b = len - 1;
            while (a < b) {
                const int m = (a + b) >> 1;
                if (col[m * 64 + l] < j) a = m + 1;
                else b = m;
            }
            return a * 64 + l;
        };
        for (int eb = B.Ic[i]; eb < B.Ic[i + 1]; eb++) {
            const int k = B.J[eb];
            const double bk = B.A[eb], dk = Dpen[k];
            for (int ec = C.Ic[k]; ec < C.Ic[k + 1]; ec++) {
                const int e = at(C.J[ec]);
                val[e] = val[e] + bk * (dk * C.A[ec]);
            }
        }
        for (int ep = P.Ic[i]; ep < P.Ic[i + 1]; ep++) {
            const int e = at(P.J[ep]);
            val[e] = val[e] - pscale * P.A[ep];
        }
        if (TIc) /* pc_type 1: the transpose's half, P(j, i) for the entries of column i */
            for (int et = TIc[i]; et < TIc[i + 1]; et++) {
                const int e = at(TJ[et]);
                val[e] = val[e] - pscale * P.A[Tsrc[et]];
            }
    }
    for (int e = 0; e < wide; e++) M.A[base + e * 64 + l] = -val[e * 64 + l];
}

/* columns of a sliced matrix from its CSR ones */
__global__ void __launch_bounds__(64) k_slice_columns(int n, const int *base, const int *Ic, const int *J, int *out) {
    const int l = threadIdx.x, i = blockIdx.x * 64 + l;
    const int b = base[blockIdx.x], wide = (base[blockIdx.x + 1] - b) >> 6;
    const int e0 = i < n ? Ic[i] : 0, len = i < n ? Ic[i + 1] - e0 : 0;
    for (int e = 0; e < wide; e++) out[b + e * 64 + l] = e < len ? J[e0 + e] : min(i, n - 1);
}

/* ------------------------------------------------------------------ */
/* sparse products and the iteration's vector steps                     */
/* ------------------------------------------------------------------ */
__device__ __forceinline__ double row_dot(const CsrView &M, int i, const double *x) {
    double s = 0.0;
    for (int e = M.Ic[i]; e < M.Ic[i + 1]; e++) s += M.A[e] * x[M.J[e]];
    return s;
}

/* the same of a sliced matrix */
__device__ __forceinline__ double slice_dot(const SliceView &M, int i, const double *x) {
    const int b = M.base[i >> 6], w = M.base[(i >> 6) + 1] - b;
    const int *J = M.J + b + (i & 63);
    const double *A = M.A + b + (i & 63);
    double s = 0.0;
    for (int e = 0; e < w; e += 512) { /* (widths are multiples of eight) */
        double p[8];
#pragma unroll
        for (int u = 0; u < 8; u++) p[u] = A[e + 64 * u] * x[J[e + 64 * u]];
#pragma unroll
        for (int u = 0; u < 8; u++) s += p[u];
    }
    return s;
}

/* row i of M x by the 8 lanes of a group, the sum in every lane */
__device__ __forceinline__ double group_dot(const CsrView &M, int i, int g, const double *x) {
    double s = 0.0;
    for (int e = M.Ic[i] + g; e < M.Ic[i + 1]; e += 8) s += M.A[e] * x[M.J[e]];
    for (int o = 4; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    return s;
}

/* b - row i of M x with products and sums carried in two doubles (the error
 * of each is exact: Ogita, Rump and Oishi 2005, Dot2).  The penalty entries
 * make a residual the difference of terms about 1e5 times larger, whose
 * rounding the soft modes amplify: in plain doubles it is what bounds the
 * correction's accuracy.  The rows are read at memory speed either way. */
struct TwoSum {
    double s, c = 0.0;
    __device__ __forceinline__ void sub(double a, double y) { /* s - a y */
        const double p = -a * y, q = __builtin_fma(-a, y, -p);
        const double t = s + p, z = t - s;
        c += ((s - (t - z)) + (p - z)) + q;
        s = t;
    }
};

__device__ __forceinline__ double row_residual(const CsrView &M, int i, const double *x, double b) {
    TwoSum r{b};
    for (int e = M.Ic[i]; e < M.Ic[i + 1]; e++) r.sub(M.A[e], x[M.J[e]]);
    return r.s + r.c;
}

/* out = b - M x, slot 0: its sum of squares */
__global__ void __launch_bounds__(SV_BLK) k_slice_residual(int n, SliceView M, const double *x, const double *b,
                                                           double *out, double *partial) {
    __shared__ double lds4[4];
    double ss = 0.0;
    for (int i = blockIdx.x * SV_BLK + threadIdx.x; i < n; i += SV_RED * SV_BLK) {
        const int e0 = M.base[i >> 6], w = M.base[(i >> 6) + 1] - e0;
        TwoSum r{b[i]};
        for (int e = e0 + (i & 63); e < e0 + w; e += 64) r.sub(M.A[e], x[M.J[e]]);
        const double f = r.s + r.c;
        out[i] = f;
        ss += f * f;
    }
    ss = block_sum(ss, lds4);
    if (threadIdx.x == 0) partial[(size_t)blockIdx.x * 32] = ss;
}

/* udum = (bu - BJ (Dpen bp)) - BJ (incomp dp)  (Solvers.c:2510-2516) */
__global__ void __launch_bounds__(SV_BLK) k_ph_udum(int n, CsrView BJ, const double *bu, const double *bp,
                                                    const double *dp, const double *Dpen, const double *incomp,
                                                    double *udum) {
    const int i = blockIdx.x * SV_BLK + threadIdx.x;
    if (i >= n) return;
    double s1 = 0.0, s2 = 0.0;
    for (int e = BJ.Ic[i]; e < BJ.Ic[i + 1]; e++) {
        const int k = BJ.J[e];
        s1 += BJ.A[e] * (Dpen[k] * bp[k]);
        s2 += BJ.A[e] * (incomp[k] * dp[k]);
    }
    udum[i] = (bu[i] - s1) - s2;
}

/* dp += Dpen ((bp - CJ du) - D1 dp)  (Solvers.c:2523-2526) */
__global__ void __launch_bounds__(SV_BLK) k_ph_dp(int np, CsrView CJ, const double *bp, const double *du,
                                                  const double *D1, const double *Dpen, double *dp) {
    const int k = blockIdx.x * SV_BLK + threadIdx.x;
    if (k >= np) return;
    const double pd = row_residual(CJ, k, du, bp[k]) - D1[k] * dp[k];
    dp[k] = Dpen[k] * pd + dp[k];
}

/* fu = (bu - AJ du) - BJ dp (8 lanes a row), with per-block maxima (slot 0) and the sums of
 * squares over u and v equations (slots 1, 2) */
__global__ void __launch_bounds__(SV_BLK) k_res_mom(int n, int nequ, CsrView AJ, CsrView BJ, const double *bu,
                                                    const double *du, const double *dp, double *fu, double *partial) {
    __shared__ double lds4[4];
    double mx = -INFINITY, su = 0.0, sv = 0.0;
    const int g = threadIdx.x & 7;
    for (int i = (blockIdx.x * SV_BLK + threadIdx.x) >> 3; i < n; i += SV_RED * SV_BLK / 8) {
        const double f = (bu[i] - group_dot(AJ, i, g, du)) - group_dot(BJ, i, g, dp);
        if (g == 0) {
            fu[i] = f;
            mx = fmax(mx, f);
            if (i < nequ) su += f * f;
            else sv += f * f;
        }
    }
    mx = block_max(mx, lds4);
    su = block_sum(su, lds4);
    sv = block_sum(sv, lds4);
    if (threadIdx.x == 0) {
        partial[(size_t)blockIdx.x * 32 + 0] = mx;
        partial[(size_t)blockIdx.x * 32 + 1] = su;
        partial[(size_t)blockIdx.x * 32 + 2] = sv;
    }
}

/* fp = (bp - CJ du) - D1 dp, with per-block maxima (slot 3) and sums of
 * squares (slot 4) */
__global__ void __launch_bounds__(SV_BLK) k_res_cont(int np, CsrView CJ, const double *bp, const double *du,
                                                     const double *D1, const double *dp, double *fp, double *partial) {
    __shared__ double lds4[4];
    double mx = -INFINITY, sp = 0.0;
    for (int k = blockIdx.x * SV_BLK + threadIdx.x; k < np; k += SV_RED * SV_BLK) {
        const double f = (bp[k] - row_dot(CJ, k, du)) - D1[k] * dp[k];
        fp[k] = f;
        mx = fmax(mx, f);
        sp += f * f;
    }
    mx = block_max(mx, lds4);
    sp = block_sum(sp, lds4);
    if (threadIdx.x == 0) {
        partial[(size_t)blockIdx.x * 32 + 3] = mx;
        partial[(size_t)blockIdx.x * 32 + 4] = sp;
    }
}

/* sum of one row of SV_RED slots, by a wave (in every lane) */
__device__ __forceinline__ double slots_sum(const double *row) {
    double x = 0.0;
#pragma unroll
    for (int b = 0; b < SV_RED; b += 64) x += row[b + (threadIdx.x & 63)];
    return wave_sum(x);
}

/* A GCR direction after the preconditioner is three launches, each taking
 * the sums that the one before left per block (every block adds them again,
 * in the same order: a few KB from L2, less than a launch to do it once).
 * At 257 x 129 cells these and the norm's take 27 us a direction, against 50
 * for nine launches on CSR rows and a copy of the norm (the product alone 13
 * for 16, at 513 x 257 cells 18 for 168: one lane a row of CSR reads lines
 * of 64 rows for each entry).
 *
 * v = Js s; row q of dots: v . VV[q], q < nq */
__global__ void __launch_bounds__(SV_BLK) k_gcr_product(int n, SliceView M, const double *s, const double *VV,
                                                        size_t ldv, int nq, double *v, double *dots) {
    __shared__ double lds[SV_RESTART][4];
    double acc[SV_RESTART];
#pragma unroll
    for (int q = 0; q < SV_RESTART; q++) acc[q] = 0.0;
    for (int i = blockIdx.x * SV_BLK + threadIdx.x; i < n; i += SV_RED * SV_BLK) {
        const double vi = slice_dot(M, i, s);
        v[i] = vi;
#pragma unroll
        for (int q = 0; q < SV_RESTART; q++)
            if (q < nq) acc[q] += vi * VV[q * ldv + i];
    }
    const int w = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < SV_RESTART; q++) {
        if (q < nq) {
            const double x = wave_sum(acc[q]);
            if ((threadIdx.x & 63) == 0) lds[q][w] = x;
        }
    }
    __syncthreads();
    if (threadIdx.x < nq) {
        const int q = threadIdx.x;
        dots[q * SV_RED + blockIdx.x] = (lds[q][0] + lds[q][1]) + (lds[q][2] + lds[q][3]);
    }
}

/* v -= sum_q val[q] VV[q] and s -= sum_q val[q] SS[q], one term after the
 * other (Solvers.c:164-168): val[q] = v . VV[q] for q < i1, and from the
 * second cycle on val[i1] of the cycle before -- but for the last direction
 * of a cycle, whose val is set in none (0 in the reference, never written
 * here); rows 0, 1 of fv: f . v, v . v */
__global__ void __launch_bounds__(SV_BLK) k_gcr_orth(int n, int i1, int cycle, const double *dots, double *val,
                                                     const double *VV, const double *SS, size_t ldv, const double *f,
                                                     double *v, double *s, double *fv) {
    __shared__ double sval[SV_RESTART], lds4[4];
    const int w = threadIdx.x >> 6, nq = i1 + (cycle > 0 && i1 < SV_RESTART - 1);
    for (int q = w; q < nq; q += 4) {
        const double x = q < i1 ? slots_sum(dots + q * SV_RED) : val[q];
        if ((threadIdx.x & 63) == 0) {
            sval[q] = x;
            if (blockIdx.x == 0 && q < i1) val[q] = x;
        }
    }
    __syncthreads();
    double a = 0.0, b = 0.0;
    for (int i = blockIdx.x * SV_BLK + threadIdx.x; i < n; i += SV_RED * SV_BLK) {
        double vi = v[i], si = s[i];
        for (int q = 0; q < nq; q++) {
            const double fact = -sval[q];
            vi = vi + fact * VV[q * ldv + i];
            si = si + fact * SS[q * ldv + i];
        }
        v[i] = vi;
        s[i] = si;
        a += f[i] * vi;
        b += vi * vi;
    }
    a = block_sum(a, lds4);
    b = block_sum(b, lds4);
    if (threadIdx.x == 0) {
        fv[blockIdx.x] = a;
        fv[SV_RED + blockIdx.x] = b;
    }
}

/* Solvers.c:170-182: v, s scaled by 1 / |v| are direction i1 (VVq, SSq), x
 * += (f.v / |v|) s, f -= (f.v / |v|) v; slot 0: sum of squares of the new f */
__global__ void __launch_bounds__(SV_BLK) k_gcr_update(int n, const double *fv, const double *v, const double *s,
                                                       double *x, double *f, double *VVq, double *SSq,
                                                       double *partial) {
    __shared__ double lds4[4];
    const double nrm = sqrt(slots_sum(fv + SV_RED));
    const double rdv = slots_sum(fv) / nrm, fact = 1.0 / nrm;
    double ss = 0.0;
    for (int i = blockIdx.x * SV_BLK + threadIdx.x; i < n; i += SV_RED * SV_BLK) {
        const double vi = v[i] * fact, si = s[i] * fact;
        VVq[i] = vi;
        SSq[i] = si;
        x[i] = x[i] + rdv * si;
        const double fi = f[i] + (-rdv) * vi;
        f[i] = fi;
        ss += fi * fi;
    }
    ss = block_sum(ss, lds4);
    if (threadIdx.x == 0) partial[(size_t)blockIdx.x * 32] = ss;
}

__global__ void k_pdiag(int np, const int *cont_node, const int *comp_cells, const double *bet_n, const double *d,
                        double penalty, double celvol, double dt, double *Dpen, double *D1, double *incomp) {
    const int k = blockIdx.x * SV_BLK + threadIdx.x;
    if (k >= np) return;
    const int c = cont_node[k];
    const int comp = comp_cells ? comp_cells[c] : 0;
    const double dk = d ? d[k] : 1.0;
    double d1 = 1.0, dp = 1.0, inc = 1.0; /* identity where comp_cells is neither 0 nor 1 */
    if (comp == 0) {
        d1 = 0.0;
        dp = penalty;
    } else if (comp == 1) {
        d1 = bet_n[c] / dt * celvol * dk * dk;
        dp = 1.0 / d1;
        inc = 0.0;
    }
    D1[k] = d1;
    Dpen[k] = dp;
    incomp[k] = inc;
}

void mdz_solver_pdiag(int np, const int *cont_node, const int *comp_cells, const double *bet_n, const double *d,
                      double penalty, double celvol, double dt, double *Dpen, double *D1, double *incomp,
                      hipStream_t s) {
    if (np <= 0) return;
    hipLaunchKernelGGL(k_pdiag, dim3(mdz_div_up_sv(np, SV_BLK)), dim3(SV_BLK), 0, s, np, cont_node, comp_cells, bet_n,
                       d, penalty / celvol, celvol, dt, Dpen, D1, incomp);
}

/* ------------------------------------------------------------------ */
/* host side                                                            */
/* ------------------------------------------------------------------ */
int mdz_solver_create(MdzSolver **out, hipStream_t s) {
    if (!out) return sv_err(MDZ_EINVAL, "solver: null output");
    MdzSolver *S = new (std::nothrow) MdzSolver();
    if (!S) return sv_err(MDZ_ENOMEM, "solver: host memory");
    S->s = s;
    const int rc = mdz_factor_create(&S->fac, s);
    if (rc) {
        delete S;
        return rc;
    }
    hipError_t e = hipMalloc((void **)&S->partial, 2 * (size_t)SV_RED * 32 * sizeof(double));
    if (e == hipSuccess) e = hipMalloc((void **)&S->dscal, 128 * sizeof(double));
    if (e == hipSuccess) e = hipHostMalloc((void **)&S->hscal, 128 * sizeof(double), hipHostMallocDefault);
    if (e != hipSuccess) {
        mdz_solver_destroy(S);
        return sv_err(MDZ_ENOMEM, "solver scalars: %s", hipGetErrorString(e));
    }
    *out = S;
    return MDZ_OK;
}

static void free_rows(SlicedRows &m) {
    hipFree(m.base); hipFree(m.Ic); hipFree(m.J); hipFree(m.A);
    m = SlicedRows();
}

void mdz_solver_destroy(MdzSolver *S) {
    if (!S) return;
    if (S->s) hipStreamSynchronize(S->s);
    if (S->pc_exec) hipGraphExecDestroy(S->pc_exec);
    if (S->pc_graph) hipGraphDestroy(S->pc_graph);
    mdz_factor_destroy(S->fac);
    hipFree(S->work); hipFree(S->partial); hipFree(S->dscal);
    free_rows(S->ts);
    free_rows(S->js);
    hipFree(S->tr_Ic); hipFree(S->tr_J); hipFree(S->tr_src);
    if (S->hscal) hipHostFree(S->hscal);
    delete S;
}

/* Band position of each momentum equation for one ordering: x-columns
 * (v column k before u column k, z inside a column) or z-rows (u row l
 * before v row l, x inside a row); keys are distinct, so one pass over a
 * key table sorts them. */
static void band_order(int Nx, int Nz, int n, const int *mom_node, bool by_x, std::vector<int> &pos) {
    const long long nun = (long long)Nx * (Nz + 1);
    const long long K = by_x ? (2LL * (Nx + 1) + 2) * (Nz + 3) : (2LL * (Nz + 1) + 2) * (Nx + 3);
    std::vector<int> slot((size_t)K, -1);
    for (int i = 0; i < n; i++) {
        const long long node = mom_node[i];
        long long k, l, key;
        if (node < nun) {
            k = node % Nx; l = node / Nx;
            key = by_x ? (2 * k + 1) * (Nz + 3) + l : (2 * l) * (Nx + 3) + k;
        } else {
            const long long m = node - nun;
            k = m % (Nx + 1); l = m / (Nx + 1);
            key = by_x ? (2 * k) * (Nz + 3) + l : (2 * l + 1) * (Nx + 3) + k;
        }
        slot[(size_t)key] = i;
    }
    pos.assign(n, 0);
    int p = 0;
    for (long long q = 0; q < K; q++)
        if (slot[(size_t)q] >= 0) pos[slot[(size_t)q]] = p++;
}

/* Pattern of P - B C: per row the sorted unique columns of P's row and of
 * the C rows of the columns of B's row */
static void schur_pattern(int n, const int *Pi, const int *Pj, const int *Bi, const int *Bj, const int *Ci,
                          const int *Cj, std::vector<int> &Ic, std::vector<int> &J) {
    Ic.assign((size_t)n + 1, 0);
    std::mutex mu;
    std::vector<std::pair<long long, std::vector<int>>> part; /* (first row, columns of the chunk's rows) */
    mdz_host_parallel(n, 8192, [&](long long i0, long long i1) {
        std::vector<int> out, row;
        for (long long i = i0; i < i1; i++) {
            row.clear();
            for (int e = Pi[i]; e < Pi[i + 1]; e++) row.push_back(Pj[e]);
            for (int eb = Bi[i]; eb < Bi[i + 1]; eb++) {
                const int k = Bj[eb];
                for (int ec = Ci[k]; ec < Ci[k + 1]; ec++) row.push_back(Cj[ec]);
            }
            std::sort(row.begin(), row.end());
            row.erase(std::unique(row.begin(), row.end()), row.end());
            out.insert(out.end(), row.begin(), row.end());
            Ic[(size_t)i + 1] = (int)row.size();
        }
        std::lock_guard<std::mutex> g(mu);
        part.emplace_back(i0, std::move(out));
    });
    for (int i = 0; i < n; i++) Ic[(size_t)i + 1] += Ic[i];
    J.resize((size_t)Ic[n]);
    mdz_host_parallel((long long)part.size(), 1, [&](long long q0, long long q1) {
        for (long long q = q0; q < q1; q++)
            std::copy(part[(size_t)q].second.begin(), part[(size_t)q].second.end(),
                      J.begin() + Ic[(size_t)part[(size_t)q].first]);
    });
}

/* largest |pos(i) - pos(j)| over a pattern */
static long long band_width(int n, const std::vector<int> &pos, const std::vector<int> &Ic, const std::vector<int> &J) {
    long long kd = 0;
    std::mutex mu;
    mdz_host_parallel(n, 20000, [&](long long i0, long long i1) {
        long long k = 0;
        for (long long i = i0; i < i1; i++)
            for (int e = Ic[(size_t)i]; e < Ic[(size_t)i + 1]; e++)
                k = std::max(k, std::llabs((long long)pos[(size_t)i] - pos[(size_t)J[(size_t)e]]));
        std::lock_guard<std::mutex> g(mu);
        kd = std::max(kd, k);
    });
    return kd;
}

static int upload_ints(int **d, const std::vector<int> &h) {
    hipFree(*d);
    *d = nullptr;
    SVHIP(hipMalloc((void **)d, std::max(h.size(), (size_t)1) * sizeof(int)));
    if (!h.empty()) SVHIP(hipMemcpy(*d, h.data(), h.size() * sizeof(int), hipMemcpyHostToDevice));
    return MDZ_OK;
}

/* slices of a CSR pattern, on the device */
static int slice_rows(SlicedRows &m, int n, const std::vector<int> &Ic, const std::vector<int> &J, hipStream_t s) {
    const int ns = mdz_div_up_sv(n, 64);
    std::vector<int> base((size_t)ns + 1, 0);
    long long at = 0;
    m.width = 0;
    for (int q = 0; q < ns; q++) {
        int w = 0;
        for (int i = 64 * q; i < std::min(n, 64 * q + 64); i++) w = std::max(w, Ic[(size_t)i + 1] - Ic[i]);
        w = (w + 7) & ~7;
        m.width = std::max(m.width, w);
        at += 64LL * w;
        if (at > INT_MAX) return sv_err(MDZ_EUNSUPPORTED, "solver: more than 2^31 matrix entries");
        base[(size_t)q + 1] = (int)at;
    }
    int *csr = nullptr, rc;
    hipFree(m.J); hipFree(m.A);
    m.J = nullptr;
    m.A = nullptr;
    if ((rc = upload_ints(&m.base, base)) || (rc = upload_ints(&m.Ic, Ic)) || (rc = upload_ints(&csr, J))) {
        hipFree(csr);
        return rc;
    }
    const size_t len = std::max<size_t>((size_t)at, 1);
    hipError_t e = hipMalloc((void **)&m.J, len * sizeof(int));
    if (e == hipSuccess) e = hipMalloc((void **)&m.A, len * sizeof(double));
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_slice_columns, dim3(ns), dim3(64), 0, s, n, (const int *)m.base, (const int *)m.Ic,
                           (const int *)csr, m.J);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(s);
    }
    hipFree(csr);
    if (e != hipSuccess)
        return sv_err(e == hipErrorOutOfMemory ? MDZ_ENOMEM : MDZ_EHIP, "solver rows: %s", hipGetErrorString(e));
    return MDZ_OK;
}

static int check_pattern(const SolverPattern &p, int nrow, int ncol, const char *name) {
    if (!p.Ic || !p.J) return sv_err(MDZ_EINVAL, "solver ordering: pattern %s missing", name);
    if (p.Ic[0] != 0) return sv_err(MDZ_EINVAL, "solver ordering: row pointers of %s", name);
    for (int i = 0; i < nrow; i++) {
        if (p.Ic[i + 1] < p.Ic[i]) return sv_err(MDZ_EINVAL, "solver ordering: row pointers of %s", name);
        for (int e = p.Ic[i]; e < p.Ic[i + 1]; e++)
            if (p.J[e] < 0 || p.J[e] >= ncol) return sv_err(MDZ_EINVAL, "solver ordering: column %d of %s", p.J[e], name);
    }
    return MDZ_OK;
}

static int order_system(MdzSolver *S, int Nx, int Nz, int nu, int np, const int *mom_node, const SolverPattern &A,
                        const SolverPattern &B, const SolverPattern &C, const SolverPattern &AJ,
                        const SolverPattern &BJ, int pc_type, int nb) {
    if (pc_type != 0 && pc_type != 1) return sv_err(MDZ_EUNSUPPORTED, "pc_type = %d", pc_type);
    if (!S || nu < 1 || np < 1 || !mom_node) return sv_err(MDZ_EINVAL, "solver ordering: bad arguments");
    int rc;
    if ((rc = check_pattern(A, nu, nu, "A")) || (rc = check_pattern(B, nu, np, "B")) ||
        (rc = check_pattern(C, np, nu, "C")) || (rc = check_pattern(AJ, nu, nu, "AJ")) ||
        (rc = check_pattern(BJ, nu, np, "BJ")))
        return rc;
    const long long nun = (long long)Nx * (Nz + 1), nvn = (long long)(Nx + 1) * Nz;
    int nequ = 0;
    for (int i = 0; i < nu; i++) {
        if (mom_node[i] < 0 || mom_node[i] >= nun + nvn) return sv_err(MDZ_EINVAL, "solver ordering: node %d", i);
        if (mom_node[i] < nun) nequ++;
    }
    std::vector<int> tsI, tsJ, jsI, jsJ, trI, trJ, trS;
    if (pc_type == 1) {
        /* AJ's transpose by counting sort on the columns; P = AJ with the
         * transpose's columns added to each row */
        const int nnz = AJ.Ic[nu];
        trI.assign((size_t)nu + 1, 0);
        for (int e = 0; e < nnz; e++) trI[(size_t)AJ.J[e] + 1]++;
        for (int i = 0; i < nu; i++) trI[(size_t)i + 1] += trI[i];
        trJ.resize((size_t)nnz);
        trS.resize((size_t)nnz);
        std::vector<int> fill(trI.begin(), trI.end() - 1);
        for (int r = 0; r < nu; r++)
            for (int e = AJ.Ic[r]; e < AJ.Ic[r + 1]; e++) {
                const int q = fill[AJ.J[e]]++;
                trJ[q] = r;
                trS[q] = e;
            }
        std::vector<int> uI((size_t)nu + 1, 0), uJ;
        for (int i = 0; i < nu; i++) {
            for (int e = AJ.Ic[i]; e < AJ.Ic[i + 1]; e++) uJ.push_back(AJ.J[e]);
            for (int q = trI[i]; q < trI[(size_t)i + 1]; q++) uJ.push_back(trJ[q]);
            uI[(size_t)i + 1] = (int)uJ.size();
        }
        schur_pattern(nu, uI.data(), uJ.data(), B.Ic, B.J, C.Ic, C.J, tsI, tsJ);
    } else {
        schur_pattern(nu, A.Ic, A.J, B.Ic, B.J, C.Ic, C.J, tsI, tsJ);
    }
    schur_pattern(nu, AJ.Ic, AJ.J, BJ.Ic, BJ.J, C.Ic, C.J, jsI, jsJ);
    std::vector<int> px, pz;
    band_order(Nx, Nz, nu, mom_node, true, px);
    band_order(Nx, Nz, nu, mom_node, false, pz);
    const long long kx = band_width(nu, px, tsI, tsJ), kz = band_width(nu, pz, tsI, tsJ);
    const long long kd = std::max(1LL, std::min(kx, kz));
    if (nb <= 0) nb = SV_NB_DEFAULT;
    if (nb < 64 || nb % 64) return sv_err(MDZ_EINVAL, "solver block size %d (a multiple of 64)", nb);
    S->ordered = false;
    if ((rc = mdz_factor_analyse(S->fac, Nx, Nz, nu, mom_node, tsI, tsJ)) ||
        (rc = slice_rows(S->ts, nu, tsI, tsJ, S->s)) || (rc = slice_rows(S->js, nu, jsI, jsJ, S->s)) ||
        (rc = upload_ints(&S->tr_Ic, trI)) || (rc = upload_ints(&S->tr_J, trJ)) || (rc = upload_ints(&S->tr_src, trS)))
        return rc;
    S->pc_type = pc_type;
    S->n = nu;
    S->np = np;
    S->nequ = nequ;
    S->kd = (int)kd;
    S->nb = nb;
    S->ordered = true;
    return MDZ_OK;
}

int mdz_solver_order(MdzSolver *S, int Nx, int Nz, int nu, int np, const int *mom_node, const SolverPattern &A,
                     const SolverPattern &B, const SolverPattern &C, const SolverPattern &AJ, const SolverPattern &BJ,
                     int pc_type, int nb) {
    try {
        return order_system(S, Nx, Nz, nu, np, mom_node, A, B, C, AJ, BJ, pc_type, nb);
    } catch (const std::exception &e) {
        return sv_err(MDZ_ENOMEM, "solver ordering: %s", e.what());
    }
}

static int ensure_buffers(MdzSolver *S) {
    const size_t n = S->n, np = S->np > 0 ? S->np : 1;
    const size_t ldv = (n + 63) & ~(size_t)63, ldp = (np + 63) & ~(size_t)63;
    const size_t work_len = 5 * ldv + 3 * ldp + 2 * SV_RESTART * ldv;
    if (S->work_len != work_len) {
        hipFree(S->work); S->work = nullptr; S->work_len = 0;
        SVHIP(hipMalloc((void **)&S->work, work_len * sizeof(double)));
        S->work_len = work_len;
    }
    double *w = S->work;
    S->ldv = ldv;
    S->udum = w; S->f = w + ldv; S->sv = w + 2 * ldv; S->v = w + 3 * ldv; S->fu = w + 4 * ldv;
    S->pdum = w + 5 * ldv; S->fp = S->pdum + ldp; S->tc = S->fp + ldp;
    S->VV = S->tc + ldp; S->SS = S->VV + SV_RESTART * ldv;
    return MDZ_OK;
}

/* slots of the pinned scalars */
enum { SC_NORM = 0, SC_RES = 8 };

/* the scalars of the launches so far */
static int wait_scalars(MdzSolver *S) {
    SVHIP(hipGetLastError());
    SVHIP(hipStreamSynchronize(S->s));
    return MDZ_OK;
}

/* values of a sliced P - B Dpen C */
static void schur_values(const SlicedRows &m, int n, const CsrView &P, double pscale, const int *TIc, const int *TJ,
                         const int *Tsrc, const CsrView &B, const CsrView &C, const double *Dpen, hipStream_t s) {
    const dim3 grid(mdz_div_up_sv(n, 64)), blk(64);
    const size_t lds = (size_t)m.width * 64 * (sizeof(double) + sizeof(int));
    if (lds <= 64 * 1024)
        hipLaunchKernelGGL(k_schur_values<true>, grid, blk, lds, s, n, m.view(), P, pscale, TIc, TJ, Tsrc, B, C, Dpen);
    else
        hipLaunchKernelGGL(k_schur_values<false>, grid, blk, 0, s, n, m.view(), P, pscale, TIc, TJ, Tsrc, B, C, Dpen);
}

static int factorise(MdzSolver *S, const SolverInput &in) {
    const bool sym = S->pc_type == 1;
    schur_values(S->ts, S->n, view(sym ? in.AJ : in.A), sym ? 0.5 : 1.0, sym ? S->tr_Ic : nullptr, S->tr_J, S->tr_src,
                 view(in.B), view(in.C), in.Dpen, S->s);
    schur_values(S->js, S->n, view(in.AJ), 1.0, nullptr, nullptr, nullptr, view(in.BJ), view(in.C), in.Dpen, S->s);
    SVHIP(hipGetLastError());
    int bad = -1;
    const int rc = mdz_factor_numeric(S->fac, S->ts.base, S->ts.Ic, S->ts.J, S->ts.A, &bad);
    if (rc) return rc;
    if (bad >= 0)
        return sv_err(MDZ_ESOLVE, "Cholesky factor of Jts: the pivot of momentum equation %d is not positive", bad);
    return MDZ_OK;
}

/* sv = Jts^-1 f as one graph launch (two launches per level of the
 * elimination tree); captured again when the factor's layout changes */
static int run_precondition(MdzSolver *S) {
    /* MDZ_SOLVER_GRAPH=0 launches the same kernels one by one (for tracing
     * tools that do not follow graph launches) */
    static const int use_graph = [] {
        const char *e = getenv("MDZ_SOLVER_GRAPH");
        return e && e[0] == '0' ? 0 : 1;
    }();
    if (!use_graph) {
        mdz_factor_apply(S->fac, S->f, S->sv);
        return MDZ_OK;
    }
    const void *key[2] = {S->f, S->sv};
    const unsigned long long version = mdz_factor_version(S->fac);
    if (!S->pc_exec || memcmp(key, S->pc_key, sizeof(key)) || version != S->pc_version) {
        if (S->pc_exec) hipGraphExecDestroy(S->pc_exec);
        if (S->pc_graph) hipGraphDestroy(S->pc_graph);
        S->pc_exec = nullptr;
        S->pc_graph = nullptr;
        SVHIP(hipStreamBeginCapture(S->s, hipStreamCaptureModeThreadLocal));
        mdz_factor_apply(S->fac, S->f, S->sv);
        hipGraph_t g = nullptr;
        hipError_t e = hipStreamEndCapture(S->s, &g);
        if (e != hipSuccess) return sv_err(MDZ_EHIP, "preconditioner capture: %s", hipGetErrorString(e));
        S->pc_graph = g;
        SVHIP(hipGraphInstantiate(&S->pc_exec, g, nullptr, nullptr, 0));
        memcpy(S->pc_key, key, sizeof(key));
        S->pc_version = version;
    }
    SVHIP(hipGraphLaunch(S->pc_exec, S->s));
    return MDZ_OK;
}

static void final_sum(MdzSolver *S, int nq, int max_mask, int slot) {
    hipLaunchKernelGGL(k_final, dim3(nq), dim3(SV_BLK), 0, S->s, (const double *)S->partial, nq, max_mask,
                       S->hscal + slot);
}

/* kspgcr (Solvers.c:100-227) on x with right-hand side b */
static int kspgcr(MdzSolver *S, const SolverInput &in, const double *b, double *x, double eps, int *its_out) {
    const int noisy = in.noisy;
    const int n = S->n;
    hipStream_t s = S->s;
    const dim3 gR(SV_RED), blk(SV_BLK);
    double *dots = S->partial + (size_t)SV_RED * 32, *fv = dots + (size_t)SV_RED * 30;
    int rc;
    hipLaunchKernelGGL(k_slice_residual, gR, blk, 0, s, n, S->js.view(), (const double *)x, b, S->f, S->partial);
    final_sum(S, 1, 0, SC_NORM);
    if ((rc = wait_scalars(S))) return rc;
    double norm_r = sqrt(S->hscal[SC_NORM]);
    const double rnorm0 = norm_r;
    int its = 0, success = 0;
    if (!(rnorm0 > 0.0)) { /* nothing to reduce (the reference would divide 0 by 0 below) */
        *its_out = 0;
        return MDZ_OK;
    }
    for (int cycle = 0; !success && its < SV_MAXIT; cycle++) {
        for (int i1 = 0; i1 < SV_RESTART; i1++) {
            double *VVq = S->VV + (size_t)i1 * S->ldv, *SSq = S->SS + (size_t)i1 * S->ldv;
            if ((rc = run_precondition(S))) return rc;
            hipLaunchKernelGGL(k_gcr_product, gR, blk, 0, s, n, S->js.view(), (const double *)S->sv,
                               (const double *)S->VV, S->ldv, i1, S->v, dots);
            hipLaunchKernelGGL(k_gcr_orth, gR, blk, 0, s, n, i1, cycle, (const double *)dots, S->dscal,
                               (const double *)S->VV, (const double *)S->SS, S->ldv, (const double *)S->f, S->v, S->sv,
                               fv);
            hipLaunchKernelGGL(k_gcr_update, gR, blk, 0, s, n, (const double *)fv, (const double *)S->v,
                               (const double *)S->sv, x, S->f, VVq, SSq, S->partial);
            final_sum(S, 1, 0, SC_NORM);
            if ((rc = wait_scalars(S))) return rc;
            norm_r = sqrt(S->hscal[SC_NORM]);
            if (noisy > 1) {
                printf("[%1.4d] %1.4d KSP GCR Residual %1.12e %1.12e\n", its / (SV_RESTART + 1), its, norm_r,
                       norm_r / rnorm0);
                fflush(stdout);
            }
            if (norm_r < eps * rnorm0) {
                success = 1;
                break;
            }
            if (!(norm_r == norm_r)) return sv_err(MDZ_ENAN, "GCR residual is NaN at iteration %d", its);
            its++;
        }
        its++;
    }
    *its_out = its;
    return MDZ_OK;
}

/* fu, fp from du, dp; slots SC_RES + 0..4: max fu, sum fu^2 (u), sum fu^2
 * (v), max fp, sum fp^2 */
static int residuals(MdzSolver *S, const SolverInput &in, const double *du, const double *dp) {
    hipStream_t s = S->s;
    hipLaunchKernelGGL(k_res_mom, dim3(SV_RED), dim3(SV_BLK), 0, s, S->n, S->nequ, view(in.AJ), view(in.BJ), in.bu, du,
                       dp, S->fu, S->partial);
    if (S->np > 0)
        hipLaunchKernelGGL(k_res_cont, dim3(SV_RED), dim3(SV_BLK), 0, s, S->np, view(in.CJ), in.bp, du, in.D1, dp,
                           S->fp, S->partial);
    else
        return sv_err(MDZ_EINVAL, "solver: no continuity rows");
    final_sum(S, 5, (1 << 0) | (1 << 3), SC_RES);
    return wait_scalars(S);
}

int mdz_solver_solve(MdzSolver *S, const SolverInput &in, double *du, double *dp, mdz_solve_info *info) {
    if (!S || !S->ordered) return sv_err(MDZ_EINVAL, "solver: no ordering");
    if (in.nu != S->n || in.np != S->np) return sv_err(MDZ_EINVAL, "solver: ordering of another system");
    if (in.pc_type != S->pc_type)
        return sv_err(MDZ_EINVAL, "solver: ordering built for pc_type %d, solve asks for %d", S->pc_type, in.pc_type);
    int rc = ensure_buffers(S);
    if (rc) return rc;
    mdz_solve_info inf;
    memset(&inf, 0, sizeof(inf));
    inf.kd = S->kd;
    inf.nb = S->nb;
    const auto t0 = std::chrono::steady_clock::now();
    if ((rc = factorise(S, in))) return rc;
    const auto t1 = std::chrono::steady_clock::now();
    inf.factor_ms = std::chrono::duration<double, std::milli>(t1 - t0).count();

    hipStream_t s = S->s;
    SVHIP(hipMemsetAsync(du, 0, (size_t)S->n * sizeof(double), s));
    SVHIP(hipMemsetAsync(dp, 0, (size_t)S->np * sizeof(double), s));
    if ((rc = residuals(S, in, du, dp))) return rc;
    const double maxru0 = S->hscal[SC_RES];
    double maxdiv = 0.0, maxru = 0.0, maxdiv0 = 0.0;
    int k;
    for (k = 0; k < SV_NITMAX; k++) {
        hipLaunchKernelGGL(k_ph_udum, dim3(mdz_div_up_sv(S->n, SV_BLK)), dim3(SV_BLK), 0, s, S->n, view(in.BJ), in.bu,
                           in.bp, (const double *)dp, in.Dpen, in.incomp, S->udum);
        int its = 0;
        if ((rc = kspgcr(S, in, S->udum, du, in.rel_tol_KSP, &its))) return rc;
        inf.ksp_its[k] = its;
        inf.ksp_its_total += its;
        hipLaunchKernelGGL(k_ph_dp, dim3(mdz_div_up_sv(S->np, SV_BLK)), dim3(SV_BLK), 0, s, S->np, view(in.CJ), in.bp,
                           (const double *)du, in.D1, in.Dpen, dp);
        if ((rc = residuals(S, in, du, dp))) return rc;
        maxru = S->hscal[SC_RES];
        maxdiv = S->hscal[SC_RES + 3];
        if (k == 0) maxdiv0 = maxdiv;
        if (in.noisy > 0) {
            printf("PH comp it. %01d. its_KSP = %02d: max. cont. = %2.2e - rel. max. div. = %2.2e / max. mom. = %2.2e - "
                   "rel. max. mom. = %2.2e\n",
                   k, its, maxdiv, fabs(maxdiv / maxdiv0), maxru, maxru / maxru0);
            fflush(stdout);
        }
        if ((fabs(maxdiv) < in.abs_tol_div || maxdiv / maxdiv0 < in.rel_tol_div) &&
            (fabs(maxru) < in.abs_tol_div || maxru / maxru0 < in.rel_tol_div))
            break;
    }
    inf.ph_its = k < SV_NITMAX ? k + 1 : SV_NITMAX;
    inf.maxdiv0 = maxdiv0;
    inf.maxdiv = maxdiv;
    inf.maxru0 = maxru0;
    inf.maxru = maxru;
    /* Fu, Fv, Fp of the final residual (Solvers.c:2580-2610) */
    const int neqv = S->n - S->nequ;
    inf.resx = S->nequ > 0 ? sqrt(S->hscal[SC_RES + 1] / S->nequ) : 0.0;
    inf.resz = neqv > 0 ? sqrt(S->hscal[SC_RES + 2] / neqv) : 0.0;
    inf.resp = S->np > 0 ? sqrt(S->hscal[SC_RES + 4] / S->np) : 0.0;
    const auto t2 = std::chrono::steady_clock::now();
    inf.iterate_ms = std::chrono::duration<double, std::milli>(t2 - t1).count();
    if (info) *info = inf;
    if (fabs(maxdiv) > in.abs_tol_div && maxdiv / maxdiv0 > in.rel_tol_div)
        return sv_err(MDZ_ESOLVE,
                      "The code has exited since the incompressibility constrain was not satisfied to abs. tol. = "
                      "%2.2e and rel. tol. = %2.2e",
                      in.abs_tol_div, in.rel_tol_div);
    return MDZ_OK;
}
