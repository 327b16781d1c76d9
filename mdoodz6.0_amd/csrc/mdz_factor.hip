/*
 * mdz_factor.hip -- sparse Cholesky factor of the penalised momentum operator
 * Jts on the staggered grid (gfx950), in place of the supernodal CHOLMOD
 * factor of KillerSolver (Solvers.c:2459-2480).
 *
 * Ordering and layout: mdz_factor_plan.h.
 *
 * Numeric phase: one dense front per node (s own columns, b boundary rows),
 * level by level from the leaves, every node of a level in one launch.  The
 * fronts are cut into 64 x 64 tiles; a launch per 64-column panel forms the
 * panel's rows L = A Linv^T, takes their products off every trailing tile
 * (own columns and the b x b update matrix) on the FP64 matrix
 * instructions, and factors and inverts the next diagonal tile in the
 * workgroup that just finished it, so that the chain of a front is one
 * launch per panel.  A parent gathers its children's update matrices by
 * index maps; nothing is scattered and no sum depends on scheduling.
 *
 * Solves: the factor is kept as T = [L11^-1; L21 L11^-1] per node, so that
 * a level of the forward solve is y = T r and one of the backward solve
 * x = T^T (y, -x_boundary): one launch per level and direction, each a
 * stream over T with no substitution inside.
 *
 * Bound by the chain of dependent launches: 262 912 unknowns (513 x 257
 * cells) take 13 levels and about 50 launches to factor, 7.4 GFLOP and 0.29
 * GB of panels.  Measured there against the band Cholesky this replaced
 * (4100 library steps of 64 columns, 257 diagonal blocks one after the
 * other in a solve): factor 703 -> 4.4 ms, a GCR direction 5.6 -> 0.37 ms;
 * a solve at 257 x 129 cells (52 directions) 231 -> 10.4 ms.
 */
#include <limits.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <new>

#include "../../include/mdoodz_hot.h"
#include "mdz_factor.h"
#include "mdz_factor_plan.h"

#define ND_BLK 256
#define ND_CH 2048 /* entries of a vector staged in LDS at a time */

typedef double nd_d4 __attribute__((ext_vector_type(4)));

#define FCHK(x)                                                                                    \
    do {                                                                                           \
        hipError_t _e = (x);                                                                       \
        if (_e != hipSuccess) {                                                                    \
            char _b[256];                                                                          \
            snprintf(_b, sizeof(_b), "factor: %s: %s", #x, hipGetErrorString(_e));                 \
            return mdz_error(_e == hipErrorOutOfMemory ? MDZ_ENOMEM : MDZ_EHIP, _b);               \
        }                                                                                          \
    } while (0)

/* ------------------------------------------------------------------ */
/* numeric phase                                                        */
/* ------------------------------------------------------------------ */
__device__ __forceinline__ double nd_lane(double x, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), l),
                            __builtin_amdgcn_readlane(__double2loint(x), l));
}

/* LDS of the tile kernels: two 64 x 64 operands (column k of row r at
 * k 64 + (r ^ 16 (k & 1)): the two columns a half wave reads lie in
 * different banks), or the diagonal tile (65 doubles a column), its inverse
 * and the column buffers of its factorisation */
#define ND_DIAG (ND_T * (ND_T + 1))
#define ND_LDS (ND_DIAG + ND_T * ND_T + 640)
__device__ __forceinline__ int nd_sw(int k, int r) { return k * ND_T + (r ^ ((k & 1) << 4)); }

/* 1 / p and 1 / sqrt(p) of a positive normal p: the hardware's estimate and
 * two Newton steps (a divide or a square root is a chain twice as long) */
__device__ __forceinline__ double nd_rcp(double p) {
    double y = __builtin_amdgcn_rcp(p);
#pragma unroll
    for (int i = 0; i < 2; i++) y = __builtin_fma(y, __builtin_fma(-p, y, 1.0), y);
    return y;
}
__device__ __forceinline__ double nd_rsqrt(double p) {
    double y = __builtin_amdgcn_rsq(p);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const double e = __builtin_fma(-p * y, y, 1.0);
        y = __builtin_fma(y * e, __builtin_fma(0.375, e, 0.5), y);
    }
    return y;
}

/* Inverse of the Cholesky factor of the w x w lower triangle in S (LDS, 65
 * doubles a column; overwritten), written to out (64 x 64 column-major,
 * identity beyond w) and, where T is not null, to its place in a front;
 * called by a whole workgroup of 256 after a barrier.  Bound by the chain of
 * w columns.
 *
 * Elimination: lane = row, wave q holds columns 16 q .. 16 q + 15 in
 * registers.  Four columns a step: their owner eliminates among them
 * (pivots by readlane; unit-lower multipliers, no square root), passes them
 * through LDS, and after one barrier the waves take four rank-one terms off
 * the columns to the right.  The loop is rolled (straight-line steps run at
 * the pace of cold instruction fetches): the owner moves its columns down by
 * four, so that the step's are always the first four.
 *
 * Inverse: wave q inverts diagonal block q (16 x 16, lane = column), then a
 * barrier per block row and V(i, j) = -V(i, i) sum_k L(i, k) V(k, j) on the
 * matrix instructions, whose result registers are the second product's
 * operand as they are; rows are scaled by 1 / sqrt(pivot) on the way out.
 *
 * Measured for 64 columns: 22 us (with its launch); 33 with the inverse eliminated
 * along by readlane, 50 for 16-column blocks through LDS with six barriers
 * each. */
__device__ __forceinline__ void nd_potrf(double *S, int w, double *__restrict__ out, double *T, int ldt, int pos0,
                                         int *bad) {
    double *V = S + ND_DIAG, *buf = V + ND_T * ND_T;
    double *piv = buf; /* 64 pivots; then two buffers of four columns, each with 32 doubles more for the
                        * owner's reads past its sixteen */
    const int r = threadIdx.x & 63, q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nb = (w + 15) >> 4, W = nb << 4;
    double a[16];
    int fail = INT_MAX;
#pragma unroll
    for (int k = 0; k < 16; k++) {
        const int c = 16 * q + k;
        V[c * ND_T + r] = r == c ? 1.0 : 0.0;
        a[k] = r < w && c <= r ? S[c * 65 + r] : c < w ? 0.0 : r == c ? 1.0 : 0.0;
    }
#pragma unroll 1
    for (int j0 = 0; j0 < W; j0 += 4) {
        const int ow = j0 >> 4;
        double *B = buf + 64 + (j0 & 4) * 72;
        if (q == ow) { /* (its own columns of S: the other waves read theirs only) */
            double y[4];
#pragma unroll
            for (int t = 0; t < 4; t++) {
                double p = nd_lane(a[t], j0 + t);
                fail = p > 0.0 ? fail : min(fail, j0 + t);
                p = p > 0.0 ? p : 1.0;
                y[t] = nd_rcp(p);
                const double f = r > j0 + t ? a[t] * y[t] : 0.0;
                if (r == 0) piv[j0 + t] = p;
#pragma unroll
                for (int u = t + 1; u < 4; u++) a[u] = __builtin_fma(-f, nd_lane(a[t], j0 + u), a[u]);
                S[(j0 + t) * 65 + r] = f;
                B[t * 64 + r] = a[t];
            }
#pragma unroll
            for (int k = 0; k < 12; k++) a[k] = a[k + 4];
        }
        __syncthreads();
        if (q >= ow) { /* (the owner's last columns are past its sixteen: never used) */
            const double *Bc = B + (q == ow ? j0 + 4 : 16 * q);
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const double f = S[(j0 + t) * 65 + r];
                double b[16];
#pragma unroll
                for (int k = 0; k < 16; k++) b[k] = Bc[t * 64 + k];
                __builtin_amdgcn_sched_barrier(0); /* all reads in flight before the first use */
#pragma unroll
                for (int k = 0; k < 16; k++) a[k] = __builtin_fma(-f, b[k], a[k]);
            }
        }
    }
    if (fail < w && r == 0) atomicMin(bad, pos0 + fail);
    __syncthreads();
    const int li = r & 15, lk = r >> 4;
    if (q < nb) {
        double x[16];
#pragma unroll
        for (int i = 0; i < 16; i++) {
            double t = li == i ? 1.0 : 0.0;
#pragma unroll
            for (int k = 0; k < i; k++) t = __builtin_fma(-S[(16 * q + k) * 65 + 16 * q + i], x[k], t);
            x[i] = t;
        }
        if (lk == 0)
#pragma unroll
            for (int i = 0; i < 16; i++) V[(16 * q + li) * ND_T + 16 * q + i] = x[i];
    }
    for (int ib = 1; ib < nb; ib++) {
        __syncthreads();
        if (q >= ib) continue;
        nd_d4 g = {}, z = {};
        for (int kb = q; kb < ib; kb++)
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                const int k = 16 * kb + 4 * ks + lk;
                g = __builtin_amdgcn_mfma_f64_16x16x4f64(S[k * 65 + 16 * ib + li], V[(16 * q + li) * ND_T + k], g, 0, 0, 0);
            }
#pragma unroll
        for (int ks = 0; ks < 4; ks++)
            z = __builtin_amdgcn_mfma_f64_16x16x4f64(V[(16 * ib + 4 * ks + lk) * ND_T + 16 * ib + li], g[ks], z, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 4; v++) V[(16 * q + li) * ND_T + 16 * ib + 4 * v + lk] = -z[v];
    }
    __syncthreads();
    const double rs = r < w ? nd_rsqrt(piv[r]) : 1.0;
#pragma unroll
    for (int k = 0; k < 16; k++) {
        const int c = 16 * q + k;
        const double x = V[c * ND_T + r] * rs;
        out[c * ND_T + r] = x;
        if (T && r < w && c < w) T[(long long)c * ldt + r] = x;
    }
}

/* rows of a row tile: first row of the front and how many */
__device__ __forceinline__ void nd_tile(const NdNode &N, int t, int &r0, int &nr) {
    if (t < N.np) {
        r0 = t * ND_T;
        nr = min(ND_T, N.s - r0);
    } else {
        const int q = (t - N.np) * ND_T;
        r0 = N.s + q;
        nr = min(ND_T, N.b - q);
    }
}

/* the children's update entries of element (r, c) of a front, r >= c */
__device__ __forceinline__ double nd_children(const NdNode *__restrict__ nodes, const NdNode &N,
                                              const int *__restrict__ inv, const double *__restrict__ Uc, int r, int c) {
    double v = 0.0;
#pragma unroll
    for (int q = 0; q < 2; q++)
        if (N.child[q] >= 0) {
            const int ir = inv[N.inv[q] + r], ic = inv[N.inv[q] + c];
            if (ir >= 0 && ic >= 0) {
                const NdNode &K = nodes[N.child[q]];
                v += Uc[K.uoff + (long long)ic * K.ldu + ir];
            }
        }
    return v;
}

/* matrix entries to their places in the panels: one row of the lower
 * triangle per thread (one writer per element) */
__global__ void __launch_bounds__(ND_BLK) k_nd_scatter(int n, const int *__restrict__ base, const int *__restrict__ Ic,
                                                       const int *__restrict__ J, const double *__restrict__ val, const int *__restrict__ pos,
                                                       const int *__restrict__ node_of,
                                                       const NdNode *__restrict__ nodes,
                                                       const int *__restrict__ blist, double *__restrict__ P) {
    const int i = blockIdx.x * ND_BLK + threadIdx.x;
    if (i >= n) return;
    const int pi = pos[i], len = Ic[i + 1] - Ic[i];
    for (int q = 0; q < len; q++) {
        const int e = base[i >> 6] + 64 * q + (i & 63);
        const int j = J[e];
        if (j > i) continue;
        const int pj = pos[j], lo = min(pi, pj), hi = max(pi, pj);
        const NdNode N = nodes[node_of[lo]];
        int r = hi - N.ooff;
        if (r >= N.s) { /* a boundary row: its place in the sorted list (the analysis put it there) */
            int a = 0, b = N.b;
            while (a < b) {
                const int mid = (a + b) >> 1;
                if (blist[N.boff + mid] < hi) a = mid + 1;
                else b = mid;
            }
            if (a >= N.b || blist[N.boff + a] != hi) continue;
            r = N.s + a;
        }
        P[N.poff + (long long)(lo - N.ooff) * N.ld + r] = val[e];
    }
}

/* own-column tiles of a level: the children's entries are added; the first
 * diagonal tile is factored */
__global__ void __launch_bounds__(ND_BLK) k_nd_assemble(const NdTask *__restrict__ task,
                                                        const NdNode *__restrict__ nodes,
                                                        const int *__restrict__ inv, const double *__restrict__ Uc,
                                                        double *__restrict__ P, double *__restrict__ Lb,
                                                        double *__restrict__ Linv, int *bad) {
    __shared__ double sh[ND_LDS];
    const NdTask t = task[blockIdx.x];
    const NdNode N = nodes[t.node];
    int r0, nr;
    nd_tile(N, t.a, r0, nr);
    const int c0 = t.b * ND_T, nc = min(ND_T, N.s - c0);
    const bool diag = t.a == t.b, first = diag && t.a == 0;
    const int r = threadIdx.x & 63;
    for (int c = threadIdx.x >> 6; c < nc; c += 4) {
        if (r >= nr || (diag && r < c)) continue;
        double *p = P + N.poff + (long long)(c0 + c) * N.ld + r0 + r;
        const double v = *p + nd_children(nodes, N, inv, Uc, r0 + r, c0 + c);
        if (first) sh[c * 65 + r] = v;
        else *p = v;
    }
    if (!first) return;
    __syncthreads();
    nd_potrf(sh, nc, Linv + (size_t)N.lin * (ND_T * ND_T), N.np == 1 ? Lb + N.poff : nullptr, N.ld,
             N.ooff, bad);
}

/* Panel j of the nodes of a level: task = (row tile, column tile) of the
 * trailing part.  The workgroup forms the two row tiles of the panel, L = A
 * Linv^T (each is formed again by every task that needs it: 2 x 64^3
 * products that cost less than a launch in between), stores its own where
 * the tile is diagonal, and takes the product off the trailing tile: an
 * own-column tile of A, or the update matrix, which starts from the
 * children's.  The next diagonal tile is factored where it was updated. */
__global__ void __launch_bounds__(ND_BLK) k_nd_panel(const NdTask *__restrict__ task, const NdNode *__restrict__ nodes,
                                                     int j, const int *__restrict__ inv,
                                                     const double *__restrict__ Uc, double *__restrict__ U, double *P,
                                                     double *__restrict__ Lb, double *Linv, int *bad) {
    __shared__ double sh[ND_LDS];
    const NdTask t = task[blockIdx.x];
    const NdNode N = nodes[t.node];
    const int l = threadIdx.x & 63, wv = threadIdx.x >> 6, li = l & 15, lk = l >> 4;
    const int cq = (wv & 1) * 32, rq = (wv >> 1) * 32;
    const int w = max(0, min(ND_T, N.s - j * ND_T)), w4 = (w + 3) & ~3;
    const double *Vj = Linv + ((size_t)N.lin + j) * (ND_T * ND_T);
    const double *Pj = P + N.poff + (long long)j * ND_T * N.ld;
    int tr0, tnr, tc0, tnc;
    nd_tile(N, t.a, tr0, tnr);
    nd_tile(N, t.b, tc0, tnc);
    double *Lr = sh, *Lc = t.a == t.b ? sh : sh + ND_T * ND_T;
    /* the panel's rows of the two tiles */
    for (int q = 0; q < (t.a == t.b ? 1 : 2); q++) {
        const int r0 = q ? tc0 : tr0, nr = q ? tnc : tnr;
        double *dst = q ? Lc : Lr;
        nd_d4 acc[2][2] = {};
        const double *pr[2];
        bool ok[2];
#pragma unroll
        for (int ri = 0; ri < 2; ri++) {
            const int r = rq + 16 * ri + li;
            ok[ri] = r < nr;
            pr[ri] = Pj + r0 + (ok[ri] ? r : 0);
        }
#pragma unroll 4
        for (int ks = 0; ks < w4; ks += 4) {
            const int k = ks + lk;
            const bool kok = k < w;
            double a[2], b[2];
#pragma unroll
            for (int ci = 0; ci < 2; ci++) a[ci] = Vj[k * ND_T + cq + 16 * ci + li];
#pragma unroll
            for (int ri = 0; ri < 2; ri++) {
                const double v = pr[ri][(long long)(kok ? k : 0) * N.ld];
                b[ri] = kok && ok[ri] ? v : 0.0;
            }
#pragma unroll
            for (int ci = 0; ci < 2; ci++)
#pragma unroll
                for (int ri = 0; ri < 2; ri++)
                    acc[ci][ri] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[ci], b[ri], acc[ci][ri], 0, 0, 0);
        }
        const bool keep = q == 0 && t.a == t.b && N.np > 1;
#pragma unroll
        for (int ci = 0; ci < 2; ci++)
#pragma unroll
            for (int ri = 0; ri < 2; ri++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int c = cq + 16 * ci + 4 * v + lk, r = rq + 16 * ri + li;
                    dst[nd_sw(c, r)] = acc[ci][ri][v];
                    if (keep && c < w && r < nr)
                        Lb[N.poff + (long long)(j * ND_T + c) * N.ld + r0 + r] = acc[ci][ri][v];
                }
    }
    __syncthreads();
    if (N.np == 1 && t.a == t.b) {
        /* a front of one panel: its rows of T = L21 L11^-1 at once */
        nd_d4 tw[2][2] = {};
#pragma unroll 4
        for (int ks = 0; ks < w4; ks += 4) {
            const int k = ks + lk;
            double a[2], b[2];
#pragma unroll
            for (int q = 0; q < 2; q++) {
                a[q] = Vj[(cq + 16 * q + li) * ND_T + k];
                b[q] = Lr[nd_sw(k, rq + 16 * q + li)];
            }
#pragma unroll
            for (int ci = 0; ci < 2; ci++)
#pragma unroll
                for (int ri = 0; ri < 2; ri++)
                    tw[ci][ri] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[ci], b[ri], tw[ci][ri], 0, 0, 0);
        }
#pragma unroll
        for (int ci = 0; ci < 2; ci++)
#pragma unroll
            for (int ri = 0; ri < 2; ri++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int c = cq + 16 * ci + 4 * v + lk, r = rq + 16 * ri + li;
                    if (c < w && r < tnr) Lb[N.poff + (long long)c * N.ld + tr0 + r] = tw[ci][ri][v];
                }
    }
    nd_d4 acc[2][2] = {};
#pragma unroll 4
    for (int ks = 0; ks < w4; ks += 4) {
        const int k = ks + lk;
        double a[2], b[2];
#pragma unroll
        for (int ci = 0; ci < 2; ci++) a[ci] = Lc[nd_sw(k, cq + 16 * ci + li)];
#pragma unroll
        for (int ri = 0; ri < 2; ri++) b[ri] = Lr[nd_sw(k, rq + 16 * ri + li)];
#pragma unroll
        for (int ci = 0; ci < 2; ci++)
#pragma unroll
            for (int ri = 0; ri < 2; ri++)
                acc[ci][ri] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[ci], b[ri], acc[ci][ri], 0, 0, 0);
    }
    const bool own = t.b < N.np, diag = t.a == t.b, next = own && diag && t.b == j + 1;
    if (next) __syncthreads(); /* the diagonal tile takes the operands' LDS */
#pragma unroll
    for (int ci = 0; ci < 2; ci++)
#pragma unroll
        for (int ri = 0; ri < 2; ri++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int c = cq + 16 * ci + 4 * v + lk, r = rq + 16 * ri + li;
                if (r >= tnr || c >= tnc || (diag && r < c)) continue;
                if (own) {
                    double *p = P + N.poff + (long long)(tc0 + c) * N.ld + tr0 + r;
                    const double x = *p - acc[ci][ri][v];
                    if (next) sh[c * 65 + r] = x;
                    else *p = x;
                } else {
                    double *u = U + N.uoff + (long long)(tc0 - N.s + c) * N.ldu + (tr0 - N.s + r);
                    const double base = j == 0 ? nd_children(nodes, N, inv, Uc, tr0 + r, tc0 + c) : *u;
                    *u = base - acc[ci][ri][v];
                }
            }
    if (!next) return;
    __syncthreads();
    nd_potrf(sh, tnc, Linv + ((size_t)N.lin + j + 1) * (ND_T * ND_T), nullptr, 0, N.ooff + tc0, bad);
}

/* T = [L11^-1; L21 L11^-1] of the fronts of several panels, over the panel
 * storage (a front of one panel has its T in Lb already), column tiles from
 * the last to the first (all nodes of all levels at once): task = (column
 * tile j, row tile); T(:, j) = (E - sum_{i > j} T(:, i) L(i, j)) Linv_j with E
 * the rows of L21, and T(j, j) = Linv_j. */
__global__ void __launch_bounds__(ND_BLK) k_nd_invert(const NdTask *__restrict__ task,
                                                      const NdNode *__restrict__ nodes, double *P,
                                                      const double *__restrict__ Lb, const double *__restrict__ Linv) {
    __shared__ double sh[ND_T * ND_T];
    const NdTask t = task[blockIdx.x];
    const NdNode N = nodes[t.node];
    const int j = t.a, rt = t.b;
    const int l = threadIdx.x & 63, wv = threadIdx.x >> 6, li = l & 15, lk = l >> 4;
    const int cq = (wv & 1) * 32, rq = (wv >> 1) * 32;
    const int w = min(ND_T, N.s - j * ND_T);
    const double *Vj = Linv + ((size_t)N.lin + j) * (ND_T * ND_T);
    int r0, nr;
    nd_tile(N, rt, r0, nr);
    double *Tj = P + N.poff + (long long)j * ND_T * N.ld + r0;
    if (rt == j) {
        const int r = threadIdx.x & 63;
        for (int c = threadIdx.x >> 6; c < w; c += 4)
            if (r < nr) Tj[(long long)c * N.ld + r] = Vj[c * ND_T + r];
        return;
    }
    const int ilast = rt < N.np ? rt : N.np - 1;
    nd_d4 acc[2][2] = {};
    int rr[2], cc[2];
#pragma unroll
    for (int q = 0; q < 2; q++) {
        rr[q] = min(rq + 16 * q + li, nr - 1); /* rows and columns beyond the tile: clamped, not stored */
        cc[q] = min(cq + 16 * q + li, w - 1);
    }
    for (int i = j + 1; i <= ilast; i++) {
        const int wi = min(ND_T, N.s - i * ND_T), wi4 = (wi + 3) & ~3;
        const double *Ti = P + N.poff + (long long)i * ND_T * N.ld + r0;
        const double *Li = Lb + N.poff + (long long)j * ND_T * N.ld + i * ND_T;
#pragma unroll 4
        for (int ks = 0; ks < wi4; ks += 4) {
            const int k = min(ks + lk, wi - 1);
            const bool kok = ks + lk < wi;
            double a[2], b[2];
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const double x = Li[(long long)cc[q] * N.ld + k], y = Ti[(long long)k * N.ld + rr[q]];
                a[q] = kok ? x : 0.0;
                b[q] = kok ? y : 0.0;
            }
#pragma unroll
            for (int ci = 0; ci < 2; ci++)
#pragma unroll
                for (int ri = 0; ri < 2; ri++)
                    acc[ci][ri] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[ci], b[ri], acc[ci][ri], 0, 0, 0);
        }
    }
#pragma unroll
    for (int ci = 0; ci < 2; ci++)
#pragma unroll
        for (int ri = 0; ri < 2; ri++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int c = cq + 16 * ci + 4 * v + lk, r = rq + 16 * ri + li;
                double e = 0.0;
                if (rt >= N.np && c < w && r < nr) e = Lb[N.poff + (long long)(j * ND_T + c) * N.ld + r0 + r];
                sh[nd_sw(c, r)] = c < w && r < nr ? e - acc[ci][ri][v] : 0.0;
                acc[ci][ri][v] = 0.0;
            }
    __syncthreads();
    const int w4 = (w + 3) & ~3;
#pragma unroll 4
    for (int ks = 0; ks < w4; ks += 4) {
        const int k = ks + lk;
        double a[2], b[2];
#pragma unroll
        for (int q = 0; q < 2; q++) {
            a[q] = Vj[(cq + 16 * q + li) * ND_T + k];
            b[q] = sh[nd_sw(k, rq + 16 * q + li)];
        }
#pragma unroll
        for (int ci = 0; ci < 2; ci++)
#pragma unroll
            for (int ri = 0; ri < 2; ri++)
                acc[ci][ri] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[ci], b[ri], acc[ci][ri], 0, 0, 0);
    }
#pragma unroll
    for (int ci = 0; ci < 2; ci++)
#pragma unroll
        for (int ri = 0; ri < 2; ri++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int c = cq + 16 * ci + 4 * v + lk, r = rq + 16 * ri + li;
                if (c < w && r < nr) Tj[(long long)c * N.ld + r] = acc[ci][ri][v];
            }
}

/* ------------------------------------------------------------------ */
/* solves                                                               */
/* ------------------------------------------------------------------ */
/* A level of a solve is bound by its chain of dependent reads (a few MB over
 * the whole chip): the task holds all of its front, the children's update
 * vectors are found by one map, and the first ND_PRE columns or rows of T of
 * every thread are read while the vector is still being gathered (257 x 129
 * cells: 52 directions in 7.7 ms, 8.1 before).  Taking the levels at the top
 * into one front of a thousand unknowns saves launches and loses as much to
 * its panels (and its explicit inverse, one launch, is not accurate enough). */
#define ND_PRE 8

/* the children's update-vector entries of row r of a front */
__device__ __forceinline__ double nd_child_vec(const NdSolve &t, const int *__restrict__ at, const double *g, int r) {
    double v = 0.0;
    if (t.ga >= 0) v += g[at[t.ga + r]];
    if (t.gb >= 0) v += g[at[t.gb + r]];
    return v;
}

/* Forward solve of a level: one tile of RT rows of a front; y = L11^-1 r on
 * the own rows, g = (children's) - L21 L11^-1 r on the boundary rows, r =
 * f + children's.  RT rows x 256 / RT column groups per workgroup: a wave
 * reads RT contiguous rows of 64 / RT columns; the groups' sums are added in
 * a fixed order. */
template <int RT>
__global__ void __launch_bounds__(ND_BLK) k_nd_forward(const NdSolve *__restrict__ task,
                                                       const int *__restrict__ at, const int *__restrict__ eq,
                                                       const double *__restrict__ P, const double *__restrict__ Lb,
                                                       const double *__restrict__ f, double *__restrict__ y,
                                                       double *g) {
    constexpr int CG = ND_BLK / RT;
    __shared__ double rs[ND_CH];
    __shared__ double red[CG][RT];
    const NdSolve t = task[blockIdx.x];
    const int lr = threadIdx.x % RT, cg = threadIdx.x / RT;
    const int m = t.s + t.b, row0 = t.tile * RT, row = row0 + lr;
    const double *Tr = (t.panels > 1 ? P : Lb) + t.toff + (row < m ? row : 0);
    /* own rows end at the diagonal tile of the last row */
    const int last = min(row0 + RT, m) - 1;
    const int cend = last < t.s ? min(t.s, (last / ND_T + 1) * ND_T) : t.s;
    const int rend = row >= m ? 0 : row < t.s ? min(t.s, (row / ND_T + 1) * ND_T) : t.s;
    double pre[ND_PRE];
    if (t.s > 0)
#pragma unroll
        for (int u = 0; u < ND_PRE; u++) pre[u] = Tr[(long long)min(cg + u * CG, t.s - 1) * t.ld];
    double acc = 0.0;
    for (int cb = 0; cb < cend; cb += ND_CH) {
        const int ce = min(cend, cb + ND_CH);
        if (cb) __syncthreads();
        for (int c = cb + threadIdx.x; c < ce; c += ND_BLK) {
            rs[c - cb] = f[eq[t.ooff + c]] + nd_child_vec(t, at, g, c);
        }
        __syncthreads();
        const int re = min(rend, ce);
        int c = cb + cg;
        if (cb == 0) {
#pragma unroll
            for (int u = 0; u < ND_PRE; u++, c += CG)
                if (c < re) acc += pre[u] * rs[c];
        }
#pragma unroll 8
        for (; c < re; c += CG) acc += Tr[(long long)c * t.ld] * rs[c - cb];
    }
    red[cg][lr] = acc;
    __syncthreads();
    if (cg == 0 && row < m) {
        double sum = 0.0;
#pragma unroll
        for (int q = 0; q < CG; q++) sum += red[q][lr];
        if (row < t.s) y[t.ooff + row] = sum;
        else g[t.boff + row - t.s] = nd_child_vec(t, at, g, row) - sum;
    }
}

/* Backward solve of a level: one tile of CT columns of a front (inside one
 * 64-column tile); x = T^T (y, -x of the boundary): 16 lanes per column (128
 * contiguous bytes a step) */
template <int CT>
__global__ void __launch_bounds__(ND_BLK) k_nd_backward(const NdSolve *__restrict__ task,
                                                        const int *__restrict__ blist, const int *__restrict__ eq,
                                                        const double *__restrict__ P, const double *__restrict__ Lb,
                                                        const double *__restrict__ y, double *x,
                                                        double *__restrict__ out) {
    constexpr int NC = CT / 16;
    __shared__ double vs[ND_CH];
    const NdSolve t = task[blockIdx.x];
    const int l = threadIdx.x & 15, cl = threadIdx.x >> 4;
    const int m = t.s + t.b, c0 = t.tile * CT;
    const int rfirst = (c0 / ND_T) * ND_T; /* rows of the columns' diagonal tile and below */
    const double *Tc = (t.panels > 1 ? P : Lb) + t.toff + (long long)min(c0 + cl, t.s - 1) * t.ld;
    const long long step = 16LL * t.ld;
    double acc[NC], pre[NC][ND_PRE];
#pragma unroll
    for (int q = 0; q < NC; q++) {
        acc[q] = 0.0;
        const double *p = c0 + cl + 16 * q < t.s ? Tc + q * step : Tc;
#pragma unroll
        for (int u = 0; u < ND_PRE; u++) pre[q][u] = p[min(rfirst + l + 16 * u, m - 1)];
    }
    for (int rb = rfirst; rb < m; rb += ND_CH) {
        const int re = min(m, rb + ND_CH);
        if (rb > rfirst) __syncthreads();
        for (int r = rb + threadIdx.x; r < re; r += ND_BLK)
            vs[r - rb] = r < t.s ? y[t.ooff + r] : -x[blist[t.boff + r - t.s]];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < NC; q++) {
            if (c0 + cl + 16 * q < t.s) {
                double a = 0.0;
                int r = rb + l;
                if (rb == rfirst) {
#pragma unroll
                    for (int u = 0; u < ND_PRE; u++, r += 16)
                        if (r < re) a += pre[q][u] * vs[r - rb];
                }
#pragma unroll 8
                for (; r < re; r += 16) a += Tc[q * step + r] * vs[r - rb];
                acc[q] += a;
            }
        }
    }
#pragma unroll
    for (int q = 0; q < NC; q++) {
        double a = acc[q];
        for (int o = 8; o > 0; o >>= 1) a += __shfl_xor(a, o, 64);
        const int c = c0 + cl + 16 * q;
        if (l == 0 && c < t.s) {
            x[t.ooff + c] = a;
            out[eq[t.ooff + c]] = a;
        }
    }
}

/* ------------------------------------------------------------------ */
/* host side                                                            */
/* ------------------------------------------------------------------ */
template <class T>
struct NdBuf {
    T *p = nullptr;
    size_t cap = 0;
};

struct MdzFactor {
    hipStream_t s = nullptr;
    int n = 0;
    unsigned long long version = 0;
    NdPlan plan; /* after the upload: level, invert, eq and the lengths */
    NdBuf<NdNode> nodes;
    NdBuf<NdTask> tasks;
    NdBuf<NdSolve> solves;
    NdBuf<int> at, pos, eq, node_of, blist, inv, bad;
    NdBuf<double> P, Lb, Linv, U[2], y, x, g;
};

template <class T>
static int nd_reserve(NdBuf<T> &b, size_t n) {
    n = std::max<size_t>(n, 1);
    if (b.cap >= n && b.cap <= 2 * n + 4096) return MDZ_OK;
    hipFree(b.p);
    b.p = nullptr;
    b.cap = 0;
    FCHK(hipMalloc((void **)&b.p, n * sizeof(T)));
    b.cap = n;
    return MDZ_OK;
}
template <class T>
static int nd_upload(NdBuf<T> &b, const std::vector<T> &h) {
    int rc = nd_reserve(b, h.size());
    if (rc) return rc;
    if (!h.empty()) FCHK(hipMemcpy(b.p, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice));
    return MDZ_OK;
}
template <class T>
static void nd_free(NdBuf<T> &b) {
    hipFree(b.p);
    b.p = nullptr;
    b.cap = 0;
}

int mdz_factor_create(MdzFactor **out, hipStream_t s) {
    if (!out) return mdz_error(MDZ_EINVAL, "factor: null output");
    *out = new (std::nothrow) MdzFactor();
    if (!*out) return mdz_error(MDZ_ENOMEM, "factor: host memory");
    (*out)->s = s;
    return MDZ_OK;
}

void mdz_factor_destroy(MdzFactor *F) {
    if (!F) return;
    if (F->s) hipStreamSynchronize(F->s);
    nd_free(F->nodes); nd_free(F->tasks); nd_free(F->solves); nd_free(F->at);
    nd_free(F->pos); nd_free(F->eq); nd_free(F->node_of); nd_free(F->blist); nd_free(F->inv); nd_free(F->bad);
    nd_free(F->P); nd_free(F->Lb); nd_free(F->Linv); nd_free(F->U[0]); nd_free(F->U[1]);
    nd_free(F->y); nd_free(F->x); nd_free(F->g);
    delete F;
}

unsigned long long mdz_factor_version(const MdzFactor *F) { return F->version; }

int mdz_factor_analyse(MdzFactor *F, int Nx, int Nz, int n, const int *mom_node, const std::vector<int> &Ic,
                       const std::vector<int> &J) {
    if (!F || n < 1 || Nx < 1 || Nz < 1) return mdz_error(MDZ_EINVAL, "factor: bad arguments");
    F->n = 0;
    F->version++;
    NdPlan &p = F->plan;
    int rc = nd_plan(p, Nx, Nz, n, mom_node, Ic, J);
    if (rc) return rc;
    if ((rc = nd_upload(F->nodes, p.node)) || (rc = nd_upload(F->tasks, p.task)) ||
        (rc = nd_upload(F->solves, p.solve)) || (rc = nd_upload(F->at, p.at)) || (rc = nd_upload(F->pos, p.pos)) ||
        (rc = nd_upload(F->eq, p.eq)) || (rc = nd_upload(F->node_of, p.node_of)) ||
        (rc = nd_upload(F->blist, p.blist)) || (rc = nd_upload(F->inv, p.inv)) || (rc = nd_reserve(F->bad, 1)) ||
        (rc = nd_reserve(F->P, p.panel_len)) || (rc = nd_reserve(F->Lb, p.panel_len)) ||
        (rc = nd_reserve(F->Linv, p.nlin * ND_T * ND_T)) || (rc = nd_reserve(F->U[0], p.ulen[0])) ||
        (rc = nd_reserve(F->U[1], p.ulen[1])) || (rc = nd_reserve(F->y, (size_t)n)) ||
        (rc = nd_reserve(F->x, (size_t)n)) || (rc = nd_reserve(F->g, p.blist.size() + 1)))
        return rc;
    FCHK(hipMemsetAsync(F->g.p, 0, (p.blist.size() + 1) * sizeof(double), F->s));
    p.release_uploaded();
    F->n = n;
    return MDZ_OK;
}

int mdz_factor_numeric(MdzFactor *F, const int *base, const int *Ic, const int *J, const double *val, int *bad) {
    if (!F || F->n < 1) return mdz_error(MDZ_EINVAL, "factor: not analysed");
    hipStream_t s = F->s;
    const NdNode *nodes = F->nodes.p;
    const int none = INT_MAX;
    FCHK(hipMemcpyAsync(F->bad.p, &none, sizeof(int), hipMemcpyHostToDevice, s));
    FCHK(hipMemsetAsync(F->P.p, 0, F->plan.panel_len * sizeof(double), s));
    hipLaunchKernelGGL(k_nd_scatter, dim3((F->n + ND_BLK - 1) / ND_BLK), dim3(ND_BLK), 0, s, F->n, base, Ic, J, val,
                       (const int *)F->pos.p, (const int *)F->node_of.p, nodes, (const int *)F->blist.p, F->P.p);
    for (size_t lv = 0; lv < F->plan.level.size(); lv++) {
        const NdLevel &L = F->plan.level[lv];
        double *U = F->U[lv & 1].p, *Uc = F->U[(lv & 1) ^ 1].p;
        if (L.assemble.count)
            hipLaunchKernelGGL(k_nd_assemble, dim3(L.assemble.count), dim3(ND_BLK), 0, s,
                               (const NdTask *)F->tasks.p + L.assemble.first, nodes, (const int *)F->inv.p,
                               (const double *)Uc, F->P.p, F->Lb.p, F->Linv.p, F->bad.p);
        for (size_t j = 0; j < L.panel.size(); j++)
            if (L.panel[j].count)
                hipLaunchKernelGGL(k_nd_panel, dim3(L.panel[j].count), dim3(ND_BLK), 0, s,
                                   (const NdTask *)F->tasks.p + L.panel[j].first, nodes, (int)j,
                                   (const int *)F->inv.p, (const double *)Uc, U, F->P.p, F->Lb.p, F->Linv.p,
                                   F->bad.p);
    }
    for (const NdRange &r : F->plan.invert)
        hipLaunchKernelGGL(k_nd_invert, dim3(r.count), dim3(ND_BLK), 0, s, (const NdTask *)F->tasks.p + r.first, nodes,
                           F->P.p, (const double *)F->Lb.p, (const double *)F->Linv.p);
    FCHK(hipGetLastError());
    int got = none;
    FCHK(hipMemcpyAsync(&got, F->bad.p, sizeof(int), hipMemcpyDeviceToHost, s));
    FCHK(hipStreamSynchronize(s));
    *bad = got == none ? -1 : F->plan.eq[(size_t)got];
    return MDZ_OK;
}

void mdz_factor_apply(MdzFactor *F, const double *f, double *x) {
    hipStream_t s = F->s;
    const dim3 blk(ND_BLK);
    const size_t nl = F->plan.level.size();
    const double *P = F->P.p, *Lb = F->Lb.p;
    for (size_t q = 0; q < nl; q++) {
        const NdLevel &L = F->plan.level[q];
        if (!L.forward.count) continue;
        const NdSolve *t = F->solves.p + L.forward.first;
        const dim3 grid(L.forward.count);
#define FWD(RT)                                                                                                       \
    hipLaunchKernelGGL((k_nd_forward<RT>), grid, blk, 0, s, t, (const int *)F->at.p, (const int *)F->eq.p, P, Lb, f, \
                       F->y.p, F->g.p)
        if (L.rt == 64) FWD(64);
        else if (L.rt == 32) FWD(32);
        else FWD(16);
#undef FWD
    }
    for (size_t q = nl; q-- > 0;) {
        const NdLevel &L = F->plan.level[q];
        if (!L.backward.count) continue;
        const NdSolve *t = F->solves.p + L.backward.first;
        const dim3 grid(L.backward.count);
#define BWD(CT)                                                                                                     \
    hipLaunchKernelGGL((k_nd_backward<CT>), grid, blk, 0, s, t, (const int *)F->blist.p, (const int *)F->eq.p, P, Lb, \
                       (const double *)F->y.p, F->x.p, x)
        if (L.ct == 64) BWD(64);
        else if (L.ct == 32) BWD(32);
        else BWD(16);
#undef BWD
    }
}
