/*
 * mdz_markers.hip -- marker -> grid on gfx950: the per-time-step producers of
 * the rheology's phase fractions and plasticity parameters.
 *
 *   P2Mastah                      ParticleRoutines.c:3226-3538
 *   Interp_P2N                    ParticleRoutines.c:1770-1946
 *   CohesionFrictionDilationGrid  RheologyDensity.c:1422-1660
 *
 * The reference scatters each marker's tent weights into per-thread copies
 * of the node arrays.  Here the marker records (x, z, value, phase, index)
 * are put into bins by nearest node once and one lane per node gathers from
 * the bins its stencil reaches, merging them in increasing marker index: each
 * node's sums see the markers in the order the reference's sequential loop
 * adds them, with no atomics on floating-point data and the same result on
 * every run.  Bins stay valid while the markers and values do not change, so
 * the interpolations of a time step on one node family share them.
 *
 * Binning is a counting sort: a marker's rank in its bin comes from an
 * integer atomic, the counts' scan gives the bins' starts, the records are
 * placed, and each is moved to the number of smaller indices in its bin --
 * which undoes the atomics' order.  Four passes over the markers, bound by
 * the atomics and the placement's scattered 32-byte writes.  Measured, 8.0
 * million markers in random order over 2.0 million quarter cells: counts 0.31
 * ms, placement 0.28, order 0.16, the step's two gathers 0.17 and 0.16; a
 * radix sort of keys and records took 0.85 ms for each node family and the
 * six gathers 0.75 (the step 2.6 -> 1.15 ms).  The ordering is quadratic in
 * a bin's markers: where the bins hold more than BIN_DENSE on average, or
 * one holds more than BIN_LONG, a stable radix sort takes the call.
 *
 * The step of a time step with the 1-node stencil bins once for both node
 * families: by quarter cell, the pair of a marker's nearest centroid and
 * nearest vertex.  A node's markers are the four quarters around it, merged
 * by index; one launch per family forms phase fractions, plastic strain and
 * strength parameters.
 */
#include <stdlib.h>
#include <string.h>

#include <rocprim/device/device_radix_sort.hpp>

#include "mdz_kernels.h"

/* nearest node along one axis, clamped to [0, n - 1] (ParticleRoutines.c:3321-3333) */
__device__ __forceinline__ int nearest_node(double pos, double x0, double h, int n) {
    const double v = ceil((pos - x0) / h + 0.5) - 1.0;
    if (!(v >= 0.0)) return 0;
    if (v > (double)(n - 1)) return n - 1;
    return (int)v;
}

/* the same without clamping: -1 when outside [0, n - 1] (Interp_P2N:1855-1861) */
__device__ __forceinline__ int node_unclamped(double pos, double x0, double h, int n) {
    const double v = ceil((pos - x0) / h + 0.5) - 1.0;
    return v >= 0.0 && v <= (double)(n - 1) ? (int)v : -1;
}

/* Bins of one node family (quarter 0), or quarter cells: bin (2 ic + iv -
 * ic, 2 jc + jv - jc) of a marker with nearest centroid (ic, jc) and vertex
 * (iv, jv).  The centroids lie half a spacing from the vertices, so that iv -
 * ic is 0 or 1 whatever the rounding (the clamped ends included). */
struct BinGrid {
    NodeAxes a, v;
    int quarter;
    __device__ __forceinline__ int bins() const { return quarter ? 4 * a.Nx * a.Nz : a.Nx * a.Nz; }
    __device__ __forceinline__ int key(double x, double z) const {
        const int i = nearest_node(x, a.X[0], a.dx, a.Nx), j = nearest_node(z, a.Z[0], a.dz, a.Nz);
        if (!quarter) return i + j * a.Nx;
        const int iv = nearest_node(x, v.X[0], v.dx, v.Nx), jv = nearest_node(z, v.Z[0], v.dz, v.Nz);
        return min(max(i + iv, 0), 2 * a.Nx - 1) + min(max(j + jv, 0), 2 * a.Nz - 1) * (2 * a.Nx);
    }
};

/* BIN_LONG: most markers of a bin that the ordering pass takes; BIN_DENSE: markers a bin, on
 * average, up to which the counting sort is the faster one.  Measured, steps of 8.0 million markers
 * (1-node stencil) in random and in seeding order: 25 a quarter cell 1.25 and 1.18 ms against 1.35
 * and 1.34 with the radix sort; 64 a quarter cell 1.58 and 1.92 against 1.53 and 1.48 (markers in
 * seeding order meet in the counts' atomics) */
#define BIN_LONG 512
#define BIN_DENSE 32

/* rank of every marker in its bin, in no particular order; counts per bin */
__global__ void __launch_bounds__(256) k_marker_count(MarkerSet m, BinGrid g, int *__restrict__ count,
                                                     int *__restrict__ rank, int *__restrict__ long_bin) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= m.n || m.phase[k] == -1) return;
    const int r = atomicAdd(&count[g.key(m.x[k], m.z[k])], 1);
    rank[k] = r;
    if (r >= BIN_LONG) *long_bin = 1;
}

__global__ void __launch_bounds__(256) k_marker_place(MarkerSet m, const double *__restrict__ val, BinGrid g,
                                                     const int *__restrict__ start, const int *__restrict__ rank,
                                                     MarkerRec *__restrict__ rec) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= m.n) return;
    const int ph = m.phase[k];
    if (ph == -1) return;
    const double x = m.x[k], z = m.z[k];
    rec[start[g.key(x, z)] + rank[k]] = MarkerRec{x, z, val ? val[k] : 0.0, ph, k};
}

/* every record to its place by increasing marker index within its bin */
__global__ void __launch_bounds__(256) k_marker_order(BinGrid g, const int *__restrict__ start,
                                                     const MarkerRec *__restrict__ in, MarkerRec *__restrict__ out) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= start[g.bins()]) return;
    const MarkerRec r = in[p];
    const int b = g.key(r.x, r.z), s0 = start[b], s1 = start[b + 1];
    int at = s0;
    for (int q = s0; q < s1; q++) at += in[q].k < r.k;
    out[at] = r;
}

/* bin key and record of every marker (key = bins for an inactive one:
 * sorted past the last bin) */
__global__ void __launch_bounds__(256) k_marker_keys(MarkerSet m, const double *__restrict__ val, BinGrid g,
                                                    int *__restrict__ key, MarkerRec *__restrict__ rec) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= m.n) return;
    const double x = m.x[k], z = m.z[k];
    const int ph = m.phase[k];
    key[k] = ph != -1 ? g.key(x, z) : g.bins();
    rec[k] = MarkerRec{x, z, val ? val[k] : 0.0, ph, k};
}

/* start[b] = first sorted position whose key is >= b, for b = 0 .. nodes:
 * the thread of position p writes the bins in (key[p - 1], key[p]] (p = n:
 * the bins past the last key) */
__global__ void __launch_bounds__(256) k_bin_starts(const int *__restrict__ key, int n, int nodes,
                                                   int *__restrict__ start) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p > n) return;
    const int lo = p == 0 ? 0 : key[p - 1] + 1;
    const int hi = p == n ? nodes : min(key[p], nodes);
    for (int b = lo; b <= hi; b++) start[b] = p;
}

static unsigned key_bits(int nodes) {
    unsigned bits = 1;
    while ((1u << bits) <= (unsigned)nodes && bits < 31) bits++;
    return bits;
}

int mdz_markers_bin(MarkerDev &md, int fam, const NodeAxes &a, const NodeAxes *v, hipStream_t s) {
    const int quarter = fam == MDZ_FAM_QUARTER;
    const int bins = (quarter ? 4 : 1) * a.Nx * a.Nz;
    if (md.n < 0 || bins < 1 || quarter != (v != nullptr)) return mdz_error(MDZ_EINVAL, "marker binning: empty grid");
    if ((size_t)bins + 1 > md.start_cap[fam]) return mdz_error(MDZ_EINVAL, "marker binning: bin array too small");
    int *start = md.start[fam];
    if (hipMemsetAsync(start, 0, ((size_t)bins + 1) * sizeof(int), s) != hipSuccess)
        return mdz_error(MDZ_EHIP, "marker binning: counts");
    if (md.n > 0) {
        if (!md.rec[fam] && hipMalloc((void **)&md.rec[fam], (size_t)md.cap * sizeof(MarkerRec)) != hipSuccess)
            return mdz_error(MDZ_ENOMEM, "marker binning: records");
        const BinGrid g{a, quarter ? *v : a, quarter};
        const dim3 grid(mdz_div_up(md.n, 256)), blk(256);
        int *flag = md.scan + md.scan_len - 1, total = 0;
        bool sort = md.n > (long long)BIN_DENSE * bins;
        if (!sort) {
            if (hipMemsetAsync(flag, 0, sizeof(int), s) != hipSuccess) return mdz_error(MDZ_EHIP, "marker binning: flag");
            hipLaunchKernelGGL(k_marker_count, grid, blk, 0, s, md.set(), g, start, md.key, flag);
            if (hipMemcpyAsync(md.long_bin, flag, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess ||
                mdz_scan_exclusive(start, bins + 1, md.scan, md.scan_len - 1, s, &total) != MDZ_OK)
                return mdz_error(MDZ_EHIP, "marker binning: scan"); /* (the total's copy waits for the stream) */
            sort = *md.long_bin != 0;
        }
        if (!sort) {
            hipLaunchKernelGGL(k_marker_place, grid, blk, 0, s, md.set(), (const double *)md.val, g,
                               (const int *)start, (const int *)md.key, md.rec_in);
            if (total > 0)
                hipLaunchKernelGGL(k_marker_order, dim3(mdz_div_up(total, 256)), blk, 0, s, g, (const int *)start,
                                   (const MarkerRec *)md.rec_in, md.rec[fam]);
        } else {
            hipLaunchKernelGGL(k_marker_keys, grid, blk, 0, s, md.set(), (const double *)md.val, g, md.key, md.rec_in);
            const unsigned bits = key_bits(bins);
            size_t need = 0;
            if (rocprim::radix_sort_pairs(nullptr, need, md.key, md.key_out, md.rec_in, md.rec[fam], (unsigned)md.n,
                                          0, bits, s) != hipSuccess)
                return mdz_error(MDZ_EHIP, "marker binning: sort size");
            if (need > md.tmp_bytes) return mdz_error(MDZ_EINVAL, "marker binning: sort scratch too small");
            size_t have = md.tmp_bytes;
            if (rocprim::radix_sort_pairs(md.tmp, have, md.key, md.key_out, md.rec_in, md.rec[fam], (unsigned)md.n,
                                          0, bits, s) != hipSuccess)
                return mdz_error(MDZ_EHIP, "marker binning: sort");
            hipLaunchKernelGGL(k_bin_starts, dim3(mdz_div_up(md.n + 1, 256)), blk, 0, s, (const int *)md.key_out, md.n,
                               bins, start);
        }
    }
    md.binned[fam] = bins;
    return MDZ_OK;
}

size_t mdz_markers_sort_bytes(int n, int nodes) {
    if (n < 1) return 0;
    size_t need = 0;
    int *k = nullptr;
    MarkerRec *r = nullptr;
    if (rocprim::radix_sort_pairs(nullptr, need, k, k, r, r, (unsigned)n, 0, key_bits(nodes), (hipStream_t)0) !=
        hipSuccess)
        return 0;
    return need;
}

/* ------------------------------------------------------------------ */
/* gather                                                               */
/* ------------------------------------------------------------------ */
/* The bins a node's stencil reaches, one fixed slot per offset (slot
 * (dj + 1) * 3 + di + 1 of the 9-node stencil, slot 0 of the 1-node one),
 * with the position of the weight's node: the reference measures a marker's
 * distance to a neighbour as X[ip] +- dx, Z[jp] +- dz from its own nearest
 * node (ip, jp) (ParticleRoutines.c:3353-3470).  Periodic x wraps the east
 * neighbour of the last column to column 0 and the west neighbour of the
 * first to column Nx - 1.  An unreached slot is an empty range. */
template <int NS>
struct Reach {
    int pos[NS], end[NS];
    double xn[NS], zn[NS];
};

template <int NS>
__device__ __forceinline__ void reach(const NodeAxes &a, const int *__restrict__ start, int i, int j, Reach<NS> &r) {
#pragma unroll
    for (int q = 0; q < NS; q++) {
        const int di = NS == 9 ? q % 3 - 1 : 0, dj = NS == 9 ? q / 3 - 1 : 0;
        /* the marker's nearest node (bi, bj) = this node minus the offset */
        const int bj = j - dj;
        int bi = i - di;
        bool ok = bj >= 0 && bj < a.Nz;
        if (bi < 0 || bi >= a.Nx) {
            if (a.periodic && di == 1 && i == 0) bi = a.Nx - 1;
            else if (a.periodic && di == -1 && i == a.Nx - 1) bi = 0;
            else ok = false;
        }
        r.pos[q] = r.end[q] = 0;
        r.xn[q] = r.zn[q] = 0.0;
        if (ok) {
            const int b = bi + bj * a.Nx;
            r.pos[q] = start[b];
            r.end[q] = start[b + 1];
            r.xn[q] = di == 0 ? a.X[bi] : (di == 1 ? a.X[bi] + a.dx : a.X[bi] - a.dx);
            r.zn[q] = dj == 0 ? a.Z[bj] : (dj == 1 ? a.Z[bj] + a.dz : a.Z[bj] - a.dz);
        }
    }
}

/* Visits the reached markers in increasing index (a merge of the sorted
 * bins), calling f(record, xn, zn) for each. */
template <int NS, class F>
__device__ __forceinline__ void merge_visit(Reach<NS> &r, const MarkerRec *__restrict__ rec, F &&f) {
    const int NONE = 0x7fffffff;
    int head[NS];
#pragma unroll
    for (int q = 0; q < NS; q++) head[q] = r.pos[q] < r.end[q] ? rec[r.pos[q]].k : NONE;
    for (;;) {
        int best = 0, kb = head[0];
#pragma unroll
        for (int q = 1; q < NS; q++)
            if (head[q] < kb) { kb = head[q]; best = q; }
        if (kb == NONE) break;
        int pb = r.pos[0];
        double xn = r.xn[0], zn = r.zn[0];
#pragma unroll
        for (int q = 1; q < NS; q++)
            if (q == best) { pb = r.pos[q]; xn = r.xn[q]; zn = r.zn[q]; }
        f(rec[pb], xn, zn);
#pragma unroll
        for (int q = 0; q < NS; q++)
            if (q == best) {
                const int p = ++r.pos[q];
                head[q] = p < r.end[q] ? rec[p].k : NONE;
            }
    }
}

/* P2Mastah: value mode (prop = 0) or phase fractions (prop = 1) */
template <int ST, bool PROP>
__global__ void __launch_bounds__(256) k_p2mastah(NodeAxes a, const MarkerRec *__restrict__ rec,
                                                 const int *__restrict__ start, P2GArgs g) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    const int n = a.Nx * a.Nz;
    if (c >= n) return;
    const int i = c % a.Nx, j = c / a.Nx;
    double hx = a.dx / 2.0, hz = a.dz / 2.0;
    if (ST == 9) { hx = 3.0 * a.dx / 2.0; hz = 3.0 * a.dz / 2.0; }
    Reach<ST> r;
    reach<ST>(a, start, i, j, r);
    double W = 0.0, BW = 0.0;
    double Wph[MDZ_MAX_PHASES];
    if (PROP)
#pragma unroll
        for (int p = 0; p < MDZ_MAX_PHASES; p++) Wph[p] = 0.0;
    merge_visit(r, rec, [&](const MarkerRec &mr, double xn, double zn) {
        const double dxm = fabs(xn - mr.x), dzm = fabs(zn - mr.z);
        const double w = (1.0 - dxm / hx) * (1.0 - dzm / hz);
        W += w;
        if (PROP) {
#pragma unroll
            for (int p = 0; p < MDZ_MAX_PHASES; p++)
                if (p == mr.phase) Wph[p] += w;
        } else {
            double v = g.flag == 1 ? mr.val : g.pval[mr.phase];
            if (g.avg == 1) v = 1.0 / v;
            if (g.avg == 2) v = log(v);
            BW += v * w;
        }
    });
    const bool skip = fabs(W) < 1e-30 || g.ntype[c] == 30 || g.ntype[c] == 31;
    if (PROP) {
        /* un-normalised weights where the node is skipped (:3496-3520) */
#pragma unroll
        for (int p = 0; p < MDZ_MAX_PHASES; p++)
            if (p < g.nph) g.perc[(size_t)p * n + c] = skip ? Wph[p] : Wph[p] / W;
    } else if (!skip) {
        double v = BW / W;
        if (g.avg == 1) v = 1.0 / v;
        if (g.avg == 2) v = exp(v);
        g.field[c] = v;
    }
}

/* Interp_P2N: one vertex per lane, markers of its own bin whose unclamped
 * vertex is this one, tent of half-width dx / 2 */
__global__ void __launch_bounds__(256) k_interp_p2n(NodeAxes a, const MarkerRec *__restrict__ rec,
                                                   const int *__restrict__ start, P2GArgs g) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    const int n = a.Nx * a.Nz;
    if (c >= n) return;
    const int i = c % a.Nx, j = c / a.Nx;
    double W = 0.0, BW = 0.0;
    const double Xi = a.X[i], Zj = a.Z[j];
    for (int p = start[c]; p < start[c + 1]; p++) {
        const MarkerRec mr = rec[p];
        if (node_unclamped(mr.x, a.X[0], a.dx, a.Nx) != i || node_unclamped(mr.z, a.Z[0], a.dz, a.Nz) != j) continue;
        const double dxm = 2.0 * fabs(Xi - mr.x), dzm = 2.0 * fabs(Zj - mr.z);
        double v = g.flag == 1 ? mr.val : g.pval[mr.phase];
        if (g.avg == 1) v = 1.0 / v;
        if (g.avg == 2) v = log(v);
        const double w = (1.0 - dxm / a.dx) * (1.0 - dzm / a.dz);
        W += w;
        BW += v * w;
    }
    if (W < 1e-30 || g.ntype[c] == 30) return;
    double v = BW / W;
    if (g.avg == 1) v = 1.0 / v;
    if (g.avg == 2) v = exp(v);
    g.field[c] = v;
}

/* periodic x: the first and last columns take their mean (:1928-1935) */
__global__ void __launch_bounds__(256) k_periodic_mean(double *f, int Nx, int Nz) {
    const int l = blockIdx.x * 256 + threadIdx.x;
    if (l >= Nz) return;
    const double av = 0.5 * (f[l * Nx + Nx - 1] + f[l * Nx]);
    f[l * Nx + Nx - 1] = av;
    f[l * Nx] = av;
}

void mdz_launch_p2mastah(const MarkerDev &md, int fam, const NodeAxes &a, int prop, int itp_stencil,
                         const P2GArgs &g, hipStream_t s) {
    const int n = a.Nx * a.Nz;
    const dim3 grid(mdz_div_up(n, 256));
    const MarkerRec *rec = md.rec[fam];
    const int *start = md.start[fam];
    if (itp_stencil == 9) {
        if (prop) hipLaunchKernelGGL((k_p2mastah<9, true>), grid, dim3(256), 0, s, a, rec, start, g);
        else hipLaunchKernelGGL((k_p2mastah<9, false>), grid, dim3(256), 0, s, a, rec, start, g);
    } else {
        if (prop) hipLaunchKernelGGL((k_p2mastah<1, true>), grid, dim3(256), 0, s, a, rec, start, g);
        else hipLaunchKernelGGL((k_p2mastah<1, false>), grid, dim3(256), 0, s, a, rec, start, g);
    }
}

void mdz_launch_interp_p2n(const MarkerDev &md, int fam, const NodeAxes &a, const P2GArgs &g, hipStream_t s) {
    const int n = a.Nx * a.Nz;
    hipLaunchKernelGGL(k_interp_p2n, dim3(mdz_div_up(n, 256)), dim3(256), 0, s, a, (const MarkerRec *)md.rec[fam],
                       (const int *)md.start[fam], g);
    if (a.periodic) hipLaunchKernelGGL(k_periodic_mean, dim3(mdz_div_up(a.Nz, 256)), dim3(256), 0, s, g.field, a.Nx, a.Nz);
}

/* ------------------------------------------------------------------ */
/* cohesion, friction and dilatancy                                     */
/* ------------------------------------------------------------------ */
/* the smooth softening of RheologyDensity.c:1466-1490 (SmoothSoftening = 1) */
__device__ __forceinline__ double soften(double v0, double v_end, double strain, double mu, double ds) {
    const double dv = v0 - v_end;
    const double v = v0 - dv / 2.0 * erfc(-(strain - mu) / ds) - v_end;
    const double vz = v0 - dv / 2.0 * erfc(-(0.0 - mu) / ds) - v_end;
    return v * dv / vz + v_end;
}

/* one phase's share fr of a node of strain s */
__device__ __forceinline__ void soften_phase(const SoftK &sk, int p, double s, double fr, double &fa, double &da,
                                             double &ca) {
    double f = sk.phi[p], d = sk.psi[p], co = sk.C[p];
    const double ds = sk.pls_end[p] - sk.pls_start[p], mu = 0.5 * (sk.pls_end[p] + sk.pls_start[p]);
    if (sk.phi_soft[p] == 1) f = soften(sk.phi[p], sk.phi_end[p], s, mu, ds);
    if (sk.psi_soft[p] == 1) d = soften(sk.psi[p], sk.psi_end[p], s, mu, ds);
    if (sk.coh_soft[p] == 1) co = soften(sk.C[p], sk.C_end[p], s, mu, ds);
    fa += fr * f;
    da += fr * d;
    ca += fr * co;
}

/* one node: the phase-fraction weighted (arithmetic) softened friction,
 * dilatancy and cohesion; zero at air / free-surface nodes */
__global__ void __launch_bounds__(256) k_cfd_nodes(int n, const double *__restrict__ strain,
                                                  const double *__restrict__ perc, const int8_t *__restrict__ tag,
                                                  int cells, SoftK sk, double *fric, double *dil, double *C) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= n) return;
    double fa = 0.0, da = 0.0, ca = 0.0;
    const int t = tag[c];
    const bool skip = t == 30 || (cells && t == 31);
    if (!skip) {
        const double s = strain[c];
        for (int p = 0; p < sk.nph; p++) soften_phase(sk, p, s, perc[(size_t)p * n + c], fa, da, ca);
    }
    fric[c] = fa;
    dil[c] = da;
    C[c] = ca;
}

/* ------------------------------------------------------------------ */
/* a time step's producers in one launch per node family                 */
/* ------------------------------------------------------------------ */
/* One centroid (VERT = 0) or vertex per lane, 1-node stencil: the markers of
 * its four quarter cells in increasing index (the head record of each quarter
 * in registers, the next one read while the current is summed); P2Mastah's
 * phase fractions with the tent of half a spacing from the node, then the
 * plastic strain -- at centroids by the same weights, at vertices by
 * Interp_P2N's over the markers whose unclamped vertex this is -- and, where
 * SOFT, the strength parameters (else the strain is left for a periodic
 * mean). */
template <int NPH, bool VERT, bool SOFT>
__global__ void __launch_bounds__(256) k_marker_step(NodeAxes a, int qx, int qz, const MarkerRec *__restrict__ rec,
                                                    const int *__restrict__ start, const int8_t *__restrict__ ntype,
                                                    SoftK sk, double *__restrict__ perc, double *__restrict__ strain,
                                                    double *__restrict__ fric, double *__restrict__ dil,
                                                    double *__restrict__ C) {
    const int c = blockIdx.x * 256 + threadIdx.x, n = a.Nx * a.Nz;
    if (c >= n) return;
    const int i = c % a.Nx, j = c / a.Nx;
    const int NONE = 0x7fffffff, last = start[qx * qz] - 1;
    int pos[4], end[4];
    MarkerRec h[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int bx = 2 * i - VERT + (q & 1), bz = 2 * j - VERT + (q >> 1);
        pos[q] = end[q] = 0;
        if (bx >= 0 && bx < qx && bz >= 0 && bz < qz) {
            const int b = bx + bz * qx;
            pos[q] = start[b];
            end[q] = start[b + 1];
        }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        if (last >= 0) h[q] = rec[min(pos[q], last)];
        if (pos[q] >= end[q]) h[q].k = NONE;
    }
    const double Xi = a.X[i], Zj = a.Z[j], hx = a.dx / 2.0, hz = a.dz / 2.0;
    double W = 0.0, WS = 0.0, BS = 0.0, Wph[NPH];
#pragma unroll
    for (int p = 0; p < NPH; p++) Wph[p] = 0.0;
    for (;;) {
        MarkerRec m = h[0];
        int at = pos[0], to = end[0], best = 0;
#pragma unroll
        for (int q = 1; q < 4; q++)
            if (h[q].k < m.k) {
                m = h[q];
                at = pos[q];
                to = end[q];
                best = q;
            }
        if (m.k == NONE) break;
        MarkerRec next = rec[min(at + 1, last)];
        if (at + 1 >= to) next.k = NONE;
        const double w = (1.0 - fabs(Xi - m.x) / hx) * (1.0 - fabs(Zj - m.z) / hz);
        W += w;
#pragma unroll
        for (int p = 0; p < NPH; p++)
            if (p == m.phase) Wph[p] += w;
        if (!VERT) {
            BS += m.val * w;
        } else if (node_unclamped(m.x, a.X[0], a.dx, a.Nx) == i && node_unclamped(m.z, a.Z[0], a.dz, a.Nz) == j) {
            const double dxm = 2.0 * fabs(Xi - m.x), dzm = 2.0 * fabs(Zj - m.z);
            const double ws = (1.0 - dxm / a.dx) * (1.0 - dzm / a.dz);
            WS += ws;
            BS += m.val * ws;
        }
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (q == best) {
                pos[q]++;
                h[q] = next;
            }
    }
    const int t = ntype[c];
    const bool skip = fabs(W) < 1e-30 || t == 30 || t == 31;
    double s = 0.0;
    if (!VERT) {
        if (!skip) s = BS / W;
    } else if (!(WS < 1e-30 || t == 30)) {
        s = BS / WS;
    }
    const bool air = t == 30 || (!VERT && t == 31);
    double fa = 0.0, da = 0.0, ca = 0.0;
#pragma unroll
    for (int p = 0; p < NPH; p++) {
        if (p >= sk.nph) break;
        const double fr = skip ? Wph[p] : Wph[p] / W;
        perc[(size_t)p * n + c] = fr;
        if (SOFT && !air) soften_phase(sk, p, s, fr, fa, da, ca);
    }
    if (!SOFT) {
        strain[c] = s;
        return;
    }
    fric[c] = fa;
    dil[c] = da;
    C[c] = ca;
}

void mdz_launch_cfd_nodes(int n, const double *strain, const double *perc, const int8_t *tag, int cells,
                          const SoftK &sk, double *fric, double *dil, double *C, hipStream_t s) {
    hipLaunchKernelGGL(k_cfd_nodes, dim3(mdz_div_up(n, 256)), dim3(256), 0, s, n, strain, perc, tag, cells, sk, fric,
                       dil, C);
}

/* ------------------------------------------------------------------ */
/* host side: the marker store of a context                             */
/* ------------------------------------------------------------------ */
#define MCK(x)                                                                                     \
    do {                                                                                           \
        if ((x) != hipSuccess) return mdz_error(MDZ_EHIP, "markers: " #x " failed");               \
    } while (0)

struct MarkerStore {
    int Nx, Nz;
    MarkerDev md;
    double *X[MDZ_MARKER_FAMS], *Z[MDZ_MARKER_FAMS]; /* node axes of each family slot */
    double *node_f;                                  /* one node field of the largest family */
    double *strain_n, *strain_s;                     /* plastic strain at centroids / vertices */
    int8_t *ntype;                                   /* node types of the largest family */
    double *pval;                                    /* per-phase values */
};

/* node counts of a family slot on an Nx x Nz vertex grid */
void mdz_family_dims(int fam, int Nx, int Nz, int *nx, int *nz) {
    switch (fam) {
    case 0: *nx = Nx - 1; *nz = Nz - 1; break;
    case 2: *nx = Nx; *nz = Nz + 1; break;
    case 3: *nx = Nx + 1; *nz = Nz; break;
    case MDZ_FAM_QUARTER: *nx = 2 * (Nx - 1); *nz = 2 * (Nz - 1); break;
    default: *nx = Nx; *nz = Nz; break; /* vertices, and the axes of Interp_P2N */
    }
}

static void free_markers(MarkerDev &md) {
    hipFree(md.x); hipFree(md.z); hipFree(md.phase); hipFree(md.val);
    hipFree(md.key); hipFree(md.key_out); hipFree(md.rec_in); hipFree(md.tmp);
    for (int f = 0; f < MDZ_MARKER_FAMS; f++) hipFree(md.rec[f]);
    md.x = md.z = md.val = nullptr;
    md.phase = md.key = md.key_out = nullptr;
    md.rec_in = nullptr;
    md.tmp = nullptr;
    md.tmp_bytes = 0;
    for (int f = 0; f < MDZ_MARKER_FAMS; f++) { md.rec[f] = nullptr; md.binned[f] = 0; }
    md.cap = 0;
}

void mdz_mstore_destroy(MarkerStore *s) {
    if (!s) return;
    free_markers(s->md);
    for (int f = 0; f < MDZ_MARKER_FAMS; f++) { hipFree(s->md.start[f]); hipFree(s->X[f]); hipFree(s->Z[f]); }
    hipFree(s->md.scan);
    if (s->md.long_bin) hipHostFree(s->md.long_bin);
    hipFree(s->node_f); hipFree(s->strain_n); hipFree(s->strain_s); hipFree(s->ntype);
    hipFree(s->pval);
    free(s);
}

int mdz_mstore_create(MarkerStore **out, int Nx, int Nz) {
    MarkerStore *s = (MarkerStore *)calloc(1, sizeof(MarkerStore));
    if (!s) return mdz_error(MDZ_ENOMEM, "markers: store");
    s->Nx = Nx; s->Nz = Nz;
    const size_t nmax = (size_t)(Nx + 1) * (Nz + 1);
    int rc = MDZ_OK;
    for (int f = 0; f < MDZ_MARKER_FAMS && !rc; f++) {
        int nx, nz;
        mdz_family_dims(f, Nx, Nz, &nx, &nz);
        s->md.start_cap[f] = (size_t)nx * nz + 1;
        if (hipMalloc((void **)&s->md.start[f], s->md.start_cap[f] * sizeof(int)) != hipSuccess ||
            hipMalloc((void **)&s->X[f], (size_t)nx * sizeof(double)) != hipSuccess ||
            hipMalloc((void **)&s->Z[f], (size_t)nz * sizeof(double)) != hipSuccess)
            rc = mdz_error(MDZ_ENOMEM, "markers: bins");
    }
    s->md.scan_len = nmax * 4 / 1024 + 16; /* block sums of the largest scan, its total, the flag */
    if (!rc && (hipMalloc((void **)&s->md.scan, s->md.scan_len * sizeof(int)) != hipSuccess ||
                hipHostMalloc((void **)&s->md.long_bin, sizeof(int), hipHostMallocDefault) != hipSuccess))
        rc = mdz_error(MDZ_ENOMEM, "markers: bins");
    if (!rc && (hipMalloc((void **)&s->node_f, nmax * sizeof(double)) != hipSuccess ||
                hipMalloc((void **)&s->strain_n, nmax * sizeof(double)) != hipSuccess ||
                hipMalloc((void **)&s->strain_s, nmax * sizeof(double)) != hipSuccess ||
                hipMalloc((void **)&s->ntype, nmax) != hipSuccess ||
                hipMalloc((void **)&s->pval, MDZ_MAX_PHASES * sizeof(double)) != hipSuccess))
        rc = mdz_error(MDZ_ENOMEM, "markers: node buffers");
    if (rc) { mdz_mstore_destroy(s); return rc; }
    *out = s;
    return MDZ_OK;
}

/* the family's node axes from the host grid (ParticleRoutines.c:3240-3263) */
int mdz_mstore_axes(MarkerStore *s, int fam, const grid *mesh, const double *Xh, const double *Zh, int periodic,
                    hipStream_t st, NodeAxes *a) {
    int nx, nz;
    mdz_family_dims(fam, s->Nx, s->Nz, &nx, &nz);
    if (!Xh || !Zh) {
        switch (fam) {
        case 0: Xh = mesh->xc_coord; Zh = mesh->zc_coord; break;
        case 1: Xh = mesh->xg_coord; Zh = mesh->zg_coord; break;
        case 2: Xh = mesh->xg_coord; Zh = mesh->zvx_coord; break;
        case 3: Xh = mesh->xvz_coord; Zh = mesh->zg_coord; break;
        default: break;
        }
    }
    if (!Xh || !Zh) return mdz_error(MDZ_EINVAL, "markers: node coordinates missing in the grid");
    MCK(hipMemcpyAsync(s->X[fam], Xh, (size_t)nx * sizeof(double), hipMemcpyHostToDevice, st));
    MCK(hipMemcpyAsync(s->Z[fam], Zh, (size_t)nz * sizeof(double), hipMemcpyHostToDevice, st));
    *a = NodeAxes{nx, nz, s->X[fam], s->Z[fam], mesh->dx, mesh->dz, periodic};
    return MDZ_OK;
}

/* markers (x, z, phase; and per-marker values when mval != NULL) into the
 * store; phases must lie in [-1, nph) */
int mdz_mstore_upload(MarkerStore *s, const markers *m, const double *mval, int nph, hipStream_t st) {
    MarkerDev &md = s->md;
    const int n = m->Nb_part;
    if (n < 0) return mdz_error(MDZ_EINVAL, "markers: negative count");
    if (n > 0 && (!m->x || !m->z || !m->phase)) return mdz_error(MDZ_EINVAL, "markers: x, z or phase missing");
    for (int k = 0; k < n; k++)
        if (m->phase[k] < -1 || m->phase[k] >= nph || m->phase[k] >= MDZ_MAX_PHASES)
            return mdz_error(MDZ_EINVAL, "markers: a phase outside [-1, Nb_phases)");
    if (n > md.cap) {
        free_markers(md);
        const size_t c = (size_t)n;
        /* records of a family are allocated at its first binning */
        if (hipMalloc((void **)&md.x, c * 8) != hipSuccess || hipMalloc((void **)&md.z, c * 8) != hipSuccess ||
            hipMalloc((void **)&md.phase, c * 4) != hipSuccess || hipMalloc((void **)&md.val, c * 8) != hipSuccess ||
            hipMalloc((void **)&md.key, c * 4) != hipSuccess || hipMalloc((void **)&md.key_out, c * 4) != hipSuccess ||
            hipMalloc((void **)&md.rec_in, c * sizeof(MarkerRec)) != hipSuccess) {
            free_markers(md);
            return mdz_error(MDZ_ENOMEM, "markers: arrays");
        }
        md.tmp_bytes = mdz_markers_sort_bytes(n, 4 * (s->Nx + 1) * (s->Nz + 1) + 1);
        if (md.tmp_bytes && hipMalloc(&md.tmp, md.tmp_bytes) != hipSuccess) {
            free_markers(md);
            return mdz_error(MDZ_ENOMEM, "markers: sort scratch");
        }
        md.cap = n;
    }
    md.n = n;
    for (int f = 0; f < MDZ_MARKER_FAMS; f++) md.binned[f] = 0;
    if (n > 0) {
        MCK(hipMemcpyAsync(md.x, m->x, (size_t)n * 8, hipMemcpyHostToDevice, st));
        MCK(hipMemcpyAsync(md.z, m->z, (size_t)n * 8, hipMemcpyHostToDevice, st));
        MCK(hipMemcpyAsync(md.phase, m->phase, (size_t)n * 4, hipMemcpyHostToDevice, st));
        if (mval) MCK(hipMemcpyAsync(md.val, mval, (size_t)n * 8, hipMemcpyHostToDevice, st));
        else MCK(hipMemsetAsync(md.val, 0, (size_t)n * 8, st));
    }
    return MDZ_OK;
}

/* per-marker values only (the markers already in the store) */
void mdz_mstore_rebin(MarkerStore *s) {
    for (int f = 0; f < MDZ_MARKER_FAMS; f++) s->md.binned[f] = 0;
}

int mdz_mstore_values(MarkerStore *s, const double *mval, hipStream_t st) {
    if (s->md.n > 0) MCK(hipMemcpyAsync(s->md.val, mval, (size_t)s->md.n * 8, hipMemcpyHostToDevice, st));
    /* the sorted records carry the values: sort again at the next binning */
    mdz_mstore_rebin(s);
    return MDZ_OK;
}

/* bins of a family on axes a, unless the store holds them already */
int mdz_mstore_bin(MarkerStore *s, int fam, const NodeAxes &a, hipStream_t st) {
    if (s->md.binned[fam] == a.Nx * a.Nz && fam != 4) return MDZ_OK;
    return mdz_markers_bin(s->md, fam, a, nullptr, st);
}


MarkerDev &mdz_mstore_dev(MarkerStore *s) { return s->md; }
double *mdz_mstore_node_field(MarkerStore *s) { return s->node_f; }
int8_t *mdz_mstore_node_types(MarkerStore *s) { return s->ntype; }
double *mdz_mstore_phase_values(MarkerStore *s) { return s->pval; }
double *mdz_mstore_strain(MarkerStore *s, int cells) { return cells ? s->strain_n : s->strain_s; }

SoftK mdz_soft_constants(const mat_prop *mt, int nph) {
    SoftK k;
    memset(&k, 0, sizeof(k));
    k.nph = nph < MDZ_MAX_PHASES ? nph : MDZ_MAX_PHASES;
    for (int p = 0; p < k.nph; p++) {
        k.phi[p] = mt->phi[p]; k.psi[p] = mt->psi[p]; k.C[p] = mt->C[p];
        k.phi_end[p] = mt->phi_end[p]; k.psi_end[p] = mt->psi_end[p]; k.C_end[p] = mt->C_end[p];
        k.pls_start[p] = mt->pls_start[p]; k.pls_end[p] = mt->pls_end[p];
        k.phi_soft[p] = mt->phi_soft[p]; k.psi_soft[p] = mt->psi_soft[p]; k.coh_soft[p] = mt->coh_soft[p];
    }
    return k;
}

/* CohesionFrictionDilationGrid on the store's markers (strain_pl in md.val):
 * the plastic strain by P2Mastah at the centroids and by Interp_P2N at the
 * vertices, then the softened, phase-averaged strength parameters. */
int mdz_mstore_cfd(MarkerStore *s, const NodeAxes &ac, const NodeAxes &av, int itp_stencil, const SoftK &sk,
                   const double *perc_n, const double *perc_s, const int8_t *BCp, const int8_t *BCg, double *fric_n,
                   double *dil_n, double *C_n, double *fric_s, double *dil_s, double *C_s, hipStream_t st) {
    const int nc = ac.Nx * ac.Nz, nv = av.Nx * av.Nz;
    int rc = mdz_mstore_bin(s, 0, ac, st);
    if (!rc) rc = mdz_mstore_bin(s, 1, av, st);
    if (rc) return rc;
    MCK(hipMemsetAsync(s->strain_n, 0, (size_t)nc * 8, st));
    MCK(hipMemsetAsync(s->strain_s, 0, (size_t)nv * 8, st));
    P2GArgs g{1, 0, sk.nph, s->md.val, nullptr, BCp, s->strain_n, nullptr};
    mdz_launch_p2mastah(s->md, 0, ac, 0, itp_stencil, g, st);
    P2GArgs gv{1, 0, sk.nph, s->md.val, nullptr, BCg, s->strain_s, nullptr};
    mdz_launch_interp_p2n(s->md, 1, av, gv, st);
    mdz_launch_cfd_nodes(nc, s->strain_n, perc_n, BCp, 1, sk, fric_n, dil_n, C_n, st);
    mdz_launch_cfd_nodes(nv, s->strain_s, perc_s, BCg, 0, sk, fric_s, dil_s, C_s, st);
    MCK(hipGetLastError());
    return MDZ_OK;
}

int mdz_mstore_step(MarkerStore *s, const NodeAxes &ac, const NodeAxes &av, const SoftK &sk, double *perc_n,
                    double *perc_s, const int8_t *BCp, const int8_t *BCg, double *fric_n, double *dil_n, double *C_n,
                    double *fric_s, double *dil_s, double *C_s, hipStream_t st) {
    MarkerDev &md = s->md;
    const int qx = 2 * ac.Nx, qz = 2 * ac.Nz, nc = ac.Nx * ac.Nz, nv = av.Nx * av.Nz;
    int rc = md.binned[MDZ_FAM_QUARTER] == qx * qz ? MDZ_OK : mdz_markers_bin(md, MDZ_FAM_QUARTER, ac, &av, st);
    if (rc) return rc;
    const MarkerRec *rec = md.rec[MDZ_FAM_QUARTER];
    const int *start = md.start[MDZ_FAM_QUARTER];
    const dim3 gc(mdz_div_up(nc, 256)), gv(mdz_div_up(nv, 256)), blk(256);
#define STEP(NPH, VERT, SOFT, grid, ax, tag, perc, strain, fric, dil, C)                                           \
    hipLaunchKernelGGL((k_marker_step<NPH, VERT, SOFT>), grid, blk, 0, st, ax, qx, qz, rec, start, tag, sk, perc, strain, \
                       fric, dil, C)
    /* (four phases in registers, or all that a model may have) */
    if (sk.nph <= 4) {
        STEP(4, false, true, gc, ac, BCp, perc_n, s->strain_n, fric_n, dil_n, C_n);
        if (av.periodic) STEP(4, true, false, gv, av, BCg, perc_s, s->strain_s, fric_s, dil_s, C_s);
        else STEP(4, true, true, gv, av, BCg, perc_s, s->strain_s, fric_s, dil_s, C_s);
    } else {
        STEP(MDZ_MAX_PHASES, false, true, gc, ac, BCp, perc_n, s->strain_n, fric_n, dil_n, C_n);
        if (av.periodic) STEP(MDZ_MAX_PHASES, true, false, gv, av, BCg, perc_s, s->strain_s, fric_s, dil_s, C_s);
        else STEP(MDZ_MAX_PHASES, true, true, gv, av, BCg, perc_s, s->strain_s, fric_s, dil_s, C_s);
    }
#undef STEP
    if (av.periodic) {
        hipLaunchKernelGGL(k_periodic_mean, dim3(mdz_div_up(av.Nz, 256)), blk, 0, st, s->strain_s, av.Nx, av.Nz);
        mdz_launch_cfd_nodes(nv, s->strain_s, perc_s, BCg, 0, sk, fric_s, dil_s, C_s, st);
    }
    MCK(hipGetLastError());
    return MDZ_OK;
}
