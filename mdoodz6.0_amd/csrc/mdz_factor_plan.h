/*
 * mdz_factor_plan.h -- elimination tree, layout and launches of the sparse
 * Cholesky factor of mdz_factor.hip (host code, no device types).
 *
 * Ordering: geometric nested dissection on the half-spaced lattice that
 * holds the u and v nodes.  A box of unknowns is cut by a strip as wide as
 * the matrix's reach (measured on its pattern), along the axis and at the
 * place that leave the smallest strip and two equal halves; the strip's
 * unknowns are a node of the elimination tree, the halves its children,
 * boxes of at most ND_LEAF unknowns its leaves.  A node's boundary (the rows
 * its columns reach beyond its own) is the frame of one reach around its
 * box: no graph is walked.  Where the pattern wraps around in x (periodic
 * walls), a strip at the low edge joins the root.
 */
#pragma once

#include <limits.h>
#include <stdlib.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "../../include/mdoodz_hot.h"
#include "mdz_host_parallel.h"

int mdz_error(int code, const char *msg);

#define ND_T 64 /* tile */
#ifndef ND_LEAF
#define ND_LEAF 64 /* most unknowns of a leaf */
#endif
/* One node of the elimination tree.  Rows of its front: s own unknowns
 * (positions ooff ..), then b boundary unknowns (positions blist[boff ..],
 * increasing).  Panel: (s + b) x s, column-major, at poff with leading
 * dimension ld; update matrix: b x b (lower) at uoff of its level's buffer. */
struct NdNode {
    int s, b, ld, ldu, np; /* np: column tiles, ceil(s / 64) */
    int ooff, boff;
    int child[2];  /* -1: none */
    int inv[2];    /* per child: map from a row of this front to the child's boundary row (or -1) */
    int lin;       /* first 64 x 64 block of the inverses of the diagonal tiles */
    long long poff, uoff;
};
struct NdTask {
    int node, a, b;
};

/* One workgroup of a solve: its front, where the rows of T are, and its tile.
 * Maps ga, gb: from a row of the front to the update vectors of its children,
 * all levels' in one array (its last entry, always zero, where the child has
 * no such row); -1: no such child. */
struct NdSolve {
    long long toff;
    int s, b, ld, panels, ooff, boff, ga, gb, tile, pad;
};

struct NdRange {
    int first, count;
};
struct NdLevel {
    NdRange assemble, forward, backward;
    int rt, ct; /* tile sizes of the solves */
    std::vector<NdRange> panel;
};

/* the host's side of the factor: tree, layout and launches */
struct NdPlan {
    std::vector<NdLevel> level; /* leaves first, the root's level last */
    std::vector<NdRange> invert;
    std::vector<NdNode> node;
    std::vector<NdTask> task;
    std::vector<NdSolve> solve;
    std::vector<int> at; /* inv with places in the array of update vectors */
    std::vector<int> pos, eq, node_of; /* position of an equation, and back; node of a position */
    std::vector<int> blist, inv;
    size_t panel_len = 0, ulen[2] = {0, 0}, nlin = 0;

    /* gives back what only the device reads, once it is there: level, invert, eq and the
     * lengths remain */
    void release_uploaded() {
        std::vector<NdNode>().swap(node);
        std::vector<NdTask>().swap(task);
        std::vector<NdSolve>().swap(solve);
        for (std::vector<int> *v : {&at, &pos, &node_of, &blist, &inv}) std::vector<int>().swap(*v);
    }
};

namespace {

/* the unknowns on the half-spaced lattice: u node (k, l) at (2 k + 1, 2 l),
 * v node at (2 k, 2 l + 1) */
struct Lattice {
    int W, H;
    std::vector<int> at;          /* unknown at (x, z), x fastest, or -1 */
    std::vector<int> sum;         /* (W + 1) x (H + 1) prefix counts */
    int count(int x0, int x1, int z0, int z1) const {
        const size_t w = (size_t)W + 1;
        return sum[z1 * w + x1] - sum[z0 * w + x1] - sum[z1 * w + x0] + sum[z0 * w + x0];
    }
};

struct Box {
    int x0, x1, z0, z1;
};
struct TreeNode {
    Box box;
    int depth, child[2];
    int own, nown; /* range of the list of unknowns */
};

/* cut position c of [lo, hi) in one axis: the strip [c, c + reach) leaves
 * sides as equal as they get; -1 where no cut leaves two sides */
template <class Count>
int cut_at(int lo, int hi, int reach, int total, Count below) {
    int a = lo + 1, b = hi - reach - 1;
    if (a > b) return -1;
    while (a < b) {
        const int mid = (a + b) >> 1;
        /* left count >= right count */
        if (below(mid) >= total - below(mid + reach)) b = mid;
        else a = mid + 1;
    }
    return a;
}

} // namespace

static int nd_plan(NdPlan &plan, int Nx, int Nz, int n, const int *mom_node, const std::vector<int> &Ic,
                   const std::vector<int> &J) {
    Lattice G;
    G.W = 2 * Nx + 2;
    G.H = 2 * Nz + 2;
    G.at.assign((size_t)G.W * G.H, -1);
    std::vector<int> px(n), pz(n);
    const long long nun = (long long)Nx * (Nz + 1), nvn = (long long)(Nx + 1) * Nz;
    int xlo = INT_MAX, xhi = 0, zlo = INT_MAX, zhi = 0;
    for (int i = 0; i < n; i++) {
        const long long q = mom_node[i];
        if (q < 0 || q >= nun + nvn) return mdz_error(MDZ_EINVAL, "factor: node of an equation");
        if (q < nun) {
            px[i] = 2 * (int)(q % Nx) + 1;
            pz[i] = 2 * (int)(q / Nx);
        } else {
            px[i] = 2 * (int)((q - nun) % (Nx + 1));
            pz[i] = 2 * (int)((q - nun) / (Nx + 1)) + 1;
        }
        int &slot = G.at[(size_t)pz[i] * G.W + px[i]];
        if (slot >= 0) return mdz_error(MDZ_EINVAL, "factor: two equations on one node");
        slot = i;
        xlo = std::min(xlo, px[i]); xhi = std::max(xhi, px[i]);
        zlo = std::min(zlo, pz[i]); zhi = std::max(zhi, pz[i]);
    }
    G.sum.assign((size_t)(G.W + 1) * (G.H + 1), 0);
    for (int z = 0; z < G.H; z++) {
        int run = 0;
        for (int x = 0; x < G.W; x++) {
            run += G.at[(size_t)z * G.W + x] >= 0;
            G.sum[(size_t)(z + 1) * (G.W + 1) + x + 1] = G.sum[(size_t)z * (G.W + 1) + x + 1] + run;
        }
    }
    /* reach of the pattern; an entry closer around the x period than across
     * it wraps */
    const int period = 2 * (Nx - 1);
    int rx = 1, rz = 1;
    bool wrap = false;
    {
        std::mutex mu;
        mdz_host_parallel(n, 20000, [&](long long i0, long long i1) {
            int ax = 1, az = 1;
            bool w = false;
            for (long long i = i0; i < i1; i++)
                for (int e = Ic[(size_t)i]; e < Ic[(size_t)i + 1]; e++) {
                    const int k = J[(size_t)e];
                    int dx = std::abs(px[(size_t)i] - px[(size_t)k]);
                    if (dx > 1 && period - dx >= 0 && period - dx < dx) {
                        dx = period - dx;
                        w = true;
                    }
                    ax = std::max(ax, dx);
                    az = std::max(az, std::abs(pz[(size_t)i] - pz[(size_t)k]));
                }
            std::lock_guard<std::mutex> g(mu);
            rx = std::max(rx, ax);
            rz = std::max(rz, az);
            wrap = wrap || w;
        });
    }
    /* the tree */
    std::vector<TreeNode> T;
    std::vector<int> list;
    list.reserve(n);
    auto take = [&](const Box &b) {
        for (int z = b.z0; z < b.z1; z++)
            for (int x = b.x0; x < b.x1; x++) {
                const int i = G.at[(size_t)z * G.W + x];
                if (i >= 0) list.push_back(i);
            }
    };
    struct Todo {
        Box box;
        int depth, parent, slot;
    };
    std::vector<Todo> todo;
    todo.push_back({{xlo, xhi + 1, zlo, zhi + 1}, 0, -1, 0});
    while (!todo.empty()) {
        const Todo td = todo.back();
        todo.pop_back();
        const int id = (int)T.size();
        T.push_back({td.box, td.depth, {-1, -1}, (int)list.size(), 0});
        if (td.parent >= 0) T[td.parent].child[td.slot] = id;
        Box b = td.box;
        if (td.parent < 0 && wrap) {
            const Box edge{b.x0, std::min(b.x1, b.x0 + rx), b.z0, b.z1};
            take(edge);
            b.x0 = edge.x1;
        }
        const int total = b.x0 < b.x1 ? G.count(b.x0, b.x1, b.z0, b.z1) : 0;
        int cx = -1, cz = -1;
        if (total > ND_LEAF) {
            cx = cut_at(b.x0, b.x1, rx, total, [&](int c) { return G.count(b.x0, c, b.z0, b.z1); });
            cz = cut_at(b.z0, b.z1, rz, total, [&](int c) { return G.count(b.x0, b.x1, b.z0, c); });
        }
        if (cx < 0 && cz < 0) {
            if (total > 0) take(b);
        } else {
            const int nx = cx < 0 ? INT_MAX : G.count(cx, cx + rx, b.z0, b.z1);
            const int nz = cz < 0 ? INT_MAX : G.count(b.x0, b.x1, cz, cz + rz);
            Box lo = b, hi = b, strip = b;
            if (nx <= nz) {
                lo.x1 = strip.x0 = cx;
                hi.x0 = strip.x1 = cx + rx;
            } else {
                lo.z1 = strip.z0 = cz;
                hi.z0 = strip.z1 = cz + rz;
            }
            take(strip);
            if (G.count(lo.x0, lo.x1, lo.z0, lo.z1) > 0) todo.push_back({lo, td.depth + 1, id, 0});
            if (G.count(hi.x0, hi.x1, hi.z0, hi.z1) > 0) todo.push_back({hi, td.depth + 1, id, 1});
        }
        T[id].nown = (int)list.size() - T[id].own;
    }
    /* nodes by level, the deepest first; elimination positions in that order */
    int depth = 0;
    for (auto &t : T) depth = std::max(depth, t.depth);
    const int nt = (int)T.size(), nl = depth + 1;
    std::vector<int> order(nt), rank(nt), lfirst(nl + 1, 0);
    for (auto &t : T) lfirst[depth - t.depth + 1]++;
    for (int q = 0; q < nl; q++) lfirst[q + 1] += lfirst[q];
    {
        std::vector<int> at(lfirst.begin(), lfirst.end() - 1);
        for (int t = 0; t < nt; t++) {
            rank[t] = at[depth - T[t].depth]++;
            order[rank[t]] = t;
        }
    }
    std::vector<int> &pos = plan.pos, &eq = plan.eq, &node_of = plan.node_of;
    pos.resize(n);
    eq.resize(n);
    node_of.resize(n);
    std::vector<NdNode> &N = plan.node;
    N.assign(nt, NdNode());
    int at = 0;
    for (int q = 0; q < nt; q++) {
        const TreeNode &t = T[order[q]];
        NdNode &k = N[q];
        k.s = t.nown;
        k.ooff = at;
        k.np = (k.s + ND_T - 1) / ND_T;
        for (int c = 0; c < 2; c++) k.child[c] = t.child[c] < 0 ? -1 : rank[t.child[c]];
        for (int i = 0; i < t.nown; i++, at++) {
            eq[at] = list[(size_t)t.own + i];
            pos[eq[at]] = at;
            node_of[at] = q;
        }
    }
    /* boundaries: the frame of one reach around each box */
    std::vector<std::vector<int>> B(nt);
    bool ordered = true;
    {
        std::mutex mu;
        mdz_host_parallel(nt, 64, [&](long long q0, long long q1) {
            std::vector<int> cols;
            bool good = true;
            for (long long q = q0; q < q1; q++) {
                const Box &b = T[order[(size_t)q]].box;
                std::vector<int> &out = B[(size_t)q];
                cols.clear();
                for (int x = b.x0 - rx; x < b.x1 + rx; x++) {
                    if (x >= xlo && x <= xhi) cols.push_back(x);
                    if (wrap && (x < b.x0 || x >= b.x1)) {
                        if (x + period >= xlo && x + period <= xhi) cols.push_back(x + period);
                        if (x - period >= xlo && x - period <= xhi) cols.push_back(x - period);
                    }
                }
                const int za = std::max(zlo, b.z0 - rz), zb = std::min(zhi + 1, b.z1 + rz);
                for (int z = za; z < zb; z++) {
                    const bool inz = z >= b.z0 && z < b.z1;
                    for (int x : cols) {
                        if (inz && x >= b.x0 && x < b.x1) continue;
                        const int i = G.at[(size_t)z * G.W + x];
                        if (i >= 0) out.push_back(pos[i]);
                    }
                }
                std::sort(out.begin(), out.end());
                out.erase(std::unique(out.begin(), out.end()), out.end());
                if (!out.empty() && out[0] < N[(size_t)q].ooff + N[(size_t)q].s) good = false;
            }
            std::lock_guard<std::mutex> g(mu);
            ordered = ordered && good;
        });
    }
    if (!ordered) return mdz_error(MDZ_EINVAL, "factor: boundary of a separator");
    long long poff = 0, boff = 0, ioff = 0, lin = 0;
    size_t ulen[2] = {0, 0};
    for (int lv = 0; lv < nl; lv++) {
        long long uoff = 0;
        for (int q = lfirst[lv]; q < lfirst[lv + 1]; q++) {
            NdNode &k = N[q];
            k.b = (int)B[q].size();
            const int m = k.s + k.b;
            k.ld = (m + 7) & ~7;
            k.ldu = (k.b + 7) & ~7;
            k.poff = poff;
            poff += (long long)k.ld * k.s;
            k.uoff = uoff;
            uoff += (long long)k.ldu * k.b;
            if (boff + k.b >= INT_MAX || lin + k.np > INT_MAX || ioff + 2LL * m > INT_MAX)
                return mdz_error(MDZ_EUNSUPPORTED, "factor: too many unknowns");
            k.boff = (int)boff;
            boff += k.b;
            k.lin = (int)lin;
            lin += k.np;
            for (int c = 0; c < 2; c++) {
                k.inv[c] = (int)ioff;
                if (k.child[c] >= 0) ioff += m;
            }
        }
        ulen[lv & 1] = std::max(ulen[lv & 1], (size_t)uoff);
    }
    std::vector<int> &blist = plan.blist, &inv = plan.inv;
    std::vector<int> &at_g = plan.at;
    blist.resize((size_t)boff);
    inv.resize((size_t)ioff);
    at_g.resize((size_t)ioff);
    bool nested = true;
    {
        std::mutex mu;
        mdz_host_parallel(nt, 64, [&](long long q0, long long q1) {
            bool good = true;
            for (long long q = q0; q < q1; q++) {
                const NdNode &k = N[(size_t)q];
                std::copy(B[(size_t)q].begin(), B[(size_t)q].end(), blist.begin() + k.boff);
                for (int c = 0; c < 2; c++) {
                    if (k.child[c] < 0) continue;
                    const std::vector<int> &kb = B[(size_t)k.child[c]];
                    const int first = N[(size_t)k.child[c]].boff;
                    int *v = inv.data() + k.inv[c], *g = at_g.data() + k.inv[c];
                    size_t p = 0;
                    for (int r = 0; r < k.s + k.b; r++) {
                        const int at_r = r < k.s ? k.ooff + r : B[(size_t)q][r - k.s];
                        v[r] = p < kb.size() && kb[p] == at_r ? (int)p++ : -1;
                        g[r] = v[r] < 0 ? (int)boff : first + v[r];
                    }
                    if (p != kb.size()) good = false;
                }
            }
            std::lock_guard<std::mutex> g(mu);
            nested = nested && good;
        });
    }
    if (!nested) return mdz_error(MDZ_EINVAL, "factor: boundary of a child outside its parent's front");
    /* launches */
    std::vector<NdTask> &task = plan.task;
    task.clear();
    plan.solve.clear();
    plan.level.assign(nl, NdLevel());
    plan.invert.clear();
    int npmax = 0;
    for (int lv = 0; lv < nl; lv++) {
        NdLevel &L = plan.level[lv];
        const int q0 = lfirst[lv], q1 = lfirst[lv + 1];
        auto begin = [&] { return (int)task.size(); };
        auto end = [&](int first) { return NdRange{first, (int)task.size() - first}; };
        int first = begin(), panels = 0;
        long long rows = 0, cols = 0;
        for (int q = q0; q < q1; q++) {
            const NdNode &k = N[q];
            const int tiles = k.np + (k.b + ND_T - 1) / ND_T;
            const bool leaf = k.child[0] < 0 && k.child[1] < 0;
            for (int c = 0; c < k.np; c++)
                for (int r = c; r < tiles; r++)
                    if (!leaf || (r == 0 && c == 0)) task.push_back({q, r, c});
            panels = std::max(panels, std::max(1, k.np));
            npmax = std::max(npmax, k.np);
            rows += k.s + k.b;
            cols += k.s;
        }
        L.assemble = end(first);
        for (int p = 0; p < panels; p++) {
            first = begin();
            for (int q = q0; q < q1; q++) {
                const NdNode &k = N[q];
                if (p >= std::max(1, k.np)) continue;
                const int tiles = k.np + (k.b + ND_T - 1) / ND_T;
                for (int c = std::min(p + 1, k.np); c < tiles; c++)
                    for (int r = c; r < tiles; r++) task.push_back({q, r, c});
            }
            L.panel.push_back(end(first));
        }
        /* tiles of the solves: as tall as keeps two workgroups per CU busy */
        L.rt = rows >= 64 * 512 ? 64 : rows >= 32 * 512 ? 32 : 16;
        L.ct = cols >= 64 * 512 ? 64 : cols >= 32 * 512 ? 32 : 16;
        auto solve = [&](const NdNode &k, int tile) {
            return NdSolve{k.poff, k.s,    k.b,    k.ld, k.np, k.ooff, k.boff, k.child[0] < 0 ? -1 : k.inv[0],
                           k.child[1] < 0 ? -1 : k.inv[1], tile, 0};
        };
        first = (int)plan.solve.size();
        for (int q = q0; q < q1; q++)
            for (int r = 0; r < N[q].s + N[q].b; r += L.rt) plan.solve.push_back(solve(N[q], r / L.rt));
        L.forward = {first, (int)plan.solve.size() - first};
        first = (int)plan.solve.size();
        for (int q = q0; q < q1; q++)
            for (int c = 0; c < N[q].s; c += L.ct) plan.solve.push_back(solve(N[q], c / L.ct));
        L.backward = {first, (int)plan.solve.size() - first};
    }
    for (int p = 0; p < (npmax > 1 ? npmax : 0); p++) { /* (fronts of one panel need none) */
        const int first = (int)task.size();
        for (int q = 0; q < nt; q++) {
            const NdNode &k = N[q];
            const int j = k.np - 1 - p, tiles = k.np + (k.b + ND_T - 1) / ND_T;
            if (j < 0 || k.np < 2) continue;
            for (int r = j; r < tiles; r++) task.push_back({q, j, r});
        }
        plan.invert.push_back({first, (int)task.size() - first});
    }
    plan.panel_len = (size_t)poff;
    plan.nlin = (size_t)lin;
    plan.ulen[0] = ulen[0];
    plan.ulen[1] = ulen[1];
    return MDZ_OK;
}
