/*
 * Host check of the factor's plan (mdz_factor_plan.h): a multifrontal
 * Cholesky carried out on the host from the plan alone, on random symmetric
 * diagonally dominant matrices over staggered lattices, against the matrix
 * itself.  Prints one line per system and exits with the number that fail.
 */
#include <math.h>
#include <stdio.h>

#include <random>

#include "../mdoodz6.0_amd/csrc/mdz_factor_plan.h"

int mdz_error(int code, const char *msg) {
    printf("error %d %s\n", code, msg);
    return code;
}

/* u and v unknowns of an Nx x Nz grid without the outermost nodes (kept at
 * the low edge of a periodic grid), a share `drop` of them taken out; every
 * pair within `reach` half spacings is coupled, around the x period too where
 * periodic */
static int check(int Nx, int Nz, int reach, bool periodic, double drop, int seed) {
    std::mt19937 gen(seed);
    std::uniform_real_distribution<double> U(0.0, 1.0);
    const int nun = Nx * (Nz + 1), nvn = (Nx + 1) * Nz, W = 2 * Nx + 2, H = 2 * Nz + 2, per = 2 * (Nx - 1);
    std::vector<int> mom, px, pz, at((size_t)W * H, -1);
    for (int q = 0; q < nun + nvn; q++) {
        const bool u = q < nun;
        const int k = u ? q % Nx : (q - nun) % (Nx + 1), l = u ? q / Nx : (q - nun) / (Nx + 1);
        if (l == 0 || l == (u ? Nz : Nz - 1) || k == (u ? Nx - 1 : Nx) || (k == 0 && !(u && periodic))) continue;
        if (U(gen) < drop) continue;
        at[(size_t)(u ? 2 * l : 2 * l + 1) * W + (u ? 2 * k + 1 : 2 * k)] = (int)mom.size();
        mom.push_back(q);
        px.push_back(u ? 2 * k + 1 : 2 * k);
        pz.push_back(u ? 2 * l : 2 * l + 1);
    }
    const int n = (int)mom.size();
    if (n < 1) return 0;
    std::vector<int> Ic(1, 0), J;
    for (int i = 0; i < n; i++) {
        std::vector<int> row;
        for (int z = std::max(0, pz[i] - reach); z <= std::min(H - 1, pz[i] + reach); z++)
            for (int x = px[i] - reach; x <= px[i] + reach; x++)
                for (int t = periodic ? -per : 0; t <= (periodic ? per : 0); t += std::max(per, 1)) {
                    const int xx = x + t;
                    if (xx >= 0 && xx < W && at[(size_t)z * W + xx] >= 0) row.push_back(at[(size_t)z * W + xx]);
                }
        std::sort(row.begin(), row.end());
        row.erase(std::unique(row.begin(), row.end()), row.end());
        J.insert(J.end(), row.begin(), row.end());
        Ic.push_back((int)J.size());
    }
    NdPlan p;
    if (nd_plan(p, Nx, Nz, n, mom.data(), Ic, J)) return 1;
    /* launches stay inside the fronts they name */
    bool ok = true;
    auto all = [&](const NdRange &r, auto fine) {
        for (int q = r.first; q < r.first + r.count; q++)
            ok = ok && q >= 0 && q < (int)p.task.size() && fine(p.node[p.task[q].node], p.task[q]);
    };
    auto tiles = [](const NdNode &k) { return k.np + (k.b + ND_T - 1) / ND_T; };
    for (const NdLevel &L : p.level) {
        all(L.assemble, [&](const NdNode &k, NdTask t) { return t.b < k.np && t.a >= t.b && t.a < tiles(k); });
        for (int j = 0; j < (int)L.panel.size(); j++)
            all(L.panel[j], [&](const NdNode &k, NdTask t) {
                return j < std::max(1, k.np) && t.b >= std::min(j + 1, k.np) && t.a >= t.b && t.a < tiles(k);
            });
        for (const NdRange *r : {&L.forward, &L.backward})
            for (int q = r->first; q < r->first + r->count; q++) {
                const NdSolve &t = p.solve[q];
                ok = ok && t.tile * (r == &L.forward ? L.rt : L.ct) < t.s + (r == &L.forward ? t.b : 0) &&
                     t.toff + (long long)t.ld * t.s <= (long long)p.panel_len && t.ooff + t.s <= n &&
                     t.boff + t.b <= (int)p.blist.size();
                for (int m : {t.ga, t.gb})
                    ok = ok && (m < 0 || (size_t)m + t.s + t.b <= p.at.size());
            }
    }
    for (int a : p.at) ok = ok && a >= 0 && a <= (int)p.blist.size();
    for (const NdRange &r : p.invert)
        all(r, [&](const NdNode &k, NdTask t) { return t.a < k.np && t.b >= t.a && t.b < tiles(k); });
    /* the matrix, its fronts */
    std::vector<double> val(J.size(), 0.0), diag(n, 0.1);
    for (int i = 0; i < n; i++)
        for (int e = Ic[i]; e < Ic[i + 1]; e++)
            if (J[e] < i) {
                val[e] = -U(gen);
                diag[i] -= val[e];
                diag[J[e]] -= val[e];
            }
    std::vector<std::vector<double>> F(p.node.size());
    for (size_t q = 0; q < F.size(); q++) {
        const size_t m = (size_t)p.node[q].s + p.node[q].b;
        F[q].assign(m * m, 0.0);
        ok = ok && p.node[q].poff + (long long)p.node[q].ld * p.node[q].s <= (long long)p.panel_len;
    }
    for (int i = 0; i < n; i++)
        for (int e = Ic[i]; e < Ic[i + 1]; e++) {
            if (J[e] > i) continue;
            if (J[e] == i) val[e] = diag[i];
            const int lo = std::min(p.pos[i], p.pos[J[e]]), hi = std::max(p.pos[i], p.pos[J[e]]), q = p.node_of[lo];
            const NdNode &k = p.node[q];
            int r = hi - k.ooff;
            if (r >= k.s) {
                const auto b = p.blist.begin() + k.boff, f = std::lower_bound(b, b + k.b, hi);
                if (f == b + k.b || *f != hi) {
                    printf("an entry has no place\n");
                    return 1;
                }
                r = k.s + (int)(f - b);
            }
            F[q][(size_t)(lo - k.ooff) * (k.s + k.b) + r] = val[e];
        }
    std::vector<double> b(n), x(n);
    for (int i = 0; i < n; i++) b[i] = x[p.pos[i]] = U(gen) - 0.5;
    auto place = [&](const NdNode &k, int r) { return r < k.s ? k.ooff + r : p.blist[k.boff + r - k.s]; };
    for (size_t q = 0; q < F.size(); q++) {
        const NdNode &k = p.node[q];
        const int m = k.s + k.b;
        std::vector<double> &M = F[q];
        for (int c = 0; c < 2; c++) {
            if (k.child[c] < 0) continue;
            const NdNode &K = p.node[k.child[c]];
            const std::vector<double> &MK = F[k.child[c]];
            for (int cc = 0; cc < m; cc++)
                for (int r = cc; r < m; r++) {
                    const int ir = p.inv[k.inv[c] + r], ic = p.inv[k.inv[c] + cc];
                    ok = ok && ir < K.b && ic < K.b && (ir < 0 || ic < 0 || ir >= ic) &&
                         p.at[k.inv[c] + r] == (ir < 0 ? (int)p.blist.size() : K.boff + ir);
                    if (ir >= 0 && ic >= 0) M[(size_t)cc * m + r] += MK[(size_t)(K.s + ic) * (K.s + K.b) + K.s + ir];
                }
        }
        for (int c = 0; c < k.s; c++) {
            const double d = sqrt(M[(size_t)c * m + c]);
            for (int r = c; r < m; r++) M[(size_t)c * m + r] /= d;
            for (int c2 = c + 1; c2 < m; c2++)
                for (int r = c2; r < m; r++) M[(size_t)c2 * m + r] -= M[(size_t)c * m + r] * M[(size_t)c * m + c2];
            x[k.ooff + c] /= M[(size_t)c * m + c];
            for (int r = c + 1; r < m; r++) x[place(k, r)] -= M[(size_t)c * m + r] * x[k.ooff + c];
        }
    }
    for (size_t q = F.size(); q-- > 0;) {
        const NdNode &k = p.node[q];
        const int m = k.s + k.b;
        for (int c = k.s - 1; c >= 0; c--) {
            for (int r = c + 1; r < m; r++) x[k.ooff + c] -= F[q][(size_t)c * m + r] * x[place(k, r)];
            x[k.ooff + c] /= F[q][(size_t)c * m + c];
        }
    }
    std::vector<double> res(b);
    for (int i = 0; i < n; i++)
        for (int e = Ic[i]; e < Ic[i + 1]; e++) {
            if (J[e] > i) continue;
            res[i] -= val[e] * x[p.pos[J[e]]];
            if (J[e] < i) res[J[e]] -= val[e] * x[p.pos[i]];
        }
    double num = 0.0, den = 0.0;
    for (int i = 0; i < n; i++) {
        num += res[i] * res[i];
        den += b[i] * b[i];
    }
    const double err = sqrt(num / den);
    /* what the device holds is given back; the next analysis makes the same plan */
    const std::vector<int> pos = p.pos, at_kept = p.at, blist = p.blist, inv = p.inv, node_of = p.node_of;
    const size_t counts[3] = {p.node.size(), p.task.size(), p.solve.size()};
    p.release_uploaded();
    ok = ok && p.node.capacity() + p.task.capacity() + p.solve.capacity() + p.at.capacity() + p.pos.capacity() +
                       p.node_of.capacity() + p.blist.capacity() + p.inv.capacity() ==
                   0;
    ok = ok && !p.level.empty() && (int)p.eq.size() == n;
    if (nd_plan(p, Nx, Nz, n, mom.data(), Ic, J)) return 1;
    ok = ok && p.pos == pos && p.at == at_kept && p.blist == blist && p.inv == inv && p.node_of == node_of &&
         p.node.size() == counts[0] && p.task.size() == counts[1] && p.solve.size() == counts[2];
    printf("%d x %d reach %d periodic %d drop %.1f: %d unknowns, %zu fronts, %zu levels, residual %.1e\n", Nx, Nz, reach,
           (int)periodic, drop, n, F.size(), p.level.size(), err);
    return !(ok && err < 1e-12);
}

int main() {
    const int grid[7][2] = {{22, 17}, {9, 30}, {4, 4}, {3, 40}, {41, 3}, {2, 2}, {46, 23}};
    int bad = 0;
    for (const auto &g : grid)
        for (int reach = 1; reach <= 4; reach++)
            for (int periodic = 0; periodic < 2; periodic++)
                for (double drop : {0.0, 0.3, 0.9}) bad += check(g[0], g[1], reach, periodic, drop, 7);
    printf("%d failed\n", bad);
    return bad;
}
