// Host check of the dense-node plans (csrc/hdd_nodeplan.h), compiled and called by
// tests/test_nodeplan.py: plans the solves of a few factors, checks that every index the kernels
// use stays inside its array, and carries the plan out in double, operand by operand as the kernels
// do, against the factors' own solves.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <map>
#include <string>
#include <vector>
#include "../hierarchicaldd_amd/csrc/hdd_nodeplan.h"

using namespace hdd;

namespace {

constexpr int T = NodePlanHost::kTile;
struct Failed { std::string what; };
void need(bool ok, const char* what) { if (!ok) throw Failed{what}; }

// 7-point operator of a box with some cells left out, its diagonal perturbed by `seed` (0: not)
void box_matrix(int nx, int ny, int nz, int hole, unsigned seed, Csr& A, std::vector<Int3>& xyz) {
    std::vector<int> id((size_t)nx * ny * nz, -1);
    auto at = [&](int x, int y, int z) -> int& { return id[((size_t)x * ny + y) * nz + z]; };
    for (int x = 0; x < nx; ++x)
        for (int y = 0; y < ny; ++y)
            for (int z = 0; z < nz; ++z) {
                const int dx = 2 * x - nx, dy = 2 * y - ny, dz = 2 * z - nz;
                if (hole && dx * dx + dy * dy + dz * dz < hole * hole) continue;
                at(x, y, z) = (int)xyz.size();
                xyz.push_back({x, y, z});
            }
    A.rows = A.cols = (int)xyz.size();
    for (int i = 0; i < A.rows; ++i) {
        const Int3 c = xyz[i];
        std::vector<std::pair<int, float>> row;
        seed = seed ? seed * 1664525u + 1013904223u : 0;
        row.push_back({i, 6.f + (seed >> 24) / 256.f});
        const int d[6][3] = {{-1, 0, 0}, {1, 0, 0}, {0, -1, 0}, {0, 1, 0}, {0, 0, -1}, {0, 0, 1}};
        for (auto& s : d) {
            const int X = c.x + s[0], Y = c.y + s[1], Z = c.z + s[2];
            if (X < 0 || Y < 0 || Z < 0 || X >= nx || Y >= ny || Z >= nz || at(X, Y, Z) < 0) continue;
            row.push_back({at(X, Y, Z), -1.f});
        }
        std::sort(row.begin(), row.end());
        for (auto& e : row) { A.idx.push_back(e.first); A.val.push_back(e.second); }
        A.ptr.push_back((int)A.idx.size());
    }
}

void check_indices(const NodePlanHost& P) {
    const int ni = (int)P.inst_prob.size();
    std::vector<int> fcount(P.ysize / T + 1, 0), ccount(P.csize / T + 1, 0), bcount(P.ysize / T + 1, 0);
    auto item = [&](const NodeItem& it, bool fwd, const NodePlanHost::Level& L) {
        const int waves = fwd ? L.fwd_waves : L.bwd_waves;
        need(it.cnt >= 1 && it.cnt <= NodePlanHost::kRun && it.inst0 >= 0 && it.inst0 + it.cnt <= ni, "run");
        need(it.split >= 1 && (it.split & (it.split - 1)) == 0 && it.split <= waves && (waves == 4 ? it.split <= 4 : it.split == 16), "split");
        need(it.rt0 >= 0 && it.rt0 < it.rt1 && it.rt1 <= it.nk + (fwd ? it.nrk : 0), "row tiles");
        need(it.cnt * (T * (it.nk + (fwd ? 0 : it.nrk)) + 4) <= (fwd ? L.fwd_lds : L.bwd_lds), "LDS");
        need((fwd ? L.fwd_lds : L.bwd_lds) <= NodePlanHost::kMaxLdsFloats, "LDS size");
        need(it.scale >= 0 && it.scale + T * it.nk <= P.scales && it.scale % 4 == 0, "scale");
        for (int r = it.rt0; r < it.rt1; ++r) {
            if (fwd && !it.nrk) {
                need(it.tile >= 0 && it.tile + (long long)(r + 1) * it.nk <= P.tiles, "tiles");
                continue;
            }
            const long long base = it.tile + (fwd ? (r < it.nk ? (long long)r * (r + 1) / 2 : (long long)it.nk * (it.nk + 1) / 2 + (long long)(r - it.nk) * it.nk)
                                                  : (long long)r * (it.nk + it.nrk) - (long long)r * (r - 1) / 2);
            const long long nt = fwd ? (r < it.nk ? r + 1 : it.nk) : it.nk + it.nrk - r;
            need(base >= 0 && base + nt <= P.tiles, "tiles");
        }
        for (int j = 0; j < it.cnt; ++j) {
            const int y = it.y0 + j * T * it.nk, c = it.c0 + j * T * it.nrk;
            need(y >= L.y0 && y % T == 0 && y + T * it.nk <= L.y1 && L.y1 <= P.ysize, "columns");
            need(c >= L.c0 && c % T == 0 && c + T * it.nrk <= L.c1 && L.c1 <= P.csize, "boundary rows");
            if (fwd && !it.nrk) for (int r = it.rt0; r < it.rt1; ++r) ++bcount[y / T + r];  // the whole solve
            for (int r = it.rt0; r < it.rt1; ++r) ++(fwd ? (r < it.nk ? fcount[y / T + r] : ccount[c / T + r - it.nk]) : bcount[y / T + r]);
        }
    };
    for (const auto& L : P.levels) {
        for (int i = L.fwd0; i < L.fwd1; ++i) item(P.fwd[i], true, L);
        for (int i = L.bwd0; i < L.bwd1; ++i) item(P.bwd[i], false, L);
    }
    for (int i = 0; i < P.ysize / T; ++i) need(fcount[i] == 1 && bcount[i] == 1, "every column tile once per pass");
    for (int i = 0; i < P.csize / T; ++i) need(ccount[i] == 1, "every boundary tile once");
    for (int v : P.orig) need(v >= -1 && v < P.n, "orig");
    for (int v : P.zidx) need(v >= 0 && v <= P.ysize, "zidx");
    auto pos = [&](const NodePos& q) {
        need(q.p0 >= 0 && q.p0 <= P.csize, "position");
        if (q.p1 >= 0) { need(q.p1 <= P.csize, "position"); return; }
        const int m = ~q.p1;
        need(m < (int)P.more.size() && m + P.more[m] < (int)P.more.size(), "list");
        for (int e = 1; e <= P.more[m]; ++e) need(P.more[m + e] >= 0 && P.more[m + e] < P.csize, "list entry");
    };
    need((int)P.pos_y.size() == P.ysize && (int)P.pos_c.size() == P.csize, "position arrays");
    for (auto& q : P.pos_y) pos(q);
    for (auto& q : P.pos_c) pos(q);
}

// the solve in double: per block S, W and D^-2, then the two passes
double emulate(const NodePlanHost& P, const std::vector<const SupernodalFactor*>& F, const std::vector<int>& off) {
    std::vector<std::vector<double>> S(P.blocks.size()), W(P.blocks.size()), D2(P.blocks.size());
    std::map<int, int> by_fwd, by_bwd;
    for (size_t k = 0; k < P.blocks.size(); ++k) {
        const auto& B = P.blocks[k];
        const int np = T * B.nk, nr = T * B.nrk;
        std::vector<double> L((size_t)(np + nr) * np), inv((size_t)np * np, 0.0);
        node_block_columns(B, L.data());
        for (int i = 0; i < np; ++i) for (int j = 0; j <= i; ++j) inv[(size_t)j * np + i] = L[(size_t)i * np + j];
        invert_lower(inv, np);
        S[k].assign((size_t)np * np, 0.0); W[k].assign((size_t)nr * np, 0.0); D2[k].resize(np);
        if (!nr) {  // closed: the inverse
            for (int i = 0; i < np; ++i)
                for (int j = 0; j < np; ++j)
                    for (int q = std::max(i, j); q < np; ++q) S[k][(size_t)i * np + j] += inv[(size_t)i * np + q] * inv[(size_t)j * np + q];
            by_fwd[B.fwd] = (int)k;
            continue;
        }
        for (int i = 0; i < np; ++i) {
            const double d = L[(size_t)i * np + i];
            D2[k][i] = 1.0 / (d * d);
            for (int j = 0; j < i; ++j) S[k][(size_t)i * np + j] = d * inv[(size_t)j * np + i];
        }
        for (int a = 0; a < nr; ++a)
            for (int q = 0; q < np; ++q) {
                const double l = L[(size_t)(np + a) * np + q];
                if (l != 0) for (int j = 0; j <= q; ++j) W[k][(size_t)a * np + j] += l * inv[(size_t)j * np + q];
            }
        by_fwd[B.fwd] = (int)k; by_bwd[B.bwd] = (int)k;
    }
    std::vector<double> b(P.n), x(P.n, 0.0), t0(P.ysize, 0.0), y(P.ysize, 0.0), z(P.ysize + 1, 0.0), c(P.csize + 1, 0.0);
    uint32_t s = 7;
    for (auto& v : b) { s = s * 1664525u + 1013904223u; v = (s >> 8) / 16777216.0 - 0.5; }
    auto children = [&](const NodePos& q) {
        double v = c[q.p0];
        if (q.p1 >= 0) return v + c[q.p1];
        const int m = ~q.p1;
        for (int e = 1; e <= P.more[m]; ++e) v += c[P.more[m + e]];
        return v;
    };
    for (const auto& L : P.levels) {
        if (L.children) {
            for (int i = L.y0; i < L.y1; ++i) t0[i] = (P.orig[i] >= 0 ? b[P.orig[i]] : 0.0) - children(P.pos_y[i]);
            for (int i = L.c0; i < L.c1; ++i) c[i] = children(P.pos_c[i]);
        }
        for (int i = L.fwd0; i < L.fwd1; ++i) {
            const NodeItem& it = P.fwd[i];
            const int k = by_fwd.at(it.tile), np = T * it.nk;
            for (int j = 0; j < it.cnt; ++j) {
                const int yb = it.y0 + j * np, cb = it.c0 + j * T * it.nrk;
                std::vector<double> t(np);
                for (int q = 0; q < np; ++q) t[q] = L.children ? t0[yb + q] : (P.orig[yb + q] >= 0 ? b[P.orig[yb + q]] : 0.0);
                for (int r = it.rt0 * T; r < it.rt1 * T; ++r) {
                    double a = 0;
                    if (!it.nrk) {
                        for (int q = 0; q < np; ++q) a += S[k][(size_t)r * np + q] * t[q];
                        z[yb + r] = a;
                        if (P.orig[yb + r] >= 0) x[P.orig[yb + r]] = a;
                    } else if (r < np) {
                        for (int q = 0; q < r; ++q) a += S[k][(size_t)r * np + q] * t[q];
                        y[yb + r] = (a + t[r]) * D2[k][r];
                    } else {
                        for (int q = 0; q < np; ++q) a += W[k][(size_t)(r - np) * np + q] * t[q];
                        c[cb + r - np] = L.children ? c[cb + r - np] + a : a;
                    }
                }
            }
        }
    }
    for (size_t l = P.levels.size(); l-- > 0;) {
        const auto& L = P.levels[l];
        for (int i = L.bwd0; i < L.bwd1; ++i) {
            const NodeItem& it = P.bwd[i];
            const int k = by_bwd.at(it.tile), np = T * it.nk, nr = T * it.nrk;
            for (int j = 0; j < it.cnt; ++j) {
                const int yb = it.y0 + j * np, cb = it.c0 + j * T * it.nrk;
                for (int r = it.rt0 * T; r < it.rt1 * T; ++r) {
                    double a = 0;
                    for (int q = r + 1; q < np; ++q) a += S[k][(size_t)q * np + r] * y[yb + q];
                    for (int q = 0; q < nr; ++q) a -= W[k][(size_t)q * np + r] * z[P.zidx[cb + q]];
                    z[yb + r] = a + y[yb + r];
                    if (P.orig[yb + r] >= 0) x[P.orig[yb + r]] = z[yb + r];
                }
            }
        }
    }
    double err = 0, top = 0;
    for (size_t m = 0; m < F.size(); ++m) {
        std::vector<double> xr(F[m]->n);
        factor_solve(*F[m], &b[off[m]], xr.data());
        for (int i = 0; i < F[m]->n; ++i) {
            err = std::max(err, std::fabs(xr[i] - x[off[m] + i]));
            top = std::max(top, std::fabs(xr[i]));
        }
    }
    return err / top;
}

}  // namespace

// Plans `copies` solves of one box factor, one of a separately built factor of the same matrix
// (equal columns, another object) and, with other = 1, one of a different matrix. out: relative error,
// levels, blocks, instances, rows of the largest block.
extern "C" int nodeplan_check(int nx, int ny, int nz, int hole, int copies, int other, int leaf, double* out, char* msg, int len) {
    try {
        std::vector<SupernodalFactor> f(3);
        for (int k = 0; k < 3; ++k) {
            Csr A;
            std::vector<Int3> xyz;
            box_matrix(nx, ny, nz, hole, k == 2 ? 5u : 0u, A, xyz);
            factor_spd(A, xyz, 1e-5, f[k], leaf);
        }
        std::vector<const SupernodalFactor*> F(copies, &f[0]);
        F.push_back(&f[1]);
        if (other) F.push_back(&f[2]);
        std::vector<int> off, prob;
        int n = 0;
        for (auto q : F) { off.push_back(n); n += q->n; prob.push_back((int)prob.size()); }
        NodePlanHost P;
        need(build_nodeplan(F, off, prob, P), "not planned");
        need(P.n == n, "rows");
        check_indices(P);
        out[0] = emulate(P, F, off);
        out[1] = (double)P.levels.size(); out[2] = (double)P.blocks.size(); out[3] = (double)P.inst_prob.size();
        out[4] = 0;
        for (auto& B : P.blocks) out[4] = std::max(out[4], (double)B.n);
        return 0;
    } catch (const Failed& e) {
        std::string(e.what).copy(msg, len - 1);
    } catch (const std::exception& e) {
        std::string(e.what()).copy(msg, len - 1);
    }
    return 1;
}
