// Host check of the dense-node plans of nearly singular matrices (csrc/hdd_nodeplan.h), compiled and
// called by tests/test_nodeplan_singular.py: a box operator without Dirichlet cells, planned and carried
// out in float as the kernels do (operators formed in double and rounded, float sums), against the
// factor's own solve.
#include "nodeplan_check.cpp"
#include <map>

namespace {

// 7-point operator of an nx x ny x nz box whose outer faces have no neighbour; `ring`: they have one
// (a Dirichlet cell), on the low x face only with ring = 2, at one of its cells with ring = 3
void neumann_matrix(int nx, int ny, int nz, int ring, Csr& A, std::vector<Int3>& xyz) {
    box_matrix(nx, ny, nz, 0, 0u, A, xyz);
    for (int i = 0; i < A.rows; ++i) {
        const Int3 c = xyz[i];
        float d = ring == 1 ? 6.f : (float)(A.ptr[i + 1] - A.ptr[i] - 1);
        if (c.x == 0 && (ring == 2 || (ring == 3 && c.y == ny / 2 && c.z == nz / 2))) d += 1.f;
        for (int e = A.ptr[i]; e < A.ptr[i + 1]; ++e) if (A.idx[e] == i) A.val[e] = d;
    }
}

// the solve as emulate() does it, every operator, operand and sum rounded to float
std::vector<float> solve_in_float(const NodePlanHost& P, const std::vector<float>& b) {
    std::vector<std::vector<float>> S(P.blocks.size()), W(P.blocks.size()), D(P.blocks.size());
    std::map<int, int> by_fwd, by_bwd;
    for (size_t k = 0; k < P.blocks.size(); ++k) {
        const auto& B = P.blocks[k];
        const int np = T * B.nk, nr = T * B.nrk;
        std::vector<double> L((size_t)(np + nr) * np), inv((size_t)np * np, 0.0);
        node_block_columns(B, L.data());
        for (int i = 0; i < np; ++i) for (int j = 0; j <= i; ++j) inv[(size_t)j * np + i] = L[(size_t)i * np + j];
        invert_lower(inv, np);
        S[k].assign((size_t)np * np, 0.f); W[k].assign((size_t)nr * np, 0.f); D[k].resize(np);
        by_fwd[B.fwd] = (int)k; by_bwd[B.bwd] = (int)k;
        if (!nr) {  // closed: the inverse, its diagonal apart
            for (int i = 0; i < np; ++i)
                for (int j = 0; j <= i; ++j) {
                    double v = 0;
                    for (int q = i; q < np; ++q) v += inv[(size_t)i * np + q] * inv[(size_t)j * np + q];
                    if (i == j) D[k][i] = (float)v;
                    else S[k][(size_t)i * np + j] = S[k][(size_t)j * np + i] = (float)v;
                }
            continue;
        }
        for (int i = 0; i < np; ++i) {
            const double d = L[(size_t)i * np + i];
            D[k][i] = (float)(1.0 / (d * d));
            for (int j = 0; j < i; ++j) S[k][(size_t)i * np + j] = (float)(d * inv[(size_t)j * np + i]);
        }
        std::vector<double> w((size_t)nr * np, 0.0);
        for (int a = 0; a < nr; ++a)
            for (int q = 0; q < np; ++q) {
                const double l = L[(size_t)(np + a) * np + q];
                if (l != 0) for (int j = 0; j <= q; ++j) w[(size_t)a * np + j] += l * inv[(size_t)j * np + q];
            }
        std::copy(w.begin(), w.end(), W[k].begin());
    }
    std::vector<float> x(P.n, 0.f), t0(P.ysize, 0.f), y(P.ysize, 0.f), z(P.ysize + 1, 0.f), c(P.csize + 1, 0.f);
    auto children = [&](const NodePos& q) {
        float v = c[q.p0];
        if (q.p1 >= 0) return v + c[q.p1];
        const int m = ~q.p1;
        for (int e = 1; e <= P.more[m]; ++e) v += c[P.more[m + e]];
        return v;
    };
    // four sums, one per column mod 4, as the kernels keep them
    auto dot = [](const float* a, const float* t, int n) {
        float s[4] = {0.f, 0.f, 0.f, 0.f};
        for (int q = 0; q < n; ++q) s[q & 3] = std::fma(a[q], t[q], s[q & 3]);
        return (s[0] + s[1]) + (s[2] + s[3]);
    };
    for (const auto& L : P.levels) {
        if (L.children) {
            for (int i = L.y0; i < L.y1; ++i) t0[i] = (P.orig[i] >= 0 ? b[P.orig[i]] : 0.f) - children(P.pos_y[i]);
            for (int i = L.c0; i < L.c1; ++i) c[i] = children(P.pos_c[i]);
        }
        for (int i = L.fwd0; i < L.fwd1; ++i) {
            const NodeItem& it = P.fwd[i];
            const int k = by_fwd.at(it.tile), np = T * it.nk;
            for (int j = 0; j < it.cnt; ++j) {
                const int yb = it.y0 + j * np, cb = it.c0 + j * T * it.nrk;
                std::vector<float> t(np);
                for (int q = 0; q < np; ++q) t[q] = L.children ? t0[yb + q] : (P.orig[yb + q] >= 0 ? b[P.orig[yb + q]] : 0.f);
                for (int r = it.rt0 * T; r < it.rt1 * T; ++r) {
                    if (!it.nrk) {
                        z[yb + r] = dot(&S[k][(size_t)r * np], t.data(), np) + t[r] * D[k][r];
                        if (P.orig[yb + r] >= 0) x[P.orig[yb + r]] = z[yb + r];
                    } else if (r < np) {
                        y[yb + r] = (dot(&S[k][(size_t)r * np], t.data(), r) + t[r]) * D[k][r];
                    } else {
                        const float a = dot(&W[k][(size_t)(r - np) * np], t.data(), np);
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
                    float s[4] = {0.f, 0.f, 0.f, 0.f};
                    for (int q = r + 1; q < np; ++q) s[q & 3] = std::fma(S[k][(size_t)q * np + r], y[yb + q], s[q & 3]);
                    for (int q = 0; q < nr; ++q) s[q & 3] = std::fma(-W[k][(size_t)q * np + r], z[P.zidx[cb + q]], s[q & 3]);
                    z[yb + r] = (s[0] + s[1]) + (s[2] + s[3]) + y[yb + r];
                    if (P.orig[yb + r] >= 0) x[P.orig[yb + r]] = z[yb + r];
                }
            }
        }
    }
    return x;
}

}  // namespace

// Solves with `copies` factors of one box, right-hand sides without a mean where ring = 0. out: error
// relative to the solution, both less their mean; blocks without boundary rows, and those of them that
// hold their inverse; the plan's error in double.
extern "C" int nodeplan_singular_check(int nx, int ny, int nz, int ring, int copies, int leaf, double* out, char* msg, int len) {
    try {
        SupernodalFactor f;
        Csr A;
        std::vector<Int3> xyz;
        neumann_matrix(nx, ny, nz, ring, A, xyz);
        factor_spd(A, xyz, 1e-5, f, leaf);
        const std::vector<const SupernodalFactor*> F(copies, &f);
        std::vector<int> off;
        for (int k = 0; k < copies; ++k) off.push_back(k * f.n);
        NodePlanHost P;
        need(build_nodeplan(F, off, {}, P), "not planned");
        check_indices(P);
        out[1] = out[2] = 0;
        for (const auto& B : P.blocks)
            if (!B.nr) { out[1] += 1; out[2] += !B.nrk; }
        out[3] = emulate(P, F, off);
        std::vector<float> b(P.n);
        uint32_t s = 11;
        for (auto& v : b) { s = s * 1664525u + 1013904223u; v = (float)((s >> 8) / 16777216.0 - 0.5); }
        if (!ring)
            for (int k = 0; k < copies; ++k) {
                double m = 0;
                for (int i = 0; i < f.n; ++i) m += b[off[k] + i];
                for (int i = 0; i < f.n; ++i) b[off[k] + i] -= (float)(m / f.n);
            }
        const std::vector<float> x = solve_in_float(P, b);
        double err = 0, all = 0;
        for (int k = 0; k < copies; ++k) {
            std::vector<double> bd(b.begin() + off[k], b.begin() + off[k] + f.n), ref(f.n);
            factor_solve(f, bd.data(), ref.data());
            double mr = 0, mx = 0;
            for (int i = 0; i < f.n; ++i) { mr += ref[i] / f.n; mx += x[off[k] + i] / (double)f.n; }
            for (int i = 0; i < f.n; ++i) {
                const double r = ref[i] - mr, e = x[off[k] + i] - mx - r;
                err += e * e; all += r * r;
            }
        }
        out[0] = std::sqrt(err / all);
        return 0;
    } catch (const Failed& e) {
        std::string(e.what).copy(msg, len - 1);
    } catch (const std::exception& e) {
        std::string(e.what()).copy(msg, len - 1);
    }
    return 1;
}
