#include "hdd_nodeplan.h"
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <map>
#include <stdexcept>
#include <unordered_map>
#include "hdd_parallel.h"

namespace hdd {

namespace {

using P_ = NodePlanHost;
constexpr int T = NodePlanHost::kTile;
int tiles_of(int rows) { return (rows + T - 1) / T; }

// Cost of a level in microseconds, from which the cuts are chosen: its launches of dependent gathers
// and stores (forward; children's sums above the first level; backward below the last), the distinct
// blocks read from memory, the blocks that further runs read again from cache, and the workgroups'
// own latency where there are many.
constexpr double kLaunchUs = 5.0, kMemoryMBPerUs = 4.5, kCacheMBPerUs = 12.0, kRunUs = 8.0 / 1280.0;
constexpr int kMaxMergedColumns = 6144;  // a node of several heights (a taller merge costs more set-up than it saves)
constexpr int kMaxBand = 9;              // heights per band at most

struct Hash {
    uint64_t a = 0x9e3779b97f4a7c15ULL, b = 0xc2b2ae3d27d4eb4fULL;
    void word(uint64_t w) {
        a = (a ^ w) * 0xff51afd7ed558ccdULL;
        a ^= a >> 32;
        b = (b + w) * 0xc4ceb9fe1a85ec53ULL;
        b ^= b >> 29;
    }
    void doubles(const std::vector<double>& v) {
        for (double d : v) {
            uint64_t w;
            std::memcpy(&w, &d, 8);
            word(w);
        }
    }
    bool operator==(const Hash& o) const { return a == o.a && b == o.b; }
};
struct HashKey {
    size_t operator()(const Hash& h) const { return (size_t)h.a; }
};

// content of a supernode: its sizes and factor columns
Hash supernode_hash(const SupernodalFactor& f, int s) {
    Hash h;
    h.word((uint64_t)f.sn[s].n << 32 | (uint64_t)f.sn[s].rows.size());
    h.doubles(f.L11[s]);
    h.doubles(f.L21[s]);
    return h;
}

// tiles a solve reads of a block: the inverse of a closed one (no boundary rows), or one of the two operators twice
long long pass_tiles(long long nk, long long nrk) { return nrk ? nk * (nk + 1) / 2 + nk * nrk : nk * nk; }
long long block_tiles(long long nk, long long nrk) { return (nrk ? 2 : 1) * pass_tiles(nk, nrk); }

int run_limit(int k) {  // nodes per run whose operand vectors of k rows fit
    return std::max(1, std::min(P_::kRun, P_::kRunLdsFloats / (k + 4)));
}

// a node of a factor, in the factor's own numbering
struct Node {
    int root = 0, level = 0, parent = -1;
    std::vector<int> sns;
    int n = 0, nr = 0, block = -1;
    int slot0 = 0;  // first of its n + nr rows in the factor's contribution lists
};
struct Nodes {
    std::vector<Node> v;
    // children's contributions, CSR over the nodes' rows: (child node, its boundary row)
    std::vector<int> ptr, child, row;
};

// The distinct factors of a batch, how often each is solved with, and the content of their supernodes
struct Batch {
    std::vector<const SupernodalFactor*> distinct;
    std::vector<int> members, which;  // which: distinct factor of each one passed
    std::vector<std::vector<Hash>> sh;
    int H = -1;                       // tallest tree
    explicit Batch(const std::vector<const SupernodalFactor*>& F) : which(F.size()) {
        std::map<const SupernodalFactor*, int> id;
        for (size_t m = 0; m < F.size(); ++m) {
            if (F[m]->n) H = std::max(H, F[m]->max_height);
            auto e = id.emplace(F[m], (int)distinct.size());
            if (e.second) { distinct.push_back(F[m]); members.push_back(0); }
            which[m] = e.first->second;
            ++members[which[m]];
        }
        sh.resize(distinct.size());
        std::vector<std::pair<int, int>> todo;
        for (size_t d = 0; d < distinct.size(); ++d) {
            sh[d].resize(distinct[d]->sn.size());
            for (int s = 0; s < (int)sh[d].size(); ++s) todo.push_back({(int)d, s});
        }
        ParallelErrors errs;
#pragma omp parallel for schedule(dynamic, 16)
        for (size_t i = 0; i < todo.size(); ++i)
            errs.run([&] { sh[todo[i].first][todo[i].second] = supernode_hash(*distinct[todo[i].first], todo[i].second); });
        errs.rethrow();
    }
};

// the nodes of a band of heights [a, b) by content; false when one is beyond the form's limits
struct NodeKind { long long members = 0; int nk = 0, nrk = 0; };
using NodeKinds = std::unordered_map<Hash, NodeKind, HashKey>;
bool band_nodes(const Batch& B, int a, int b, NodeKinds& kinds) {
    for (size_t d = 0; d < B.distinct.size(); ++d) {
        const SupernodalFactor& f = *B.distinct[d];
        const int ns = (int)f.sn.size();
        std::vector<int> n(ns, 0);
        std::vector<Hash> h(ns);
        for (int s = 0; s < ns; ++s) {
            const Supernode& S = f.sn[s];
            if (S.height < a || S.height >= b) continue;
            n[s] += S.n;
            h[s].word(B.sh[d][s].a);
            const int p = S.parent;
            if (p >= 0 && f.sn[p].height < b) {
                n[p] += n[s];
                h[p].word(h[s].a);
                continue;
            }
            const int nk = tiles_of(n[s]), nrk = tiles_of((int)S.rows.size());
            if (T * (nk + nrk) + 4 > P_::kMaxLdsFloats || (b > a + 1 && n[s] > kMaxMergedColumns)) return false;
            NodeKind& k = kinds[h[s]];
            k.members += B.members[d];
            k.nk = nk; k.nrk = nrk;
        }
    }
    return true;
}

double estimate_level(const Batch& B, int a, int b, bool* ok) {
    NodeKinds kinds;
    *ok = band_nodes(B, a, b, kinds);
    if (!*ok || kinds.empty()) return 0;
    double distinct_mb = 0, again_mb = 0, runs = 0;
    for (auto& e : kinds) {
        const NodeKind& k = e.second;
        const int lim = run_limit(T * (k.nk + k.nrk));
        const double r = (double)((k.members + lim - 1) / lim), mb = 1024.0 * (double)block_tiles(k.nk, k.nrk) * 1e-6;
        distinct_mb += mb;
        again_mb += (r - 1) * mb;
        runs += r;
    }
    return kLaunchUs * (1 + (a > 0) + (b <= B.H)) + distinct_mb / kMemoryMBPerUs + again_mb / kCacheMBPerUs + runs * kRunUs;
}

// band boundaries 0 = c_0 < c_1 < .. = H + 1 of least estimated time (empty: none is possible)
std::vector<int> choose_cuts(const Batch& B) {
    const double inf = 1e300;
    const int H = B.H;
    struct Band { int a, b; double us; bool ok; };
    std::vector<Band> bands;
    for (int b = 1; b <= H + 1; ++b)
        for (int a = std::max(0, b - kMaxBand); a < b; ++a) bands.push_back({a, b, 0, false});
    ParallelErrors errs;
#pragma omp parallel for schedule(dynamic)
    for (size_t i = 0; i < bands.size(); ++i)
        errs.run([&] { bands[i].us = estimate_level(B, bands[i].a, bands[i].b, &bands[i].ok); });
    errs.rethrow();
    std::vector<double> best(H + 2, inf);
    std::vector<int> from(H + 2, -1);
    best[0] = 0;
    for (const Band& q : bands)  // ascending b: best[a] is final
        if (q.ok && best[q.a] < inf && best[q.a] + q.us < best[q.b]) { best[q.b] = best[q.a] + q.us; from[q.b] = q.a; }
    std::vector<int> cuts;
    if (best[H + 1] >= inf) return cuts;
    for (int b = H + 1; b > 0; b = from[b]) cuts.push_back(b);
    cuts.push_back(0);
    std::reverse(cuts.begin(), cuts.end());
    return cuts;
}

// the nodes of a factor, children before parents, and their contribution lists
void find_nodes(const SupernodalFactor& f, const std::vector<int>& level_of, Nodes& N) {
    const int ns = (int)f.sn.size();
    std::vector<int> node_of(ns, -1), sn_of(f.n), col_of(f.n);
    for (int s = ns - 1; s >= 0; --s) {
        const int p = f.sn[s].parent, l = level_of[f.sn[s].height];
        if (p >= 0 && level_of[f.sn[p].height] == l) { node_of[s] = node_of[p]; continue; }
        Node nd;
        nd.root = s; nd.level = l;
        node_of[s] = (int)N.v.size();
        N.v.push_back(nd);
    }
    std::reverse(N.v.begin(), N.v.end());  // ascending roots: children before parents
    for (int s = 0; s < ns; ++s) node_of[s] = (int)N.v.size() - 1 - node_of[s];
    for (int s = 0; s < ns; ++s) {
        Node& nd = N.v[node_of[s]];
        nd.sns.push_back(s);
        for (int k = 0; k < f.sn[s].n; ++k) { sn_of[f.sn[s].s0 + k] = s; col_of[f.sn[s].s0 + k] = nd.n + k; }
        nd.n += f.sn[s].n;
    }
    int slots = 0;
    for (Node& nd : N.v) {
        const Supernode& R = f.sn[nd.root];
        nd.nr = (int)R.rows.size();
        nd.parent = R.parent >= 0 ? node_of[R.parent] : -1;
        nd.slot0 = slots;
        slots += nd.n + nd.nr;
    }
    // target row of every child boundary row: a column of the parent node or one of its boundary rows
    std::vector<int> target, owner, arow;
    N.ptr.assign(slots + 1, 0);
    for (size_t k = 0; k < N.v.size(); ++k) {
        const Node& nd = N.v[k];
        if (nd.parent < 0) {
            if (nd.nr) throw std::runtime_error("node plan: a root with boundary rows");
            continue;
        }
        const Node& par = N.v[nd.parent];
        const std::vector<int>& rows = f.sn[nd.root].rows;
        const std::vector<int>& prow = f.sn[par.root].rows;
        size_t q = 0;
        for (int a = 0; a < nd.nr; ++a) {
            int t;
            if (node_of[sn_of[rows[a]]] == nd.parent) {
                t = par.slot0 + col_of[rows[a]];
            } else {
                while (q < prow.size() && prow[q] < rows[a]) ++q;
                if (q == prow.size() || prow[q] != rows[a]) throw std::runtime_error("node plan: a boundary row its parent does not hold");
                t = par.slot0 + par.n + (int)q;
            }
            target.push_back(t); owner.push_back((int)k); arow.push_back(a);
            ++N.ptr[t + 1];
        }
    }
    for (int t = 0; t < slots; ++t) N.ptr[t + 1] += N.ptr[t];
    N.child.resize(target.size()); N.row.resize(target.size());
    std::vector<int> fill(N.ptr.begin(), N.ptr.end() - 1);
    for (size_t e = 0; e < target.size(); ++e) {
        const int i = fill[target[e]]++;
        N.child[i] = owner[e]; N.row[i] = arow[e];
    }
}

// row of the block (columns, then boundary rows from `n` on) of every sub-diagonal row of its supernodes
void local_rows(const SupernodalFactor& f, const std::vector<int>& sns, int n, std::vector<int>& out) {
    const std::vector<int>& bound = f.sn[sns.back()].rows;
    out.clear();
    for (int s : sns) {
        size_t own = 0, q = 0;  // next supernode that may hold the row (both ascending), next boundary row
        int col = 0;            // first column of sns[own]
        for (int r : f.sn[s].rows) {
            while (own < sns.size() && f.sn[sns[own]].s0 + f.sn[sns[own]].n <= r) col += f.sn[sns[own++]].n;
            if (own < sns.size() && f.sn[sns[own]].s0 <= r) {
                out.push_back(col + r - f.sn[sns[own]].s0);
                continue;
            }
            while (q < bound.size() && bound[q] < r) ++q;
            if (q == bound.size() || bound[q] != r) throw std::runtime_error("node plan: a row outside its node");
            out.push_back(n + (int)q);
        }
    }
}

bool same_columns(const SupernodalFactor& fa, const std::vector<int>& a, const SupernodalFactor& fb, const std::vector<int>& b) {
    if (a.size() != b.size()) return false;
    for (size_t i = 0; i < a.size(); ++i) {
        const auto &x = fa.L11[a[i]], &y = fb.L11[b[i]], &u = fa.L21[a[i]], &v = fb.L21[b[i]];
        if (fa.sn[a[i]].n != fb.sn[b[i]].n || x.size() != y.size() || u.size() != v.size()) return false;
        if (std::memcmp(x.data(), y.data(), x.size() * 8) || std::memcmp(u.data(), v.data(), u.size() * 8)) return false;
    }
    return true;
}

// Share of the constant in the rows of a block's inverse, in units of the diagonal's: with m rows that are
// coupled to each other, sum of all entries over sum of the diagonal q, and the constant nearly an
// eigenvector, the inverse's rows have a part of 2-norm 1 / (q sqrt(m)) along it. Rounded to float, the
// inverse leaves 0.3 * 2^-24 of that in every row, also where the right-hand side has no such part (a domain
// without Dirichlet cells: its right-hand sides sum to zero, its operator annihilates the constant but for
// the 1e-5 on the diagonal). The triangles leave their rounding in the constant itself, where the operator
// does not see it. So a block beyond kMaxConstant keeps the two passes.
// Measured as the error outside the smallest mode, inverse against two passes (blocks of 27 to 4129 columns,
// in float): 0.2 to 4.8 times for shares below 1.2 (every block of the Dirichlet domains looked at, 32^3 to
// 160^3, and of a channel of 3 x 3 x 126 cells), 3.3 times at 42 (four Dirichlet cells on a 32^3 box), 32 times at
// 510 (one on a 64^3 box), 390 to 710 times at 13,000 to 23,000 (none on 32^3 to 64^3). At 100 it is 2e-6, what the
// two passes have at the last of these.
constexpr double kMaxConstant = 100;
double constant_share(const P_::Block& B) {
    const SupernodalFactor& f = *B.f;
    std::vector<int> at, part(B.n);
    local_rows(f, B.sns, B.n, at);
    for (int i = 0; i < B.n; ++i) part[i] = i;
    auto find = [&](int a) {
        while (part[a] != a) a = part[a] = part[part[a]];
        return a;
    };
    // of each column of the triangle the square of its sum and the sum of its squares; its rows are coupled to it
    std::vector<double> all(B.n), diag(B.n);
    int col = 0;
    const int* row = at.data();
    for (int s : B.sns) {
        const int n = f.sn[s].n, nr = (int)f.sn[s].rows.size();
        for (int j = 0; j < n; ++j) {
            double sum = 0, squares = 0;
            int root = find(col + j);
            auto entry = [&](int i, double l) {
                sum += l;
                squares += l * l;
                if (l != 0 && part[i] != root) part[find(i)] = root;
            };
            const double *l11 = &f.L11[s][(size_t)j * n], *l21 = nr ? &f.L21[s][(size_t)j * nr] : nullptr;
            for (int r = j; r < n; ++r) entry(col + r, l11[r]);
            for (int a = 0; a < nr; ++a) entry(row[a], l21[a]);
            all[col + j] = sum * sum;
            diag[col + j] = squares;
        }
        col += n;
        row += nr;
    }
    std::vector<int> m(B.n, 0);  // rows of a part, at its root
    for (int j = 0; j < B.n; ++j) {
        const int p = find(j);
        if (p != j) { all[p] += all[j]; diag[p] += diag[j]; }
        ++m[p];
    }
    double share = 0;
    for (int p = 0; p < B.n; ++p)
        if (m[p] > 1) share = std::max(share, diag[p] / (all[p] * std::sqrt((double)m[p])));
    return share;
}

// Work items of one run in one pass: `rows` row tiles of up to `len` tiles, `level_rows` row tiles in
// the level. A wave streams about four tiles per memory round trip, so the waves of a workgroup share
// a row tile (split) until each has at most kWaveTiles of its tiles, or 4 where the chip has waves to
// spare. A workgroup takes several row tiles, so that its operand vectors are read once for them,
// where that leaves kGroups workgroups and its waves at most kWorkTiles tiles each. (All flat: 16, 24
// and 1024 are within 4% of half and double themselves from the 64^3 to the 256^3 domain.)
void push_items(std::vector<NodeItem>& out, NodeItem it, int rows, int len, int waves, long long level_rows) {
    constexpr int kWaveTiles = 16, kWorkTiles = 24, kGroups = 1024, kMaxRows = 16;
    int split = waves == 16 ? 16 : 1;
    while (split < waves && (len > kWaveTiles * split || (len > 4 * split && level_rows * split < 2048))) split *= 2;
    it.split = split;
    const long long step = waves / split, by_work = (long long)kWorkTiles * waves / std::max(1, len);
    const long long want = std::max(1LL, std::min({by_work, level_rows / kGroups, (long long)kMaxRows}));
    const int chunk = (int)((want + step - 1) / step * step);
    for (int r = 0; r < rows; r += chunk) {
        it.rt0 = r; it.rt1 = std::min(rows, r + chunk);
        out.push_back(it);
    }
}

// waves per workgroup of a level's pass: the few long row tiles of the big separators go to sixteen
// (without them the interface solves take 330 us instead of 306 at 256^3, 70 instead of 62 at 100^3)
int level_waves(long long row_tiles, double mean_tiles) { return row_tiles < 640 && mean_tiles >= 48 ? 16 : 4; }

}  // namespace

PlanBytes nodeplan_bytes(const std::vector<const SupernodalFactor*>& F) {
    PlanBytes out;
    const Batch B(F);
    if (B.H < 0) return out;
    const std::vector<int> cuts = choose_cuts(B);
    out.planned = !cuts.empty();
    double total = 0, largest = 0;
    for (size_t l = 0; l + 1 < cuts.size(); ++l) {
        NodeKinds kinds;
        band_nodes(B, cuts[l], cuts[l + 1], kinds);
        for (auto& e : kinds) {
            const NodeKind& k = e.second;
            const int lim = run_limit(T * (k.nk + k.nrk));
            const double runs = (double)((k.members + lim - 1) / lim), doubles = 256.0 * (k.nk + k.nrk) * k.nk;
            out.held += 1024.0 * (double)block_tiles(k.nk, k.nrk) + 4.0 * T * k.nk;
            // per padded column t, y, z, its row and its children's positions; per boundary row c, its column and the
            // same; a work item per row tile
            out.held += k.members * (24.0 * T * k.nk + 20.0 * T * k.nrk + 4.0) + runs * 48.0 * (2.0 * k.nk + k.nrk);
            total += doubles;
            largest = std::max(largest, doubles);
        }
    }
    // set-up: a chunk of the blocks' columns, their inverses, and the factor columns on their way
    out.setup = 8.0 * 2.5 * std::min(total, std::max(largest, (double)P_::kSetupChunk));
    return out;
}

bool build_nodeplan(const std::vector<const SupernodalFactor*>& F, const std::vector<int>& offsets, const std::vector<int>& prob_of,
                    NodePlanHost& P) {
    P = NodePlanHost();
    for (size_t m = 0; m < F.size(); ++m) P.n = std::max(P.n, offsets[m] + F[m]->n);
    const Batch batch(F);
    const std::vector<const SupernodalFactor*>& distinct = batch.distinct;
    const std::vector<int>& which = batch.which;
    const std::vector<std::vector<Hash>>& sh = batch.sh;
    const int H = batch.H;
    if (P.n == 0 || H < 0) return false;
    const std::vector<int> cuts = choose_cuts(batch);
    if (cuts.empty()) return false;
    const int NL = (int)cuts.size() - 1;
    std::vector<int> level_of(H + 1, 0);
    for (int l = 0; l < NL; ++l)
        for (int h = cuts[l]; h < cuts[l + 1]; ++h) level_of[h] = l;
    // nodes of the distinct factors, and the distinct blocks among them
    std::vector<Nodes> nodes(distinct.size());
    std::vector<std::vector<Hash>> nh(distinct.size());
    {
        ParallelErrors errs;
#pragma omp parallel for schedule(dynamic)
        for (size_t d = 0; d < distinct.size(); ++d)
            errs.run([&] {
                find_nodes(*distinct[d], level_of, nodes[d]);
                std::vector<int> rows;
                for (const Node& nd : nodes[d].v) {
                    Hash h;
                    h.word((uint64_t)nd.n << 32 | (uint64_t)nd.nr);
                    for (int s : nd.sns) { h.word(sh[d][s].a); h.word(sh[d][s].b); }
                    local_rows(*distinct[d], nd.sns, nd.n, rows);
                    for (int r : rows) h.word((uint64_t)r);
                    nh[d].push_back(h);
                }
            });
        errs.rethrow();
        std::unordered_map<Hash, std::vector<int>, HashKey> seen;
        std::vector<int> ra, rb;
        for (size_t d = 0; d < distinct.size(); ++d)
            for (size_t k = 0; k < nodes[d].v.size(); ++k) {
                Node& nd = nodes[d].v[k];
                std::vector<int>& bucket = seen[nh[d][k]];
                for (int c : bucket) {
                    const P_::Block& B = P.blocks[c];
                    if (B.n != nd.n || B.nr != nd.nr || !same_columns(*B.f, B.sns, *distinct[d], nd.sns)) continue;
                    local_rows(*B.f, B.sns, B.n, ra);
                    local_rows(*distinct[d], nd.sns, nd.n, rb);
                    if (ra == rb) { nd.block = c; break; }
                }
                if (nd.block >= 0) continue;
                nd.block = (int)P.blocks.size();
                bucket.push_back(nd.block);
                P_::Block B;
                B.f = distinct[d]; B.sns = nd.sns; B.n = nd.n; B.nr = nd.nr;
                B.nk = tiles_of(nd.n); B.nrk = tiles_of(nd.nr);
                P.blocks.push_back(B);
            }
    }
    // a nearly singular block without boundary rows gets a boundary tile of zeros, and with it the two passes
    {
        ParallelErrors errs;
#pragma omp parallel for schedule(dynamic)
        for (size_t k = 0; k < P.blocks.size(); ++k)
            errs.run([&] {
                P_::Block& B = P.blocks[k];
                if (!B.nr && !(constant_share(B) <= kMaxConstant)) B.nrk = 1;
            });
        errs.rethrow();
        for (const P_::Block& B : P.blocks)
            if (T * (B.nk + B.nrk) + 4 > P_::kMaxLdsFloats) return false;
    }
    for (P_::Block& B : P.blocks) {
        const long long t = block_tiles(B.nk, B.nrk);
        if (P.tiles + t > INT_MAX || (long long)P.scales + T * B.nk > INT_MAX) return false;
        B.scale = P.scales; P.scales += T * B.nk;
        B.fwd = B.bwd = (int)P.tiles;
        if (B.nrk) B.bwd += (int)(t / 2);
        P.tiles += t;
    }
    // instances: every node of every member, its padded columns and boundary rows. A level's rows are
    // contiguous, largest blocks first, and the nodes that share a block follow each other.
    struct Inst { int y, c, prob, block, m, k; };
    std::vector<std::vector<Inst>> at_level(NL);
    std::vector<std::vector<int>> ybase(F.size()), cbase(F.size());
    for (size_t m = 0; m < F.size(); ++m) {
        const size_t n = nodes[which[m]].v.size();
        ybase[m].resize(n); cbase[m].resize(n);
        for (size_t k = 0; k < n; ++k) {
            const Node& nd = nodes[which[m]].v[k];
            at_level[nd.level].push_back({0, 0, prob_of.empty() ? 0 : prob_of[m], nd.block, (int)m, (int)k});
        }
    }
    P.levels.resize(NL);
    long long ny = 0, nc = 0;
    for (int l = 0; l < NL; ++l) {
        P_::Level& L = P.levels[l];
        std::stable_sort(at_level[l].begin(), at_level[l].end(), [&](const Inst& a, const Inst& b) {
            if (a.block == b.block) return false;
            const P_::Block &x = P.blocks[a.block], &y = P.blocks[b.block];
            const long long s = block_tiles(x.nk, x.nrk), t = block_tiles(y.nk, y.nrk);
            return s != t ? s > t : a.block < b.block;
        });
        L.y0 = (int)ny; L.c0 = (int)nc;
        for (Inst& i : at_level[l]) {
            const P_::Block& B = P.blocks[i.block];
            ybase[i.m][i.k] = i.y = (int)ny; cbase[i.m][i.k] = i.c = (int)nc;
            ny += T * B.nk; nc += T * B.nrk;
            if (ny > INT_MAX - 64 || nc > INT_MAX - 64) return false;
        }
        L.y1 = (int)ny; L.c1 = (int)nc;
    }
    P.ysize = (int)ny; P.csize = (int)nc;
    P.orig.assign(P.ysize, -1);
    P.zidx.assign(P.csize, P.ysize);
    P.pos_y.assign(P.ysize, {P.csize, P.csize});
    P.pos_c.assign(P.csize, {P.csize, P.csize});
    for (size_t m = 0; m < F.size(); ++m) {
        const SupernodalFactor& f = *F[m];
        const Nodes& N = nodes[which[m]];
        std::vector<int> ypos(f.n);  // permuted position -> padded column
        for (size_t k = 0; k < N.v.size(); ++k) {
            int q = ybase[m][k];
            for (int s : N.v[k].sns)
                for (int i = 0; i < f.sn[s].n; ++i, ++q) {
                    P.orig[q] = offsets[m] + f.perm[f.sn[s].s0 + i];
                    ypos[f.sn[s].s0 + i] = q;
                }
        }
        for (size_t k = 0; k < N.v.size(); ++k) {
            const Node& nd = N.v[k];
            const std::vector<int>& rows = f.sn[nd.root].rows;
            for (int a = 0; a < nd.nr; ++a) P.zidx[cbase[m][k] + a] = ypos[rows[a]];
            for (int r = 0; r < nd.n + nd.nr; ++r) {
                const int e0 = N.ptr[nd.slot0 + r], e1 = N.ptr[nd.slot0 + r + 1];
                if (e0 == e1) continue;
                auto where = [&](int e) { return cbase[m][N.child[e]] + N.row[e]; };
                NodePos& q = r < nd.n ? P.pos_y[ybase[m][k] + r] : P.pos_c[cbase[m][k] + r - nd.n];
                q.p0 = where(e0);
                if (e1 - e0 == 2) q.p1 = where(e0 + 1);
                if (e1 - e0 > 2) {
                    if (P.more.size() > (size_t)INT_MAX - 1024) return false;
                    q.p1 = ~(int)P.more.size();
                    P.more.push_back(e1 - e0 - 1);
                    for (int e = e0 + 1; e < e1; ++e) P.more.push_back(where(e));
                }
            }
        }
    }
    // per level: runs of instances that share a block, and their work items
    for (int l = 0; l < NL; ++l) {
        P_::Level& L = P.levels[l];
        L.children = l > 0;
        const auto& v = at_level[l];
        struct Run { int i0, cnt, block, y, c; };
        std::vector<int> longest(P.blocks.size(), 0);  // run of each block
        std::vector<Run> runs;
        long long frows = 0, brows = 0, ftiles = 0, btiles = 0;
        for (size_t i = 0; i < v.size();) {
            const P_::Block& B = P.blocks[v[i].block];
            const int lim = run_limit(T * (B.nk + B.nrk));
            int k = 1;
            while (k < lim && i + k < v.size() && v[i + k].block == v[i].block) ++k;
            longest[v[i].block] = std::max(longest[v[i].block], k);
            runs.push_back({(int)P.inst_prob.size(), k, v[i].block, v[i].y, v[i].c});
            for (int j = 0; j < k; ++j) P.inst_prob.push_back(v[i + j].prob);
            frows += B.nk + B.nrk;
            ftiles += pass_tiles(B.nk, B.nrk);
            L.fwd_lds = std::max(L.fwd_lds, k * (T * B.nk + 4));
            if (B.nrk) {
                brows += B.nk;
                btiles += pass_tiles(B.nk, B.nrk);
                L.bwd_lds = std::max(L.bwd_lds, k * (T * (B.nk + B.nrk) + 4));
            }
            i += k;
        }
        L.fwd_waves = level_waves(frows, frows ? (double)ftiles / frows : 0);
        L.bwd_waves = level_waves(brows, brows ? (double)btiles / brows : 0);
        L.fwd0 = (int)P.fwd.size(); L.bwd0 = (int)P.bwd.size();
        for (const Run& r : runs) {
            const P_::Block& B = P.blocks[r.block];
            NodeItem it = {B.fwd, r.i0, r.y, r.c, r.cnt, 1, B.nk, B.nrk, 0, 0, longest[r.block] == 1, B.scale};
            push_items(P.fwd, it, B.nk + B.nrk, B.nk, L.fwd_waves, frows);
            if (!B.nrk) continue;
            it.tile = B.bwd;
            push_items(P.bwd, it, B.nk, B.nk + B.nrk, L.bwd_waves, brows);
        }
        L.fwd1 = (int)P.fwd.size(); L.bwd1 = (int)P.bwd.size();
    }
    return true;
}

void node_block_rows(const NodePlanHost::Block& B, std::vector<int>& rows) {
    local_rows(*B.f, B.sns, B.n, rows);
    for (int& r : rows)
        if (r >= B.n) r += T * B.nk - B.n;
}

void node_block_columns(const NodePlanHost::Block& B, double* L) {
    const SupernodalFactor& f = *B.f;
    const int np = T * B.nk, rows = np + T * B.nrk;
    std::fill(L, L + (size_t)rows * np, 0.0);
    std::vector<int> at;
    node_block_rows(B, at);
    for (int i = B.n; i < np; ++i) L[(size_t)i * np + i] = 1.0;
    int col = 0;
    size_t first = 0;
    for (int s : B.sns) {
        const int n = f.sn[s].n, nr = (int)f.sn[s].rows.size();
        for (int j = 0; j < n; ++j) {
            for (int r = j; r < n; ++r) L[(size_t)(col + r) * np + col + j] = f.L11[s][(size_t)j * n + r];
            for (int a = 0; a < nr; ++a) L[(size_t)at[first + a] * np + col + j] = f.L21[s][(size_t)j * nr + a];
        }
        col += n;
        first += nr;
    }
}

}  // namespace hdd
