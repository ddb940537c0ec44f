// Host check of a failed hdd_set_sigma_refinement (SigmaDevice::set_refinement,
// csrc/hdd_sigma_device.hip), compiled and run by tests/test_refinement_setup.py as a program of its
// own: the HIP memory calls below take the place of the runtime's, device memory is host memory, and
// the k-th allocation fails as it does out of memory. Nothing here reaches a GPU.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>
#include "../hierarchicaldd_amd/csrc/hdd_sigma_device.h"

static int g_left = -1;  // allocations until one fails (-1: none does)
static int g_count = 0, g_live = 0;

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    ++g_count;
    if (g_left == 0) { *p = nullptr; return hipErrorOutOfMemory; }
    if (g_left > 0) --g_left;
    *p = std::malloc(n);
    ++g_live;
    return hipSuccess;
}
hipError_t hipFree(void* p) { std::free(p); --g_live; return hipSuccess; }
hipError_t hipMemset(void* p, int v, size_t n) { std::memset(p, v, n); return hipSuccess; }
hipError_t hipMemcpy(void* to, const void* from, size_t n, hipMemcpyKind) { std::memcpy(to, from, n); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
}

using namespace hdd;

static Csr box(int n, std::vector<Int3>& xyz) {
    Csr A;
    A.rows = A.cols = n * n * n;
    for (int i = 0; i < A.rows; ++i) {
        const int x = i / (n * n), y = i / n % n, z = i % n;
        xyz.push_back({x, y, z});
        auto add = [&](bool in, int j, float v) { if (in) { A.idx.push_back(j); A.val.push_back(v); } };
        add(x > 0, i - n * n, -1.f); add(y > 0, i - n, -1.f); add(z > 0, i - 1, -1.f);
        add(true, i, 6.f);
        add(z + 1 < n, i + 1, -1.f); add(y + 1 < n, i + n, -1.f); add(x + 1 < n, i + n * n, -1.f);
        A.ptr.push_back((int)A.idx.size());
    }
    return A;
}

// one level: two subdomains of one shape and an interface, planned as dense nodes are (without their blocks)
struct Setup {
    SigmaHost host;
    SupernodalFactor fi, fr;
    SigmaDevice S;
    Setup() {
        std::vector<Int3> ci, cr;
        const Csr Ai = box(9, ci), Ar = box(7, cr);
        factor_spd(Ai, ci, 1e-5, fi, 24);
        factor_spd(Ar, cr, 1e-5, fr, 24);
        host.levels = 1; host.nsub = 2;
        host.n_if = {Ar.rows};
        host.Arr = {Ar};
        host.Aii = {{Ai, Ai}};
        S.levels = 1; S.nprob = 1;
        S.lv.resize(1);
        SigmaLevel& L = S.lv[0];
        L.n_if = Ar.rows; L.n_int = 2 * Ai.rows;
        L.Lii.n = 2 * Ai.rows; L.Lii.use_nodes = true; L.Lii.F = {&fi, &fi}; L.Lii.offsets = {0, Ai.rows};
        L.Lrr.n = Ar.rows; L.Lrr.use_nodes = true; L.Lrr.F = {&fr}; L.Lrr.offsets = {0};
        S.plan_bytes = 1000000;  // the rest of the context
    }
    bool refine(int steps) {
        try {
            S.set_refinement({&host}, steps, nullptr);
            return true;
        } catch (const std::exception&) {
            return false;
        }
    }
};

// every array of the per-height form holds what the undisturbed one holds
template <class T>
static bool same(const DBuf<T>& a, const DBuf<T>& b) { return a.n == b.n && (a.n == 0 || (a.p && b.p && !std::memcmp(a.p, b.p, a.n * sizeof(T)))); }
static bool same_plan(const TriPlan& a, const TriPlan& b) {
    return a.H == b.H && a.H >= 0 && a.fused == b.fused && a.sl_begin == b.sl_begin && same(a.sn_prob, b.sn_prob) && same(a.run_q, b.run_q) &&
           same(a.run_n, b.run_n) && same(a.orig_of, b.orig_of) && same(a.s0, b.s0) && same(a.sz, b.sz) && same(a.nr, b.nr) && same(a.roff, b.roff) &&
           same(a.srows, b.srows) && same(a.sn_of, b.sn_of) && same(a.sn_list, b.sn_list) && same(a.sl_sn, b.sl_sn) && same(a.sl_r0, b.sl_r0) &&
           same(a.rowlist, b.rowlist) && same(a.inc_ptr, b.inc_ptr) && same(a.ci_sn, b.ci_sn) && same(a.ci_a0, b.ci_a0) && same(a.ci_a1, b.ci_a1) &&
           same(a.bi_sn, b.bi_sn) && same(a.bi_c, b.bi_c) && same(a.bi_j0, b.bi_j0) && same(a.loff, b.loff) && same(a.doff, b.doff) &&
           same(a.cofs, b.cofs) && same(a.cpos, b.cpos) && same(a.bofs, b.bofs) && same(a.diag, b.diag) && same(a.diagT, b.diagT) &&
           same(a.l21, b.l21) && a.c.n == b.c.n && a.bpart.n == b.bpart.n && a.t.n == b.t.n && a.y.n == b.y.n && a.t.p && a.y.p && a.c.p && a.bpart.p;
}

#define NEED(ok, ...)            \
    do {                         \
        if (!(ok)) {             \
            std::printf(__VA_ARGS__); \
            std::printf("\n");   \
            return 1;            \
        }                        \
    } while (0)

int main() {
    Setup whole;
    NEED(whole.refine(1), "the undisturbed call failed");
    const int allocations = g_count;
    const size_t heights = whole.S.lv[0].Lii.bytes() + whole.S.lv[0].Lrr.bytes();
    NEED(whole.S.plan_bytes == 1000000 + heights, "plan bytes of the undisturbed call");
    NEED(allocations > 40, "only %d allocations", allocations);
    for (int k = 0; k < allocations; ++k) {
        Setup q;
        const int live = g_live;
        g_left = k;
        NEED(!q.refine(1), "allocation %d failed and the call did not", k);
        const bool first = q.S.lv[0].Lii.H >= 0, second = q.S.lv[0].Lrr.H >= 0;
        NEED(q.S.refine_steps == 0 && q.S.lv[0].Lii.refine == 0 && q.S.lv[0].Lrr.refine == 0, "allocation %d: solves refined after a failure", k);
        NEED(q.S.plan_bytes == 1000000 + (first ? q.S.lv[0].Lii.bytes() : 0) + (second ? q.S.lv[0].Lrr.bytes() : 0), "allocation %d: plan bytes", k);
        NEED(!q.refine(1), "allocation %d failed again and the second call did not", k);  // still out of memory
        g_left = -1;
        NEED(q.refine(1), "allocation %d: no retry", k);
        NEED(same_plan(q.S.lv[0].Lii, whole.S.lv[0].Lii) && same_plan(q.S.lv[0].Lrr, whole.S.lv[0].Lrr), "allocation %d: the retry's plans", k);
        NEED(q.S.plan_bytes == 1000000 + heights, "allocation %d: plan bytes of the retry", k);
        NEED(g_live - live == allocations, "allocation %d: %d arrays left, %d in the undisturbed call", k, g_live - live, allocations);
    }
    std::printf("%d allocations, each failed once\n", allocations);
    return 0;
}
