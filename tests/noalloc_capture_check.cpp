// Host check of a captured hdd_inner_product_noalloc (csrc/hdd_kernels.hip), compiled and run by
// tests/test_noalloc_capture.py as a program of its own: the HIP calls below take the place of the
// runtime's, and a launch does to the tickets what its kernel does (one thread: clears its own; a grid of
// g workgroups: draws g, whose last one clears it, and clears the one half a round away).
#include <cstdio>
#include <cstring>
#include <vector>
#include <hip/hip_runtime.h>
#include "../include/hdd.h"

constexpr int kParts = 1024, kTickets = 64;
struct Scratch {
    double part[kParts];
    unsigned ticket[kTickets];
};
static Scratch g_scratch;
struct Launch { int grid, ticket; };
static std::vector<Launch> g_graph;
static bool g_capturing = false;
static int g_wrong = 0;  // sums that a workgroup other than the last would have ended

static void run(const Launch& l) {
    unsigned& t = g_scratch.ticket[l.ticket];
    if (l.grid == 0) { t = 0; return; }
    g_scratch.ticket[(l.ticket + kTickets / 2) % kTickets] = 0;
    for (int i = 0; i < l.grid; ++i)
        if (t++ == (unsigned)l.grid - 1u) {
            g_wrong += i != l.grid - 1;
            t = 0;
        } else {
            g_wrong += i == l.grid - 1;
        }
}

extern "C" {
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = &g_scratch; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    *s = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
static dim3 g_dim, g_block;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t) { g_dim = g; g_block = b; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
    *g = g_dim; *b = g_block; *m = 0; *s = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3 g, dim3 b, void** args, size_t, hipStream_t) {
    Launch l;
    if (b.x == 1) {  // (scratch, ticket)
        l.grid = 0;
        std::memcpy(&l.ticket, args[1], 4);
    } else {         // (a, b, groups, g, scratch, ticket, out)
        l.grid = (int)g.x;
        std::memcpy(&l.ticket, args[5], 4);
    }
    if (g_capturing) g_graph.push_back(l);
    else run(l);
    return hipSuccess;
}
}

#define NEED(ok, what) do { if (!(ok)) { std::printf("%s\n", what); return 1; } } while (0)

int main() {
    alignas(16) static float a[4096];
    double out;
    int own;
    const hipStream_t s = (hipStream_t)&own;
    auto call = [&](int pages) { return hdd_inner_product_noalloc(a, a, pages, &out, s); };
    for (int i = 0; i < 3; ++i) NEED(call(50 + i) == HDD_OK && !g_wrong, "an eager call");
    g_capturing = true;
    NEED(call(200) == HDD_OK && call(17) == HDD_OK, "capture");
    g_capturing = false;
    auto replay = [&] { for (const Launch& l : g_graph) run(l); };
    for (int i = 0; i < 5; ++i) { replay(); NEED(!g_wrong, "a replay"); }
    // calls that overlapped leave any count behind, in the eager calls' tickets and in the graph's: the
    // replays after them are right, and the eager calls from half a round on
    for (unsigned& t : g_scratch.ticket) t = 7;
    for (int i = 0; i < 3; ++i) replay();
    NEED(!g_wrong, "a replay after calls that overlapped");
    for (int i = 0; i < kTickets / 2; ++i) call(100);
    g_wrong = 0;
    for (int i = 0; i < 3 * kTickets; ++i) { call(60 + i % 9); replay(); }
    NEED(!g_wrong, "later calls");
    std::printf("%zu nodes a graph\n", g_graph.size());
    return 0;
}
