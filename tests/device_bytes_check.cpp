// Host check of the device bytes a problem is estimated to need (ProblemHost::device_bytes), by which the
// server admits requests, compiled and run by tests/test_device_bytes.py as a program of its own: the HIP
// calls below take the place of the runtime's, device memory is host memory and launches do nothing, so a
// whole context is set up on the CPU and every allocation counted.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <vector>
#include "../hierarchicaldd_amd/csrc/hdd_runtime.h"
#include "../hierarchicaldd_amd/csrc/hdd_server.h"
#include "../hierarchicaldd_amd/csrc/hdd_sigma_device.h"

static std::mutex g_mu;
static std::map<void*, size_t> g_live;
static size_t g_held = 0, g_peak = 0;

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    *p = std::calloc(1, n);
    std::lock_guard<std::mutex> l(g_mu);
    g_live[*p] = n;
    g_held += n;
    if (g_held > g_peak) g_peak = g_held;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    std::lock_guard<std::mutex> l(g_mu);
    g_held -= g_live[p];
    g_live.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = std::calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipMemset(void* p, int v, size_t n) { std::memset(p, v, n); return hipSuccess; }
hipError_t hipMemcpy(void* to, const void* from, size_t n, hipMemcpyKind) { std::memcpy(to, from, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(to, from, n); return hipSuccess; }
hipError_t hipMemcpyToSymbol(const void*, const void*, size_t, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)std::malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { std::free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)std::malloc(1); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)std::malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
    *g = *b = dim3(1);
    *m = 0;
    *s = nullptr;
    return hipSuccess;
}
}

using namespace hdd;

struct Input {
    SolverParams P;
    std::vector<uint64_t> offsets;
    std::vector<uint32_t> flags;
    std::vector<float> b;
};
// edge, subdomain edge, V-cycle levels, pages; then the pages' offsets, flags and right-hand side
static Input read_input(const char* path) {
    Input in;
    int h[4];
    FILE* f = std::fopen(path, "rb");
    bool ok = f && std::fread(h, 4, 4, f) == 4;
    if (ok) {
        in.P.size = {h[0], h[0], h[0]}; in.P.sub = {h[1], h[1], h[1]}; in.P.vlevels = h[2];
        const size_t n = h[3];
        in.offsets.resize(n); in.flags.resize(n * 256); in.b.resize(n * 256);
        ok = std::fread(in.offsets.data(), 8, n, f) == n && std::fread(in.flags.data(), 4, n * 256, f) == n * 256 &&
             std::fread(in.b.data(), 4, n * 256, f) == n * 256;
    }
    if (f) std::fclose(f);
    if (!ok) { std::printf("no input %s\n", path); std::_Exit(2); }
    return in;
}
static std::shared_ptr<ProblemHost> host_of(const Input& in) {
    auto q = std::make_shared<ProblemHost>(in.P, (int)in.offsets.size(), in.offsets.data(), in.flags.data(), in.b.data());
    q->factorize();
    return q;
}

// "bytes <heights> file..": one context of the problems; prints estimate, set-up estimate, bytes held, peak
// "server <budget> file": one request; prints "done" or "failed: .."
int main(int argc, char** argv) {
    if (argc < 4) return 2;
    const std::string what = argv[1];
    if (what == "server") {
        const Input in = read_input(argv[3]);
        ServerParams p;
        p.setup_threads = 1; p.hbm_budget = std::atof(argv[2]);
        Server s(p);
        const int64_t id = s.submit(in.P, (int)in.offsets.size(), in.offsets.data(), in.flags.data(), in.b.data(), 1e-3, 5);
        const auto r = s.wait(id);
        if (r->failed) std::printf("failed: %s\n", r->error.c_str());
        else std::printf("done %d\n", (int)r->heights);
    } else {
        const bool heights = std::atoi(argv[2]) != 0;
        std::vector<std::shared_ptr<ProblemHost>> hosts;
        size_t est = 0, setup = 0;
        for (int a = 3; a < argc; ++a) {
            size_t t = 0;
            hosts.push_back(host_of(read_input(argv[a])));
            est += hosts.back()->device_bytes(heights, &t);
            setup += t;
        }
        Solver S(hosts, heights);
        std::printf("%zu %zu %zu %zu\n", est, setup, g_held, g_peak);
    }
    std::fflush(stdout);
    std::_Exit(0);
}
