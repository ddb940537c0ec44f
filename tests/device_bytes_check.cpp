// Host check of the device bytes a problem is estimated to need (ProblemHost::device_bytes), by which the
// server admits requests, compiled and run by tests/test_device_bytes.py as a program of its own with the
// HIP calls of host_hip.h: a whole context is set up on the CPU and every allocation counted.
#include <cstdio>
#include <cstdlib>
#include <memory>
#include <string>
#include <vector>
#include "../hierarchicaldd_amd/csrc/hdd_runtime.h"
#include "../hierarchicaldd_amd/csrc/hdd_server.h"
#include "../hierarchicaldd_amd/csrc/hdd_sigma_device.h"
#include "host_hip.h"

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

// "create <memory> file": a context with that much device memory; prints the peak and whether its solves use
//     dense nodes, or "failed: .."
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
    } else if (what == "create") {
        const auto host = host_of(read_input(argv[3]));
        g_memory = (size_t)std::atof(argv[2]);
        try {
            Solver S({host});
            std::printf("%zu %d\n", g_peak, (int)S.sigma->lv[0].Lrr.use_nodes);
        } catch (const std::exception& e) {
            std::printf("failed: %s\n", e.what());
        }
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
