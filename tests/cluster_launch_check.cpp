// Host check of the V-cycle's cluster launches (csrc/hdd_kernels.hip), compiled and run by
// tests/test_cluster_launches.py with the HIP calls of host_hip.h: kernel attributes are set with the plan
// and not again by a V-cycle. A full box of n^3 cells, subdomains of `sub`.
#include <cstdio>
#include <memory>
#include <vector>
#include "../hierarchicaldd_amd/csrc/hdd_runtime.h"
#include "../hierarchicaldd_amd/csrc/hdd_sigma_device.h"
#include "host_hip.h"

using namespace hdd;

int main(int argc, char** argv) {
    const int n = argc > 1 ? std::atoi(argv[1]) : 41, sub = argc > 2 ? std::atoi(argv[2]) : 20;
    PagedLevel grid;
    grid.init({n, n, n});
    for (int x = 0; x < n; ++x)
        for (int y = 0; y < n; ++y)
            for (int z = 0; z < n; ++z) {
                const int p = grid.add_page(x >> 2, y >> 3, z >> 3);
                const bool ring = x == 0 || y == 0 || z == 0 || x == n - 1 || y == n - 1 || z == n - 1;
                grid.flags[(size_t)p * kPageCells + page_cell(x, y, z)] = ring ? kDirichlet : kActive;
            }
    grid.sort_pages();
    std::vector<uint64_t> offsets;
    for (const Int3& o : grid.page_base) offsets.push_back(page_key(o.x >> 2, o.y >> 3, o.z >> 3) << 12);
    SolverParams P;
    P.size = {n, n, n}; P.sub = {sub, sub, sub}; P.vlevels = 2;
    const std::vector<float> b(grid.flags.size(), 1.f);
    Solver S(P, grid.npages(), offsets.data(), grid.flags.data(), b.data());
    const DevClusters W = S.lv[0].clusters();
    const int set = g_attributes, launched = g_launches;
    S.vcycle();
    S.vcycle();
    std::printf("%d cells a workgroup, %d values of LDS, %d attributes set up, %d by %d launches\n", W.slots, W.entries, set, g_attributes - set,
                g_launches - launched);
    std::fflush(stdout);
    std::_Exit(W.nwg > 0 && 2 * W.entries * (int)sizeof(float) > 64 * 1024 && set > 0 && g_launches > launched && g_attributes == set ? 0 : 1);
}
