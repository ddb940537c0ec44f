// Host check of HostStage (csrc/hdd_runtime.cpp), compiled and run by tests/test_host_stage.py with the HIP
// calls of host_hip.h: copies of pinned memory go to the runtime as one copy, of pageable memory through the
// ring, and all arrive whole.
#include <cstdint>
#include <cstdio>
#include <vector>
#include "../hierarchicaldd_amd/csrc/hdd_runtime.h"
#include "host_hip.h"

static int g_answer = 0;  // hipPointerGetAttributes: 0 unregistered, 1 pinned, 2 an error
extern "C" hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
    a->type = g_answer == 1 ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return g_answer == 2 ? hipErrorInvalidValue : hipSuccess;
}

using namespace hdd;

int main() {
    HostStage stage;
    const size_t n = (size_t(17) << 20) + 12;  // five chunks, the last of a part
    stage.init(n);
    std::vector<char> host(n), dev(n, 0), back(n, 0);
    for (size_t i = 0; i < n; ++i) host[i] = (char)(i * 2654435761u >> 13);
    for (g_answer = 0; g_answer < 3; ++g_answer)
        for (const size_t bytes : {n, size_t(HostStage::kMin), size_t(HostStage::kMin) - 4}) {
            std::fill(dev.begin(), dev.end(), 0);
            std::fill(back.begin(), back.end(), 0);
            const int c0 = g_copies;
            stage.to_device(dev.data(), host.data(), bytes, nullptr);
            const int c1 = g_copies;
            stage.to_host(back.data(), dev.data(), bytes, nullptr);
            const int c2 = g_copies, chunks = (int)((bytes + HostStage::kChunk - 1) / HostStage::kChunk);
            const int want = g_answer == 1 || bytes < HostStage::kMin ? 1 : chunks;
            if (c1 - c0 != want || c2 - c1 != want || std::memcmp(back.data(), host.data(), bytes)) {
                std::printf("memory of kind %d, %zu bytes: %d and %d copies, %d expected\n", g_answer, bytes, c1 - c0, c2 - c1, want);
                return 1;
            }
        }
    return 0;
}
