// The HIP calls of a context's set-up and solves, for programs that run them on the CPU (the *_check.cpp
// of this folder): they take the place of the runtime's, device memory is host memory, copies are made at
// once and launches do nothing. Counts what its programs check.
#pragma once
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <hip/hip_runtime.h>

static std::mutex g_mu;
static std::map<void*, size_t> g_live;
static size_t g_held = 0, g_peak = 0, g_memory = ~size_t(0);  // device bytes; as many as there are
static int g_attributes = 0, g_launches = 0, g_copies = 0;

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    std::lock_guard<std::mutex> l(g_mu);
    *p = nullptr;
    if (n > g_memory - g_held) return hipErrorOutOfMemory;
    *p = std::calloc(1, n);
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
hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind, hipStream_t) { ++g_copies; std::memcpy(to, from, n); return hipSuccess; }
hipError_t hipMemcpyToSymbol(const void*, const void*, size_t, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)std::malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { std::free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)std::malloc(1); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)std::malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { ++g_attributes; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { ++g_launches; return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
    *g = *b = dim3(1);
    *m = 0;
    *s = nullptr;
    return hipSuccess;
}
}
