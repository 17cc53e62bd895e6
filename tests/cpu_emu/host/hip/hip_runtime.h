// The HIP calls of the library's host code on the CPU, for tests of what it
// plans: memory is host memory, copies are immediate, a launch is recorded
// (name, grid) and runs nothing.
#pragma once
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>
#include "../../hip/hip_runtime.h"

inline uint32_t __umulhi(uint32_t a, uint32_t b) { return (uint32_t)(((uint64_t)a * b) >> 32); }
inline int __builtin_amdgcn_readfirstlane(int v) { return v; }

struct EmuLaunch {
    std::string name;
    dim3 grid;
};
inline std::vector<EmuLaunch> emu_launches;
#undef hipLaunchKernelGGL
#undef hipExtLaunchKernelGGL
#define hipLaunchKernelGGL(kernel, grid, block, shmem, stream, ...) \
    emu_launches.push_back({#kernel, dim3(grid)})
#define hipExtLaunchKernelGGL(kernel, grid, ...) emu_launches.push_back({#kernel, dim3(grid)})

typedef void *hipGraph_t;
typedef void *hipGraphExec_t;
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
enum { hipHostMallocMapped = 1, hipHostMallocCoherent = 2 };
enum { hipStreamCaptureModeThreadLocal = 0 };
inline const char *hipGetErrorString(hipError_t) { return "error"; }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    memcpy(d, s, n);
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = calloc(1, n);
    return *p ? hipSuccess : hipErrorInvalidValue;
}
inline hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) {
    *d = h;
    return hipSuccess;
}
inline hipError_t hipHostFree(void *p) {
    free(p);
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipStreamBeginCapture(hipStream_t, int) { return hipSuccess; }
inline hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipSuccess; }
inline hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, void *, char *, size_t) {
    return hipSuccess;
}
inline hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
inline hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
inline hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventCreate(hipEvent_t *) { return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 0.f;
    return hipSuccess;
}
