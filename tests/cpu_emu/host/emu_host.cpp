// definitions of the emulation's work-item state for the host-code tests
#include <hip/hip_runtime.h>
thread_local dim3 threadIdx, blockIdx;
dim3 gridDim, blockDim;
pthread_barrier_t emu_barrier;
double emu_shfl[1024];
