// A stand-in for the HIP runtime on the CPU: one device that works off a queue on a thread of its own, which a test can
// hold.  Only what host_io.hip uses.  Fresh memory is filled with a pattern, so that nothing passes by luck.
#pragma once
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <functional>

#define __global__
#define __host__
#define __device__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __restrict__
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __HIP_MEMORY_SCOPE_SYSTEM 0
#define __hip_atomic_fetch_add(p, v, order, scope) __atomic_fetch_add(p, v, order)
#define __hip_atomic_store(p, v, order, scope) __atomic_store_n(p, v, order)

struct dim3 {
    unsigned x, y, z;
    dim3(unsigned x_ = 1, unsigned y_ = 1, unsigned z_ = 1) : x(x_), y(y_), z(z_) {}
};
struct uint4 { uint32_t x, y, z, w; };
extern thread_local dim3 blockIdx, threadIdx, gridDim;
inline void __syncthreads() {}
inline void __threadfence_system() {}

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
typedef struct fakeStream* hipStream_t;
enum { hipHostMallocCoherent = 0 };

namespace fake {
void enqueue(std::function<void()> f);
void hold();                 // the device stops taking work until release()
void release();
size_t pending();            // work not finished yet
extern size_t syncs, host_mallocs, host_frees, host_bytes, host_bytes_limit;
}  // namespace fake

hipError_t hipStreamSynchronize(hipStream_t);  // nullptr: the null stream
hipError_t hipDeviceSynchronize();
hipError_t hipMalloc(void** p, size_t n);
hipError_t hipFree(void* p);
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags);
hipError_t hipHostFree(void* p);
hipError_t hipMemset(void* p, int v, size_t n);  // on the null stream, which has no order with the others: done when that is waited for
inline hipError_t hipGetLastError() { return hipSuccess; }
inline const char* hipGetErrorString(hipError_t) { return "error"; }

// The threads of a launch one after the other (the kernels at hand keep no state across a barrier).
template <typename K, typename... A>
void hipLaunchKernelGGL(K kernel, dim3 grid, dim3 block, size_t, hipStream_t, A... args) {
    fake::enqueue([=] {
        gridDim = grid;
        for (blockIdx.x = 0; blockIdx.x < grid.x; blockIdx.x++)
            for (unsigned t = block.x; t-- > 0;) {  // thread 0 last: it counts the workgroup off
                threadIdx.x = t;
                kernel(args...);
            }
    });
}
