// Kernel launches of the host library and its drivers.
#pragma once

#include <hip/hip_runtime.h>

namespace nvshmem_amd {

template <typename T>
struct same_type {
    typedef T type;
};
// One call into the runtime.  <<<...>>> (and hipLaunchKernelGGL, which is the same) makes three: the launch shape is pushed,
// the kernel's stub pops it, and only then launches.  On the small on-stream calls the host is what bounds a row of them: us
// per launch on an idle host thread 2.35 / 2.17.  The error is left to hipGetLastError.
template <typename... P>
inline void launch_kernel(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t stream,
                          typename same_type<P>::type... args) {
    void *pointers[] = {(void *)&args...};
    (void)hipLaunchKernel((const void *)kernel, grid, block, pointers, lds, stream);
}

}  // namespace nvshmem_amd
