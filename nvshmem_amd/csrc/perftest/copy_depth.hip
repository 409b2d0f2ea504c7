// A block's put in a translation unit of its own, built with a depth of the long rounds that is no power of two: the depth is
// a setting of the including unit, and every one of them has to move the same bytes.
#include <hip/hip_runtime.h>

#define NVSHMEMI_AMD_COPY_DEEP_UNROLL 12

#include "nvshmem_perftest.h"
#include "nvshmemx.h"
#include "perftest_common.hpp"

namespace {

__global__ __launch_bounds__(1024) void put_depth12_kernel(char *dest, const char *src, size_t bytes) {
    const int me = nvshmem_my_pe();
    nvshmemx_putmem_block(dest, src, bytes, (me + 1 == nvshmem_n_pes()) ? 0 : me + 1);
}

}  // namespace

extern "C" int nvshmem_perftest_put_depth12(void *dest, const void *src, size_t bytes, int threads, void *stream) {
    if (!perftest::ready() || !perftest::check_launch(1, threads) || !perftest::check_range(dest, bytes) ||
        !perftest::check_range(src, bytes))
        return NVSHMEMX_ERROR_INVALID_VALUE;
    nvshmem_amd::launch_kernel(put_depth12_kernel, dim3(1, 1, (unsigned)nvshmem_n_pes()), dim3(threads), 0, (hipStream_t)stream,
                       (char *)dest, (const char *)src, bytes);
    return perftest::launch_status("put_depth12");
}
