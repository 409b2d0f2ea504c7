// The token dispatch that signals every row: one nvshmemx_putmem_signal_nbi per row copy, the form
// the reference's signalling idiom takes (examples/ring-reduce.cu:111-127) on the token shuffle of
// examples/moe_shuffle.cu:240-289.  A translation unit of its own because of its copy depth: a row of
// 14336 bytes is 14 vectors per lane of a wavefront, and with rounds of 14 a put is one run of loads
// followed by one run of stores (4.53 -> 4.90 TB/s against rounds of 8 + 4 + 2); the 56 vector
// registers that costs would take occupancy from the one-wavefront blocks of the other shuffle kernels.
#include <hip/hip_runtime.h>

#define NVSHMEMI_AMD_COPY_UNROLL 14

#include "moe_rowsignal.hpp"

namespace perftest {

int launch_moe_rowsignal(bool warp, bool full, int blocks_per_pe, int threads, void **args, hipStream_t stream) {
    const void *fn = !warp ? (const void *)moe_dispatch_rowsignal_kernel<false, false>
                     : full ? moe_rowsignal_full()
                            : (const void *)moe_dispatch_rowsignal_kernel<true, false>;
    return launch_senders(fn, blocks_per_pe, threads, args, stream);
}

}  // namespace perftest
