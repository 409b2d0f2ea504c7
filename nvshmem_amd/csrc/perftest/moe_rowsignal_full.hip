// The token dispatch that signals every row, for more data than the caches take (launch_moe_rowsignal says when): a wavefront
// keeps three of a row's stores outstanding.  All fourteen at once crowd out other wavefronts' loads where the writes go to
// memory, and are the better form where they do not.  us for 8 PEs, all at once / three: 4096 tokens to 8 experts in rows of
// 14 KiB 853 / 829, 8192 1702 / 1660, 8192 to 4 937 / 901, 16384 to 2 1136 / 1108, 6000 to 2 in rows of 12 544 bytes 365 / 353, 2048
// to 8 of 9216 235 / 224 (the cascade of rounds that the one-round copy replaced: 832, 1660, 907, 1104, 400, 225).  Two would
// gain another 1 %, and lose 6 in processes whose heap lies so that all at once takes 1299 us for 1702.
#include <hip/hip_runtime.h>

#define NVSHMEMI_AMD_COPY_UNROLL 14
#define NVSHMEMI_AMD_COPY_STORES 3

#include "moe_rowsignal.hpp"

namespace perftest {

const void *moe_rowsignal_full() { return (const void *)moe_dispatch_rowsignal_kernel<true, true>; }

}  // namespace perftest
