// A HIP runtime without a GPU, for tests of what the library launches: memory is address space, kernels are not run,
// every launch is recorded.  Loaded globally before the library, whose calls then bind to these.  A launch of 2^32
// threads or more in one dimension is refused, as on the GPU.
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
struct Launch {
    std::string kernel;
    int cooperative;
    dim3 grid, block;
    size_t lds;
};
std::vector<Launch> launches;
std::map<const void *, std::string> kernels;
std::map<void *, size_t> allocations;
Launch configured;  // <<<...>>>
hipError_t last = hipSuccess;

hipError_t record(const void *func, int cooperative, dim3 grid, dim3 block, size_t lds) {
    if ((unsigned long long)grid.x * block.x >> 32 || grid.y > 65535 || grid.z > 65535) return last = hipErrorInvalidConfiguration;
    launches.push_back({kernels.count(func) ? kernels[func] : "?", cooperative, grid, block, lds});
    return hipSuccess;
}
}  // namespace

extern "C" {
int recorder_count() { return (int)launches.size(); }
void recorder_clear() { launches.clear(); }
const char *recorder_kernel(int i) { return launches[i].kernel.c_str(); }
void recorder_shape(int i, unsigned long long *out) {
    const Launch &l = launches[i];
    const unsigned long long v[8] = {(unsigned long long)l.cooperative, l.grid.x, l.grid.y, l.grid.z,
                                     l.block.x, l.block.y, l.block.z, l.lds};
    memcpy(out, v, sizeof v);
}

void **__hipRegisterFatBinary(const void *) { return (void **)&launches; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *, int *) {
    kernels[host] = name;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t) {
    configured = {"", 0, grid, block, lds};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *stream) {
    *grid = configured.grid, *block = configured.block, *lds = configured.lds, *stream = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **, size_t lds, hipStream_t) {
    return record(f, 0, grid, block, lds);
}
hipError_t hipExtLaunchKernel(const void *f, dim3 grid, dim3 block, void **, size_t lds, hipStream_t, hipEvent_t, hipEvent_t, int) {
    return record(f, 0, grid, block, lds);
}
hipError_t hipLaunchCooperativeKernel(const void *f, dim3 grid, dim3 block, void **, unsigned lds, hipStream_t) {
    return record(f, 1, grid, block, lds);
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *blocks, const void *, int threads, size_t) {
    *blocks = 2048 / threads;
    return hipSuccess;
}

hipError_t hipMalloc(void **p, size_t bytes) {
    *p = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (*p == MAP_FAILED) return last = hipErrorOutOfMemory;
    allocations[*p] = bytes;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (p) munmap(p, allocations[p]);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { return hipMalloc(p, bytes); }
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipMemcpy(void *to, const void *from, size_t bytes, hipMemcpyKind) { memcpy(to, from, bytes); return hipSuccess; }
hipError_t hipMemcpyAsync(void *to, const void *from, size_t bytes, hipMemcpyKind kind, hipStream_t) { return hipMemcpy(to, from, bytes, kind); }
hipError_t hipMemcpy2DAsync(void *, size_t, const void *, size_t, size_t, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemcpyToSymbol(const void *, const void *, size_t, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemset(void *p, int value, size_t bytes) { memset(p, value, bytes); return hipSuccess; }
hipError_t hipMemsetAsync(void *p, int value, size_t bytes, hipStream_t) { return hipMemset(p, value, bytes); }

hipError_t hipGetDevice(int *device) { *device = 0; return hipSuccess; }
hipError_t hipGetDeviceCount(int *count) { *count = 1; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *prop, int) {
    memset(prop, 0, sizeof *prop);
    prop->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *status) { *status = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *event, unsigned) { *event = (hipEvent_t)&launches; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return hipErrorInvalidValue; }
hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t) { return "refused"; }
}
