// A stand-in for the HIP runtime, preloaded so that libgca.so's host code runs without a GPU: "device"
// memory is host memory, copies are memcpy, kernels do nothing.  An allocation beyond a budget set by
// the test fails as the runtime's does, and the error stays until hipGetLastError takes it.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::map<void *, size_t> blocks;
size_t live = 0, budget = ~size_t(0);
hipError_t last = hipSuccess;
dim3 cfg_grid, cfg_block;
size_t cfg_lds;
hipStream_t cfg_stream;
std::map<const void *, std::string> kernels;
void *bounds_of = nullptr;  // the last k_bounds_keys launch's workgroup bounds

hipError_t alloc(void **p, size_t n)
{
    *p = nullptr;
    if (n > budget || live > budget - n) return last = hipErrorOutOfMemory;
    *p = calloc(1, n ? n : 1);
    blocks[*p] = n;
    live += n;
    return hipSuccess;
}
}  // namespace

extern "C" {
void host_runtime_budget(size_t bytes) { budget = bytes; }
size_t host_runtime_live() { return live; }
void *host_runtime_bounds() { return bounds_of; }

void **__hipRegisterFatBinary(const void *)
{
    static void *handle;
    return &handle;
}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    kernels[f] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s)
{
    cfg_grid = g, cfg_block = b, cfg_lds = lds, cfg_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s)
{
    *g = cfg_grid, *b = cfg_block, *lds = cfg_lds, *s = cfg_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t)
{
    if (kernels[f].find("k_bounds_keys") != std::string::npos) bounds_of = *(void **)args[0];
    return hipSuccess;
}

hipError_t hipGetLastError()
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipMalloc(void **p, size_t n) { return alloc(p, n); }
hipError_t hipFree(void *p)
{
    auto it = blocks.find(p);
    if (it != blocks.end()) {
        live -= it->second;
        blocks.erase(it);
        free(p);
    }
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    *p = calloc(1, n ? n : 1);
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    memmove(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    memmove(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t)
{
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    memset(p, 0, sizeof(*p));
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *)
{
    static char scratch[1 << 19];
    return *p = scratch, hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = (hipStream_t)malloc(1), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return free(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *c)
{
    return *c = hipStreamCaptureStatusNone, hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t)malloc(1), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return free(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 0.f, hipSuccess; }
}
