// device_double.cpp - stands in for the HIP runtime in CPU tests of the host
// code: device memory is host memory, kernels are not run, only noted.
// Loaded with RTLD_GLOBAL before libradhip.so, whose calls then land here.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {

std::map<void *, size_t> live;          // allocations not freed yet
size_t live_bytes, limit = SIZE_MAX;    // hipMalloc refuses what would exceed limit,
size_t largest = SIZE_MAX;              // and any single one beyond largest
std::map<const void *, std::string> kernels;
void (*launched)(const char *name, void **args);
size_t streams, unstreamed; // streams alive; launches on none of them
float elapsed; // each hipEventElapsedTime reads 1 ms more than the last

} // namespace

extern "C" {

size_t double_live(void) { return live.size(); }
size_t double_streams(void) { return streams; }
size_t double_unstreamed(void) { return unstreamed; }
size_t double_live_bytes(void) { return live_bytes; }
void double_limit(size_t bytes) { limit = bytes; }
void double_largest(size_t bytes) { largest = bytes; }
void double_on_launch(void (*f)(const char *, void **)) { launched = f; }

hipError_t hipMalloc(void **p, size_t n)
{
    if (n > largest || n > limit || live_bytes > limit - n)
        return hipErrorOutOfMemory;
    *p = calloc(n, 1);
    live[*p] = n;
    live_bytes += n;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    if (!p)
        return hipSuccess;
    auto it = live.find(p);
    if (it == live.end())
        return hipErrorInvalidValue;
    live_bytes -= it->second;
    live.erase(it);
    free(p);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *fr, size_t *total)
{
    *total = limit;
    *fr = limit - live_bytes;
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n)
{
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t)
{
    memset(d, v, n);
    return hipSuccess;
}

void **__hipRegisterFatBinary(const void *)
{
    static void *handle;
    return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *)
{
    kernels[host] = name;
}
static hipStream_t called_on;
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t st)
{
    called_on = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *st)
{
    *st = called_on;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t st)
{
    unstreamed += st == nullptr;
    if (launched)
        launched(kernels[f].c_str(), args);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *)
{
    static char space[64 << 20];
    *p = space;
    return hipSuccess;
}

hipError_t hipGetDevice(int *d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int)
{
    *v = 256;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t e)
{
    return e == hipErrorOutOfMemory ? "out of memory" : "error";
}
hipError_t hipGetLastError(void) { return hipSuccess; }

static hipError_t handle(void **h)
{
    *h = malloc(1);
    return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t *s)
{
    ++streams;
    return handle((void **)s);
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    --streams;
    free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t st, hipEvent_t e, unsigned)
{
    return st && e ? hipSuccess : hipErrorInvalidHandle;
}
hipError_t hipEventCreate(hipEvent_t *e) { return handle((void **)e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return handle((void **)e); }
hipError_t hipEventDestroy(hipEvent_t e)
{
    free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st)
{
    return st && e ? hipSuccess : hipErrorInvalidHandle;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = elapsed += 1.0f;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return handle((void **)g); }
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    return handle((void **)x);
}
hipError_t hipGraphUpload(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g)
{
    free(g);
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x)
{
    free(x);
    return hipSuccess;
}

} // extern "C"
