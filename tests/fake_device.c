/* The HIP calls that the library makes, on host memory of a set size: plans can be created without
 * a GPU, and allocations fail where a device's memory would end.  Kernels do not run. */
#include <hip/hip_runtime_api.h>
#include <stdlib.h>
#include <string.h>

static size_t limit = (size_t)-1, live, pinned;
static hipError_t last;

void fake_limit(size_t bytes) { limit = bytes; }
size_t fake_live(void) { return live; }
size_t fake_pinned(void) { return pinned; }

static hipError_t take(void **p, size_t n, size_t *sum, size_t most) {
    if (n > most || *sum > most - n) return last = hipErrorOutOfMemory;
    size_t *b = calloc(1, n + 64);
    if (!b) return last = hipErrorOutOfMemory;
    *b = n;
    *sum += n;
    *p = (char *)b + 64;
    return hipSuccess;
}
static hipError_t give(void *p, size_t *sum) {
    if (p) {
        size_t *b = (size_t *)((char *)p - 64);
        *sum -= *b;
        free(b);
    }
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) { return take(p, n, &live, limit); }
hipError_t hipFree(void *p) { return give(p, &live); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned f) { return take(p, n, &pinned, (size_t)-1); }
hipError_t hipHostFree(void *p) { return give(p, &pinned); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemset(void *d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipGetLastError(void) { hipError_t e = last; last = hipSuccess; return e; }

hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t n, hipStream_t s) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *n, hipStream_t *s) {
    *g = *b = (dim3){1, 1, 1};
    *n = 0;
    *s = 0;
    return hipSuccess;
}
static size_t launches;
size_t fake_launches(void) { return launches; }
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **a, size_t n, hipStream_t s) { launches++; return hipSuccess; }

hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int d) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int d) {
    memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    p->sharedMemPerBlock = 65536;
    p->totalGlobalMem = (size_t)288 << 30;
    strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *s) { return hipErrorInvalidSymbol; }
hipError_t hipStreamCreate(hipStream_t *s) { *s = (hipStream_t)malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t s) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned f) { return hipEventCreate(e); }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f) { return hipStreamCreate(s); }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned f) { return hipSuccess; }
